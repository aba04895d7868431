// nf4_gemm.hip - entry points of the NF4-dequant-fused bf16 GEMMs: argument
// checks, the choice of kernel and its workspace (kernels: nf4_gemm_core.hpp
// and, for few tokens, nf4_skinny.hip).
#include "abi_common.hpp"
#include "gemm_common.hpp"
#include "nf4_gemm_core.hpp"
#include "nf4_skinny.hpp"

namespace nf4s {

static AbsmaxRef absmax_of(const nf4s_tensor &t) {
  AbsmaxRef a;
  a.absmax = t.absmax;
  a.q = t.absmax_q;
  a.scale = t.absmax_scale;
  a.group_shift = t.dq_group > 0 ? group_shift(t.dq_group) : 0;
  a.block_shift = t.block_size > 64 ? group_shift(t.block_size / 64) : 0;
  return a;
}

// Shared argument checks of the two GEMM entry points.  W is [wn, wk].  With
// m == 0 (no tokens) nothing is read or written: the activation and output
// pointers may be NULL or unaligned (an empty tensor's or vector's data
// pointer), and only the weight's shape is checked.
static int32_t check_gemm(const uint16_t *act, const nf4s_tensor *w, int64_t m, int64_t wn,
                          int64_t wk, const uint16_t *out) {
  if (m != 0 && (act == nullptr || out == nullptr))
    return fail(NF4S_ERR_INVALID_ARGUMENT, "activation or output is NULL");
  if (m < 0 || wn <= 0 || wk <= 0)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "bad GEMM shape m=%lld n=%lld k=%lld",
                (long long)m, (long long)wn, (long long)wk);
  // Keeps the tile counts of each dimension (at least 64 rows or columns a
  // tile) and their sums over four weights far inside 64 bits; plan_launch
  // bounds their product.
  constexpr int64_t kMaxDim = (int64_t)1 << 39;
  if (m > kMaxDim || wn > kMaxDim || wk > kMaxDim)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "GEMM dimension beyond 2^39: m=%lld n=%lld k=%lld",
                (long long)m, (long long)wn, (long long)wk);
  int64_t numel;
  if (__builtin_mul_overflow(wn, wk, &numel))
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "weight of %lld x %lld elements overflows 64 bits",
                (long long)wn, (long long)wk);
  const int32_t rc = validate_tensor(w, numel);
  if (rc != NF4S_OK) return rc;
  // A 64-deep reduction step must lie in one absmax block: block sizes 64,
  // 128, 256, ... (64 << s), with whole blocks per row.
  const int32_t bsz = w->block_size;
  if (bsz < 64 || bsz > (1 << 20) || (bsz & (bsz - 1)) != 0)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE,
                "fused GEMM needs block_size 64 << s (64, 128, 256, ...), got %d", bsz);
  if (wk % 64 != 0)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "fused GEMM needs k %% 64 == 0, got %lld",
                (long long)wk);
  if (wk % bsz != 0)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE,
                "fused GEMM needs k %% block_size == 0 (whole blocks per row), got k %lld, "
                "block_size %d", (long long)wk, bsz);
  if (m == 0) return NF4S_OK;
  if (!aligned(act, 16) || !aligned(w->packed, 16))
    return fail(NF4S_ERR_MISALIGNED, "activation and packed weights must be 16-byte aligned");
  if (!aligned(out, 2)) return fail(NF4S_ERR_MISALIGNED, "output must be 2-byte aligned");
  return NF4S_OK;
}

// The activation loads address a wave's 128 rows with 32-bit offsets.  The
// bound also keeps the kernels' 32-bit step counts (R / 64 <= 2^16) exact.
static int32_t check_offsets(int64_t lda) {
  if (lda > (int64_t)1 << 22)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "activation row of %lld elements is too long",
                (long long)lda);
  return NF4S_OK;
}

// A forward group can take the batched weight loads: whole 4-block absmax
// groups per row (k % 256), aligned group loads, and 4-block groups inside
// one double-quant scale.
static bool fwd_batchable(const nf4s_tensor &w, int64_t k) {
  if (k % 256 != 0 || w.block_size != 64) return false;
  if (w.absmax_q != nullptr) return aligned(w.absmax_q, 4) && w.dq_group >= 4;
  return aligned(w.absmax, 16);
}

static GemmGroup group_of(const nf4s_tensor &w, int64_t wn) {
  GemmGroup q{};
  q.packed = w.packed;
  q.am = absmax_of(w);
  q.wn = wn;
  return q;
}

// Reduction steps of an input-gradient launch: its groups' steps in order.
static int64_t dgrad_steps(const int64_t *ns, int32_t count) {
  int64_t steps = 0;
  for (int32_t i = 0; i < count; ++i) steps += ns[i] / kStep;
  return steps;
}

// Workspace bytes the split-K input gradient over these weights needs (0: no
// split), for either producer's step granularity.
static int64_t dgrad_workspace_bytes(const int64_t *ns, int32_t count, int64_t m, int64_t k) {
  constexpr int64_t kMaxDim = (int64_t)1 << 39;  // beyond it the GEMM rejects the shape
  if (m <= 0 || m > kMaxDim || k <= 0 || k > kMaxDim || k % 64 != 0) return 0;
  for (int32_t i = 0; i < count; ++i)
    if (ns[i] <= 0 || ns[i] > kMaxDim || ns[i] % 64 != 0) return 0;
  const int64_t tiles_o = (k + kTileO - 1) / kTileO;
  const int64_t steps = dgrad_steps(ns, count);
  int64_t best = 0;
  for (int unroll : {2, 4}) {
    const int64_t b = plan_bytes(m, tiles_o, steps, unroll);
    if (b > best) best = b;
  }
  return best;
}


// Forward over `count` weights W_i [ns[i], k] sharing x [m, k]: y_i = x . W_i^T.
// Weights of one kind (double-quantized or not, batched loads or not) share
// a launch; a mixed set runs as one launch per kind.
static int32_t gemm_fwd_groups(const uint16_t *x, const nf4s_tensor *ws, const int64_t *ns,
                               uint16_t *const *ys, int32_t count, int64_t m, int64_t k,
                               hipStream_t s, void *work = nullptr, int64_t work_bytes = 0) {
  if (count <= 0 || count > kMaxGroups)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "count must be 1..%d, got %d", kMaxGroups, count);
  if (ws == nullptr || ns == nullptr || ys == nullptr)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "weights, sizes or outputs are NULL");
  int32_t rc = NF4S_OK;
  for (int32_t i = 0; i < count && rc == NF4S_OK; ++i)
    rc = check_gemm(x, &ws[i], m, ns[i], k, ys[i]);
  if (rc == NF4S_OK) rc = check_offsets(k);
  if (rc != NF4S_OK) return rc;
  if (m == 0) return NF4S_OK;
  if (skinny_takes(ns, count, m)) {
    SkinnyArgs a{};
    a.x = x;
    a.m = m;
    a.k = k;
    a.ngroups = count;
    for (int32_t i = 0; i < count; ++i) {
      a.grp[i].packed = ws[i].packed;
      a.grp[i].am = absmax_of(ws[i]);
      a.grp[i].out = ys[i];
      a.grp[i].n = ns[i];
    }
    return skinny_fwd(a, s, work, work_bytes);
  }
  // Kind of each weight: bit 0 double-quant, bit 1 batched loads.
  int kind[kMaxGroups];
  for (int32_t i = 0; i < count; ++i)
    kind[i] = (ws[i].absmax_q != nullptr ? 1 : 0) | (fwd_batchable(ws[i], k) ? 2 : 0);
  bool done[kMaxGroups] = {false, false, false, false};
  for (int32_t i = 0; i < count; ++i) {
    if (done[i]) continue;
    GroupedArgs ga{};
    GemmArgs &g = ga.base;
    g.a = x;
    g.lda = k;
    g.M = m;
    g.R = k;
    g.wk = k;
    int64_t tiles = 0;
    for (int32_t j = i; j < count; ++j) {
      if (done[j] || kind[j] != kind[i]) continue;
      GemmGroup q = group_of(ws[j], ns[j]);
      q.out = ys[j];
      q.ldo = ns[j];
      const int64_t tiles_o = (ns[j] + kTileO - 1) / kTileO;
      tiles += tiles_o;
      if (tiles > kMaxTiles) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
      q.tiles_o = (int32_t)tiles_o;
      ga.grp[ga.ngroups++] = q;
      done[j] = true;
    }
    ga.tiles_o = (int32_t)tiles;
    rc = launch_fwd(ga, (kind[i] & 1) != 0, (kind[i] & 2) != 0, s, work, work_bytes);
    if (rc != NF4S_OK) return rc;
  }
  return NF4S_OK;
}

// hidden [m, ff] = silu(x . Wg^T) * (x . Wu^T), Wg and Wu [ff, k] of one kind.
static int32_t gemm_swiglu(const uint16_t *x, const nf4s_tensor *wg, const nf4s_tensor *wu,
                           int64_t m, int64_t ff, int64_t k, uint16_t *hidden, hipStream_t s) {
  if (wg == nullptr || wu == nullptr)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "weight descriptor is NULL");
  int32_t rc = check_gemm(x, wg, m, ff, k, hidden);
  if (rc == NF4S_OK) rc = check_gemm(x, wu, m, ff, k, hidden);
  if (rc == NF4S_OK) rc = check_offsets(k);
  if (rc != NF4S_OK) return rc;
  const bool dq = wg->absmax_q != nullptr;
  const bool batch = fwd_batchable(*wg, k) && fwd_batchable(*wu, k);
  if ((wu->absmax_q != nullptr) != dq)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE,
                "gate and up weights must both be double-quantized or both not");
  if (m == 0) return NF4S_OK;
  if (skinny_takes(&ff, 1, m)) {
    SkinnyArgs a{};
    a.x = x;
    a.m = m;
    a.k = k;
    a.ngroups = 2;
    const nf4s_tensor *w[2] = {wg, wu};
    for (int i = 0; i < 2; ++i) {
      a.grp[i].packed = w[i]->packed;
      a.grp[i].am = absmax_of(*w[i]);
      a.grp[i].out = hidden;
      a.grp[i].n = ff;
    }
    return skinny_swiglu(a, s);
  }
  GroupedArgs ga{};
  GemmArgs &g = ga.base;
  g.a = x;
  g.lda = k;
  g.out = hidden;
  g.ldo = ff;
  g.M = m;
  g.O = ff;
  g.R = k;
  g.wk = k;
  const int64_t tiles_h = (ff + kTileO / 2 - 1) / (kTileO / 2);
  if (tiles_h > kMaxTiles) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  ga.tiles_o = (int32_t)tiles_h;
  ga.grp[0] = group_of(*wg, ff);
  ga.grp[1] = group_of(*wu, ff);
  ga.ngroups = 2;
  return launch_swiglu(ga, dq, batch, s);
}

// Input gradient dx [m, k] = sum_i dy_i [m, ns[i]] . W_i [ns[i], k].
static int32_t gemm_dgrad_groups(const uint16_t *const *dys, const nf4s_tensor *ws,
                                 const int64_t *ns, int32_t count, int64_t m, int64_t k,
                                 uint16_t *dx, hipStream_t s, void *work = nullptr,
                                 int64_t work_bytes = 0) {
  if (count <= 0 || count > kMaxGroups)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "count must be 1..%d, got %d", kMaxGroups, count);
  if (dys == nullptr || ws == nullptr || ns == nullptr)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "gradients, weights or sizes are NULL");
  const bool dq = ws[0].absmax_q != nullptr;
  for (int32_t i = 0; i < count; ++i) {
    int32_t rc = check_gemm(dys[i], &ws[i], m, ns[i], k, dx);
    if (rc == NF4S_OK) rc = check_offsets(ns[i]);
    if (rc != NF4S_OK) return rc;
    if (ns[i] % 64 != 0)
      return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "dgrad needs n %% 64 == 0, got %lld",
                  (long long)ns[i]);
    if ((ws[i].absmax_q != nullptr) != dq)
      return fail(NF4S_ERR_UNSUPPORTED_SHAPE,
                  "summed dgrad needs all weights double-quantized or none");
  }
  if (m == 0) return NF4S_OK;
  GroupedArgs ga{};
  GemmArgs &g = ga.base;
  g.out = dx;
  g.ldo = k;
  g.M = m;
  g.O = k;
  g.wk = k;
  const int64_t tiles_o = (k + kTileO - 1) / kTileO;
  if (tiles_o > kMaxTiles) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  g.tiles_o = (int32_t)tiles_o;
  for (int32_t i = 0; i < count; ++i) {
    GemmGroup q = group_of(ws[i], ns[i]);
    q.a = dys[i];
    q.lda = ns[i];
    ga.grp[ga.ngroups++] = q;
  }
  // Batched absmax loads: whole 4-step groups for every weight, both blocks
  // of a 128-column tile in every row (k % 128), aligned pair loads, and
  // the two blocks of a pair inside one double-quant scale group.
  bool batch = k % 128 == 0;
  for (int32_t i = 0; i < count && batch; ++i) {
    batch = ns[i] % 256 == 0 && ws[i].block_size == 64;
    if (dq)
      batch = batch && aligned(ws[i].absmax_q, 2) && ws[i].dq_group >= 2;
    else
      batch = batch && aligned(ws[i].absmax, 8);
  }
  const int64_t nsteps = dgrad_steps(ns, count);
  return launch_dgrad(ga, nsteps, dq, batch, s, work, work_bytes);
}

// Workspace bytes the split-K forward over these weights needs (0: no split
// would help, or a shape the GEMM itself rejects, which the GEMM reports).
// Weights of one kind share a launch and a mixed set runs one launch per
// kind, so this is the largest plan over every subset of the weights and
// both producers' step multiples: enough for any partition into launches.
static int64_t fwd_workspace_bytes(const int64_t *ns, int32_t count, int64_t m, int64_t k) {
  constexpr int64_t kMaxDim = (int64_t)1 << 39;  // beyond it the GEMM rejects the shape
  if (m <= 0 || m > kMaxDim || k <= 0 || k > kMaxDim || k % 64 != 0) return 0;
  for (int32_t i = 0; i < count; ++i)
    if (ns[i] <= 0 || ns[i] > kMaxDim) return 0;
  if (skinny_takes(ns, count, m)) return skinny_workspace_bytes(ns, count, m, k);
  int64_t best = 0;
  for (uint32_t set = 1; set < (1u << count); ++set) {
    int64_t tiles_o = 0;
    for (int32_t i = 0; i < count; ++i)
      if (set & (1u << i)) tiles_o += (ns[i] + kTileO - 1) / kTileO;
    for (int unroll : {2, 4}) {
      const int64_t b = plan_bytes(m, tiles_o, k / kStep, unroll);
      if (b > best) best = b;
    }
  }
  return best;
}

static_assert(partial_floats(4) * (int64_t)sizeof(float) == kGemmPartialTileBytes,
              "partial tile size shared with nf4_noalloc.hip");

int32_t fwd_workspace_query(const int64_t *ns, int32_t count, int64_t m, int64_t k,
                            int64_t *bytes) {
  if (bytes == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = 0;
  if (count <= 0 || count > kMaxGroups || ns == nullptr)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "count must be 1..%d with sizes", kMaxGroups);
  *bytes = fwd_workspace_bytes(ns, count, m, k);
  return NF4S_OK;
}

int32_t gemm_fwd_grouped_on(const uint16_t *x, const nf4s_tensor *ws, const int64_t *ns,
                            uint16_t *const *ys, int32_t count, int64_t m, int64_t k,
                            hipStream_t s, void *work, int64_t work_bytes) {
  return gemm_fwd_groups(x, ws, ns, ys, count, m, k, s, work, work_bytes);
}

}  // namespace nf4s

using namespace nf4s;

extern "C" {

int32_t nf4s_gemm_fwd(const uint16_t *x, const nf4s_tensor *w, int64_t m, int64_t n, int64_t k,
                      uint16_t *y, void *stream) {
  clear_error();
  if (w == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "weight descriptor is NULL");
  uint16_t *ys[1] = {y};
  return gemm_fwd_groups(x, w, &n, ys, 1, m, k, as_stream(stream));
}

int32_t nf4s_gemm_dgrad(const uint16_t *dy, const nf4s_tensor *w, int64_t m, int64_t n,
                        int64_t k, uint16_t *dx, void *stream) {
  clear_error();
  if (w == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "weight descriptor is NULL");
  const uint16_t *dys[1] = {dy};
  return gemm_dgrad_groups(dys, w, &n, 1, m, k, dx, as_stream(stream));
}

int32_t nf4s_gemm_fwd_grouped(const uint16_t *x, const nf4s_tensor *ws, const int64_t *ns,
                              uint16_t *const *ys, int32_t count, int64_t m, int64_t k,
                              void *stream) {
  clear_error();
  return gemm_fwd_groups(x, ws, ns, ys, count, m, k, as_stream(stream));
}

int32_t nf4s_gemm_fwd_grouped_ws(const uint16_t *x, const nf4s_tensor *ws, const int64_t *ns,
                                 uint16_t *const *ys, int32_t count, int64_t m, int64_t k,
                                 void *workspace, int64_t workspace_bytes, void *stream) {
  clear_error();
  if (workspace_bytes < 0)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "negative workspace size %lld",
                (long long)workspace_bytes);
  if (workspace != nullptr && !aligned(workspace, 16))
    return fail(NF4S_ERR_MISALIGNED, "workspace must be 16-byte aligned");
  return gemm_fwd_groups(x, ws, ns, ys, count, m, k, as_stream(stream), workspace,
                         workspace_bytes);
}

int32_t nf4s_gemm_fwd_workspace_size(const int64_t *ns, int32_t count, int64_t m, int64_t k,
                                     int64_t *bytes) {
  clear_error();
  return fwd_workspace_query(ns, count, m, k, bytes);
}

int32_t nf4s_gemm_fwd_swiglu(const uint16_t *x, const nf4s_tensor *w_gate,
                             const nf4s_tensor *w_up, int64_t m, int64_t ff, int64_t k,
                             uint16_t *hidden, void *stream) {
  clear_error();
  return gemm_swiglu(x, w_gate, w_up, m, ff, k, hidden, as_stream(stream));
}

int32_t nf4s_gemm_dgrad_sum(const uint16_t *const *dys, const nf4s_tensor *ws, const int64_t *ns,
                            int32_t count, int64_t m, int64_t k, uint16_t *dx, void *stream) {
  clear_error();
  return gemm_dgrad_groups(dys, ws, ns, count, m, k, dx, as_stream(stream));
}

int32_t nf4s_gemm_dgrad_sum_ws(const uint16_t *const *dys, const nf4s_tensor *ws,
                               const int64_t *ns, int32_t count, int64_t m, int64_t k,
                               uint16_t *dx, void *workspace, int64_t workspace_bytes,
                               void *stream) {
  clear_error();
  if (workspace_bytes < 0)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "negative workspace size %lld",
                (long long)workspace_bytes);
  if (workspace != nullptr && !aligned(workspace, 16))
    return fail(NF4S_ERR_MISALIGNED, "workspace must be 16-byte aligned");
  return gemm_dgrad_groups(dys, ws, ns, count, m, k, dx, as_stream(stream), workspace,
                           workspace_bytes);
}

int32_t nf4s_gemm_dgrad_workspace_size(const int64_t *ns, int32_t count, int64_t m, int64_t k,
                                       int64_t *bytes) {
  clear_error();
  if (bytes == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = 0;
  if (count <= 0 || count > kMaxGroups || ns == nullptr)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "count must be 1..%d with sizes", kMaxGroups);
  *bytes = dgrad_workspace_bytes(ns, count, m, k);
  return NF4S_OK;
}

}  // extern "C"
