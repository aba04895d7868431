// nf4_skinny.hip - NF4-dequant-fused forward GEMM for few tokens (m <= 128)
// on gfx950: y[m,n] = x[m,k] . W^T, and its SwiGLU form.
//
// With few tokens the product is bound by reading W (0.52 B per element) and
// by dequantizing it (29 VALU lane-instructions per 8 elements: about 4 TB/s
// of NF4 bytes over the chip at most), not by the matrix pipe.  So each weight is
// dequantized exactly once, by the lane that feeds it to the MFMA, straight
// from registers:
//   * lane l of a wave owns W row l % 32 and, of every 128-deep step, the
//     64-element block g = l / 32.  Reduction slot e of the step's j-th
//     v_mfma_f32_32x32x16_bf16 is element 8j + e of that block for both
//     operands, so the block's packed bytes (32 contiguous ones) and its one
//     product table stay in the lane;
//   * the wave keeps all the tokens (TR) of its 32 weight rows in its
//     accumulators;
//   * x goes through LDS: per step and k-group, TR token rows of 256 B moved
//     by direct-to-LDS loads, double buffered, read as 16-byte fragments.
// A workgroup has WN x WK waves: WN blocks of 32 weight rows that share the
// x tile, times WK k-groups, each over its own contiguous part of K, whose
// accumulators are summed in LDS in k-group order.  Splitting K inside the
// workgroup fills the chip without partial sums in memory; only a launch
// whose tiles still leave CUs idle adds K slices over workgroups (fp32
// partials in the caller's workspace, summed in slice order by
// nf4_skinny_sum_kernel).
//
// MI355X, double-quantized weights read from HBM, GPU time against the tiled
// kernel of nf4_gemm.hip (512-row tiles, split-K) on the same box:
//   n x k          m = 1          m = 16-17      m = 32         m = 64
//   4096 x 4096    43.0 -> 8.6    42.4 -> 9.0    42.4 -> 13.1   42.7 -> 15.9 us
//   10240 x 8192   83.3 -> 24.0   77.7 -> 27.0   78.5 -> 26.9   78.5 -> 33.4 us
//   28672 x 8192   181 -> 43.4    174 -> 52.5    174 -> 54.9    170 -> 68.6 us
// What is left, from K = 8192 to 16384: a 128-deep step of a wave costs 0.55 us
// of its SIMD with four waves on it (3.8 TB/s of NF4 bytes), beside a fixed 5 us
// of launch, first loads and the final sum.  Counters: q/k/v of 8192 at 17
// tokens issue VALU work 39 % of the cycles and MFMAs 9 %, and the waves wait
// for loads and barriers 38 % of their time; 4096 x 4096 at one token waits
// 51 %; gate and up of 13824 x 5120 at 100 tokens: MFMA 24 %, VALU 30 %, waits
// 40 %, one LDS read per MFMA and no bank conflicts.
#include "gemm_common.hpp"
#include "nf4_skinny.hpp"

namespace nf4s {

constexpr int kSkStep = 128;    // reduction depth per step: two absmax blocks
constexpr int kSkRowUnits = 16; // 16-byte units of one token row per step

// x tile: token row r, logical 16-byte unit u (reduction elements 8u..8u+7 of
// the step) at r * 16 + (u ^ (r & 15)): the 16 lanes that a ds_read_b128
// serves at a time cover 16 rows at one unit, 16 distinct bank windows.
__device__ __forceinline__ int sk_unit(int r, int u) {
  return r * kSkRowUnits + (u ^ (r & 15));
}

// Partial tile of one wave in LDS: token t, chunk c (weight rows 4c..4c+3) as
// one floatx4 at t * 8 + (c ^ (t & 7)).
__device__ __forceinline__ int sk_chunk(int t, int c) { return t * 8 + (c ^ (t & 7)); }

// silu(x) = x / (1 + e^-x) (doublepass/src/math.rs:91-93), as the SwiGLU
// epilogue of the many-token kernel computes it.
__device__ __forceinline__ float sk_silu(float x) {
  const float e = __builtin_amdgcn_exp2f(-x * 1.4426950408889634f);
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// One lane's weights of one step: its block's packed words and raw absmax.
struct SkBlock {
  u32x4 w0, w1;
  float s;
  uint32_t q;
};

// An offset past every buffer resource here: such a load returns zero and
// touches no memory.
constexpr uint32_t kPast = 0x7ffffff0u;

// The wave's 32 weight rows (uniform) and the lane's offsets into them.
// Block b of the lane's row: packed bytes at poff + 32 b, absmax index
// (idx + b) >> block_shift, scale index (sidx + (b >> block_shift)) >>
// group_shift, all relative to the wave's first row.
struct SkRow {
  const void *packed, *am, *scale;
  int32_t packed_bytes, am_bytes, scale_bytes;
  uint32_t poff, idx, sidx;
  int32_t block_shift, group_shift;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t sk_rsrc(const void *p, int32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, kBufferFlags);
}

// Loads the lane's block of the step that starts at block b (uniform).  A
// step past the wave's range (!live, uniform) and a lane without a block
// (past: the second one of a step that has only one) get zero words and a
// zero absmax: code and scale both, since the blocks that follow belong to
// other rows, and an infinite or NaN scale of theirs times a zero code would
// put NaN into this row.
template <bool kDQ>
__device__ __forceinline__ void sk_load(const SkRow &r, int b, bool live, bool past, SkBlock &v) {
  const uint32_t off = past ? kPast : r.poff;
  const __amdgpu_buffer_rsrc_t pk = sk_rsrc(r.packed, live ? r.packed_bytes : 0);
  const __amdgpu_buffer_rsrc_t am = sk_rsrc(r.am, live ? r.am_bytes : 0);
  const int pb = __builtin_amdgcn_readfirstlane(32 * b);
  v.w0 = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(pk, (int)off, pb, 0));
  v.w1 = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(pk, (int)(off + 16), pb,
                                                                         0));
  const uint32_t blk = (r.idx + (uint32_t)b) >> r.block_shift;
  if constexpr (kDQ) {
    v.q = __builtin_amdgcn_raw_buffer_load_b8(am, (int)(past ? kPast : blk), 0, 0);
    const uint32_t sc = (r.sidx + (uint32_t)(b >> r.block_shift)) >> r.group_shift;
    const __amdgpu_buffer_rsrc_t rs = sk_rsrc(r.scale, live ? r.scale_bytes : 0);
    const uint32_t sv = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)(past ? kPast : 4 * sc), 0,
                                                             0);
    v.s = __builtin_bit_cast(float, sv);
  } else {
    const uint32_t av = __builtin_amdgcn_raw_buffer_load_b32(am, (int)(past ? kPast : 4 * blk), 0,
                                                             0);
    v.s = __builtin_bit_cast(float, av);
  }
}

// Dequantizes one packed word into the MFMA's 8 bf16 in three stages that the
// step spreads between MFMAs (NatLookup's lookup; `base` holds 0x03020100 in
// a vector register, which lets the and-or be one instruction).
__device__ __forceinline__ void sk_select(uint32_t w, uint32_t base, NatLookup &x) {
  nat_select(w, x);
  x.ctlA = ((x.selA >> 1) & 0x04040404u) | base;
  x.ctlB = ((x.selB >> 1) & 0x04040404u) | base;
  x.selA &= 0x07070707u;
  x.selB &= 0x07070707u;
}

// The step's MFMAs: 8 packed words of the lane's block against TM token
// tiles of the x tile `xt`; word j + 1 is dequantized while word j's MFMAs
// run.
template <int TM, int TR, bool kDQ>
__device__ __forceinline__ void sk_step(floatx16 (&acc)[TM], const SkBlock &blk, uint32_t base,
                                        const u32x4 *__restrict__ xt, int lane) {
  const int jl = lane & 31, g = lane >> 5;
  const Lut16 lut = make_lut<false>(kDQ ? (float)blk.q * blk.s : blk.s);
  auto word = [&](int j) { return j < 4 ? blk.w0[j & 3] : blk.w1[j & 3]; };
  auto read_x = [&](int j, u32x4 (&xf)[TM]) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
      xf[tm] = xt[sk_unit(TR < 32 ? jl & (TR - 1) : 32 * tm + jl, 8 * g + j)];
  };
  uint32_t o[2][4];
  {
    NatLookup n;
    sk_select(word(0), base, n);
    nat_planes_a(lut, n);
    nat_planes_b(lut, n);
    nat_merge(n, o[0]);
  }
  static_for<0, 8>([&](auto J) {
    constexpr int j = decltype(J)::value, c = j & 1;
    NatLookup n;
    u32x4 xf[TM];
    read_x(j, xf);
    if constexpr (j < 7) sk_select(word(j + 1), base, n);
    const u32x4 wf = {o[c][0], o[c][1], o[c][2], o[c][3]};
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
      acc[tm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, wf), __builtin_bit_cast(bf16x8, xf[tm]), acc[tm], 0, 0, 0);
    if constexpr (j < 7) {
      nat_planes_a(lut, n);
      nat_planes_b(lut, n);
      nat_merge(n, o[c ^ 1]);
    }
  });
}

// Stores 4 adjacent outputs of one token row: columns c .. c+3 of `row`, those below n.
__device__ __forceinline__ void sk_store4(uint16_t *row, int64_t c, int64_t n, bool vec_ok,
                                          const float v[4]) {
  const uint32_t lo = pack_bf16x2(v[0], v[1]), hi = pack_bf16x2(v[2], v[3]);
  if (vec_ok && c + 4 <= n) {
    *reinterpret_cast<u32x2 *>(row + c) = (u32x2){lo, hi};
  } else {
    if (c < n) row[c] = (uint16_t)(lo & 0xffffu);
    if (c + 1 < n) row[c + 1] = (uint16_t)(lo >> 16);
    if (c + 2 < n) row[c + 2] = (uint16_t)(hi & 0xffffu);
    if (c + 3 < n) row[c + 3] = (uint16_t)(hi >> 16);
  }
}

__device__ __forceinline__ bool sk_vec_ok(const uint16_t *out, int64_t ldo) {
  return ((reinterpret_cast<uintptr_t>(out) & 7) == 0) && ((ldo & 3) == 0);
}

// TR: token rows in LDS (4, 16, 32, 64, 96, 128 >= m).  SwiGLU: even waves of a
// k-group take 32 gate rows, odd ones the same 32 up rows, and hidden is
// elementwise between their partial tiles.
template <int TR, int WN, int WK, bool kSwiglu, bool kDQ>
__global__ void __launch_bounds__(64 * WN * WK, TR <= 64 ? 4 : 2)
    nf4_skinny_kernel(const SkinnyArgs a) {
  static_assert(!kSwiglu || WN % 2 == 0, "gate and up rows in pairs of waves");
  constexpr int TM = TR < 32 ? 1 : TR / 32;
  constexpr int kCols = 32 * (kSwiglu ? WN / 2 : WN);  // output columns of the workgroup
  constexpr int kXUnits = TR * kSkRowUnits;     // one x tile
  constexpr int kXLds = 2 * WK * kXUnits;
  constexpr int kRedLds = WN * WK * TR * 8;
  __shared__ u32x4 lds[kXLds > kRedLds ? kXLds : kRedLds];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int tile = blockIdx.x / a.slices;
  const int slice = blockIdx.x - tile * a.slices;
  // The weight of this tile (uniform).
  int gi = 0;
  if (!kSwiglu) {
#pragma unroll
    for (int j = 1; j < kSkinnyMaxGroups; ++j) gi += (j < a.ngroups && tile >= a.grp[j].tile0);
  }
  const int64_t c0 = (int64_t)(tile - a.grp[gi].tile0) * kCols;  // first column
  const int64_t n = a.grp[gi].n;
  const int jl = lane & 31, g = lane >> 5;
  const int blocks = (int)(a.k >> 6);  // 64-element blocks per row
  SkRow row;
  {
    // Rows from this wave's first one, r0 (or the last row: a wave past it
    // stores nothing), clamped to the rows that exist.
    const SkinnyGroup &w = a.grp[kSwiglu ? (wn & 1) : gi];
    int64_t r0 = c0 + 32 * (kSwiglu ? (wn >> 1) : wn);
    if (r0 > n - 1) r0 = n - 1;
    const int32_t last = (n - 1 - r0 < 31) ? (int32_t)(n - 1 - r0) : 31;
    const uint32_t r = (uint32_t)(jl < last ? jl : last);
    const int64_t b0 = r0 * blocks;  // first 64-element block of row r0
    const int bs = w.am.block_shift, gs = w.am.group_shift;
    const int64_t a0 = b0 >> bs;     // its absmax block
    row.packed = w.packed + b0 * 32;
    row.packed_bytes = (last + 1) * blocks * 32;
    const int nblk = ((last + 1) * blocks) >> bs;
    if constexpr (kDQ) {
      row.am = w.am.q + a0;
      row.am_bytes = nblk;
      row.scale = w.am.scale + (a0 >> gs);
      row.scale_bytes = 4 * (int)(((a0 + nblk - 1) >> gs) - (a0 >> gs) + 1);
    } else {
      row.am = w.am.absmax + a0;
      row.am_bytes = 4 * nblk;
    }
    row.poff = r * (uint32_t)(blocks * 32) + 32u * (uint32_t)g;
    row.idx = r * (uint32_t)blocks + (uint32_t)g;
    // Scale groups are not aligned to rows: keep the first block's place in its group.
    row.sidx = (uint32_t)(a0 & (((int64_t)1 << gs) - 1)) + (row.idx >> bs);
    row.block_shift = bs;
    row.group_shift = gs;
  }
  uint32_t base = 0x03020100u;
  asm("" : "+v"(base));

  // This k-group's steps s0 .. s1-1: the slice's steps in WK contiguous
  // parts.  Every wave runs the same number of steps; those past s1 load
  // zeros.
  const int steps = (blocks + 1) >> 1;
  const int sl0 = slice * a.slice_steps;
  const int sl1 = (sl0 + a.slice_steps < steps) ? sl0 + a.slice_steps : steps;
  const int per = (sl1 - sl0 + WK - 1) / WK;
  const int s0 = sl0 + wk * per;
  const int s1 = (s0 + per < sl1) ? s0 + per : sl1;

  // Direct-to-LDS loads of the x tile: instruction i covers token rows 4i ..
  // 4i+3 (lane p: row 4i + p / 16, physical unit p % 16); the WN waves of a
  // k-group take them in turn.  Rows past m, steps past s1 and the second
  // block of a last step that has only one read as zero.
  constexpr int kDma = TR / 4 / WN;
  static_assert(kDma > 0, "a DMA for every wave");
  uint32_t xoff[kDma];
  uint32_t second = 0;  // bit i: the lane's unit of DMA i is in the second block
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = 4 * (WN * i + wn) + (lane >> 4);
    const int u = (lane & 15) ^ (r & 15);
    xoff[i] = r < a.m ? (uint32_t)(r * a.k * 2 + 16 * u) : kPast;
    second |= (uint32_t)(u >> 3) << i;
  }
  const int32_t xbytes = (int32_t)(a.m * a.k * 2);
  u32x4 *x0 = lds + wk * kXUnits, *x1 = lds + (WK + wk) * kXUnits;
  auto load_x = [&](u32x4 *dst, int s) {
    const __amdgpu_buffer_rsrc_t rs = sk_rsrc(a.x, s < s1 ? xbytes : 0);
    const int so = __builtin_amdgcn_readfirstlane(s * (kSkStep * 2));
    const bool half = 2 * s + 1 >= blocks;  // uniform
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (lds_void_t *)(dst + 64 * (WN * i + wn)), 16,
          (int)(half && ((second >> i) & 1) ? kPast : xoff[i]), so, 0, 0);
  };
  auto load_w = [&](SkBlock &v, int s) {
    sk_load<kDQ>(row, 2 * s, s < s1, 2 * s + 1 >= blocks && g != 0, v);
  };

  floatx16 acc[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;

  // Step s issues the loads of step s + 1; the wait that closes it then finds
  // them landed, since the SIMD's other waves had their turn meanwhile (two
  // and three steps ahead took registers from the waves and measured 15-25 %
  // slower).
  SkBlock w[2];
  load_x(x0, s0);
  load_w(w[0], s0);
  auto close = [&] {
    if constexpr (WN > 1) {
      step_barrier<0>();
    } else {  // the wave's own x tile
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  close();
  auto step = [&](auto U, int s) {
    constexpr int u = decltype(U)::value;
    load_x(u ? x0 : x1, s + 1);
    load_w(w[u ^ 1], s + 1);
    __builtin_amdgcn_sched_barrier(0);
    sk_step<TM, TR, kDQ>(acc, w[u], base, u ? x1 : x0, lane);
    close();
  };
  const int end = s0 + per;
#pragma unroll 1
  for (int s = s0; s < end; s += 2) {
    step(IC<0>{}, s);
    if (s + 1 >= end) break;
    step(IC<1>{}, s + 1);
  }
  // No DMA may still write the x tiles that the partials below replace.
  step_barrier<0>();

  // Partial tiles to LDS (the x tiles are done with), then each thread sums
  // the k-groups' chunk in order and stores 4 outputs of one token.
  floatx4 *red = reinterpret_cast<floatx4 *>(lds);
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int tok = 32 * t + jl;
    if (tok < a.m) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        red[wave * (TR * 8) + sk_chunk(tok, 2 * j + g)] =
            (floatx4){acc[t][4 * j], acc[t][4 * j + 1], acc[t][4 * j + 2], acc[t][4 * j + 3]};
    }
  }
  __syncthreads();
  constexpr int kQuads = kCols / 4;
  const int m = (int)a.m;
  for (int e = threadIdx.x; e < m * kQuads; e += 64 * WN * WK) {
    const int tok = e / kQuads, q = e - tok * kQuads;
    const int rn = (q >> 3) * (kSwiglu ? 2 : 1), c = q & 7;
    floatx4 v = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < WK; ++kk) {
      v += red[(kk * WN + rn) * (TR * 8) + sk_chunk(tok, c)];
      if constexpr (kSwiglu) u += red[(kk * WN + rn + 1) * (TR * 8) + sk_chunk(tok, c)];
    }
    if (!kSwiglu && a.slices > 1) {
      const int64_t width = (int64_t)a.tiles * kCols;
      *reinterpret_cast<floatx4 *>(a.ws + ((int64_t)slice * m + tok) * width +
                                   (int64_t)tile * kCols + 4 * q) = v;
    } else {
      float o[4] = {v.x, v.y, v.z, v.w};
      if constexpr (kSwiglu) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = sk_silu(v[i]) * u[i];
      }
      uint16_t *out = a.grp[gi].out;
      sk_store4(out + tok * n, c0 + 4 * q, n, sk_vec_ok(out, n), o);
    }
  }
}

// Sums the K slices' partials [slice][token][width] in slice order: one
// thread takes 4 adjacent columns of one token.
__global__ void __launch_bounds__(256) nf4_skinny_sum_kernel(const SkinnyArgs a, int tile_rows) {
  const int64_t width = (int64_t)a.tiles * tile_rows;
  const int64_t quads = width >> 2;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= a.m * quads) return;
  const int64_t tok = e / quads, q = e - tok * quads;
  const floatx4 *p = reinterpret_cast<const floatx4 *>(a.ws) + tok * quads + q;
  floatx4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < a.slices; ++s) v += p[(int64_t)s * a.m * quads];
  const int tile = (int)(4 * q / tile_rows);
  int gi = 0;
#pragma unroll
  for (int j = 1; j < kSkinnyMaxGroups; ++j) gi += (j < a.ngroups && tile >= a.grp[j].tile0);
  const int64_t n = a.grp[gi].n;
  const int64_t col = 4 * q - (int64_t)a.grp[gi].tile0 * tile_rows;
  const float o[4] = {v.x, v.y, v.z, v.w};
  uint16_t *out = a.grp[gi].out;
  sk_store4(out + tok * n, col, n, sk_vec_ok(out, n), o);
}

// The workgroup shape for m tokens: up to 64 tokens 64 KB of LDS or less, two
// workgroups a CU.
// As few weight rows as the x traffic allows (each 32-row block re-reads x
// from L2), so that the K split stays inside the workgroup.  Measured against
// it, 28672 x 8192 and 4096 x 4096: four-wave workgroups for m <= 16, 44.9
// and 9.9 us (43.4 and 8.6); {32, 4, 4} for m = 32, 55.2 and 17.1 (54.9 and
// 13.2); {64, 4, 4} for m = 64, 78.3 and 22.5 (68.6 and 15.9).
// Up to 128 tokens, 128 KB: every x fragment still feeds only one MFMA per
// wave, so the LDS reads of all waves take as long as the MFMAs, but at 100
// tokens it beats the tiled kernel's 128-row tiles (28672 x 8192 88 us against
// 96, 4096 x 4096 21 against 25; 512-row tiles took 175 and 42).  Beyond them
// the wave has no registers for more tokens: the tiled kernel, whose waves
// share the dequantized weights instead, takes over.
// 96-token tiles (96 KB) between: the MFMAs and x reads of a quarter fewer token
// tiles; at 80 tokens against 128-token ones 28672 x 8192 84.2 -> 76.2 us,
// 4096 x 4096 19.4 -> 17.9, SwiGLU of 13824 x 5120 52.5 -> 47.2.
struct SkShape {
  int tr, wn, wk;
};
static SkShape sk_shape(int64_t m, bool swiglu) {
  if (m <= 4 && !swiglu) return {4, 1, 8};
  if (m <= 16) return swiglu ? SkShape{16, 2, 4} : SkShape{16, 1, 8};
  if (m <= 32) return {32, 2, 4};
  if (m <= 64) return {64, 4, 2};
  if (m <= 96) return {96, 4, 2};
  return {128, 4, 2};
}

// SwiGLU tiles of 64 hidden columns that would leave half the CUs without a
// workgroup run as 32-column tiles instead: twice the workgroups, and for 64
// and 96 tokens more k-groups in each (128 and 144 KB of LDS, one a CU).
// Against the wide shapes, gate and up of 4096 x 4096: 64 tokens 28.7 -> 19.1
// us, 96 tokens 38.5 -> 26.8, 128 tokens 39.2 -> 33.2; of 8192 x 8192 56.2 ->
// 37.9, 78.6 -> 53.3, 79.0 -> 66.0.  Beyond 8192 columns the narrow tiles no
// longer fit one round.
static SkShape sk_narrow(const SkShape &sh) {
  return {sh.tr, 2, sh.tr == 64 ? 4 : sh.tr == 96 ? 3 : 2};
}

// K slices of a launch of `tiles` output tiles: as many as two workgroups a
// CU take at once, each wave keeping at least 4 steps (fewer would spend more
// on the partials than on the weights).
static int sk_slices(int64_t tiles, int64_t steps, const SkShape &sh) {
  const int64_t slots = (sh.tr > 64 ? 1 : 2) * (int64_t)cu_slots();  // 96 KB of LDS or more: one
  int64_t s = slots / tiles;
  const int64_t most = steps / (4 * sh.wk);  // at least 4 steps per wave
  if (s > most) s = most;
  if (s < 2) return 1;
  const int64_t per = (steps + s - 1) / s;
  return (int)((steps + per - 1) / per);  // slices of `per` steps that are not empty
}

static int64_t sk_tiles(int64_t n, int rows) { return (n + rows - 1) / rows; }

// Weights of one kind share a launch and a mixed set runs one launch per
// kind, each with the whole workspace: the largest plan over every subset.
int64_t skinny_workspace_bytes(const int64_t *ns, int32_t count, int64_t m, int64_t k) {
  const SkShape sh = sk_shape(m, false);
  const int rows = 32 * sh.wn;
  const int64_t steps = (k / 64 + 1) / 2;
  int64_t best = 0;
  for (uint32_t set = 1; set < (1u << count); ++set) {
    int64_t tiles = 0;
    for (int32_t i = 0; i < count; ++i)
      if (set & (1u << i)) tiles += sk_tiles(ns[i], rows);
    const int64_t s = sk_slices(tiles, steps, sh);
    const int64_t bytes = s < 2 ? 0 : s * m * tiles * rows * (int64_t)sizeof(float);
    if (bytes > best) best = bytes;
  }
  return best;
}

template <bool kSwiglu, bool kDQ>
static void sk_launch(const SkinnyArgs &a, const SkShape &sh, uint32_t grid, hipStream_t s) {
  const dim3 g(grid), b(64 * sh.wn * sh.wk);
  if constexpr (kSwiglu) {
    if (sh.wn == 2 && sh.tr >= 64) {
      if (sh.tr == 64)
        hipLaunchKernelGGL((nf4_skinny_kernel<64, 2, 4, true, kDQ>), g, b, 0, s, a);
      else if (sh.tr == 96)
        hipLaunchKernelGGL((nf4_skinny_kernel<96, 2, 3, true, kDQ>), g, b, 0, s, a);
      else
        hipLaunchKernelGGL((nf4_skinny_kernel<128, 2, 2, true, kDQ>), g, b, 0, s, a);
      return;
    }
  }
  switch (sh.tr) {
    case 4:
      if constexpr (!kSwiglu)
        hipLaunchKernelGGL((nf4_skinny_kernel<4, 1, 8, false, kDQ>), g, b, 0, s, a);
      break;
    case 16:
      if constexpr (kSwiglu)
        hipLaunchKernelGGL((nf4_skinny_kernel<16, 2, 4, true, kDQ>), g, b, 0, s, a);
      else
        hipLaunchKernelGGL((nf4_skinny_kernel<16, 1, 8, false, kDQ>), g, b, 0, s, a);
      break;
    case 32: hipLaunchKernelGGL((nf4_skinny_kernel<32, 2, 4, kSwiglu, kDQ>), g, b, 0, s, a); break;
    case 64: hipLaunchKernelGGL((nf4_skinny_kernel<64, 4, 2, kSwiglu, kDQ>), g, b, 0, s, a); break;
    case 96: hipLaunchKernelGGL((nf4_skinny_kernel<96, 4, 2, kSwiglu, kDQ>), g, b, 0, s, a); break;
    default: hipLaunchKernelGGL((nf4_skinny_kernel<128, 4, 2, kSwiglu, kDQ>), g, b, 0, s, a); break;
  }
}

// One launch over the weights of `all` that are (dq) or are not
// double-quantized.
static int32_t sk_fwd_kind(const SkinnyArgs &all, bool dq, hipStream_t s, void *work,
                           int64_t work_bytes) {
  SkinnyArgs a = all;
  a.ngroups = 0;
  const SkShape sh = sk_shape(a.m, false);
  const int rows = 32 * sh.wn;
  int64_t tiles = 0;
  for (int32_t i = 0; i < all.ngroups; ++i) {
    if ((all.grp[i].am.q != nullptr) != dq) continue;
    SkinnyGroup &w = a.grp[a.ngroups++];
    w = all.grp[i];
    w.tile0 = (int32_t)tiles;
    tiles += sk_tiles(w.n, rows);
  }
  if (a.ngroups == 0) return NF4S_OK;
  a.tiles = (int32_t)tiles;
  const int steps = (int)((a.k / 64 + 1) / 2);
  a.slices = sk_slices(tiles, steps, sh);
  const int64_t per_slice = a.m * tiles * rows * (int64_t)sizeof(float);
  const int64_t fit = work != nullptr ? work_bytes / per_slice : 0;
  if (a.slices > fit) a.slices = fit < 2 ? 1 : (int)fit;
  a.slice_steps = (steps + a.slices - 1) / a.slices;
  a.slices = (steps + a.slice_steps - 1) / a.slice_steps;
  a.ws = static_cast<float *>(work);
  if (dq)
    sk_launch<false, true>(a, sh, (uint32_t)(tiles * a.slices), s);
  else
    sk_launch<false, false>(a, sh, (uint32_t)(tiles * a.slices), s);
  int32_t rc = check_launch("nf4_skinny");
  if (rc == NF4S_OK && a.slices > 1) {
    const int64_t quads = a.m * tiles * rows / 4;
    hipLaunchKernelGGL(nf4_skinny_sum_kernel, dim3((uint32_t)((quads + 255) / 256)), dim3(256), 0,
                       s, a, rows);
    rc = check_launch("nf4_skinny_sum");
  }
  return rc;
}

int32_t skinny_fwd(const SkinnyArgs &a, hipStream_t s, void *work, int64_t work_bytes) {
  const int32_t rc = sk_fwd_kind(a, true, s, work, work_bytes);
  return rc != NF4S_OK ? rc : sk_fwd_kind(a, false, s, work, work_bytes);
}

int32_t skinny_swiglu(SkinnyArgs &a, hipStream_t s) {
  SkShape sh = sk_shape(a.m, true);
  if (sh.wn == 4 && 2 * sk_tiles(a.grp[0].n, 64) <= cu_slots()) sh = sk_narrow(sh);
  const int64_t tiles = sk_tiles(a.grp[0].n, 16 * sh.wn);
  a.grp[0].tile0 = a.grp[1].tile0 = 0;
  a.tiles = (int32_t)tiles;
  a.slices = 1;
  a.slice_steps = (int)((a.k / 64 + 1) / 2);
  a.ws = nullptr;
  if (a.grp[0].am.q != nullptr)
    sk_launch<true, true>(a, sh, (uint32_t)tiles, s);
  else
    sk_launch<true, false>(a, sh, (uint32_t)tiles, s);
  return check_launch("nf4_skinny_swiglu");
}

}  // namespace nf4s
