// bf16_wgrad.hip - weight gradient dW = dY^T . X for gfx950 (MI355X).
//
//   dw[n, k] (+)= sum_m dy[m, n] * x[m, k]
// the d_wd / d_wg / d_wu / d_wo / d_wq / d_wk / d_wv loops of
// single_layer_backward (doublepass/src/backward.rs:87-93, 117-129, 160-168,
// 284-300), with the micro-batch accumulation of backward.rs:478-502 as the
// `accumulate` flag.  dy [M, N] and x [M, K] are bf16, row-major; dw [N, K]
// fp32.  The reduction runs over the token index m, the row index of both
// operands, so both MFMA operands are columns of row-major tiles.
//
// Workgroup = 4 waves in 2 x 2, tile = 64 kMT dW rows (n) x 256 dW columns (k),
// kMT = 4 or 2; each wave owns 32 kMT x 128 in 64 kMT accumulator registers
// (4 kMT tiles of v_mfma_f32_32x32x16_bf16).  kMT = 4 takes a CU for itself,
// of kMT = 2 two workgroups share one (wg_tile_mt says which is launched).
// Per 32-token step the dy tile (32 x 64 kMT bf16) and the x tile (32 x 256)
// move into LDS with direct-to-LDS loads, into a ring of kWgStages stages of
// 32 (24) KB that keeps the next kWgStages - 1 steps in
// flight while step t computes (3 stages measured faster than 2 of 64
// tokens, and than 4 or 5 of 32), and each wave reads its fragments with
// the transposing ds_read_b64_tr_b16: 8 consecutive tokens of one column
// per lane.
#include <cmath>

#include "abi_common.hpp"
#include "gemm_common.hpp"
#include "nf4_device.hpp"

namespace nf4s {

constexpr int kWgThreads = 256;
constexpr int kWgTile = 256;  // dW columns per workgroup
constexpr int kWgStep = 32;   // tokens per step
constexpr int kWgStages = 3;  // LDS ring stages

constexpr int kMaxWgGroups = 4;  // products per launch that share x

// The products of one launch stack their dW row tiles: product i owns tile
// rows tile0[i] .. tile0[i+1]-1 of a tiles_n x tiles_k grid.
struct WgradArgs {
  const uint16_t *dy[kMaxWgGroups];  // [M, N_i], row stride N_i
  float *dw[kMaxWgGroups];           // [N_i, K], row stride K
  int64_t N[kMaxWgGroups];
  int32_t tile0[kMaxWgGroups + 1];
  int32_t ngroups;
  const uint16_t *x;  // [M, K], row stride K
  int64_t M, K;
  int32_t tiles_n, tiles_k;
  int32_t blk_n, blk_k;  // XCD block of blk_n x blk_k tiles (0: strips)
  int32_t strip;         // tile columns per strip (wg_map_tile)
};

// a[i] for a wave-uniform i < kMaxWgGroups, as a chain of selects: indexing
// the kernel-argument arrays with a variable would copy them to scratch.
template <typename T>
__device__ __forceinline__ T wg_pick(const T (&a)[kMaxWgGroups], int i) {
  T v = a[0];
#pragma unroll
  for (int j = 1; j < kMaxWgGroups; ++j) v = (i == j) ? a[j] : v;
  return v;
}

// Tile order.  An XCD's resident workgroups should form a square-ish patch of
// the tile grid: they then read few dy and x column blocks per step from
// memory and the rest from the XCD's L2.
// A launch whose rounds are all full (T a multiple of the grid G, G / 8 slots
// per XCD): in round r, XCD x (workgroups b with b % 8 == x) takes block
// 8 r + x of blk_n x blk_k tiles, blk_n * blk_k = G / 8, slot i = (b % G) / 8
// the tile (i / blk_k, i % blk_k) of the block.
// Any other launch: the tiles are numbered row by row within strips of
// `strip` tile columns (the last one narrower) and each XCD takes a
// contiguous range of them.  Rows over the whole width instead read every x
// block for each dy block: 11008 x 16384 over 8192 tokens 2498 us, strips
// 2295 (256-row tiles); 4096 x 11008 over 4096, 429 and 317 (128-row).
__device__ __forceinline__ void wg_map_tile(const WgradArgs &g, int b, int &tn, int &tk) {
  if (g.blk_n == 0) {
    const int T = g.tiles_n * g.tiles_k;
    const int x = b & 7, base = T >> 3, rem = T & 7;
    const int L = x * base + (x < rem ? x : rem) + (b >> 3);
    const int per = g.tiles_n * g.strip;  // tiles of a whole strip
    const int s = L / per, i = L - s * per;
    const int left = g.tiles_k - s * g.strip;
    const int w = left < g.strip ? left : g.strip;
    tn = i / w;
    tk = s * g.strip + i - tn * w;
    return;
  }
  const int G = gridDim.x;
  const int r = b / G, c = b - r * G;
  const int blk = 8 * r + (c & 7), i = c >> 3;
  const int nbk = g.tiles_k / g.blk_k;
  const int bn = blk / nbk, bk = blk - bn * nbk;
  tn = bn * g.blk_n + i / g.blk_k;
  tk = bk * g.blk_k + i % g.blk_k;
}

// LDS tile: 32 token rows x 256 columns (512 B = 32 units of 16 B per row), or
// 128 columns (16 units) of dy when kMT = 2.  A wave reads one half of the
// columns.  Unit u of row r lives at
// physical unit (u & 16) | ((u & 15) ^ 5 (r % 4)): with it, each 32-lane
// half of a transposed fragment read covers 16 distinct 16-B units of one
// half-row's 64 banks (rows are 512 B or 256 B = 128 or 64 banks apart, so every
// row starts at bank 0), and each 16-lane quarter of a DMA writes one row's 16
// contiguous units.
__device__ __forceinline__ int wg_unit(int row, int u) {
  return (u & 16) | ((u & 15) ^ (5 * (row & 3)));
}

// 16-byte units of one token row of the dy tile, and of one stage (dy tile,
// then x tile).
template <int kMT>
constexpr int kWgDyUnits = 8 * kMT;
template <int kMT>
constexpr int kWgStageUnits = kWgStep * (kWgDyUnits<kMT> + 32);

// Byte offset (from its tile's base) of lane `lane`'s first transposed read
// of fragment j: column 32j + lane % 32 of the wave's half h, token rows
// 8 (lane / 32) + 0..3 of sub-step 0.  ds_read_b64_tr_b16 transposes 4 x 4
// blocks of 16-bit values within each 16-lane group: lane i receives element
// i % 4 of the 8 bytes that lane 4e + i / 4 addresses, so lane 4e + c
// addresses row e, columns 4c..4c+3 of the group's 16-column strip.  A second
// read 4 rows lower completes the 8 tokens.
template <int kUnits>
__device__ __forceinline__ uint32_t wg_read_off(int lane, int h, int j) {
  const int l16 = lane & 15, e = l16 >> 2;
  const int row = 8 * (lane >> 5) + e;
  const int u = kUnits / 2 * h + 4 * j + 2 * ((lane >> 4) & 1) + ((l16 >> 1) & 1);
  return (uint32_t)(16 * (kUnits * row + wg_unit(row, u)) + 8 * (l16 & 1));
}

// Fragment (8 tokens of one column, sub-step s) from the tile at `base`, whose
// rows are kUnits 16-byte units long.
template <int kUnits>
__device__ __forceinline__ u32x4 wg_frag(const char *base, uint32_t off, int s) {
  typedef __attribute__((address_space(3))) char lds_char_t;
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16_t;
  lds_char_t *p = (lds_char_t *)const_cast<char *>(base) + off + 256 * kUnits * s;
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t *)p);
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t *)(p + 64 * kUnits));
  const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
  return (u32x4){l2.x, l2.y, h2.x, h2.y};
}

// Fragment read q (0 .. kMT + 3) of a sub-step in the order the sub-step's first
// MFMAs use them: dy0, x0, x1, x2, x3, dy1, dy2, dy3.
template <int kMT>
__device__ __forceinline__ void wg_read(const char *tdy, const char *tx, const uint32_t (&rdy)[kMT],
                                        const uint32_t (&rx)[4], u32x4 (&fd)[kMT], u32x4 (&fx)[4],
                                        int s, int q) {
  if (q == 0 || q >= 5) {
    const int j = (q == 0) ? 0 : q - 4;
    fd[j] = wg_frag<kWgDyUnits<kMT>>(tdy, rdy[j], s);
  } else {
    fx[q - 1] = wg_frag<32>(tx, rx[q - 1], s);
  }
}

// One 32-token step t from stage `cur`: 2 sub-steps of 4 kMT MFMAs (the
// counts below are kMT = 4's).  The
// fragments of sub-step 1 are read (one per MFMA slot) during sub-step 0.
// The kMT + 4 DMAs of this wave for step t + kWgStages - 1 (8 token rows of dy
// and of x, 1 KB per instruction) go into stage `nxt` after
// MFMAs 9, 11, .., 23 (the same DMAs in sub-step 0's first half measured
// 1-2 % slower on 70B shapes); that stage held step t-1, whose reads all
// ended before the barrier that closed step t-1.  The caller's barrier
// after MFMA 7 of sub-step 1 waits for step t+1's DMAs (leaving the later
// steps' in flight) and every LDS read; the last 8 MFMAs (operands in
// registers) open the next call, each followed by one of the next step's
// sub-step 0 reads.
// `more` (that step exists) is a branch around the DMAs, which keeps each
// DMA after its slot's MFMA and reads.  The LDS stages come in as distinct
// __restrict__ pointers: the compiler then knows that DMAs into `nxt` never
// alias the reads of `cur` and waits (vmcnt) only at the barriers.
template <int kMT>
__device__ __forceinline__ void wgrad_step(floatx16 (&acc)[kMT][4], u32x4 (&fd)[2][kMT],
                                           u32x4 (&fx)[2][4], const char *__restrict__ cur_dy,
                                           const char *__restrict__ cur_x,
                                           char *__restrict__ nxt_dy, char *__restrict__ nxt_x,
                                           const uint32_t (&rdy)[kMT], const uint32_t (&rx)[4],
                                           __amdgpu_buffer_rsrc_t rs_dy,
                                           __amdgpu_buffer_rsrc_t rs_x,
                                           uint32_t (&vdy)[kMT], uint32_t (&vx)[4],
                                           uint32_t step_dy, uint32_t step_x, bool more, int wave) {
  constexpr int kReads = kMT + 4, kDmas = kMT + 4;
  constexpr int kPost = 2 * kMT;           // MFMAs that open the next step
  constexpr int kFront = 8 * kMT - kPost;  // the others
  // Previous step's last MFMAs, then this step's sub-step 0 reads.
  static_for<0, kPost>([&](auto I) {
    constexpr int i = decltype(I)::value;
    constexpr int mt = kMT / 2 + (i >> 2), nt = i & 3;
    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, fx[1][nt]), __builtin_bit_cast(bf16x8, fd[1][mt]),
        acc[mt][nt], 0, 0, 0);
    static_for<0, kReads>([&](auto Q) {
      constexpr int q = decltype(Q)::value;
      if constexpr (q * kPost / kReads == i)
        wg_read<kMT>(cur_dy, cur_x, rdy, rx, fd[0], fx[0], 0, q);
    });
    __builtin_amdgcn_sched_barrier(0);
  });
  static_for<0, kFront>([&](auto N) {
    constexpr int n = decltype(N)::value;
    constexpr int s = n / (4 * kMT), i = n % (4 * kMT);
    constexpr int mt = i >> 2, nt = i & 3;
    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, fx[s][nt]), __builtin_bit_cast(bf16x8, fd[s][mt]),
        acc[mt][nt], 0, 0, 0);
    if constexpr (s == 0 && i < kReads)
      wg_read<kMT>(cur_dy, cur_x, rdy, rx, fd[1], fx[1], 1, i);
    // DMA d, after MFMAs 9, 11, .., 23 (kMT = 4) or 6, 7, .., 11 (kMT = 2): the
    // kMT of dy, then the 4 of x.
    constexpr int kGap = kMT / 2;
    constexpr int back = kFront - 1 - n;  // MFMAs after this one
    if constexpr (back % kGap == 0 && back / kGap < kDmas) {
      constexpr int d = kDmas - 1 - back / kGap;
      if (more) {
        if constexpr (d < kMT) {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              rs_dy, (lds_void_t *)(nxt_dy + 1024 * (kMT * wave + d)), 16,
              (int)vdy[d], 0, 0, 0);
          vdy[d] += step_dy;
        } else {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              rs_x, (lds_void_t *)(nxt_x + 1024 * (4 * wave + d - kMT)), 16, (int)vx[d - kMT], 0,
              0, 0);
          vx[d - kMT] += step_x;
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  });
}

// The barrier that closes step t: this wave's DMAs of step t+1 have landed
// and every LDS read of step t has ended.  Its DMAs of the later steps in
// the ring (t+2 .. t+kWgStages-1, kMT + 4 each, issued after t+1's, those that
// exist) may still be in flight: vmcnt retires in issue order.
template <int kMT>
__device__ __forceinline__ void wgrad_close_step(int64_t t, int64_t nsteps) {
  int64_t later = nsteps - t - 2;  // steps after t+1 that exist, clamped below
  later = (later < 0) ? 0 : (later > kWgStages - 2) ? kWgStages - 2 : later;
  static_for<0, kWgStages - 1>([&](auto I) {
    constexpr int a = decltype(I)::value;  // exactly one a == later
    if (later == a) step_barrier<(kMT + 4) * a>();
  });
}

// Direct epilogue, for outputs without 16-byte stores: four adjacent fp32 per
// store or less.
template <bool kAcc, int kMT>
__device__ __forceinline__ void wg_store(const WgradArgs &g, const floatx16 (&acc)[kMT][4],
                                         float *dw, int64_t n0, int64_t k0, int64_t N, int lane,
                                         bool vec_ok) {
  asm volatile("" : "+v"(lane));  // as in wg_store_lds
  const int jl = lane & 31, grp = lane >> 5;
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt) {
    const int64_t n = n0 + 32 * mt + jl;
    if (n < N) {
      float *row = dw + n * g.K;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t k = k0 + 32 * nt + 8 * j + 4 * grp;
          floatx4 v = {acc[mt][nt][4 * j], acc[mt][nt][4 * j + 1], acc[mt][nt][4 * j + 2],
                       acc[mt][nt][4 * j + 3]};
          if (vec_ok && k + 4 <= g.K) {
            floatx4 *p = reinterpret_cast<floatx4 *>(row + k);
            if constexpr (kAcc) v += *p;
            *p = v;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (k + i < g.K) row[k + i] = kAcc ? row[k + i] + v[i] : v[i];
          }
        }
    }
  }
}

// Epilogue through LDS for outputs that take 16-byte stores: the direct stores
// write 32 rows x 32 bytes per instruction, these two whole 512-byte rows.
// Per 32-row block mt the wave writes its 32 x 128 fp32 to its own 16 KB of
// the idle ring (row r, 16-byte chunk c at physical chunk c ^ r: the lanes of a
// ds_write_b128 share c, those of a ds_read_b128 r, both spread over all
// banks), reads it back by rows and stores; to accumulate, 8 of dW's old row
// pairs are loaded at a time.  Chunks past the last column are dropped: K is a
// multiple of 8, so none is partial.  (Direct stores for the tiles of a ragged
// last column, all on the XCD that takes the last strip, kept it busy after
// the others: 15696 x 6120 over 100 tokens 118 -> 94 us, accumulating 270 ->
// 165.)
// The tile's output burst (64 MB a round over the chip) is what a short
// reduction waits for: against the direct stores, same box, 2 x 11008 x 4096
// over 1000 tokens 245 -> 231 us (326 -> 273 accumulating), 28672 x 8192 over
// 512 tokens 384 -> 319 (600 -> 484), 8192 x 8192 over 8192 tokens 846 -> 826
// (909 -> 867).
// kNt: non-temporal stores (wg_nontemporal).  Accumulating and the store policy
// are instantiations: as a run-time test accumulating spilled 51 registers in
// both, the policy 9.
template <bool kAcc, int kMT, bool kNt>
__device__ __forceinline__ void wg_store_lds(const WgradArgs &g, const floatx16 (&acc)[kMT][4],
                                             floatx4 *lds, float *dw, int64_t n0, int64_t k0,
                                             int64_t N, int lane) {
  // An opaque lane index keeps the per-lane addresses below from being hoisted
  // out of the tile loop and spilled.
  asm volatile("" : "+v"(lane));
  const int jl = lane & 31, grp = lane >> 5;
  const int r0 = lane >> 5, c = lane & 31;  // read-back: row 2i + r0, chunk c
  // The wave's rows below N through a buffer resource that ends after the last.
  const int64_t left = N - n0;
  const int64_t cols = g.K - k0;  // <= 0 for a wave past the last column
  const int64_t rows = left <= 0 || cols <= 0 ? 0 : (left > 32 * kMT ? 32 * kMT : left);
  const uint32_t ld4 = (uint32_t)(g.K * 4);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(rows > 0 ? dw + n0 * g.K + k0 : dw), 0,
      rows > 0 ? (int32_t)((rows - 1) * ld4 + 4 * (uint32_t)(cols < 128 ? cols : 128)) : 0,
      kBufferFlags);
  typedef unsigned int uvec4 __attribute__((ext_vector_type(4)));
  constexpr int kPolicy = kNt ? 2 : 0;
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt) {
    const uint32_t base = (uint32_t)(32 * mt + r0) * ld4 + 16u * (uint32_t)c;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        lds[jl * 32 + ((8 * nt + 2 * j + grp) ^ jl)] =
            (floatx4){acc[mt][nt][4 * j], acc[mt][nt][4 * j + 1], acc[mt][nt][4 * j + 2],
                      acc[mt][nt][4 * j + 3]};
    // Other lanes' writes are read below, and the reads end before the next
    // block's writes.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int h = 0; h < 16; h += 8) {
      if (4 * c >= cols) continue;  // a lane past the last column
      floatx4 v[8], old[8];
      if constexpr (kAcc) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          old[i] = __builtin_bit_cast(
              floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                           rs, (int)(base + 2u * (uint32_t)(h + i) * ld4), 0, 0));
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = 2 * (h + i) + r0;
        v[i] = lds[r * 32 + (c ^ r)];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (kAcc) v[i] += old[i];
        __builtin_amdgcn_raw_buffer_store_b128(
            __builtin_bit_cast(uvec4, v[i]), rs,
            (int)(base + 2u * (uint32_t)(h + i) * ld4), 0, kPolicy);
      }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    asm volatile("" ::: "memory");
  }
}

// One output tile: its 64 kMT x 256 dW block over all M tokens.
template <bool kAcc, int kMT, bool kNt>
__global__ void __launch_bounds__(kWgThreads, 4 / kMT) wgrad_kernel(const WgradArgs g) {
  const int T = g.tiles_n * g.tiles_k;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int hn = wave >> 1, hk = wave & 1;  // the wave's halves of n and k
  __shared__ u32x4 lds[kWgStages][kWgStageUnits<kMT>];
  uint32_t rdy[kMT], rx[4];
#pragma unroll
  for (int j = 0; j < kMT; ++j) rdy[j] = wg_read_off<kWgDyUnits<kMT>>(lane, hn, j);
#pragma unroll
  for (int j = 0; j < 4; ++j) rx[j] = wg_read_off<32>(lane, hk, j);
  char *ldy[kWgStages], *lx[kWgStages];
#pragma unroll
  for (int i = 0; i < kWgStages; ++i) {
    ldy[i] = reinterpret_cast<char *>(&lds[i][0]);
    lx[i] = reinterpret_cast<char *>(&lds[i][kWgStep * kWgDyUnits<kMT>]);
  }
  // 16 KB of the ring for each wave's epilogue.
  floatx4 *lds_wave = reinterpret_cast<floatx4 *>(&lds[0][0]) + 1024 * wave;
  const int64_t nsteps = (g.M + kWgStep - 1) / kWgStep;
  const uint32_t step_x = (uint32_t)(kWgStep * g.K * 2);
#pragma unroll 1
  for (int b = blockIdx.x; b < T; b += gridDim.x) {
    int tn, tk;
    wg_map_tile(g, b, tn, tk);
    // The product that owns tile row tn.
    int gi = 0;
#pragma unroll
    for (int j = 1; j < kMaxWgGroups; ++j) gi += (j < g.ngroups && tn >= g.tile0[j]) ? 1 : 0;
    const uint16_t *dy = wg_pick(g.dy, gi);
    float *dw = wg_pick(g.dw, gi);
    const int64_t N = wg_pick(g.N, gi);
    int32_t t0 = g.tile0[0];
#pragma unroll
    for (int j = 1; j < kMaxWgGroups; ++j) t0 = (gi == j) ? g.tile0[j] : t0;
    const int64_t n0 = (int64_t)(tn - t0) * (64 * kMT), k0 = (int64_t)tk * kWgTile;
    const uint32_t step_dy = (uint32_t)(kWgStep * N * 2);
    // Buffer resources based at the tiles' first columns; num_records ends
    // at the matrix end, so token rows >= M (and the last row's columns past
    // the end) read as zero.  Columns past N or K of other rows read the next
    // row's values and only reach outputs that are never stored.
    const __amdgpu_buffer_rsrc_t rs_dy = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(dy + n0), 0, (int)(g.M * N * 2 - n0 * 2), kBufferFlags);
    const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(g.x + k0), 0, (int)(g.M * g.K * 2 - k0 * 2), kBufferFlags);
    // Lane offsets of this wave's DMAs for step 0: x instruction d writes rows
    // 8 wave + 2d + (lane / 32), physical unit lane % 32; of dy, whose rows are
    // kWgDyUnits long, each writes 64 / kWgDyUnits rows.
    uint32_t vdy[kMT], vx[4];
    constexpr int kDyRows = 64 / kWgDyUnits<kMT>;
#pragma unroll
    for (int d = 0; d < kMT; ++d) {
      const int r = 8 * wave + kDyRows * d + lane / kWgDyUnits<kMT>;
      const int u = wg_unit(r, lane % kWgDyUnits<kMT>);  // the logical unit stored there
      vdy[d] = (uint32_t)(r * N * 2 + 16 * u);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int r = 8 * wave + 2 * d + (lane >> 5);
      vx[d] = (uint32_t)(r * g.K * 2 + 16 * wg_unit(r, lane & 31));
    }
    // Prologue: steps 0 .. kWgStages-2 (those that exist) into their
    // stages, then wait for step 0.
#pragma unroll
    for (int p = 0; p < kWgStages - 1; ++p) {
      if (p < nsteps) {
#pragma unroll
        for (int d = 0; d < kMT; ++d) {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              rs_dy, (lds_void_t *)(ldy[p] + 1024 * (kMT * wave + d)), 16, (int)vdy[d], 0, 0, 0);
          vdy[d] += step_dy;
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              rs_x, (lds_void_t *)(lx[p] + 1024 * (4 * wave + d)), 16, (int)vx[d], 0, 0, 0);
          vx[d] += step_x;
        }
      }
    }
    wgrad_close_step<kMT>(-1, nsteps);

    floatx16 acc[kMT][4];
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[mt][nt][v] = 0.0f;
    u32x4 fd[2][kMT], fx[2][4];
#pragma unroll
    for (int i = 0; i < kMT; ++i) fd[1][i] = (u32x4){0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 4; ++i) fx[1][i] = (u32x4){0u, 0u, 0u, 0u};
    // Step t computes from stage t % kWgStages and loads step
    // t + kWgStages - 1 into the stage before it.
    int64_t t = 0;
#pragma unroll 1
    for (; t + kWgStages <= nsteps; t += kWgStages) {
      static_for<0, kWgStages>([&](auto I) {
        constexpr int i = decltype(I)::value;
        constexpr int c = i, nx = (i + kWgStages - 1) % kWgStages;
        wgrad_step<kMT>(acc, fd, fx, ldy[c], lx[c], ldy[nx], lx[nx], rdy, rx, rs_dy, rs_x, vdy, vx,
                        step_dy, step_x, t + i + kWgStages - 1 < nsteps, wave);
        wgrad_close_step<kMT>(t + i, nsteps);
      });
    }
    static_for<0, kWgStages - 1>([&](auto I) {
      constexpr int i = decltype(I)::value;
      constexpr int c = i, nx = (i + kWgStages - 1) % kWgStages;
      if (t + i < nsteps) {
        wgrad_step<kMT>(acc, fd, fx, ldy[c], lx[c], ldy[nx], lx[nx], rdy, rx, rs_dy, rs_x, vdy, vx,
                        step_dy, step_x, false, wave);
        wgrad_close_step<kMT>(t + i, nsteps);
      }
    });
    // The last step's final MFMAs.
#pragma unroll
    for (int i = 0; i < 2 * kMT; ++i) {
      const int mt = kMT / 2 + (i >> 2), nt = i & 3;
      acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, fx[1][nt]), __builtin_bit_cast(bf16x8, fd[1][mt]),
          acc[mt][nt], 0, 0, 0);
    }

    // Epilogue.  Lane l holds dW row n = n0 + 32 kMT hn + 32 mt + l % 32 and
    // columns k = k0 + 128 hk + 32 nt + 8 j + 4 (l / 32) + i in registers
    // 4 j + i of tile [mt][nt].
    const bool vec_ok = ((reinterpret_cast<uintptr_t>(dw) & 15) == 0) && ((g.K & 3) == 0);
    if (vec_ok && g.K < ((int64_t)1 << 22))  // 32-bit row offsets
      wg_store_lds<kAcc, kMT, kNt>(g, acc, lds_wave, dw, n0 + 32 * kMT * hn, k0 + 128 * hk, N,
                                   lane);
    else
      wg_store<kAcc, kMT>(g, acc, dw, n0 + 32 * kMT * hn, k0 + 128 * hk, N, lane, vec_ok);
    // The next tile's prologue DMAs overwrite the LDS that the last step and
    // the epilogues read: every wave's reads (not its stores) end before this.
    step_barrier<63>();
  }
}

__global__ void fill_zero_f32(float *__restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0.0f;
}

// dW rows per tile / 64: 4 (256-row tiles, one workgroup a CU) or 2 (128-row
// tiles, two workgroups a CU).  Two workgroups hide one's stores and first
// loads behind the other's products, and half tiles leave less of a last round
// idle; but each x fragment feeds half the products.  The costs below are in
// full rounds of 256-row tiles, fitted to 1214 calls (16 to 8192 tokens, 512 to
// 56000 rows, 1024 to 16384 columns, stored and accumulated, a tenth of a round
// to 27): the choice takes 0.3 % more time than the better of the two on
// average.
// One round of 128-row tiles (two a CU) takes 0.78 at 256 tokens and 0.055 more
// with each doubling, in a row of rounds 0.84 and 0.045 (8192 x 8192: 256
// tokens 57 us against 76, 1000 tokens 130 against 146, 2048 tokens 234 against
// 242, 4096 tokens 432 against 421, 8192 tokens 850 against 808); past the third
// the workgroups of a patch run out of step and share less, 0.06 a round
// (accumulated 35816 x 8840 over 2282 tokens, 19 rounds: 1853 us against 1504;
// stored 27928 x 9144 over 2219, 15 rounds: 1078 against 1003).  Once the
// operands come near the Infinity Cache's 256 MB, dy comes from memory in rows
// of 256 bytes: up to 1.3 times that (27176 x 2528 over 8000 tokens 1138 us
// against 977, 39848 x 7184 over 6783 tokens 1.45 times).
// A round that fills a share f of the chip is no full one, its workgroups run
// faster: 0.62 to 0.70 up to half the chip and in proportion beyond; with
// 128-row tiles 0.4 to 0.6, then 0.75 as soon as a CU has two (0.82 after whole
// rounds, whose ends are not in step).
// tiles4: 256-row tile rows of all products.  Called on sizes whose tile count
// fits 31 bits (a 128-row tiling that would not keeps the 256-row one).
static int wg_tile_mt(const int64_t *ns, int32_t count, int64_t m, int64_t k, int64_t tiles4,
                      int64_t tiles_k) {
  const int64_t cus = cu_slots();
  int64_t tiles2 = 0;
  for (int i = 0; i < count; ++i) tiles2 += (ns[i] + 127) / 128;
  if (tiles2 * tiles_k > 0x7fffffff) return 4;
  const int64_t t2 = tiles2 * tiles_k;
  double n = (double)k;
  for (int i = 0; i < count; ++i) n += (double)ns[i];
  const double doublings = std::log2((double)(m < 128 ? 128 : m)) - 8.0;
  const double past = (2e-6 * n * (double)m - 220.0) / 450.0;  // MB of dy and x
  const double far = past < 0.0 ? 1.0 : (past > 0.3 ? 1.3 : 1.0 + past);
  const int64_t t4 = tiles4 * tiles_k;
  const double f2 = (double)(t2 % (2 * cus)) / (double)(2 * cus);
  const double f4 = (double)(t4 % cus) / (double)cus;
  const double two = t2 < 2 * cus ? 0.50 : 0.57;
  const double part2 = f2 == 0.0 ? 0.0 : (f2 <= 0.5 ? 0.40 + 0.4 * f2 : two + 0.5 * f2);
  const double part4 = f4 == 0.0 ? 0.0 : (f4 <= 0.5 ? 0.62 + 0.16 * f4 : 0.40 + 0.6 * f4);
  const double whole = (double)(t2 / (2 * cus));
  const double late = whole > 3.0 ? 0.06 * (whole - 3.0) : 0.0;
  const double cost2 = far * ((0.84 + 0.045 * doublings) * whole + late +
                              (0.78 + 0.055 * doublings) * part2);
  const double cost4 = (double)(t4 / cus) + part4;
  return cost2 < cost4 ? 2 : 4;
}

// Whether dW (not accumulated) is stored non-temporally: 28672 x 8192 over 512
// tokens 319 us with, 367 without.  Rows that are no multiple of 128 bytes
// share their first and last cache lines with their neighbours, and only a
// cache merges the two parts.  So they keep the default policy while the stores
// set the time and dW (nearly) fits in the Infinity Cache of 256 MB (times with
// / without non-temporal stores, us):
//   16000 x 4104 (250 MiB), 16 tokens 69 / 45, 128 67 / 52, 1024 150 / 146,
//   3000 355 / 357, 4096 474 / 501;
//   24000 x 4104 (376 MiB), 128 tokens 97 / 89, 256 101 / 110, 1024 219 / 241.
// A larger dW of very few tokens keeps it too, unless whole 64-byte halves of
// the lines are written (28672 x 5000, 128 tokens 166 / 145; 28672 x 8208, a
// multiple of 16, 171 / 203).
constexpr int64_t kWgFewTokens = 160;
static bool wg_nontemporal(const int64_t *ns, int32_t count, int64_t m, int64_t k) {
  if (k % 32 == 0 || m > 3072) return true;
  int64_t bytes = 0;
  for (int i = 0; i < count; ++i) bytes += 4 * ns[i] * k;
  return bytes > ((int64_t)288 << 20) && (k % 16 == 0 || m > kWgFewTokens);
}

static int32_t wgrad_grouped(const uint16_t *const *dys, const int64_t *ns, float *const *dws,
                             int32_t count, const uint16_t *x, int64_t m, int64_t k,
                             int32_t accumulate, hipStream_t s) {
  if (count < 1 || count > kMaxWgGroups)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "weight-gradient product count %d outside [1, %d]",
                count, kMaxWgGroups);
  if (dys == nullptr || ns == nullptr || dws == nullptr)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "dys, ns or dws is NULL");
  if (m < 0 || k <= 0)
    return fail(NF4S_ERR_INVALID_ARGUMENT, "bad weight-gradient shape m=%lld k=%lld",
                (long long)m, (long long)k);
  constexpr int64_t kMaxDim = (int64_t)1 << 39;  // tile counts below are 32-bit
  if (k > kMaxDim)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "weight-gradient k=%lld beyond 2^39", (long long)k);
  if (k % 8 != 0)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "weight gradient needs k %% 8 == 0, got k=%lld",
                (long long)k);
  if (m > 0 && x == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "x is NULL");
  if (m > 0 && !aligned(x, 16)) return fail(NF4S_ERR_MISALIGNED, "x must be 16-byte aligned");
  // Lane offsets are 32-bit and must stay below 2^31 for every row a step
  // addresses, including the rows past m of the last 32-token step (which
  // read as zero only while their offsets do not wrap onto real rows).
  // The comparisons divide instead of multiplying, so no caller size can
  // overflow them.
  const int64_t lim = ((int64_t)1 << 31) - 1;
  const int64_t rows = m / kWgStep * kWgStep + (m % kWgStep ? kWgStep : 0);
  if (rows > 0 && k > lim / 2 / rows)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE,
                "x larger than 2 GiB with m rounded up to 32 (m=%lld k=%lld)", (long long)m,
                (long long)k);
  WgradArgs g{};
  g.ngroups = count;
  g.x = x;
  g.M = m;
  g.K = k;
  g.tiles_k = (int32_t)((k + kWgTile - 1) / kWgTile);
  int64_t tiles_n = 0;
  for (int i = 0; i < count; ++i) {
    const int64_t n = ns[i];
    if (dws[i] == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "dw %d is NULL", i);
    if (m > 0 && dys[i] == nullptr) return fail(NF4S_ERR_INVALID_ARGUMENT, "dy %d is NULL", i);
    if (n <= 0)
      return fail(NF4S_ERR_INVALID_ARGUMENT, "bad weight-gradient shape m=%lld n=%lld k=%lld",
                  (long long)m, (long long)n, (long long)k);
    if (n > kMaxDim)
      return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "weight-gradient n=%lld beyond 2^39", (long long)n);
    if (n % 8 != 0)
      return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "weight gradient needs n %% 8 == 0 and k %% 8 == 0, "
                  "got n=%lld k=%lld", (long long)n, (long long)k);
    if (m > 0 && !aligned(dys[i], 16))
      return fail(NF4S_ERR_MISALIGNED, "dy and x must be 16-byte aligned");
    if (!aligned(dws[i], 4)) return fail(NF4S_ERR_MISALIGNED, "dw must be 4-byte aligned");
    int64_t nk;
    if (__builtin_mul_overflow(n, k, &nk))
      return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "dW of %lld x %lld elements overflows 64 bits",
                  (long long)n, (long long)k);
    if (rows > 0 && n > lim / 2 / rows)
      return fail(NF4S_ERR_UNSUPPORTED_SHAPE,
                  "dy or x larger than 2 GiB with m rounded up to 32 (m=%lld n=%lld k=%lld)",
                  (long long)m, (long long)n, (long long)k);
    g.dy[i] = dys[i];
    g.dw[i] = dws[i];
    g.N[i] = n;
    tiles_n += (n + 255) / 256;
    if (tiles_n > 0x7fffffff) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  }
  if (tiles_n * g.tiles_k > 0x7fffffff)
    return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  const int mt = wg_tile_mt(ns, count, m, k, tiles_n, g.tiles_k);
  tiles_n = 0;
  for (int i = 0; i < count; ++i) {
    g.tile0[i] = (int32_t)tiles_n;
    tiles_n += (ns[i] + 64 * mt - 1) / (64 * mt);
  }
  for (int i = count; i <= kMaxWgGroups; ++i) g.tile0[i] = (int32_t)tiles_n;
  g.tiles_n = (int32_t)tiles_n;
  const int64_t T = tiles_n * g.tiles_k;
  if (m == 0) {
    // An empty sum: dw += 0, or dw = 0 (a fill kernel rather than
    // hipMemsetAsync, so that a caller may capture the call in a HIP graph).
    // The main kernel's buffer bounds assume m > 0.
    if (accumulate) return NF4S_OK;
    for (int i = 0; i < count; ++i) {
      const int64_t cnt = ns[i] * k;
      const int64_t blocks = (cnt + 255) / 256;
      hipLaunchKernelGGL(fill_zero_f32, dim3((uint32_t)(blocks < 65536 ? blocks : 65536)),
                         dim3(256), 0, s, dws[i], cnt);
      const int32_t rc = check_launch("fill_zero_f32");
      if (rc != NF4S_OK) return rc;
    }
    return NF4S_OK;
  }
  const int64_t slots = (int64_t)cu_slots() * (4 / mt);
  const int64_t G = T < slots ? T : slots;
  // Strips of about 8 tile columns; the 64 slots of an XCD with 128-row tiles
  // read less per step from strips of about 4, which pays once the steps
  // outweigh the stores (28672 x 8192 over 256 tokens: 188 us with 8, 203 with
  // 4; 2 x 11008 x 4096 over 1000: 181 and 176, over 8192: 1289 and 1232).  All
  // of one width: a last strip of one column reads all of dy for it (56000 x
  // 1080 over 2841 tokens, 4 + 1 columns 446 us, 5 412).
  const int want = (mt == 2 && m > 512) ? 4 : 8;
  const int strips = g.tiles_k < want ? 1 : (g.tiles_k + want / 2) / want;
  g.strip = (g.tiles_k + strips - 1) / strips;
  // Stores of the default policy meet their neighbours' halves of a line in the
  // cache if whole rows of dW are under way at once: with so few tokens that
  // the operands hardly count, the strip is the whole width (16000 x 10808
  // over 81 tokens 181 -> 168 us, 32840 x 12072 439 -> 400).
  const bool nt = accumulate || wg_nontemporal(ns, count, m, k);
  if (!nt && m <= kWgFewTokens) g.strip = g.tiles_k;
  // XCD blocks (wg_map_tile) when every round is full: the squarest
  // blk_n x blk_k = G / 8 that divides the tile grid (the products' tile
  // rows stacked), if an XCD then reads no more per step than with strips (59
  // x 8 tiles only divide into 59 x 1, which reads all of dy on every XCD).
  if (G % 8 == 0 && T % G == 0 && (nt || m > kWgFewTokens)) {
    const int S = (int)(G / 8), w = g.strip < S ? g.strip : S;
    int best = mt * ((S + w - 1) / w) + 4 * w;  // columns read per XCD and step, in 64s
    for (int bn = 1; bn <= S; ++bn) {
      if (S % bn != 0 || g.tiles_n % bn != 0 || g.tiles_k % (S / bn) != 0) continue;
      const int bk = S / bn;
      const int cost = mt * bn + 4 * bk;
      if (cost < best || (cost == best && g.blk_n == 0)) {
        best = cost;
        g.blk_n = bn;
        g.blk_k = bk;
      }
    }
  }
  auto *kernel = mt == 4 ? wgrad_kernel<true, 4, true> : wgrad_kernel<true, 2, true>;
  if (!accumulate && nt)
    kernel = mt == 4 ? wgrad_kernel<false, 4, true> : wgrad_kernel<false, 2, true>;
  else if (!accumulate)
    kernel = mt == 4 ? wgrad_kernel<false, 4, false> : wgrad_kernel<false, 2, false>;
  hipLaunchKernelGGL(kernel, dim3((uint32_t)G), dim3(kWgThreads), 0, s, g);
  return check_launch("wgrad_kernel");
}

}  // namespace nf4s

using namespace nf4s;

extern "C" {

int32_t nf4s_gemm_wgrad(const void *dy, const void *x, int64_t m, int64_t n, int64_t k,
                        float *dw, int32_t accumulate, void *stream) {
  clear_error();
  const uint16_t *dys[1] = {static_cast<const uint16_t *>(dy)};
  float *dws[1] = {dw};
  return wgrad_grouped(dys, &n, dws, 1, static_cast<const uint16_t *>(x), m, k, accumulate,
                       as_stream(stream));
}

int32_t nf4s_gemm_wgrad_grouped(const void *const *dys, const int64_t *ns, float *const *dws,
                                int32_t count, const void *x, int64_t m, int64_t k,
                                int32_t accumulate, void *stream) {
  clear_error();
  return wgrad_grouped(reinterpret_cast<const uint16_t *const *>(dys), ns, dws, count,
                       static_cast<const uint16_t *>(x), m, k, accumulate, as_stream(stream));
}

}  // extern "C"
