// nf4_skinny.hpp - the forward GEMM for few tokens (nf4_skinny.hip), as
// nf4_gemm.hip dispatches to it.
#pragma once

#include "abi_common.hpp"
#include "nf4_device.hpp"

namespace nf4s {

// Largest token count the few-token forward takes.
constexpr int64_t kSkinnyMaxM = 128;

constexpr int kSkinnyMaxGroups = 4;

// Whether the few-token forward takes these weights: one workgroup per tile
// of at least 32 rows, bounded so that a launch stays far below 2^32 threads
// (the tiled kernel, a fixed grid, takes taller weights).
inline bool skinny_takes(const int64_t *ns, int32_t count, int64_t m) {
  if (m > kSkinnyMaxM) return false;
  int64_t rows = 0;
  for (int32_t i = 0; i < count; ++i) {
    if (ns[i] > ((int64_t)1 << 26)) return false;
    rows += ns[i];
  }
  return rows <= ((int64_t)1 << 26);
}

struct SkinnyGroup {
  const uint8_t *packed;
  AbsmaxRef am;
  uint16_t *out;      // y_i [m, n] (SwiGLU: hidden, in group 0)
  int64_t n;          // rows of W_i
  int32_t tile0;      // first output tile of this weight in the launch
};

// One launch: y_i = x . W_i^T for up to 4 weights that share x [m, k], or
// hidden = silu(x . Wg^T) * (x . Wu^T).
struct SkinnyArgs {
  const uint16_t *x;
  int64_t m, k;
  SkinnyGroup grp[kSkinnyMaxGroups];
  int32_t ngroups;
  int32_t tiles;        // output tiles over all weights
  int32_t slices;       // K slices (workgroups per tile)
  int32_t slice_steps;  // 128-deep steps per slice
  float *ws;            // slices > 1: partials [slice][m][tiles * tile rows]
};

// Workspace bytes skinny_fwd uses for these shapes (0: no K slices).
int64_t skinny_workspace_bytes(const int64_t *ns, int32_t count, int64_t m, int64_t k);

// Runs the launch described by a (x, m, k, the groups' packed, am, out and
// n); the plan (tiles, slices) is filled in here: as many K slices as the
// workspace holds, none with a NULL one.  0 < m <= kSkinnyMaxM.
int32_t skinny_fwd(const SkinnyArgs &a, hipStream_t s, void *work, int64_t work_bytes);
int32_t skinny_swiglu(SkinnyArgs &a, hipStream_t s);

}  // namespace nf4s
