// Launchers shared between the router, decode and prefill translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mimo {

struct RouterSmallArgs {
  const uint16_t* x;       // [T, H] bf16
  const uint16_t* Wg;      // [E, H] bf16
  const float* bias;       // [E]
  int T, H, E, k, nlog;    // nlog = E logits blocks (set by the launcher)
  float* logits;           // [T, E]
  float* scores;           // [T, E] sigmoid (optional)
  float* keys;             // [T, E] sigmoid + bias (optional)
  // optional RMSNorm of the rows first (the post-attention norm of a decoder layer): the logits are then of
  // r = RMSNorm(x) * norm_w, and r itself goes to r_out when given (H a multiple of 256)
  const uint16_t* norm_w;  // [H] bf16
  float eps;
  uint16_t* r_out;         // [T, H] bf16 (optional)
};

int launch_router_logits_small(const RouterSmallArgs& a, hipStream_t st);   // logits, sigmoid, keys, normalised rows

struct SelectGroupArgs {
  const float *scores, *keys;   // [T, E]
  int T, E, k;
  const int32_t* slot_of;
  int R, n_slots, Umax;
  int32_t* inds_out;
  float* w_out;
  int32_t *uids, *urows, *ucnt;
  float* uw;
  uint32_t* gidx;
  int32_t *n_unique, *status;
};
// top-k + renormalisation per row and grouping by slot (one block; T <= 8, T*k <= 64, Umax*R <= 512)
int launch_select_group(const float* scores, const float* keys, int T, int E, int k, const int32_t* slot_of, int R,
                        int n_slots, int Umax, int32_t* inds_out, float* w_out, int32_t* uids, int32_t* urows,
                        int32_t* ucnt, float* uw, uint32_t* gidx, int32_t* n_unique, int32_t* status,
                        hipStream_t st);
// zero_status (optional): a status word the launch clears (its first block), for the kernels queued after it
int launch_router_logits(const uint16_t* x, const uint16_t* W, int T, int H, int E, float* logits, hipStream_t st,
                         int32_t* zero_status = nullptr);
int launch_router_select(const float* logits, const float* bias, int T, int E, int k, float scaling, int32_t* inds,
                         float* w, const int32_t* slot_of, int32_t* slot_inds, int n_slots, int32_t* status,
                         hipStream_t st, bool parts = false);
// Logits of a chunk of at most kRlPartsMax tokens as kRlParts partial sums [kRlParts, T, E], which
// launch_router_select(parts) adds; router_logits_parts: whether the inputs allow it.
// Beyond, the blocks of whole reductions fill the chip: 512 tokens 14.8 us in parts, 25.5 whole; 640 20.0 and 25.3, 768
// 20.7 and 25.6, 1024 26.8 and 25.6, and the selection takes 0.5 to 1.4 us more to add the parts.
constexpr int kRlPartsMax = 640, kRlParts = 8;
bool router_logits_parts(const uint16_t* x, const uint16_t* W, int T, int H);
int launch_router_logits_parts(const uint16_t* x, const uint16_t* W, int T, int H, int E, float* part, hipStream_t st,
                               int32_t* zero_status);
// Row tiles of the grouped GEMM: a slot with 1..narrow_max routes is one narrow tile; a larger one is cut into wide
// tiles of wide_rows routes and one of the remainder.
// tiles[0] = (wide count, narrow count, 0, 0), wide tile t at tiles[kTileHead + t], narrow tile t at
// tiles[kTileHead + wcap + t], each (slot, first route, end route, 0).  tiles[1 + x] cuts the wide tiles into eight
// shares of equal cost, a tile costing kTileCost plus its chunks of 16 routes: share x starts off / (8 cost) of the way
// through tile t, for (t, off, cost, 0) (not written without wide tiles).
constexpr int kTileHead = 9, kTileCost = 2;
struct TileSpec {
  int narrow_max, wide_rows, wcap;
};
int launch_dispatch(const int32_t* slots, int n, int n_slots, int32_t* hist, int32_t* perm, int32_t* offsets,
                    int32_t* inv, const TileSpec* spec, int4* tiles, int32_t* status, bool zero_status, hipStream_t st);
size_t dispatch_workspace(int n, int n_slots);

}  // namespace mimo
