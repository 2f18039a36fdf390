// GEMM launch planner for MI355X: (m, n, k) → tile variant + split-K, for every
// epilogue alike.
// decide's counterpart is gemm_configs::plan / recommend
// (crates/decide-metal/src/gemm_configs.rs:290-314), a table measured on an
// M1 Pro. This one is a table measured on an MI355X for decide's engine
// shapes, with a calibrated cost model (rounds of 256 workgroups, per-stage
// time per tile height, HBM floor, split-K reduction) for every other shape.
// Pure host code: no device needed.
#pragma once

#include <stdint.h>

namespace dh {

struct Plan {
  int variant;
  uint32_t splits;
  uint32_t kps;       // K per split (multiple of 64)
  uint32_t mtiles, stripes;
  uint32_t grid;      // workgroups of the tile kernel
  uint64_t ws_bytes;  // split-K workspace
  double est_us;      // model estimate
};

// Plan.variant of the small-M weight-streaming kernel (gemm_stream.hip): 32
// output columns per workgroup, M <= 16, K a multiple of 128.
constexpr int kStreamVariant = 64;  // DH_GEMM_STREAM_VARIANT
constexpr uint32_t kStreamMaxM = 16;
// Widest N (summed over a grouped launch's members) the streaming kernel takes, where the table has no choice of its
// own. Against the best split of the 32 x 96 tile, weights from HBM, 1 to 16 rows: k|v (2560 -> 2048) 9.2-10.6 us
// streaming, 9.5-10.1 tiled, so it streams; out (4096 -> 2560) 12.0-12.9 against 10.7-11.4 and down (9216 -> 2560)
// 15.7-17.5 against 14.9-15.3, so the table's tiles take them. Of other shapes, N = 1024 to 4096 at 3 and 12 rows, the
// best split of that tile is level to 25 % ahead, but the cost model does not find it (1024 -> 1024 at 17 rows: eight
// splits, 9.1 us; streaming at 12 rows 7.8; best split 6.4), so they stream. Wider N (q|gate, gate|up) streams slower.
constexpr uint32_t kStreamMaxN = 4096;

// Model estimate for one (variant, splits) choice; +inf if the choice is not
// valid for the shape.
double plan_estimate_us(int variant, uint32_t splits, uint32_t m, uint32_t n, uint32_t k);
// Builds the plan for (variant, splits), filling the derived fields.
Plan plan_make(int variant, uint32_t splits, uint32_t m, uint32_t n, uint32_t k);
// The weight-streaming kernel's plan (M <= kStreamMaxM, K % 128 == 0, N % 32 == 0).
Plan plan_stream(uint32_t m, uint32_t n, uint32_t k, uint64_t max_ws);
// Best plan for a single GEMM. `max_ws` caps the split-K workspace bytes.
Plan plan_gemm(uint32_t m, uint32_t n, uint32_t k, uint64_t max_ws);
// The largest split-K workspace plan_gemm asks for over every M in 1..max_m at
// (n, k): the workspace a caller must hold so that no call of
// up to max_m rows grows it. The table switches split counts between measured
// rows, so the need is not monotone in M; this sweeps every M.
uint64_t plan_ws_need(uint32_t max_m, uint32_t n, uint32_t k, uint64_t max_ws);
// Best plan for a grouped launch of `count` members of widths ns[] that share
// X (no split-K). Each member rounds up to whole column stripes of its own.
Plan plan_grouped(uint32_t m, uint32_t k, const uint32_t* ns, uint32_t count);
// The tile kernels' work order for plan p (TileArgs::ngroup): the hardware
// deals workgroups to the 8 XCDs round-robin and xcd_remap gives each XCD a
// contiguous run of work ids, so the order decides which X row blocks and W
// column stripes share one XCD's L2. Returns the stripe-group width (0 = M
// tiles fastest) that minimises the bytes of distinct X and W tiles each XCD
// fetches per round of one workgroup per CU, over a few candidates.
// DH_GEMM_TILE_GROUP=<g> (0..64) in the environment fixes it (for measurements).
uint32_t plan_order(const Plan& p);

}  // namespace dh
