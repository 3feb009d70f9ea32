// gemm_wreg.hpp -- host interface of the grouped expert products whose
// weights go straight to registers (gemm_wreg.hip).
#pragma once

#include "common.hpp"
#include "dispatch.hpp"
#include "router.hpp"

namespace grim {

// Rows per tile of the routed rows (INT4 batches have at most two routes per
// expert on average).  The down product takes two activation planes, so half
// the rows fill its tile.
constexpr int wreg_mc(int fmt, bool gate_up) {
    return fmt == GRIM_FMT_INT4 || fmt == GRIM_FMT_INT4_F16 ? 16 : gate_up ? 128 : 64;
}

struct WregArgs {
    WView w, w_sh;             // routed experts, shared expert
    int N;                     // gate_up: I (row pairs); down: H (rows)
    int K;                     // reduction length: gate_up H, down I
    const uint16_t* A;         // bf16 rows [a_rows][planes][wreg_kpad]
    const uint16_t* A_sh;      // the shared expert's
    int64_t a_rows, a_rows_sh;
    const int32_t* a_lo;       // gate_up, two planes: per row of A, whether its lo plane is non-zero
    const int32_t* map;        // gate_up: route row -> row of A (the token); down: null
    uint16_t* h;               // gate_up out: bf16 pair rows [R][2][wreg_kpad(N)]
    uint16_t* h_sh;
    float* y;                  // down out: fp32 rows [R][N]
    float* y_sh;
    const TileDesc* tiles;     // row tiles of at most wreg_mc rows
    const int32_t* n_live;     // how many (device)
    int max_tiles;             // their bound, which the grid is sized for
    int T_sh;                  // shared-expert rows (0 = none)
};

// Whether a weight [.][K] of this format can take the path.
bool wreg_weight_ok(const grim_quant_weight& w, int rows_per_expert, int K);
// Reduction length padded to whole segments of the format.
int wreg_kpad(int fmt, int K);
// Activation planes of gate_up: INT4 experts split fp32 x in two bf16 halves
// (exact for 16 significant bits, within 2^-17 of x otherwise), the others
// round x to bf16.
int wreg_x_planes(int fmt);
// x fp32 [T][H] -> bf16 rows [T][planes][wreg_kpad] (+ per row lo != 0), and
// in the same launch the dispatch of the routes in tk.out_e (its first
// work-group) with the top-k before it when `topk` -- where
// wreg_one_dispatch / wreg_one_topk hold; otherwise d is null and both ran
// before.
bool wreg_one_dispatch(int T, int K, int E);
bool wreg_one_topk(int T);
hipError_t wreg_route_launch(hipStream_t st, int fmt, const float* x, int H, uint16_t* dst, int32_t* lo,
                             const TopkArgs& tk, const DispatchArgs* d, bool topk);
hipError_t wreg_launch(hipStream_t st, int fmt, const WregArgs& a, bool gate_up);

}  // namespace grim
