// Launch side of the mid tiles (gemm_mid.h): the kernel of each tile shape and mode that MID_SHAPES lists, instantiated
// once per output dtype in gemm_mid_bf16.hip and gemm_mid_f16.hip.
#pragma once
#include "gemm_launch.h"
#include "gemm_mid.h"

namespace wq8 {

template <int BM, int BN, int STAGES, int MODE, bool WG, int DT, bool SEG>
static int launch_mid(GemmArgs& g, int pieces, hipStream_t stream) {
    g.tiles_m = (g.m + BM - 1) / BM;
    g.tiles_n = (g.n + BN - 1) / BN;
    g.n_first = g.dp_tiles = 0;
    g.pieces = pieces;
    g.defer = pieces > 1;
    gemm_mid<BM, BN, 4, 2, STAGES, MODE, WG, DT, SEG><<<g.tiles_m * g.tiles_n * pieces, 512, 0, stream>>>(g);
    if (const int rc = int(hipGetLastError())) return rc;
    return pieces > 1 ? launch_finish<DT, MODE, WG>(g, stream) : 0;
}

// STAGES: as many as the LDS holds, at most 5 (with hi and lo rows a stage holds twice the tokens)
template <int MODE, bool WG, int DT, bool SEG>
static int launch_mid_shape(GemmArgs& g, const MidShape& shape, int pieces, hipStream_t stream) {
    constexpr bool HILO = MODE == MODE_EXACT;
    auto is = [&](int bm, int bn) { return shape.bm == bm && shape.bn == bn; };
    if (is(64, 64)) return launch_mid<64, 64, 5, MODE, WG, DT, SEG>(g, pieces, stream);
    if (is(128, 128)) return launch_mid<128, 128, HILO ? 3 : 4, MODE, WG, DT, SEG>(g, pieces, stream);
    if constexpr (!SEG) {
        if (is(64, 32)) return launch_mid<64, 32, 5, MODE, WG, DT, SEG>(g, pieces, stream);
        if (is(128, 64)) return launch_mid<128, 64, HILO ? 3 : 5, MODE, WG, DT, SEG>(g, pieces, stream);
        if constexpr (HILO) {
            if (is(64, 128)) return launch_mid<64, 128, 4, MODE, WG, DT, SEG>(g, pieces, stream);
        } else {
            if (is(128, 160)) return launch_mid<128, 160, 3, MODE, WG, DT, SEG>(g, pieces, stream);
            if (is(128, 192)) return launch_mid<128, 192, 3, MODE, WG, DT, SEG>(g, pieces, stream);
            if constexpr (!WG)
                if (is(256, 128)) return launch_mid<256, 128, 3, MODE, WG, DT, SEG>(g, pieces, stream);
        }
    }
    return -3;
}

template <int DT>
int dispatch_mid(GemmArgs& g, const Variant& v, int split, hipStream_t stream) {
    const MidPlan plan = mid_plan(g, v, split);
    if (plan.shape < 0) return -3;
    const MidShape& shape = MID_SHAPES[plan.shape];
    if (g.seg_rows) {
        if (v.wgroup) return -4;
        if (v.mode == MODE_ROW) return launch_mid_shape<MODE_ROW, false, DT, true>(g, shape, 1, stream);
        if (v.mode == MODE_EXACT) return launch_mid_shape<MODE_EXACT, false, DT, true>(g, shape, 1, stream);
        return launch_mid_shape<MODE_BLOCK, false, DT, true>(g, shape, 1, stream);
    }
    if (v.mode == MODE_ROW) return launch_mid_shape<MODE_ROW, false, DT, false>(g, shape, plan.pieces, stream);
    if (v.mode == MODE_EXACT && !v.wgroup) return launch_mid_shape<MODE_EXACT, false, DT, false>(g, shape, plan.pieces, stream);
    if (v.mode == MODE_EXACT) return launch_mid_shape<MODE_EXACT, true, DT, false>(g, shape, plan.pieces, stream);
    if (v.wgroup) return launch_mid_shape<MODE_BLOCK, true, DT, false>(g, shape, plan.pieces, stream);
    return launch_mid_shape<MODE_BLOCK, false, DT, false>(g, shape, plan.pieces, stream);
}

}  // namespace wq8
