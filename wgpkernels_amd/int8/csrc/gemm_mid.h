// INT8 GEMM mainloop for launches of about one tile per CU (tens of tokens to about a thousand at the Wan widths), every
// mode.
//
// What bounds such a launch: the bytes each CU copies into LDS. Its weights come from HBM or the Infinity Cache and its
// token rows are new to the XCD's L2 on every k-tile, and a CU takes in lines that miss the L2 at about 45 B/ns (32 KiB of
// them in flight, 0.7 us each) against 110-147 B/ns for lines that hit (copies alone, 128-byte pieces of rows, 80-256
// CUs). gemm_pingpong's 256-token tiles waste half of that on padding at these sizes, give a copy half a k-tile to land,
// and wait for a launch that transposes the scales. Here:
// - tiles of 64-256 tokens x 32-192 channels, chosen (gemm_launch.h, mid_plan) so that the launch fills the CUs over the
//   whole of K or a few pieces of it;
// - the ring is 3-5 stages deep and a copy has STAGES - 1 k-tiles to land;
// - the fragments of k-tile kt + 1 are read from LDS into a second set of registers between the MFMAs of k-tile kt: a
//   stage is free for its next copy as soon as its fragments are read, with one barrier per k-tile;
// - block scales are read as the quantizer stores them (row-major, four k-blocks of a row at a time).
// Measured (bare GEMM, weights from HBM, against the best of the other tiles with their scale transpose): block K = 5120,
// N = 13824: M = 64 31.4 -> 22.3 us, M = 256 45.6 -> 35.4; K = 13824, N = 5120: M = 64 32.0 -> 23.0, M = 256 48.0 -> 38.0;
// block+g K = 3072, N = 12288, M = 333: 46.5 -> 31.6. With the copies left out the same loops run 24-48% faster, with the
// MFMAs left out no faster: the copies set the time. Four waves that only copy beside four that only compute measured the
// same.
//
// LDS layout and swizzle of the operand rows as in gemm_pingpong.h; the arithmetic and the order of every element's sums
// are the other kernels' (block: the biased single-FMA fold; block+g: the reference's order), except exact+g, whose
// combined block sums are scaled by sb and the result by 1 / 254 (the other kernel takes sb / 254 from a launch of its
// own).
#pragma once
#include "gemm_ring.h"

namespace wq8 {

// The work of a workgroup: consecutive workgroups go round robin over the 8 XCDs, each XCD taking a contiguous range of
// (piece, tile) with the tiles of a piece next to each other, so that an XCD reads one K range of the activations and
// neighbouring weight panels.
WQ8_DEVICE Work mid_work(const GemmArgs& g) {
    const int tiles = g.tiles_m * g.tiles_n, total = tiles * g.pieces, b = blockIdx.x;
    const int q = total / 8, r = total % 8, xcd = b % 8, idx = b / 8;
    const int v = xcd * q + (xcd < r ? xcd : r) + idx;
    Work w{0, 0, 0, g.kblocks, -1, 0};
    w.piece = v / tiles;
    const int t = v - w.piece * tiles;
    w.tn = t / g.tiles_m;
    w.tm = t - w.tn * g.tiles_m;
    w.kb0 = w.piece * g.kblocks / g.pieces;
    w.kb1 = (w.piece + 1) * g.kblocks / g.pieces;
    w.tm = __builtin_amdgcn_readfirstlane(w.tm);
    w.tn = __builtin_amdgcn_readfirstlane(w.tn);
    w.kb0 = __builtin_amdgcn_readfirstlane(w.kb0);
    w.kb1 = __builtin_amdgcn_readfirstlane(w.kb1);
    w.piece = __builtin_amdgcn_readfirstlane(w.piece);
    return w;
}

// bdma4 with only the lanes of `mask` (a branch on the lane would split the mainloop into blocks scheduled apart). Every
// lane of the wave is active before and after.
WQ8_DEVICE void bdma4_lanes(sgpr4 rsrc, uint32_t voffset, void* dst, uint64_t mask) {
    asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tbuffer_load_dword %0, %1, 0 offen lds\n\ts_mov_b64 exec, -1"
                 :: "v"(voffset), "s"(rsrc), "s"(lds_addr(dst)), "s"(mask)
                 : "memory", "m0");
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int MODE, bool WG, int DT, bool SEG>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_mid(GemmArgs g) {
    static_assert(WAVES_N * WAVES_M == 8, "eight waves");
    static_assert(!(WG && SEG), "segments take per-channel scales");
    constexpr bool BLOCK = MODE == MODE_BLOCK, HILO = MODE == MODE_EXACT;
    constexpr bool BIAS_FOLD = BLOCK && !WG;
    constexpr bool FOLD = BLOCK || WG;  // FP32 accumulators, one fold per k-tile
    constexpr int WAVES = 8, BK = 128, MF = 16, KSTEPS = 2, EPT = 4;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, FM = WM / MF, FN = WN / MF, T = FN * FM;
    static_assert(WM % MF == 0 && WN % MF == 0 && FM >= 1 && FN >= 1, "wave tile");
    constexpr int AR = HILO ? 2 * BM : BM, ROWS = AR + BN;  // stage rows: tokens (hi, then lo), channels
    // 1 KiB copies (8 rows) per wave; where they do not divide evenly the last waves copy one group twice (branch free, and
    // the same count in every wave)
    constexpr int GROUPS = ROWS / 8, L = (GROUPS + WAVES - 1) / WAVES;
    static_assert(AR % 8 == 0 && BN % 8 == 0, "whole copies");
    constexpr int STAGE_BYTES = ROWS * BK;
    // scales: three slots of four k-blocks, [token or channel][k-block] (a wave copies SA_W tokens and SB_W channels a k-tile)
    constexpr int SA_W = BLOCK ? (BM / 4 + WAVES - 1) / WAVES : 0, SB_W = WG ? (BN / 4 + WAVES - 1) / WAVES : 0;
    static_assert(BM % 4 == 0 && BN % 4 == 0 && SA_W < 16 && SB_W < 16, "one scale copy per wave and k-tile");
    constexpr int SA_SLOT = BLOCK ? (BM * 3 / 4 + WAVES * SA_W) * 16 : 0, SB_SLOT = WG ? (BN * 3 / 4 + WAVES * SB_W) * 16 : 0;
    constexpr int SCALE_BYTES = 3 * (SA_SLOT + SB_SLOT);
    constexpr int COPIES = L + (BLOCK ? 1 : 0) + (WG ? 1 : 0);  // per wave and k-tile
    constexpr int EPI_BYTES = WAVES * epilogue_stage_bytes<WN, WM>();
    constexpr int RING_BYTES = STAGES * STAGE_BYTES > EPI_BYTES ? STAGES * STAGE_BYTES : EPI_BYTES;
    using Params = EpilogueParams<DT, MODE, WG, SEG, BM, BN>;
    static_assert(STAGES >= 3 && RING_BYTES + SCALE_BYTES + Params::BYTES <= 160 * 1024, "LDS");
    // scale chunks issued at k-tile kt are read from k-tile kt + 4 on; the wait there covers copies STAGES - 1 k-tiles old
    static_assert(STAGES <= 5, "scale chunks have landed when they are read");
    static_assert((STAGES - 1) * COPIES < 64, "vmcnt");
    __shared__ __attribute__((aligned(1024))) uint8_t ring[RING_BYTES];
    __shared__ __attribute__((aligned(16))) uint8_t scale_lds[SCALE_BYTES > 0 ? SCALE_BYTES : 16];
    __shared__ __attribute__((aligned(16))) uint8_t params_lds[Params::BYTES];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WAVES_N, wm = wave / WAVES_N;
    const int m = g.m, n = g.n, k = g.k, kblocks = g.kblocks;
    const Work w = mid_work(g);
    const int m0 = w.tm * BM, n0 = w.tn * BN;
    const long long in_shift = g.counter && (g.in_first || g.in_step) ? g.in_first + __ldg(g.counter) * g.in_step : 0;
    const float* sa = g.sa + in_shift * (BLOCK ? kblocks : 1);
    // the epilogue's parameters: their loads go first, and stay in registers until the mainloop is done
    Params params;
    params.load(g, m0, n0, sa, tid);

    // ---- DMA: wave w copies the 8-row groups w + 8 j of a stage; lane l fills physical chunk l % 8 of row l / 8
    constexpr uint32_t OUT_OF_RANGE = 0x80000000u;
    const int kbase = w.kb0, k_tiles = w.kb1 - w.kb0;
    const int lr = lane >> 3;
    const uint32_t chunk = uint32_t((lane & 7) ^ ((4 * wave + (lr >> 1)) & 7)) * 16u;
    const uint32_t lane_part = uint32_t(lr) * uint32_t(k) + chunk;
    const int k_lim = k - int(chunk) - kbase * BK;  // this lane's chunk of k-tile kt lies inside the row when kt * BK < k_lim
    const sgpr4 rs_a = buffer_rsrc(g.a + in_shift * k, uint32_t(m) * uint32_t(k));
    const sgpr4 rs_lo = HILO ? buffer_rsrc(g.a_lo + in_shift * k, uint32_t(m) * uint32_t(k)) : rs_a;
    auto group_of = [&](int j) { return wave + WAVES * j < GROUPS ? wave + WAVES * j : wave + WAVES * (j - 1); };
    sgpr4 rs_row[L];
    uint32_t base_row[L];
#pragma unroll
    for (int j = 0; j < L; ++j) {
        const int r0 = group_of(j) * 8;
        if (r0 < AR) {
            rs_row[j] = HILO && r0 >= BM ? rs_lo : rs_a;
            base_row[j] = uint32_t(m0 + (r0 < BM ? r0 : r0 - BM)) * uint32_t(k);
        } else {
            const int c0 = n0 + (r0 - AR);
            if constexpr (SEG) {
                const int count = n / g.seg_rows;
                int s = c0 / g.seg_rows;
                s = s < count ? s : count - 1;
                rs_row[j] = buffer_rsrc(g.seg_b[s], uint32_t(g.seg_rows) * uint32_t(k));
                base_row[j] = uint32_t(c0 - s * g.seg_rows) * uint32_t(k);
            } else {
                rs_row[j] = buffer_rsrc(g.b, uint32_t(n) * uint32_t(k));
                base_row[j] = uint32_t(c0) * uint32_t(k);
            }
        }
        base_row[j] += uint32_t(kbase) * 128u;
    }
    // copy j of k-tile kt (into stage `st` bytes from the ring's start); past the last k-tile: zeros, no memory traffic
    auto copy_rows = [&](int kt, int j, int st) {
        const uint32_t kk = uint32_t(kt) * uint32_t(BK);
        const int lim = kt < k_tiles ? k_lim : 0;
        const uint32_t off = lane_part + (base_row[j] + kk);
        bdma16(rs_row[j], int(kk) < lim ? off : OUT_OF_RANGE, ring + st + group_of(j) * 1024);
    };
    // scales: chunk kt % 4 (a quarter of the tokens / channels) of the four k-blocks 4 (kt / 4) .. + 3, into slot (kt / 4) % 3.
    // k-blocks past the piece and rows past M / N read zeros.
    const sgpr4 rs_s = buffer_rsrc(sa, BLOCK ? uint32_t(m) * uint32_t(kblocks) * 4u : 0u);
    const sgpr4 rs_c = buffer_rsrc(g.sb, WG ? uint32_t(n) * uint32_t(kblocks) * 4u : 0u);
    auto copy_scales = [&](int kt, bool channels) {
        const int per = channels ? SB_W : SA_W, part = (channels ? BN : BM) / 4;
        const int quad = kt >> 2, kb = 4 * quad + (lane & 3), local = (kt & 3) * part + wave * per, row = local + (lane >> 2);
        const int grow = (channels ? n0 : m0) + row;
        const bool in = bool(int(kb < k_tiles) & int(grow < (channels ? n : m)));
        const uint32_t off = in ? (uint32_t(grow) * uint32_t(kblocks) + uint32_t(kbase + kb)) * 4u : OUT_OF_RANGE;
        uint8_t* dst = scale_lds + (channels ? 3 * SA_SLOT + (quad % 3) * SB_SLOT : (quad % 3) * SA_SLOT) + local * 16;
        bdma4_lanes(channels ? rs_c : rs_s, off, dst, (1ull << (4 * per)) - 1);
    };
    // copy number p of the COPIES of an iteration: operand rows of k-tile kt, then the scale chunks two quads ahead
    auto issue = [&](int kt, int scale_kt, int st, int p) {
        if (p < L) copy_rows(kt, p, st);
        else if (BLOCK && p == L) copy_scales(scale_kt, false);
        else if (WG && p == L + (BLOCK ? 1 : 0)) copy_scales(scale_kt, true);
    };

    // ---- fragments (two sets), accumulators
    const int frag_row = lane & 15;
    uint32_t off_a[KSTEPS], off_b[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        const uint32_t swz = uint32_t((4 * ks + (lane >> 4)) ^ ((frag_row >> 1) & 7)) << 4;
        off_a[ks] = uint32_t((wm * WM + frag_row) * BK) + swz;
        off_b[ks] = uint32_t((AR + wn * WN + frag_row) * BK) + swz;
    }
    v4i af[2][FM][KSTEPS], bf[2][FN][KSTEPS], lf[2][HILO ? FM : 1][KSTEPS];
    float s_tok[2][FM], s_ch[2][WG ? FN : 1][4];
    v4i acc[FOLD ? 1 : FN][FOLD ? 1 : FM], acc_lo[HILO && !FOLD ? FN : 1][HILO && !FOLD ? FM : 1];
    v4f accf[FOLD ? FN : 1][FOLD ? FM : 1];
    float corr[FM];
    v4i start = {};
    if constexpr (BIAS_FOLD) {
#pragma unroll
        for (int x = 0; x < EPT; ++x) start[x] = FOLD_BIAS_BITS;
    }
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
            if constexpr (FOLD) accf[i][j] = v4f{};
            else acc[i][j] = v4i{};
            if constexpr (HILO && !FOLD) acc_lo[i][j] = v4i{};
        }
#pragma unroll
    for (int j = 0; j < FM; ++j) corr[j] = 0.0f;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int j = 0; j < FM; ++j) s_tok[b][j] = 0.0f;
#pragma unroll
        for (int i = 0; i < (WG ? FN : 1); ++i)
#pragma unroll
            for (int x = 0; x < 4; ++x) s_ch[b][i][x] = 0.0f;
    }
    // read number r of the fragments of the k-tile in stage `st` into set B: channel fragments, token fragments (hi, lo)
    constexpr int RD = KSTEPS * (FN + FM * (HILO ? 2 : 1));
    auto read = [&](auto set, int st, int r) {
        constexpr int B = decltype(set)::value;
        const uint8_t* s = ring + st;
        const int ks = r / (RD / KSTEPS), q = r % (RD / KSTEPS);
        if (q < FM) af[B][q][ks] = *reinterpret_cast<const v4i*>(s + off_a[ks] + q * MF * BK);
        else if (HILO && q < 2 * FM) lf[B][HILO ? q - FM : 0][ks] = *reinterpret_cast<const v4i*>(s + off_a[ks] + BM * BK + (q - FM) * MF * BK);
        else {
            const int i = q - FM * (HILO ? 2 : 1);
            bf[B][i][ks] = *reinterpret_cast<const v4i*>(s + off_b[ks] + i * MF * BK);
        }
    };
    auto read_scales = [&](auto set, int kt) {
        constexpr int B = decltype(set)::value;
        if constexpr (BLOCK) {
            const float* s = reinterpret_cast<const float*>(scale_lds + ((kt >> 2) % 3) * SA_SLOT) + (wm * WM + frag_row) * 4 + (kt & 3);
#pragma unroll
            for (int j = 0; j < FM; ++j) s_tok[B][j] = s[j * MF * 4];
        }
        if constexpr (WG) {
            const float* s = reinterpret_cast<const float*>(scale_lds + 3 * SA_SLOT + ((kt >> 2) % 3) * SB_SLOT) + (wn * WN + 4 * (lane >> 4)) * 4 + (kt & 3);
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int x = 0; x < 4; ++x) s_ch[B][i][x] = s[(i * MF + x) * 4];
        }
    };
    auto fold = [&](auto set, int i, int j, const v4i& sum, const v4i& sum_lo) {
        constexpr int B = decltype(set)::value;
        if constexpr (BIAS_FOLD) {
            const v4f bits = __builtin_bit_cast(v4f, sum);
#pragma unroll
            for (int x = 0; x < EPT; ++x) accf[i][j][x] = __builtin_fmaf(bits[x], s_tok[B][j], accf[i][j][x]);
        } else if constexpr (BLOCK) {
#pragma unroll
            for (int x = 0; x < EPT; ++x) accf[i][j][x] = __builtin_fmaf(float(sum[x]), s_tok[B][j] * s_ch[B][WG ? i : 0][x], accf[i][j][x]);
        } else {
            // hi and lo block sums combined exactly in INT32 (|hi| <= 128 * 127^2 < 2^23)
#pragma unroll
            for (int x = 0; x < EPT; ++x)
                accf[i][j][x] = __builtin_fmaf(float(__mul24(sum[x], 254) + sum_lo[x]), s_ch[B][WG ? i : 0][x], accf[i][j][x]);
        }
    };

    // a tile's block sums fold LAG tiles behind its chain; the last LAG tiles of a k-tile fold in the next one
    constexpr int LAG = T > 2 ? 2 : 1;
    constexpr int TR = T - T / 4;
    v4i prev[LAG], prev_lo[LAG];
#pragma unroll
    for (int l = 0; l < LAG; ++l) prev[l] = start, prev_lo[l] = v4i{};

    // k-tile kt, whose fragments are in set C: its MFMAs with the copies of k-tile kt + STAGES (stage `st`, which it frees)
    // and the fragment reads of k-tile kt + 1 (stage `st_next`) spread between them
    auto step = [&](auto set, int kt, int st, int st_next) {
        constexpr int C = decltype(set)::value;
        using Cur = IntC<C>;
        using Other = IntC<1 - C>;
        wait_vmcnt<(STAGES - 2) * COPIES>();
        wait_lgkm0();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (BIAS_FOLD) {
#pragma unroll
            for (int j = 0; j < FM; ++j) corr[j] = __builtin_fmaf(FOLD_BIAS, s_tok[C][j], corr[j]);
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int i = t / FM, j = t % FM;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = t * COPIES / T; p < (t + 1) * COPIES / T; ++p) issue(kt + STAGES, kt + 8, st, p);
            // (the reads end before the last tiles, so that the next step does not wait for them)
            const int r0 = t * RD / TR < RD ? t * RD / TR : RD, r1 = (t + 1) * RD / TR < RD ? (t + 1) * RD / TR : RD;
            if constexpr (FOLD) {
                v4i c = start, c_lo = v4i{};
                c = MfmaI8<MF>::run(bf[C][i][0], af[C][j][0], c);
                if constexpr (HILO) c_lo = MfmaI8<MF>::run(bf[C][i][0], lf[C][j][0], c_lo);
#pragma unroll
                for (int r = r0; r < r1; ++r) read(Other{}, st_next, r);
                c = MfmaI8<MF>::run(bf[C][i][1], af[C][j][1], c);
                if constexpr (HILO) c_lo = MfmaI8<MF>::run(bf[C][i][1], lf[C][j][1], c_lo);
                if (t >= LAG) fold(Cur{}, (t - LAG) / FM, (t - LAG) % FM, prev[LAG - 1], prev_lo[LAG - 1]);
                else fold(Other{}, (T + t - LAG) / FM, (T + t - LAG) % FM, prev[LAG - 1], prev_lo[LAG - 1]);
#pragma unroll
                for (int l = LAG - 1; l > 0; --l) prev[l] = prev[l - 1], prev_lo[l] = prev_lo[l - 1];
                prev[0] = c;
                prev_lo[0] = c_lo;
                // the other set's scales belong to k-tile kt - 1 until its last tiles have folded
                if (t == LAG - 1) read_scales(Other{}, kt + 1);
            } else {
                acc[i][j] = MfmaI8<MF>::run(bf[C][i][0], af[C][j][0], acc[i][j]);
                if constexpr (HILO) acc_lo[i][j] = MfmaI8<MF>::run(bf[C][i][0], lf[C][j][0], acc_lo[i][j]);
#pragma unroll
                for (int r = r0; r < r1; ++r) read(Other{}, st_next, r);
                acc[i][j] = MfmaI8<MF>::run(bf[C][i][1], af[C][j][1], acc[i][j]);
                if constexpr (HILO) acc_lo[i][j] = MfmaI8<MF>::run(bf[C][i][1], lf[C][j][1], acc_lo[i][j]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- prologue: k-tiles 0 .. STAGES - 1 and, behind k-tile 0's rows, the first two scale slots; each k-tile with as
    // many copies as an iteration of the loop issues (the last scale chunk again), so that the waits count the same from
    // the start
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
#pragma unroll
        for (int p = 0; p < COPIES; ++p) issue(s, 7, s * STAGE_BYTES, p);
        if constexpr (BLOCK || WG) {
            if (s == 0) {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    if constexpr (BLOCK) copy_scales(c, false);
                    if constexpr (WG) copy_scales(c, true);
                }
            }
        }
    }
    // k-tile 0 and the scales landed: the STAGES - 1 later k-tiles' copies stay in flight
    wait_vmcnt<(STAGES - 1) * COPIES>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < RD; ++r) read(IntC<0>{}, 0, r);
    read_scales(IntC<0>{}, 0);
    int st = 0;
    auto next = [](int s) { return s + STAGE_BYTES == STAGES * STAGE_BYTES ? 0 : s + STAGE_BYTES; };
    int kt = 0;
    for (; kt + 1 < k_tiles; kt += 2) {
        int nx = next(st);
        step(IntC<0>{}, kt, st, nx);
        st = nx;
        nx = next(st);
        step(IntC<1>{}, kt + 1, st, nx);
        st = nx;
    }
    const bool odd = kt < k_tiles;
    if (odd) step(IntC<0>{}, kt, st, next(st));
    if constexpr (FOLD) {
#pragma unroll
        for (int l = LAG - 1; l >= 0; --l) {
            const int t = T - 1 - l;
            if (odd) fold(IntC<0>{}, t / FM, t % FM, prev[l], prev_lo[l]);
            else fold(IntC<1>{}, t / FM, t % FM, prev[l], prev_lo[l]);
        }
    }
    params.park(params_lds, tid);
    wait_vmcnt<0>();  // no copy in flight (the zero-filled ones past the last k-tile included)
    __syncthreads();  // every wave is done with the ring
    auto value = [&](int i, int j, int x) -> float {
        if constexpr (BIAS_FOLD) return accf[i][j][x] - corr[j];
        else if constexpr (BLOCK) return accf[i][j][x];
        else if constexpr (WG) return accf[i][j][x] * (1.0f / 254.0f);
        else if constexpr (HILO) return __builtin_fmaf(float(acc_lo[i][j][x]), 1.0f / 254.0f, float(acc[i][j][x]));
        else return float(acc[i][j][x]);
    };
    if constexpr (!SEG) {
        if (g.pieces > 1) {
            defer_store<FN, FM, WN, WM, MF, HILO && !FOLD ? 2 : 1>(g, m0, n0, wn, wm, w.piece, [&](int i, int j, int x, int h) -> uint32_t {
                if constexpr (FOLD) return __builtin_bit_cast(uint32_t, value(i, j, x));
                else if constexpr (HILO) return uint32_t(h == 0 ? acc[i][j][x] : acc_lo[i][j][x]);
                else return uint32_t(acc[i][j][x]);
            });
            return;
        }
    }
    uint8_t* stage = ring + wave * epilogue_stage_bytes<WN, WM>();
    gemm_epilogue<DT, MODE, WG, SEG, BM, BN, FN, FM, WN, WM, MF>(g, m0, n0, wn, wm, params_lds, stage, value);
}

}  // namespace wq8
