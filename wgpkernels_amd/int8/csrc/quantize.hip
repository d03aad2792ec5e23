// Activation preparation on gfx950: per-block INT8 (block path), per-row INT8 with an optional hi/lo split
// (row / exact paths), and the unquantized few-token prologue (transform_rows, rotate_groups).
//
// One 256-thread workgroup (4 waves of 64) per row; few rows are spread over more workgroups or threads (launch_prep). The
// row is cut into 8-element chunks; thread t takes chunks t, t + 256, ... (16-byte loads, consecutive threads on
// consecutive chunks: coalesced). Up to 2048 * CPW elements a thread keeps its chunks in registers (one read of the row);
// longer rows are read again per pass.
// Reference: wgpkernels/int8/int8_gemm.cu (K8) :253-485 (kernels), :1354-1414 and :1860-1977 (launch / C ABI).
#include "wq8_common.h"
#include "wq8_abi.h"

namespace wq8 {

enum { PREP_BLOCKS = 0, PREP_ROWS = 1, PREP_TRANSFORM = 2 };

struct PrepArgs {
    const void* x;          // input rows (ldx elements apart)
    int8_t* q;              // BLOCKS: q; ROWS: hi
    int8_t* lo;             // ROWS: optional lo
    float* scale;           // BLOCKS: (m, ceil(k/128)); ROWS: (m)
    void* out;              // TRANSFORM: (m, k) in x's dtype
    float* inv_rms;         // optional: 1 / RMS per row (RMSNorm only)
    const void* act_weight; // RMSNorm weight (k values) or null
    const long long* counter; long long first, step;  // row offset first + counter[0] * step of x (graph loops)
    int64_t ldx;
    int k, group, act;
    float eps;
};

// Sum over the 4 waves of a workgroup in the fixed order ((w0 + w1) + w2) + w3.
WQ8_DEVICE float block_sum4(float wave_value, float* lds4) {
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds4[wave] = wave_value;
    __syncthreads();
    return ((lds4[0] + lds4[1]) + lds4[2]) + lds4[3];
}

WQ8_DEVICE float block_max4(float wave_value, float* lds4) {
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds4[wave] = wave_value;
    __syncthreads();
    return fmaxf(fmaxf(lds4[0], lds4[1]), fmaxf(lds4[2], lds4[3]));
}

// ---- one prepared chunk c (8 elements) of row r -> memory ----------------------------------------------------------------
// Block codes: one FP32 scale per 128-element block = 16 consecutive lanes (one DPP row; every lane of the wave calls).
template <int DT> WQ8_DEVICE void store_block_codes(const PrepArgs& p, int64_t r, int k, int c, int chunks, const float* v) {
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, __builtin_fabsf(v[j]));
    amax = row16_max(amax);
    const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
    if (c >= chunks) return;
    if ((c & 15) == 0) p.scale[r * ((k + 127) >> 7) + (c >> 4)] = div127(amax * group_norm(p.group));
    int qv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        // |v inv| <= 127: the code is the low byte. FP32 rows keep the conversion, whose NaN result is 0 whatever the
        // NaN's payload (a BF16 / FP16 input NaN has a zero low byte either way)
        if constexpr (DT == DT_F32) qv[j] = rne_int(v[j] * inv);
        else qv[j] = rne_low_byte(v[j] * inv);
    }
    *reinterpret_cast<u32x2*>(p.q + r * k + 8 * c) = u32x2{pack_s8x4(qv[0], qv[1], qv[2], qv[3]), pack_s8x4(qv[4], qv[5], qv[6], qv[7])};
}
// Row codes, with the remainder's codes where p.lo asks for them.
WQ8_DEVICE void store_row_codes(const PrepArgs& p, int64_t r, int k, int c, int chunks, float inv, const float* v) {
    if (c >= chunks) return;
    int hv[8], lv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float t = v[j] * inv;
        hv[j] = rne_int(t);
        lv[j] = rne_int((t - float(hv[j])) * 254.0f);
    }
    *reinterpret_cast<u32x2*>(p.q + r * k + 8 * c) = u32x2{pack_s8x4(hv[0], hv[1], hv[2], hv[3]), pack_s8x4(hv[4], hv[5], hv[6], hv[7])};
    if (p.lo) *reinterpret_cast<u32x2*>(p.lo + r * k + 8 * c) = u32x2{pack_s8x4(lv[0], lv[1], lv[2], lv[3]), pack_s8x4(lv[4], lv[5], lv[6], lv[7])};
}
// Rows in x's dtype.
template <int DT> WQ8_DEVICE void store_transformed(const PrepArgs& p, int64_t r, int k, int c, int chunks, const float* v) {
    using raw = typename Elem<DT>::raw;
    if (c >= chunks) return;
    const float norm = group_norm(p.group);
    raw* out = static_cast<raw*>(p.out) + r * k;
    if constexpr (DT == DT_F32) {
#pragma unroll
        for (int j = 0; j < 8; ++j) out[8 * c + j] = v[j] * norm;
    } else {
        u32x4 packed;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            packed[j] = uint32_t(Elem<DT>::from_f(v[2 * j] * norm)) | (uint32_t(Elem<DT>::from_f(v[2 * j + 1] * norm)) << 16);
        *reinterpret_cast<u32x4*>(out + 8 * c) = packed;
    }
}

// Waves per SIMD asked of the register allocator: a thread caches 8 * CPW floats, and these budgets (64, 96, 128 VGPRs)
// keep the occupancy that the cache alone allows. FP16 rows of the block quantizer and of transform_rows need more
// registers to convert and would spill under them; there the budget only holds 4 waves at 6 chunks of the quantizer.
constexpr int prep_waves(int dt, int mode, int cpw) {
    return dt == DT_F16 && mode != PREP_ROWS ? (mode == PREP_BLOCKS && cpw == 6 ? 4 : 1) : cpw <= 4 ? 8 : cpw <= 7 ? 5 : 4;
}

template <int DT, int MODE, int CPW>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(prep_waves(DT, MODE, CPW)))) prep_rows(PrepArgs p) {
    using raw = typename Elem<DT>::raw;
    __shared__ float lds4[4];
    const int tid = threadIdx.x;
    const int k = p.k, chunks = k >> 3, act = p.act, group = p.group;
    const long long shift = p.counter ? p.first + __ldg(p.counter) * p.step : 0;
    const raw* row = static_cast<const raw*>(p.x) + (int64_t(blockIdx.x) + shift) * p.ldx;
    const raw* aw = static_cast<const raw*>(p.act_weight);
    const int64_t r = blockIdx.x;
    const int iters = CPW ? CPW : (chunks + 255) >> 8;

    // RMSNorm: sum of squares in the fixed tree (per thread: chunks in order, fmaf per element; wave butterfly;
    // ((w0 + w1) + w2) + w3).
    float cache[CPW ? CPW : 1][8];
    float inv_rms = 1.0f;
    if (CPW) {
#pragma unroll
        for (int i = 0; i < (CPW ? CPW : 1); ++i) {
            const int c = tid + 256 * i;
            load_act<DT>(row, k, 8 * c, cache[i], c < chunks, act == ACT_RMS ? ACT_NONE : act);
        }
    }
    if (act == ACT_RMS) {
        float ss = 0.0f;
        for (int i = 0; i < iters; ++i) {
            float v[8];
            const int c = tid + 256 * i;
            if (CPW) {
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = cache[CPW ? i : 0][j];
            } else {
                load8<DT>(row + 8 * c, v, c < chunks);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(v[j], v[j], ss);
        }
        inv_rms = rms_inverse(block_sum4(wave_sum(ss), lds4), k, p.eps);
        if (p.inv_rms && tid == 0) p.inv_rms[r] = inv_rms;
    }
    // the prepared (op, RMSNorm, rotated) chunk i of this thread
    auto chunk = [&](int i, float* v) {
        const int c = tid + 256 * i;
        const bool valid = c < chunks;
        if (CPW) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = cache[CPW ? i : 0][j];
        } else {
            load_act<DT>(row, k, 8 * c, v, valid, act == ACT_RMS ? ACT_NONE : act);
        }
        if (act == ACT_RMS) apply_rms<DT>(v, inv_rms, aw, 8 * c, valid);
        rotate_chunk(v, group);
    };
    if constexpr (MODE == PREP_BLOCKS) {
        for (int i = 0; i < iters; ++i) {
            // a wave whose chunks all lie past the row has nothing to store (its blocks are another wave's)
            if (256 * i + (tid & ~63) >= chunks) break;
            float v[8];
            chunk(i, v);
            store_block_codes<DT>(p, r, k, tid + 256 * i, chunks, v);
        }
    } else if constexpr (MODE == PREP_ROWS) {
        float amax = 0.0f;
        for (int i = 0; i < iters; ++i) {
            float v[8];
            chunk(i, v);
            if (CPW) {
#pragma unroll
                for (int j = 0; j < 8; ++j) cache[CPW ? i : 0][j] = v[j];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) amax = fmaxf(amax, __builtin_fabsf(v[j]));
        }
        amax = block_max4(wave_max(amax), lds4);
        const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
        if (tid == 0) p.scale[r] = div127(amax * group_norm(group));
        for (int i = 0; i < iters; ++i) {
            float v[8];
            if (CPW) {
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = cache[CPW ? i : 0][j];
            } else {
                chunk(i, v);
            }
            store_row_codes(p, r, k, tid + 256 * i, chunks, inv, v);
        }
    } else {
        for (int i = 0; i < iters; ++i) {
            // a wave whose chunks all lie past the row has nothing to store (its blocks are another wave's)
            if (256 * i + (tid & ~63) >= chunks) break;
            float v[8];
            chunk(i, v);
            store_transformed<DT>(p, r, k, tid + 256 * i, chunks, v);
        }
    }
}

// The same preparation with a row spread over several workgroups of one chunk a thread (block codes, transform_rows):
// workgroup (row, part) takes chunks 256 part .. 256 part + 255. For RMSNorm every part sums the whole row's squares in
// prep_rows's tree (the row comes from L2 after the first).
// Few rows leave prep_rows on as many CUs, each thread working through up to 8 chunks of a gelu of 26 operations.
template <int DT, int MODE>
__global__ void __launch_bounds__(256) prep_parts(PrepArgs p, int parts) {
    static_assert(MODE != PREP_ROWS, "a row's scale needs the whole row");
    using raw = typename Elem<DT>::raw;
    __shared__ float lds4[4];
    const int tid = threadIdx.x, part = blockIdx.x % parts;
    const int64_t r = blockIdx.x / parts;
    const int k = p.k, chunks = k >> 3, act = p.act, c = 256 * part + tid;
    const long long shift = p.counter ? p.first + __ldg(p.counter) * p.step : 0;
    const raw* row = static_cast<const raw*>(p.x) + (r + shift) * p.ldx;
    const bool valid = c < chunks;
    float v[8];
    load_act<DT>(row, k, 8 * c, v, valid, act == ACT_RMS ? ACT_NONE : act);
    if (act == ACT_RMS) {
        float ss = 0.0f;
        for (int i = 0; i < parts; ++i) {
            float u[8];
            const int ci = tid + 256 * i;
            load8<DT>(row + 8 * ci, u, ci < chunks);
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(u[j], u[j], ss);
        }
        const float inv_rms = rms_inverse(block_sum4(wave_sum(ss), lds4), k, p.eps);
        if (p.inv_rms && tid == 0 && part == 0) p.inv_rms[r] = inv_rms;
        apply_rms<DT>(v, inv_rms, static_cast<const raw*>(p.act_weight), 8 * c, valid);
    }
    if ((c & ~63) >= chunks) return;  // a wave whose chunks all lie past the row
    rotate_chunk(v, p.group);
    if constexpr (MODE == PREP_BLOCKS) store_block_codes<DT>(p, r, k, c, chunks, v);
    else store_transformed<DT>(p, r, k, c, chunks, v);
}

// Row codes (and hi / lo) with G x 256 threads a row, ceil(chunks / (256 G)) chunks a thread: few rows then have G times
// the waves at work on each. Thread 256 q + s takes chunks s + 256 (q + G j); RMSNorm's sum of squares keeps prep_rows's
// tree, its 256 chains handed from one group of 256 threads to the next through LDS.
template <int DT, int G, int CPT>
__global__ void __launch_bounds__(256 * G) prep_wide(PrepArgs p) {
    using raw = typename Elem<DT>::raw;
    __shared__ float lds[4 * G], chain[256];
    const int tid = threadIdx.x, slot = tid & 255, q = tid >> 8;
    const int k = p.k, chunks = k >> 3, act = p.act;
    const int64_t r = blockIdx.x;
    const long long shift = p.counter ? p.first + __ldg(p.counter) * p.step : 0;
    const raw* row = static_cast<const raw*>(p.x) + (r + shift) * p.ldx;
    float v[CPT][8];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        const int c = slot + 256 * (q + G * j);
        load_act<DT>(row, k, 8 * c, v[j], c < chunks, act == ACT_RMS ? ACT_NONE : act);
    }
    if (act == ACT_RMS) {
        if (q == 0) chain[slot] = 0.0f;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CPT; ++j)
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if (q == g) {
                    float ss = chain[slot];
#pragma unroll
                    for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(v[j][e], v[j][e], ss);
                    chain[slot] = ss;
                }
                __syncthreads();
            }
        // every group takes the 256 chains' butterfly sum itself: wave w of a group holds the sum of chains 64 w ..
        const float w = wave_sum(chain[slot]);
        if ((tid & 63) == 0) lds[tid >> 6] = w;
        __syncthreads();
        const float inv_rms = rms_inverse(((lds[4 * q] + lds[4 * q + 1]) + lds[4 * q + 2]) + lds[4 * q + 3], k, p.eps);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int c = slot + 256 * (q + G * j);
            apply_rms<DT>(v[j], inv_rms, static_cast<const raw*>(p.act_weight), 8 * c, c < chunks);
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
        rotate_chunk(v[j], p.group);
#pragma unroll
        for (int e = 0; e < 8; ++e) amax = fmaxf(amax, __builtin_fabsf(v[j][e]));
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) lds[tid >> 6] = amax;
    __syncthreads();
    amax = lds[0];
#pragma unroll
    for (int w = 1; w < 4 * G; ++w) amax = fmaxf(amax, lds[w]);
    const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
    if (tid == 0) p.scale[r] = div127(amax * group_norm(p.group));
#pragma unroll
    for (int j = 0; j < CPT; ++j) store_row_codes(p, r, k, slot + 256 * (q + G * j), chunks, inv, v[j]);
}

// Whether the rows or codes are written over input rows: prep_parts's parts each read the whole of a normalised row, where
// one workgroup a row has it in registers (or reads its own chunk last) before it stores.
template <int DT> static bool stores_over_input(const PrepArgs& p, int m) {
    constexpr uintptr_t SIZE = sizeof(typename Elem<DT>::raw);
    const uintptr_t x = reinterpret_cast<uintptr_t>(p.x), out = reinterpret_cast<uintptr_t>(p.out ? p.out : p.q);
    return x < out + uintptr_t(m) * p.k * (p.out ? SIZE : 1) && out < x + (uintptr_t(m - 1) * p.ldx + p.k) * SIZE;
}

template <int DT, int MODE>
static int launch_prep(const PrepArgs& p, int m, hipStream_t stream) {
    const int chunks = p.k / 8, parts = (chunks + 255) / 256;
    // Few rows: spread over the chip (prep_parts, prep_wide). The lines lie where the two forms measured equal, BF16, in us
    // (a row per 256 threads -> spread), K = 5120 and 13824:
    //   gelu codes        M = 1: 3.9 -> 2.5, 7.2 -> 2.6; M = 512: 4.9 -> 4.4, 9.2 -> 7.6; M = 1024: 6.6 -> 6.6, 15.0 -> 13.0
    //   RMSNorm codes     M = 128: 4.4 -> 3.7, 7.3 -> 5.1; M = 256: 4.5 -> 4.0, 7.6 -> 10.7 (every part reads the whole row)
    //   hi / lo, no op    M = 1: 3.2 -> 2.6, 4.8 -> 3.5; M = 512: 4.5 -> 4.3, 8.1 -> 7.2; M = 1024: 5.9 -> 6.6, 12.4 -> 12.9
    //   hi / lo, RMSNorm  M = 256: 4.9 -> 4.6, 8.1 -> 7.0; M = 512: 5.6 -> 5.9, 10.1 -> 9.9
    // Rows of one part (K <= 2048) have nothing to spread, and rows of more than 8 (K > 16384) stay with the looping form.
    if (parts > 1 && parts <= 8) {
        if constexpr (MODE == PREP_ROWS) {
            if (m <= (p.act == ACT_RMS ? 256 : 512)) {
                if (parts == 2) prep_wide<DT, 2, 1><<<m, 512, 0, stream>>>(p);
                else if (parts == 3) prep_wide<DT, 3, 1><<<m, 768, 0, stream>>>(p);
                else if (parts == 4) prep_wide<DT, 4, 1><<<m, 1024, 0, stream>>>(p);
                else prep_wide<DT, 4, 2><<<m, 1024, 0, stream>>>(p);
                return int(hipGetLastError());
            }
        } else if (p.act == ACT_RMS ? m * parts <= 1024 && !stores_over_input<DT>(p, m) : m <= 256 * (parts < 4 ? parts : 4)) {
            prep_parts<DT, MODE><<<m * parts, 256, 0, stream>>>(p, parts);
            return int(hipGetLastError());
        }
    }
    // one row per workgroup; chunks per thread: the smallest count that covers the row (K = 5120 -> 3, 13824 -> 7), so no
    // thread evaluates the activation on chunks past the row
    if (chunks <= 256) prep_rows<DT, MODE, 1><<<m, 256, 0, stream>>>(p);
    else if (chunks <= 512) prep_rows<DT, MODE, 2><<<m, 256, 0, stream>>>(p);
    else if (chunks <= 768) prep_rows<DT, MODE, 3><<<m, 256, 0, stream>>>(p);
    else if (chunks <= 1024) prep_rows<DT, MODE, 4><<<m, 256, 0, stream>>>(p);
    else if (chunks <= 1536) prep_rows<DT, MODE, 6><<<m, 256, 0, stream>>>(p);
    else if (chunks <= 1792) prep_rows<DT, MODE, 7><<<m, 256, 0, stream>>>(p);
    else if (chunks <= 2048) prep_rows<DT, MODE, 8><<<m, 256, 0, stream>>>(p);
    else prep_rows<DT, MODE, 0><<<m, 256, 0, stream>>>(p);
    return int(hipGetLastError());
}

template <int MODE>
static int dispatch_prep(const PrepArgs& p, int m, int dtype, hipStream_t stream) {
    if (dtype == DT_F16) return launch_prep<DT_F16, MODE>(p, m, stream);
    if (dtype == DT_BF16) return launch_prep<DT_BF16, MODE>(p, m, stream);
    if (dtype == DT_F32 && !p.act) return launch_prep<DT_F32, MODE>(p, m, stream);
    return -1;
}

// argument checks shared by the preparation entry points (before any launch)
static int check_prep(int m, int k, int dtype, int group, int act) {
    if (dtype < 0 || dtype > 2) return -1;
    if (group != 0 && group != 16 && group != 64 && group != 256) return -1;
    if (act < 0 || act > 3) return -1;
    if (dtype == DT_F32 && act) return -1;
    if (m < 0 || k <= 0 || k % 8 || (group && k % group)) return -2;
    return 0;
}

thread_local RowOffsetArgs g_prep_offset = {nullptr, 0, 0};

}  // namespace wq8

using namespace wq8;

WQ8_API int wq8_quantize(const void* x, int8_t* hi, int8_t* lo, float* scale, int m, int k, int64_t ldx, int dtype, int group, int act,
                         const void* act_weight, float eps, hipStream_t stream) {
    if (!m) return 0;
    if (int rc = check_prep(m, k, dtype, group, act)) return rc;
    PrepArgs p{x, hi, lo, scale, nullptr, nullptr, act_weight, g_prep_offset.counter, g_prep_offset.first, g_prep_offset.step,
               ldx, k, group, act, eps};
    return dispatch_prep<PREP_ROWS>(p, m, dtype, stream);
}

WQ8_API int wq8_quantize_blocks(const void* x, int8_t* q, float* scale, int m, int k, int64_t ldx, int dtype, int group, int act,
                                const void* act_weight, float eps, float* inv_rms, hipStream_t stream) {
    if (!m) return 0;
    if (int rc = check_prep(m, k, dtype, group, act)) return rc;
    // the reference's caller supplies inv_rms scratch for RMSNorm rows longer than 16384 (K8:1887-1890); kept as a
    // contract: this library fills it with the rows' 1 / RMS
    if (act == ACT_RMS && k > 16384 && !inv_rms) return -2;
    PrepArgs p{x, q, nullptr, scale, nullptr, inv_rms, act_weight, g_prep_offset.counter, g_prep_offset.first, g_prep_offset.step,
               ldx, k, group, act, eps};
    return dispatch_prep<PREP_BLOCKS>(p, m, dtype, stream);
}

WQ8_API int wq8_quantize_at(const void* x, int8_t* hi, int8_t* lo, float* scale, int m, int k, int64_t ldx, int dtype, int group, int act,
                            const void* act_weight, float eps, const long long* counter, long long first, long long step, hipStream_t stream) {
    g_prep_offset = {counter, first, step};
    const int rc = wq8_quantize(x, hi, lo, scale, m, k, ldx, dtype, group, act, act_weight, eps, stream);
    g_prep_offset = {nullptr, 0, 0};
    return rc;
}

WQ8_API int wq8_quantize_blocks_at(const void* x, int8_t* q, float* scale, int m, int k, int64_t ldx, int dtype, int group, int act,
                                   const void* act_weight, float eps, float* inv_rms, const long long* counter, long long first, long long step,
                                   hipStream_t stream) {
    g_prep_offset = {counter, first, step};
    const int rc = wq8_quantize_blocks(x, q, scale, m, k, ldx, dtype, group, act, act_weight, eps, inv_rms, stream);
    g_prep_offset = {nullptr, 0, 0};
    return rc;
}

WQ8_API int wq8_transform_rows(const void* x, void* out, int m, int k, int64_t ldx, int dtype, int group, int act, const void* act_weight,
                               float eps, hipStream_t stream) {
    if (!m) return 0;
    if (dtype != DT_F16 && dtype != DT_BF16) return -1;
    if (int rc = check_prep(m, k, dtype, group, act)) return rc;
    PrepArgs p{x, nullptr, nullptr, nullptr, out, nullptr, act_weight, nullptr, 0, 0, ldx, k, group, act, eps};
    return dispatch_prep<PREP_TRANSFORM>(p, m, dtype, stream);
}

WQ8_API int wq8_rotate_groups(const void* x, void* out, int m, int k, int64_t ldx, int dtype, int group, hipStream_t stream) {
    if (!m) return 0;
    if (dtype != DT_F16 && dtype != DT_BF16) return -1;
    if (group != 16 && group != 64 && group != 256) return -1;
    if (k <= 0 || k % group) return -2;
    PrepArgs p{x, nullptr, nullptr, nullptr, out, nullptr, nullptr, nullptr, 0, 0, ldx, k, group, ACT_NONE, 0.0f};
    return dispatch_prep<PREP_TRANSFORM>(p, m, dtype, stream);
}
