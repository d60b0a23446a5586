// tl_float.hip -- the float32 model of model/tinyllama.py (TL), the baseline
// the INT8 path is compared against by the analysis report (GI:470-626):
//   linear_f32_kernel     TL:106-110  y = x . W (+ b) (+ residual), W [K][N]
//   attention_f32_kernel  TL:122-156  scores, causal mask, softmax, P . V
// Float32 sums here run in tile order, not NumPy's, so results agree with the
// reference to float32 rounding, not bit for bit.  Not on the INT8 hot path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "tl_device.h"
#include "tl_internal.h"

namespace tl {

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

// y = x . W on v_mfma_f32_32x32x2_f32 (one multiply-add per product, float32
// accumulators): a workgroup of 8 wavefronts per 32 x (32 NB) output tile, each
// over an eighth of K, partial tiles added in LDS in a fixed order.  In a chunk
// of 8 k's lane l holds x[row l % 32][4 (l / 32) .. + 3] (one 16-byte load) and
// multiplies k = s and k = 4 + s in step s, so its W operand is row
// 4 (l / 32) + s, column l % 32 of each column block: 128-byte runs of W
// straight into registers, no LDS and no barrier in the main loop.
// What bounds it: the float32 matrix rate at hundreds of rows (640 x 5632 x
// 2048: 90 TFLOP/s; 100 x 5632 x 2048 puts 236 of 256 CUs at work), launch and
// latency at a few.  The whole call at 100 x 5632 x 2048: 245 us with 64 x 64 vector-FMA
// tiles through LDS, 50 us now; 640 rows 407 -> 170; one row 238 -> 28.  Eight
// partial sums per output also round less: 2.9e-7 relative to 64 bits where
// one chain of 2048 had 8.1e-7.
constexpr int kLinWaves = 8;

// WIDE: the form for every size.  The other one counts tiles in one grid
// dimension and lane offsets and columns in 32 bits (launch_linear_f32 says up to
// where); its shorter start is worth 0.5-0.7 us of a whole call (38.3 against 39.0 us
// at 33 x 5632 x 2048, 50.3 against 51.0 at 100 rows).
template <int NB, bool VEC, bool WIDE>
__global__ __launch_bounds__(kLinWaves * 64) void linear_f32_kernel(const float* __restrict__ x,
                                                                    const float* __restrict__ w,
                                                                    const float* __restrict__ b,
                                                                    const float* __restrict__ residual, int32_t m,
                                                                    int32_t n, int32_t k, int32_t tiles_m,
                                                                    int32_t tiles_n, float* __restrict__ y) {
    using Off = std::conditional_t<WIDE, int64_t, unsigned>;
    using Col = std::conditional_t<WIDE, unsigned, int>;   // the last tile's columns may pass 2^31
    constexpr int PD = NB == 1 ? 8 : 4, HW = kLinWaves / 2;   // chunks in flight; LDS partial tiles
    __shared__ float red[HW][NB * 16][64];
    // workgroups go to the 8 XCDs round-robin: the row tiles of a column tile
    // stay on one XCD, whose L2 then holds the column tile's weights.  One
    // dimension, or (wide) 8 x the row tiles in x and groups of 8 column tiles in y
    // and z: the same order
    int tm, tn;
    if constexpr (WIDE) {
        tm = (int)blockIdx.x >> 3;
        tn = (int)(blockIdx.z * gridDim.y + blockIdx.y) * 8 + ((int)blockIdx.x & 7);
    } else {
        const int q = (int)blockIdx.x >> 3;
        tn = q / tiles_m * 8 + ((int)blockIdx.x & 7);
        tm = q % tiles_m;
    }
    if (tn >= tiles_n) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), col = lane & 31, hi = lane >> 5;
    const int64_t row0 = (int64_t)tm * 32;
    const Col col0 = (Col)tn * 32 * NB;
    const int nfull = k >> 3, nch = WIDE ? nfull + ((k & 7) != 0) : (k + 7) >> 3, per = (nch + kLinWaves - 1) / kLinWaves;
    const int c0 = min(wave * per, nfull), c1 = min(c0 + per, nfull);   // this wavefront's whole chunks
    // one wavefront-uniform base per chunk, and lane offsets formed once
    const float* xb = x + row0 * k;
    const Off xo = (Off)min(col, (int)(m - 1 - row0)) * (Off)k + 4 * hi;
    Off wo[4][NB];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int j = 0; j < NB; j++) wo[s][j] = (Off)(4 * hi + s) * (Off)n + (unsigned)min(col0 + 32 * j + col, (Col)n - 1);
    v16f acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = (v16f){};
    float av[PD][4], bv[PD][4][NB];
    auto load = [&](int set, int c) {
        const float* xc = xb + 8 * (int64_t)c;
        const float* wc = w + 8 * (int64_t)c * n;
        if constexpr (VEC) {
            const float4 v = *(const float4*)(xc + xo);
            av[set][0] = v.x; av[set][1] = v.y; av[set][2] = v.z; av[set][3] = v.w;
        } else {
#pragma unroll
            for (int s = 0; s < 4; s++) av[set][s] = xc[xo + s];
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < NB; j++) bv[set][s][j] = wc[wo[s][j]];
    };
    auto mma = [&](int set) {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[set][s], bv[set][s][j], acc[j], 0, 0, 0);
    };
    if (c0 < c1) {
#pragma unroll
        for (int u = 0; u < PD; u++) load(u, min(c0 + u, c1 - 1));
        int c = c0;
        for (; c + PD <= c1; c += PD) {
#pragma unroll
            for (int u = 0; u < PD; u++) {
                mma(u);
                load(u, min(c + u + PD, c1 - 1));   // past the end: a redundant load in bounds
                __builtin_amdgcn_sched_barrier(0);  // the loads stay here: PD - 1 chunks of MFMAs cover them
            }
        }
#pragma unroll
        for (int u = 0; u < PD - 1; u++)
            if (c + u < c1) mma(u);
    }
    if (nch > nfull && wave == kLinWaves - 1) {   // the last k % 8: zeros past k on both sides
        const int64_t kk = 8 * (int64_t)nfull + 4 * hi;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const bool in = kk + s < k;
            av[0][s] = in ? xb[8 * (int64_t)nfull + xo + s] : 0.0f;
#pragma unroll
            for (int j = 0; j < NB; j++) bv[0][s][j] = in ? w[8 * (int64_t)nfull * n + wo[s][j]] : 0.0f;
        }
        mma(0);
    }
    // wavefront h + 4's tile into LDS, wavefront h adds its own, then every
    // thread adds four partial sums per output in wavefront order
    if (wave >= HW) {
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) red[wave - HW][j * 16 + e][lane] = acc[j][e];
    }
    __syncthreads();
    if (wave < HW) {
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) red[wave][j * 16 + e][lane] = acc[j][e] + red[wave][j * 16 + e][lane];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * NB; i++) {   // output register e of block j: 16 NB of them over 8 wavefronts
        const int je = i * kLinWaves + wave, e = je & 15;
        const int64_t r = row0 + 8 * (e >> 2) + 4 * hi + (e & 3);
        const Col c = col0 + 32 * (je >> 4) + col;
        if (r >= m || c >= (Col)n) continue;
        float v = (red[0][je][lane] + red[1][je][lane]) + (red[2][je][lane] + red[3][je][lane]);
        if (b) v = v + b[c];
        const int64_t idx = r * n + c;
        if (residual) v = residual[idx] + v;
        y[idx] = v;
    }
}

template <int NB>
void go_linear(hipStream_t s, const float* x, const float* w, const float* b, const float* residual, int32_t m,
               int32_t n, int32_t k, int32_t tm, int32_t tn, float* y) {
    const dim3 grid((unsigned)((tn + 7) / 8 * 8) * (unsigned)tm), block(kLinWaves * 64);
    if (k % 4 == 0 && (uintptr_t)x % 16 == 0)
        TL_KLAUNCH((linear_f32_kernel<NB, true, false>), grid, block, 0, s, x, w, b, residual, m, n, k, tm, tn, y);
    else TL_KLAUNCH((linear_f32_kernel<NB, false, false>), grid, block, 0, s, x, w, b, residual, m, n, k, tm, tn, y);
}

void go_linear_wide(hipStream_t s, const float* x, const float* w, const float* b, const float* residual, int32_t m,
                    int32_t n, int32_t k, float* y) {
    constexpr int32_t kMaxY = 32768;
    const int32_t tm = (int32_t)(((int64_t)m + 31) / 32), tn = (int32_t)(((int64_t)n + 31) / 32), g = (tn + 7) / 8;
    const dim3 grid(8u * (unsigned)tm, std::min(g, kMaxY), (g + kMaxY - 1) / kMaxY), block(kLinWaves * 64);
    TL_KLAUNCH((linear_f32_kernel<1, false, true>), grid, block, 0, s, x, w, b, residual, m, n, k, tm, tn, y);
}

// one (query row i, query head h) per workgroup; the row's scores live in LDS
__global__ __launch_bounds__(256) void attention_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                            const float* __restrict__ v, int32_t seq, int32_t n_heads,
                                                            int32_t n_kv, float scale, float* __restrict__ out,
                                                            float* __restrict__ scores, float* __restrict__ weights) {
    extern __shared__ float s[];   // [seq] scores -> exps -> probabilities, then [nblk] block sums
    __shared__ float qv[64];
    __shared__ float red[16];
    __shared__ float total_s;
    __shared__ float part[4][64];
    const int i = blockIdx.x, h = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int G = n_heads / n_kv, g = h / G;
    const int D = n_heads * kHeadDim, KVD = n_kv * kHeadDim;
    if (tid < kHeadDim) qv[tid] = q[(int64_t)i * D + h * kHeadDim + tid];
    __syncthreads();
    const int64_t srow = ((int64_t)h * seq + i) * seq;
    float mx = -INFINITY;
    for (int t = tid; t < seq; t += blockDim.x) {
        float val = -1e9f;   // TL:90-91 causal mask value
        if (t <= i) {
            const float* kr = k + (int64_t)t * KVD + g * kHeadDim;
            float acc = 0.0f;
#pragma unroll 16
            for (int d = 0; d < kHeadDim; d++) acc = __builtin_fmaf(qv[d], kr[d], acc);
            val = acc * scale;
        }
        s[t] = val;
        if (scores) scores[srow + t] = val;
        mx = fmaxf(mx, val);
    }
    const float m = block_max(mx, red);
    const int nblk = (seq + 63) >> 6;
    float* bsum = s + seq;
    for (int bi = wave; bi < nblk; bi += blockDim.x >> 6) {
        const int t = bi * 64 + lane;
        float e = 0.0f;
        if (t < seq) {
            e = tl_expf(s[t] - m);
            s[t] = e;
        }
        const float bsv = wave_butterfly_sum(e);
        if (lane == 0) bsum[bi] = bsv;
    }
    __syncthreads();
    if (tid == 0) {
        float tot = 0.0f;
        for (int bi = 0; bi < nblk; bi++) tot = tot + bsum[bi];
        total_s = tot;
    }
    __syncthreads();
    const float tot = total_s;
    for (int t = tid; t < seq; t += blockDim.x) {
        const float p = __fdiv_rn(s[t], tot);
        s[t] = p;
        if (weights) weights[srow + t] = p;
    }
    __syncthreads();
    // keys past i have probability 0 exactly and are skipped
    float acc = 0.0f;
    for (int t = wave; t <= i; t += 4) acc = __builtin_fmaf(s[t], v[(int64_t)t * KVD + g * kHeadDim + lane], acc);
    part[wave][lane] = acc;
    __syncthreads();
    if (tid < kHeadDim)
        out[(int64_t)i * D + h * kHeadDim + tid] = ((part[0][tid] + part[1][tid]) + part[2][tid]) + part[3][tid];
}

}  // namespace

hipError_t launch_linear_f32(hipStream_t s, const float* x, const float* w, const float* b, const float* residual,
                             int32_t m, int32_t n, int32_t k, float* y) {
    if (m <= 0 || n <= 0) return hipSuccess;
    // column blocks per tile: the fewest MFMAs on the busiest CU (rounds of 256
    // tiles times blocks); of equals the widest, which reads x least often
    const int64_t tm = ((int64_t)m + 31) / 32;
    int nb = 1;
    int64_t best = INT64_MAX, tn = 0;
    for (int c = 1; c <= 4; c++) {
        const int64_t t = ((int64_t)n + 32 * c - 1) / (32 * c), cost = (tm * t + 255) / 256 * c;
        if (cost <= best) {
            best = cost;
            nb = c;
            tn = t;
        }
    }
    // offsets inside a tile below 2^32 (31 k + 8 and 8 n), and a grid below 2^32
    // threads of one dimension
    if (k >= 1 << 27 || n > 1 << 29 || (tn + 7) / 8 * 8 * tm >= 1 << 23) {
        go_linear_wide(s, x, w, b, residual, m, n, k, y);
        return hipGetLastError();
    }
    const int32_t m32 = (int32_t)tm, n32 = (int32_t)tn;
    switch (nb) {
        case 1: go_linear<1>(s, x, w, b, residual, m, n, k, m32, n32, y); break;
        case 2: go_linear<2>(s, x, w, b, residual, m, n, k, m32, n32, y); break;
        case 3: go_linear<3>(s, x, w, b, residual, m, n, k, m32, n32, y); break;
        default: go_linear<4>(s, x, w, b, residual, m, n, k, m32, n32, y); break;
    }
    return hipGetLastError();
}

hipError_t launch_attention_f32(hipStream_t s, const float* q, const float* k, const float* v, int32_t seq,
                                int32_t n_heads, int32_t n_kv, float scale, float* out, float* scores,
                                float* weights) {
    if (seq <= 0) return hipSuccess;
    const size_t lds = sizeof(float) * ((size_t)seq + (seq + 63) / 64);
    TL_KLAUNCH(attention_f32_kernel, dim3(seq, n_heads), dim3(256), lds, s, q, k, v, seq, n_heads, n_kv, scale, out,
               scores, weights);
    return hipGetLastError();
}

}  // namespace tl
