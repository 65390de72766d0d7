// Best-matching-unit search kernels for gfx950.
//
// Three precisions, one output contract: for every sample i the reference's top-2 BMUs
// (decontamination/algo/som_abstract.py:815-878 update rule = lexicographic (distance, index)),
// written as c1[i], c2[i] (int32, -1 when absent; c1 falls back to `default_index`) and d1[i]
// (FP64 squared distance of c1, NaN when absent).
//
//   EXACT       bmu_exact_kernel: one sample per lane, weights streamed through LDS, the exact
//               distance formula (reference FP32-difference/FP64-sum, or FP64) for every neuron.
//               Also the fallback for samples the MFMA path flags.
//   FP32        bmu_fp32_kernel: |w'|^2 - 2 x'.w' on v_mfma_f32_32x32x2_f32 (x', w' centred on the
//               weight centroid), top-2 on those values (the plain FP32 form).
//   BF16_RERANK bmu_f16_kernel: the same GEMM on v_mfma_f32_32x32x16_f16, from high and low FP16 parts of x' and
//               w' along directions chosen at preparation. Phase A scans half of a coarse sub-lattice of the
//               map for the top-2 of per-lane block minima; phase B scans every other neuron,
//               recording every neuron inside a provable error window of the running second minimum
//               while it tightens the window; phase C records phase A's neurons under the final window.
//               Then the exact distance formula on the recorded set, of FP32 or FP64 rows. Samples whose
//               list overflows, or whose bound is not finite, go to an exact scan.
#include "bmu_f16.hpp"

#include <algorithm>
#include <vector>

// instantiated in k_f16_*.hip
extern template int somhip_search_f16<16, float>(somhip_model *, const float *, int64_t, int, int, int, int32_t *, int32_t *,
                                              double *, float *, int64_t *, unsigned int *, const int32_t *);
extern template int somhip_search_f16<32, float>(somhip_model *, const float *, int64_t, int, int, int, int32_t *, int32_t *,
                                              double *, float *, int64_t *, unsigned int *, const int32_t *);
extern template int somhip_search_f16<64, float>(somhip_model *, const float *, int64_t, int, int, int, int32_t *, int32_t *,
                                              double *, float *, int64_t *, unsigned int *, const int32_t *);
extern template int somhip_search_f16<16, double>(somhip_model *, const double *, int64_t, int, int, int, int32_t *, int32_t *,
                                              double *, float *, int64_t *, unsigned int *, const int32_t *);
extern template int somhip_search_f16<32, double>(somhip_model *, const double *, int64_t, int, int, int, int32_t *, int32_t *,
                                              double *, float *, int64_t *, unsigned int *, const int32_t *);
extern template int somhip_search_f16<64, double>(somhip_model *, const double *, int64_t, int, int, int, int32_t *, int32_t *,
                                              double *, float *, int64_t *, unsigned int *, const int32_t *);

namespace {

// ------------------------------------------------------------------------------------------------
// EXACT: direct-difference scan. Grid: one thread per listed sample. T = float: the reference's
// FP32-difference formula (MODE REF32) or FP64 differences of the FP32 values (MODE FP64); T = double
// (float64 SOMs): FP64 differences of FP64 data and weights, no |x| maxima (xmax_part must be null).
// ------------------------------------------------------------------------------------------------
template <int DP, int MODE, bool NEED_C2, class T = float>
__global__ __launch_bounds__(256) void bmu_exact_kernel(const T *__restrict__ x, int64_t n, int dim,
                                                        const int64_t *__restrict__ list,
                                                        const unsigned int *__restrict__ list_count,
                                                        const T *__restrict__ w, int mn, int default_index,
                                                        int32_t *__restrict__ c1, int32_t *__restrict__ c2,
                                                        double *__restrict__ d1, float *__restrict__ xmax_part)
{
    constexpr bool F64 = sizeof(T) == sizeof(double);
    constexpr int CH = F64 ? 64 : 128;  // neurons per LDS chunk
    __shared__ T ws[CH * DP];
    const int64_t total = list ? (int64_t)(*list_count) : n;
    float amax[DP];
#pragma unroll
    for (int k = 0; k < DP; k++) amax[k] = 0.f;
    // Grid-stride over samples; every thread of the block takes part in the chunk loads.
    for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < total; base += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = base + threadIdx.x;
        const bool active = t < total;
        const int64_t i = active ? (list ? list[t] : t) : 0;
        T xr[DP];
#pragma unroll
        for (int k = 0; k < DP; k++) {
            xr[k] = (active && k < dim) ? x[i * dim + k] : (T)0;
            if constexpr (!F64) {
                const float a = fabsf(xr[k]);
                amax[k] = fmaxf(amax[k], a < __builtin_inff() ? a : 0.f);
            }
        }
        double md1 = 1.0e99, md2 = 1.0e99;
        int mi1 = -1, mi2 = -1;
        for (int j0 = 0; j0 < mn; j0 += CH) {
            __syncthreads();
            for (int e = threadIdx.x; e < CH * DP; e += blockDim.x) {
                int jj = j0 + e / DP, k = e % DP;
                ws[e] = (jj < mn && k < dim) ? w[(int64_t)jj * dim + k] : (T)0;
            }
            __syncthreads();
            const int jn = min(CH, mn - j0);
            for (int jj = 0; jj < jn; jj++) {
                double d;  // zero padding adds exact zeros
                if constexpr (F64) d = sqd_f64(&ws[jj * DP], xr, DP);
                else d = sqd_mode<MODE>(&ws[jj * DP], xr, DP);
                if (d != d) continue;
                const int j = j0 + jj;
                if (NEED_C2) {
                    if (md1 > d) {
                        md2 = md1; mi2 = mi1; md1 = d; mi1 = j;
                    } else if (md2 > d) {
                        md2 = d; mi2 = j;
                    }
                } else if (md1 > d) {
                    md1 = d; mi1 = j;
                }
            }
        }
        if (active) {
            c1[i] = mi1 >= 0 ? mi1 : default_index;
            if (c2) c2[i] = mi2;
            if (d1) d1[i] = mi1 >= 0 ? md1 : __builtin_nan("");
        }
    }
    if (!F64 && xmax_part) {
        const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
        for (int k = 0; k < DP; k++) {
            float v = amax[k];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, WAVE));
            amax[k] = v;
        }
        if (lane == 0) {
            const int64_t wid = (int64_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
#pragma unroll
            for (int k = 0; k < DP; k++) xmax_part[wid * DP + k] = amax[k];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// FP32 plain form. Wave = G groups of 32 samples; block = 32 neurons (natural order).
// ------------------------------------------------------------------------------------------------
template <int DP, int G>
__global__ __launch_bounds__(BMU_WAVES * WAVE) void bmu_fp32_kernel(
    const float *__restrict__ x, int64_t n, int dim, const float *__restrict__ centre,
    const f32x4 *__restrict__ frag, const f32x4 *__restrict__ norms4, int nblk, int mn, int default_index,
    int32_t *__restrict__ c1, int32_t *__restrict__ c2, double *__restrict__ d1, float *__restrict__ xmax_part)
{
    constexpr int KS = DP / 2;  // MFMA k-steps of 2
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = threadIdx.x / WAVE;
    const int64_t sbase = ((int64_t)blockIdx.x * BMU_WAVES + wave) * (G * 32);
    const int col = lane & 31;
    const int khalf = lane >> 5;

    // B operand: b[g][s] = -2 * x'[sample][2s + khalf]
    float b[G][KS];
    float xn[G];  // |x'|^2 partial (this lane's dims), combined below
    float amax[KS];
#pragma unroll
    for (int st = 0; st < KS; st++) amax[st] = 0.f;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int64_t s = sbase + g * 32 + col;
        float acc = 0.f;
#pragma unroll
        for (int st = 0; st < KS; st++) {
            const int k = 2 * st + khalf;
            const float raw = (s < n && k < dim) ? x[s * dim + k] : 0.f;
            const float a = fabsf(raw);
            amax[st] = fmaxf(amax[st], a < __builtin_inff() ? a : 0.f);
            float v = (k < dim) ? __fsub_rn(raw, centre[k]) : 0.f;
            b[g][st] = -2.f * v;
            acc = fmaf(v, v, acc);
        }
        xn[g] = acc + xchg32(acc);
    }
    if (xmax_part) {
#pragma unroll
        for (int st = 0; st < KS; st++) {
            float v = amax[st];
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, WAVE));
            amax[st] = v;
        }
        if ((lane & 31) == 0) {
            const int64_t wid = (int64_t)blockIdx.x * BMU_WAVES + wave;
#pragma unroll
            for (int st = 0; st < KS; st++) xmax_part[wid * DP + 2 * st + khalf] = amax[st];
        }
    }

    float m1[G], m2[G];
    int i1[G], i2[G];
#pragma unroll
    for (int g = 0; g < G; g++) { m1[g] = m2[g] = __builtin_inff(); i1[g] = i2[g] = -1; }

    auto load_block = [&](int blk, f32x4 (&a4)[KS / 4], f32x16 &cin) {
#pragma unroll
        for (int q = 0; q < KS / 4; q++) a4[q] = frag[((int64_t)blk * (KS / 4) + q) * WAVE + lane];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            f32x4 t = norms4[blk * 8 + 2 * q + khalf];
            cin[4 * q + 0] = t[0]; cin[4 * q + 1] = t[1]; cin[4 * q + 2] = t[2]; cin[4 * q + 3] = t[3];
        }
    };
    f32x4 a4[KS / 4];
    f32x16 cin;
    if (nblk > 0) load_block(0, a4, cin);
    for (int blk = 0; blk < nblk; blk++) {
        // prefetch the next block's fragments while this one computes
        f32x4 na4[KS / 4];
        f32x16 ncin;
        if (blk + 1 < nblk) load_block(blk + 1, na4, ncin);
        const int jbase = blk * 32 + 4 * khalf;
#pragma unroll
        for (int g = 0; g < G; g++) {
            f32x16 acc = cin;
#pragma unroll
            for (int st = 0; st < KS; st++)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[st / 4][st % 4], b[g][st], acc, 0, 0, 0);
            // in-order top-2 with strict '<' (lowest index wins ties within the lane):
            // values by min/med3, indices by selects
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float v = acc[r];
                const int j = jbase + 8 * (r >> 2) + (r & 3);
                const bool lt1 = v < m1[g];
                const bool lt2 = v < m2[g];
                const int t2 = lt2 ? j : i2[g];
                i2[g] = lt1 ? i1[g] : t2;
                i1[g] = lt1 ? j : i1[g];
                m2[g] = __builtin_amdgcn_fmed3f(m1[g], m2[g], v);
                m1[g] = fminf(m1[g], v);
            }
        }
        if (blk + 1 < nblk) {
#pragma unroll
            for (int q = 0; q < KS / 4; q++) a4[q] = na4[q];
            cin = ncin;
        }
    }

#pragma unroll
    for (int g = 0; g < G; g++) {
        // merge with the partner lane (lexicographic on (value, index))
        float pm1 = xchg32(m1[g]), pm2 = xchg32(m2[g]);
        int pi1 = xchg32i(i1[g]), pi2 = xchg32i(i2[g]);
        float a1 = m1[g], a2 = m2[g];
        int j1 = i1[g], j2 = i2[g];
        auto lessv = [](float da, int ia, float db, int ib) {
            return da < db || (da == db && (unsigned)ia < (unsigned)ib);
        };
        // insert partner's two candidates
        float cd[2] = {pm1, pm2};
        int ci[2] = {pi1, pi2};
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (ci[t] < 0) continue;
            if (lessv(cd[t], ci[t], a1, j1)) { a2 = a1; j2 = j1; a1 = cd[t]; j1 = ci[t]; }
            else if (lessv(cd[t], ci[t], a2, j2)) { a2 = cd[t]; j2 = ci[t]; }
        }
        const int64_t s = sbase + g * 32 + col;
        if (lane < 32 && s < n) {
            const bool ok1 = j1 >= 0 && j1 < mn;
            c1[s] = ok1 ? j1 : default_index;
            if (c2) c2[s] = (j2 >= 0 && j2 < mn) ? j2 : -1;
            if (d1) d1[s] = ok1 ? (double)fmaxf(a1 + xn[g], 0.f) : __builtin_nan("");
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Preparation of the derived weight data: centroid, for longer searches a rotation, then the plan, the
// fragments and the maxima of what they leave out.
// ------------------------------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(256) void prep_centre_kernel(const T *__restrict__ w, int mn, int ncol, int dim, int dpad,
                                                          float *__restrict__ centre, BmuPlan *__restrict__ plan)
{
    // one block per padded dimension; fixed-order FP64 sum, the extent about the centroid and the steps between
    // neighbours of a map row (those within a wave). Also clears the maxima that the next kernels raise (same stream).
    const int k = blockIdx.x;
    if (k == 0 && threadIdx.x >= 2 * F16_MAX_DIM && threadIdx.x < sizeof(BmuPlan) / sizeof(unsigned int))
        ((unsigned int *)plan)[threadIdx.x] = 0u;
    __shared__ double red[256];
    __shared__ float mm[2][256];
    double acc = 0.0;
    float st = 0.f;
    T lo = (T)__builtin_inf(), hi = -(T)__builtin_inf();
    const bool last = (threadIdx.x & (WAVE - 1)) == WAVE - 1;
    auto step = [&](int j, T v) {
        const float d = (float)(__shfl_down(v, 1, WAVE) - v);
        if (!last && j + 1 < mn && (j + 1) % ncol) st = fmaf(d, d, st);
    };
    if (k < dim) {
        // 8 loads in flight, added in index order
        int j = threadIdx.x;
        for (; j + 7 * 256 < mn; j += 8 * 256) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = w[(int64_t)(j + u * 256) * dim + k];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                acc += (double)v[u];
                step(j + u * 256, v[u]);
                lo = fmin(lo, v[u]);
                hi = fmax(hi, v[u]);
            }
        }
        for (; j < mn; j += 256) {
            const T v = w[(int64_t)j * dim + k];
            acc += (double)v;
            step(j, v);
            lo = fmin(lo, v);
            hi = fmax(hi, v);
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    const float c = (float)(red[0] / (double)mn);
    __shared__ float steps[4];
    for (int o = WAVE / 2; o > 0; o >>= 1) st += __shfl_xor(st, o, WAVE);
    if (threadIdx.x % WAVE == 0) steps[threadIdx.x / WAVE] = st;
    // the centred extremes: subtraction and rounding are monotonic
    mm[0][threadIdx.x] = k < dim && lo <= hi ? fabsf(centred(lo, c)) : 0.f;
    mm[1][threadIdx.x] = k < dim && lo <= hi ? fabsf(centred(hi, c)) : 0.f;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
            for (int q = 0; q < 2; q++) mm[q][threadIdx.x] = fmaxf(mm[q][threadIdx.x], mm[q][threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        plan->step2[k] = steps[0] + steps[1] + steps[2] + steps[3];
        centre[k] = k < dim ? c : 0.f;
        // dimension k is direction t = 8 (k / 16) + k % 8 of half (k / 8) % 2
        const int at = (k / 8 % 2) * (dpad / 2) + 8 * (k / 16) + k % 8;
        plan->wmax[at] = __builtin_bit_cast(unsigned int, fmaxf(mm[0][0], mm[1][0]));
    }
}

// The rotation: an orthonormal basis of the row space, its leading directions close to the map's principal
// ones. One workgroup: FP64 second moments C of up to basis_rows centred neurons (spread over the map by a
// golden-ratio sequence, which no row or column of the map stays in step with), then a Householder
// factorisation of C with column pivoting in FP64, which applies every reflection to the identity too. Any
// orthonormal basis gives correct bounds (the maxima are measured afterwards, the departure from orthonormality
// here). On trained maps the bound comes within a quarter of the eigenvectors'; with the neurons themselves as
// pivots it is half as large again, and FP32 moments lose the directions below 3e-4 of the first.
// Four lanes hold a column, a quarter of its values each. Latency bound: a serial chain of up to dpad steps of one
// barrier each: 16, 31 and 84 us at
// D = 16, 20 and 40 (one wave alone, a lane per column in LDS: 27, 60 and 182 us).
template <int DP>
constexpr int basis_rows() { return DP <= 32 ? 256 : 128; }
constexpr int BASIS_NT = 512;

// Sum over the four lanes of a vector, in each of them.
__device__ __forceinline__ double quad_sum(double v)
{
    auto dpp = [](double x, auto ctrl) {
        const uint64_t u = __builtin_bit_cast(uint64_t, x);
        const int lo = (int)(unsigned)u, hi = (int)(unsigned)(u >> 32);
        const unsigned a = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, decltype(ctrl)::value, 0xF, 0xF, true);
        const unsigned b = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, decltype(ctrl)::value, 0xF, 0xF, true);
        return __builtin_bit_cast(double, ((uint64_t)b << 32) | a);
    };
    v += dpp(v, std::integral_constant<int, 0xB1>{});  // quad_perm 1,0,3,2
    v += dpp(v, std::integral_constant<int, 0x4E>{});  // quad_perm 2,3,0,1
    return v;
}

template <int DP, class T>
__global__ __launch_bounds__(BASIS_NT) void prep_basis_kernel(const T *__restrict__ w, int mn, int dim,
                                                              const float *__restrict__ centre,
                                                              double *__restrict__ basis, float *__restrict__ rot,
                                                              BmuPlan *__restrict__ plan)
{
    constexpr int NR = basis_rows<DP>();
    constexpr int LD = DP + 1, LR = DP + 4;
    constexpr int QUADS = DP * DP / 4;          // (i, 4 k) groups of C
    constexpr int PARTS = BASIS_NT / QUADS > 0 ? BASIS_NT / QUADS : 1;  // row parts
    static_assert(QUADS * PARTS % BASIS_NT == 0, "whole groups of four per thread");
    constexpr int R = DP / 4;             // values per lane
    constexpr int NCW = 4 * DP / WAVE;    // waves of C's columns; the identity's follow
    static_assert(2 * NCW * WAVE <= BASIS_NT, "a column per four threads");
    // first the sampled rows, then the moments' parts, then the product of the reflections (rows: directions)
    constexpr size_t ROWS_B = sizeof(float) * NR * LR, PARTS_B = sizeof(double) * PARTS * DP * DP, Q_B = sizeof(double) * DP * LD;
    constexpr size_t LDS_B = ROWS_B > PARTS_B ? (ROWS_B > Q_B ? ROWS_B : Q_B) : (PARTS_B > Q_B ? PARTS_B : Q_B);
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDS_B];
    float *rows = (float *)lds;
    double *parts = (double *)lds, *Q = (double *)lds;
    __shared__ __attribute__((aligned(16))) double vb[2][NCW][DP];  // each wave's candidate
    __shared__ float nb[2][NCW];                                    // and its squared length
    __shared__ float red[BASIS_NT / WAVE];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE, vec = tid / 4, l = tid & 3;
    // scaled to about one, so the moments and their squares stay in range
    float big = lane < DP ? __builtin_bit_cast(float, plan->wmax[lane]) : 0.f;
    for (int o = WAVE / 2; o > 0; o >>= 1) big = fmaxf(big, __shfl_xor(big, o, WAVE));
    const float sc = big > 0.f && big < __builtin_inff() ? exp2i(min(126, max(-126, -expo(big)))) : 1.f;
    const int nr = min(mn, NR);
#pragma unroll 8
    for (int e = tid; e < NR * DP; e += BASIS_NT) {
        const int r = e / DP, k = e % DP;
        const int j = mn <= NR ? min(r, mn - 1) : (int)(((uint64_t)((unsigned)r * 2654435769u) * (unsigned)mn) >> 32);
        const float v = r < nr && k < dim ? centred(w[(int64_t)j * dim + k], centre[k]) * sc : 0.f;
        rows[r * LR + k] = __builtin_isfinite(v) ? v : 0.f;
    }
    __syncthreads();
    if (tid < F16_MAX_DIM) plan->wmax[tid] = 0u;  // the maxima of the rotated directions follow
    constexpr int PER = QUADS * PARTS / BASIS_NT;
    double c[PER][4];
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int at = tid + u * BASIS_NT, g = at % QUADS, part = at / QUADS, i = g / (DP / 4), k = 4 * (g % (DP / 4));
#pragma unroll
        for (int e = 0; e < 4; e++) c[u][e] = 0.0;
#pragma unroll 8
        for (int r = part * (NR / PARTS); r < (part + 1) * (NR / PARTS); r++) {
            const double a = (double)rows[r * LR + i];
            const f32x4 b = *(const f32x4 *)&rows[r * LR + k];
#pragma unroll
            for (int e = 0; e < 4; e++) c[u][e] = fma(a, (double)b[e], c[u][e]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) parts[4 * (tid + u * BASIS_NT) + e] = c[u][e];
    __syncthreads();
    const bool isc = wave < NCW, on = wave < 2 * NCW;  // uniform over the wave
    double x[R];
    float nrm = 0.f;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int k = l * R + r;
        x[r] = 0.0;
        if (isc) {
            for (int q = 0; q < PARTS; q++) x[r] += parts[q * DP * DP + k * DP + vec];
        } else if (on) {
            x[r] = vec - DP == k ? 1.0 : 0.0;
        }
    }
    auto length2 = [&]() {
        double m = 0.0;
#pragma unroll
        for (int r = 0; r < R; r++) m = fma(x[r], x[r], m);
        nrm = (float)quad_sum(m);
    };
    length2();
    __syncthreads();  // the moments have been read: Q takes their place
    const int steps = min(dim, DP - 1);
    float floor2 = 0.f;
    int i = 0;
    for (; i < steps; i++) {
        const int buf = i & 1;
        if (isc) {
            float m = half_max(nrm), ma, mb;
            pair32(m, ma, mb);
            m = fmaxf(ma, mb);
            const unsigned long long at_max = __builtin_amdgcn_ballot_w64(nrm == m);
            const int top = at_max ? __builtin_ctzll(at_max) & ~3 : 0;
            if ((lane & ~3) == top) {
#pragma unroll
                for (int r = 0; r < R; r++) vb[buf][wave][l * R + r] = x[r];
                if (l == 0) nb[buf][wave] = m;
            }
        }
        __syncthreads();  // two buffers: the next step's candidates are written while these are read
        float best = nb[buf][0];
        int s = 0;
#pragma unroll
        for (int q = 1; q < NCW; q++) {
            const float m = nb[buf][q];
            if (m > best) { best = m; s = q; }
        }
        // uniform: nothing left to the rounding of FP64, the rest of the basis stays as it is
        if (!(best > floor2 && best < __builtin_inff())) break;
        if (i == 0) floor2 = 1e-29f * best;
        if (!on) continue;
        s = __builtin_amdgcn_readfirstlane(s);
        // v = the candidate (zero before value i), its value i moved away from zero by its length
        const double head = vb[buf][s][i];
        const int own = i - l * R;  // value i among this lane's
        double v[R], d = 0.0, tail = 0.0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            v[r] = vb[buf][s][l * R + r];
            if (r != own) tail = fma(v[r], v[r], tail);
        }
        tail = quad_sum(tail);
        const double len = sqrt(fma(head, head, tail)), v0 = head + (head >= 0.0 ? len : -len);
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r == own) v[r] = v0;
            d = fma(v[r], x[r], d);
        }
        const double f = -2.0 * quad_sum(d) / fma(v0, v0, tail);
#pragma unroll
        for (int r = 0; r < R; r++) {
            x[r] = fma(f, v[r], x[r]);
            if (r == own) {
                // final: a row of the product; of C's columns the rest alone is needed
                if (!isc) Q[i * LD + vec - DP] = x[r];
                else x[r] = 0.0;
            }
        }
        if (isc) length2();
    }
    if (on && !isc)
#pragma unroll
        for (int r = 0; r < R; r++)
            if (l * R + r >= i) Q[(l * R + r) * LD + vec - DP] = x[r];
    __syncthreads();
    // the basis as used: rounded to FP32, so products with FP32 rows are exact in FP64. Direction i is
    // t = i / 2 of half i % 2, row half * DP/2 + t.
    for (int e = tid; e < DP * DP; e += BASIS_NT) {
        const int i = e / DP, k = e % DP;
        double q = (double)(float)Q[i * LD + k];
        if (!__builtin_isfinite(q)) q = i == k ? 1.0 : 0.0;
        Q[i * LD + k] = q;
        basis[(i % 2 * (DP / 2) + i / 2) * DP + k] = q;
    }
    __syncthreads();
    constexpr int NQ = (DP / 2 + 15) / 16;
    for (int e = tid; e < (DP / 16) * NQ * WAVE * 8; e += BASIS_NT) {
        // MFMA 32x32x2 A operand q of step kc*8 + e8: lane (row, half) holds K index kc*16 + 8*half + e8
        const int e8 = e % 8, l = e / 8 % WAVE, q = e / (8 * WAVE) % NQ, kc = e / (8 * WAVE * NQ);
        const int r = l & 31, h = (r >> 2) & 1, t = 16 * q + 4 * (r >> 3) + (r & 3), i = 2 * t + h;
        rot[e] = i < DP ? (float)Q[i * LD + kc * 16 + 8 * (l >> 5) + e8] : 0.f;
    }
    float dd = 0.f;
    for (int e = tid; e < DP * DP; e += BASIS_NT) {
        const int a = e / DP, b = e % DP;
        double g = a == b ? -1.0 : 0.0;
#pragma unroll 8
        for (int i = 0; i < DP; i++) g = fma(Q[i * LD + a], Q[i * LD + b], g);
        dd = fmaf((float)g, (float)g, dd);
    }
    for (int o = WAVE / 2; o > 0; o >>= 1) dd += __shfl_xor(dd, o, WAVE);
    if (lane == 0) red[tid / WAVE] = dd;
    __syncthreads();
    if (tid == 0) {
        float f = 0.f;
        for (int v = 0; v < BASIS_NT / WAVE; v++) f += red[v];
        plan->defect = sqrtf(f) * 1.01f;
    }
}

// Raw rows of the slot-ordered copy, the centred rows rotated in FP64 (kept as FP32), their norms, and the maxima
// per direction. 16 slots per workgroup, 16 threads a slot with every 16th direction each: a map has too few
// neurons for a thread per slot to fill the chip (one wave per 64 slots took 73 us at 1,024 neurons of 40 dims).
constexpr int ROT_SLOTS = 16, ROT_NT = 256;
template <int DP, class T>
__global__ __launch_bounds__(ROT_NT) void prep_rotate_kernel(const T *__restrict__ w, int mn, int dim, int pblk,
                                                             const float *__restrict__ centre,
                                                             const double *__restrict__ basis,
                                                             const int *__restrict__ perm, T *__restrict__ wslot,
                                                             float *__restrict__ wrot, double *__restrict__ norms,
                                                             BmuPlan *__restrict__ plan)
{
    __shared__ double bs[DP][DP + 1];
    __shared__ double v[ROT_SLOTS][DP + 1];
    __shared__ unsigned int mx[DP];
    const int tid = threadIdx.x;
    const int p0 = blockIdx.x * ROT_SLOTS;  // whole blocks of 32 slots: always in range
    for (int e = tid; e < DP * DP; e += ROT_NT) bs[e / DP][e % DP] = basis[e];
    for (int e = tid; e < ROT_SLOTS * DP; e += ROT_NT) {
        const int p = p0 + e / DP, d = e % DP, j = perm[p];
        const T raw = (j >= 0 && d < dim) ? w[(int64_t)j * dim + d] : (T)0;
        wslot[(int64_t)p * DP + d] = raw;
        v[e / DP][d] = (j >= 0 && d < dim) ? (double)centred(raw, centre[d]) : 0.0;
    }
    if (tid < DP) mx[tid] = 0u;
    __syncthreads();
    const int sl = tid / 16, g = tid % 16;
    double r[DP / 16];
#pragma unroll
    for (int u = 0; u < DP / 16; u++) r[u] = 0.0;
#pragma unroll 8
    for (int k = 0; k < DP; k++) {
        const double x = v[sl][k];
#pragma unroll
        for (int u = 0; u < DP / 16; u++) r[u] = fma(bs[g + 16 * u][k], x, r[u]);
    }
#pragma unroll
    for (int u = 0; u < DP / 16; u++) {
        const int i = g + 16 * u;
        const float f = (float)r[u];
        wrot[(int64_t)(p0 + sl) * DP + i] = f;
        if (fabsf(f) > 0.f) atomicMax(&mx[i], __builtin_bit_cast(unsigned int, fabsf(f)));
    }
    if (tid < ROT_SLOTS) {
        double nrm = 0.0;
        for (int k = 0; k < DP; k++) nrm = fma(v[tid][k], v[tid][k], nrm);
        norms[p0 + tid] = perm[p0 + tid] >= 0 ? nrm : __builtin_inf();
    }
    __syncthreads();
    if (tid < DP && mx[tid]) atomicMax(&plan->wmax[tid], mx[tid]);
}

// One neuron's slots of one lane half (values -2 w'' pieces; the norm piece last), and the squares of what the
// plan leaves out.
template <int NK, int HD, int Q3>
__device__ __forceinline__ void neuron_slots(const float (&om)[HD], _Float16 norm, f16x8 (&a)[NK], float &lt, float &nt,
                                             float &rt, float &ns, float &rs, float &nd)
{
    constexpr int Q1 = F16Split<NK, HD>::q1(Q3);
#pragma unroll
    for (int c = 0; c < NK; c++)
#pragma unroll
        for (int e = 0; e < 8; e++) a[c][e] = (_Float16)0.f;
#pragma unroll
    for (int t = 0; t < HD; t++) {
        const float v = om[t];
        const _Float16 h = (_Float16)v;
        const float r1 = v - (float)h;
        if (t < Q3) {
            const _Float16 l = (_Float16)r1;
            const float lf = (float)l, r2 = r1 - lf;
            lt = fmaf(lf, lf, lt);
            nt = fmaf(v, v, nt);
            rt = fmaf(r2, r2, rt);
            // -2 x the pieces is exact: an exponent step
            const _Float16 h2 = (_Float16)(-2.f * (float)h), l2 = (_Float16)(-2.f * lf);
            a[(3 * t) / 8][(3 * t) % 8] = h2;
            a[(3 * t + 1) / 8][(3 * t + 1) % 8] = h2;
            a[(3 * t + 2) / 8][(3 * t + 2) % 8] = l2;
        } else if (t < Q3 + Q1) {
            constexpr int S0 = 2 * Q3;
            ns = fmaf(v, v, ns);
            rs = fmaf(r1, r1, rs);
            a[(S0 + t) / 8][(S0 + t) % 8] = (_Float16)(-2.f * (float)h);
        } else {
            nd = fmaf(v, v, nd);
        }
    }
    a[NK - 1][7] = norm;
}
template <int NK, int HD, int Q3 = F16Split<NK, HD>::QMIN>
__device__ __forceinline__ void neuron_slots_q(int q3, const float (&om)[HD], _Float16 norm, f16x8 (&a)[NK], float &lt,
                                               float &nt, float &rt, float &ns, float &rs, float &nd)
{
    if constexpr (Q3 < F16Split<NK, HD>::QMAX) {
        if (q3 != Q3) return neuron_slots_q<NK, HD, Q3 + 1>(q3, om, norm, a, lt, nt, rt, ns, rs, nd);
    }
    neuron_slots<NK, HD, Q3>(om, norm, a, lt, nt, rt, ns, rs, nd);
}

// Least bound (relative to the map) over the splits of NK slices, from the maxima per direction (LDS): high parts
// alone are off by about 2^-12 of a direction's extent, directions left out by all of it.
template <int NK, int HD>
__device__ __forceinline__ float plan_bound(const float *wm, int &q3)
{
    using S = F16Split<NK, HD>;
    float least = __builtin_inff();
    for (int c = S::QMIN; c <= S::QMAX; c++) {
        const int held = c + S::q1(c);
        float et = 0.f, es = 0.f, ed = 0.f;
        for (int t = 0; t < HD; t++) {
            const float v = wm[t] * wm[t] + wm[HD + t] * wm[HD + t];
            et += t < c ? v : 0.f;
            es += t >= c && t < held ? v : 0.f;
            ed += t >= held ? v : 0.f;
        }
        const float e = sqrtf(ed) + 2.9e-4f * sqrtf(es) + 1.5e-7f * sqrtf(et);
        if (e < least) { least = e; q3 = c; }
    }
    return least;
}

// One thread per permuted slot: the plan from the maxima (the same in every workgroup), then the FP16 fragments
// and the maxima of what they leave out. ROT: rows of the rotation (wrot, norms); else the centred weights
// themselves, whose raw rows it also copies in slot order.
template <int DP, bool ROT, class T>
__global__ __launch_bounds__(WAVE) void prep_frag_kernel(const T *__restrict__ w, int mn, int dim, int pblk,
                                                         const float *__restrict__ centre, const int *__restrict__ perm,
                                                         T *__restrict__ wslot, const float *__restrict__ wrot,
                                                         const double *__restrict__ norms, f16x8 *__restrict__ frag,
                                                         int nk_max, BmuPlan *__restrict__ plan)
{
    constexpr int HD = DP / 2;
    __shared__ float wm[DP];
    const int lane = threadIdx.x;
    const int p = blockIdx.x * WAVE + lane;
    if (lane < DP) wm[lane] = __builtin_bit_cast(float, plan->wmax[lane]);
    __syncthreads();
    float big = lane < DP ? wm[lane] : 0.f, all = big * big, gap = lane < DP ? plan->step2[lane] : 0.f;
    for (int o = WAVE / 2; o > 0; o >>= 1) {
        big = fmaxf(big, __shfl_xor(big, o, WAVE));
        all += __shfl_xor(all, o, WAVE);
        gap += __shfl_xor(gap, o, WAVE);
    }
    // the largest value to [2^5, 2^6): norms / 16 stay below 2^15
    const int k = big > 0.f ? min(100, max(-100, 5 - expo(big))) : 0;
    // The fewest slices whose bound is small against the map or against the squared distance of neighbouring
    // neurons, or close to what more of them give. A slice costs about a quarter of the block loop: the first
    // epoch of a training on 64x64 at D = 16, from random weights far apart, takes 4.9 ms with two and 6.2 ms with
    // three. A wide window on a smooth map, dozens of candidates: errors of 140,000 rows on 100x90, 506 and 281 us. The
    // sixth lies between trained maps where two slices are better (winners of 1,000,003 rows on 64x64 at D = 13, a
    // ninth: 405 and 470 us) and where three are (errors of 1,000,000 rows on 40x50 at D = 32, two fifths: 790 and 570).
    int nk = 2, q3 = 0;
    float e = plan_bound<2, HD>(wm, q3);
    const float fine = fmaxf(3e-5f * sqrtf(all), gap / (float)mn / (6.f * sqrtf(all)));
    {
        int q = 0;
        const float e3 = plan_bound<3, HD>(wm, q);
        if (e > fine && e > 2.f * e3) { nk = 3; q3 = q; e = e3; }
    }
    if constexpr (DP > 32) {
        int q = 0;
        const float e5 = plan_bound<5, HD>(wm, q);
        if (nk_max >= 5 && e > fine && e > 2.f * e5) { nk = 5; q3 = q; e = e5; }
    }
    float nw = 0.f, lt = 0.f, nt = 0.f, rt = 0.f, ns = 0.f, rs = 0.f, nd = 0.f, rn = 0.f;
    if (p < pblk * 32) {
        const float sc = exp2i(k);
        float om[2][HD];
        double nrm;
        if constexpr (ROT) {
            nrm = norms[p];
#pragma unroll
            for (int i = 0; i < DP; i++) om[i / HD][i % HD] = wrot[(int64_t)p * DP + i];
        } else {
            const int j = perm[p];
            nrm = j >= 0 ? 0.0 : __builtin_inf();
#pragma unroll
            for (int d = 0; d < DP; d++) {
                const T raw = (j >= 0 && d < dim) ? w[(int64_t)j * dim + d] : (T)0;
                wslot[(int64_t)p * DP + d] = raw;
                const float v = (j >= 0 && d < dim) ? centred(raw, centre[d]) : 0.f;
                nrm = fma((double)v, (double)v, nrm);
                om[d / 8 % 2][8 * (d / 16) + d % 8] = v;
            }
        }
        const bool real = nrm < __builtin_inf();  // not padding (nor NaN)
        const double nu = nrm * ((double)sc * (double)sc) * 0.0625;
        const _Float16 nh = (_Float16)(float)nu;
        const double r1 = nu - (double)(float)nh;
        const _Float16 nl = real ? (_Float16)(float)r1 : (_Float16)0.f;
        if (real) {
            rn = 16.f * (float)fabs(r1 - (double)(float)nl) * (1.f + 2.f * U32);
            nw = (float)nrm * (1.f + 2.f * U32);
        }
        const int blk = p >> 5, row = p & 31;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int t = 0; t < HD; t++) om[h][t] = real ? om[h][t] * sc : 0.f;
            const _Float16 np = h == 0 ? nh : nl;
            auto put = [&](auto &a, int slices) {
#pragma unroll
                for (int c = 0; c < (int)(sizeof(a) / sizeof(a[0])); c++)
                    frag[((int64_t)blk * slices + c) * WAVE + row + 32 * h] = a[c];
            };
            if (nk == 2) {
                f16x8 a[2];
                neuron_slots_q<2, HD>(q3, om[h], np, a, lt, nt, rt, ns, rs, nd);
                put(a, 2);
            }
            if (nk == 3) {
                f16x8 a[3];
                neuron_slots_q<3, HD>(q3, om[h], np, a, lt, nt, rt, ns, rs, nd);
                put(a, 3);
            }
            if constexpr (DP > 32) {
                if (nk == 5) {
                    f16x8 a[5];
                    neuron_slots_q<5, HD>(q3, om[h], np, a, lt, nt, rt, ns, rs, nd);
                    put(a, 5);
                }
            }
        }
    }
    const float m[8] = {nw, lt, nt, rt, ns, rs, nd, rn};
    unsigned int *out[8] = {&plan->nw2, &plan->lt2, &plan->nt2, &plan->rt2, &plan->ns2, &plan->rs2, &plan->nd2, &plan->rn};
#pragma unroll
    for (int i = 0; i < 8; i++) {
        float v = m[i] * (1.f + 2.f * DP * U32);
        for (int o = WAVE / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, WAVE));
        if (lane == 0 && v > 0.f) atomicMax(out[i], __builtin_bit_cast(unsigned int, v));
    }
    if (p == 0) {
        float s1 = 0.f;
        for (int i = 0; i < DP; i++) s1 += wm[i];
        plan->s1 = s1 * (1.f + 2.f * DP * U32);
        plan->rotated = ROT ? 1 : 0;
        plan->nk = nk;
        plan->q3h = q3;
        plan->k = k;
    }
}

// Plain FP32 search: fragments and norms in natural order, one thread per neuron slot.
template <int DP>
__global__ __launch_bounds__(256) void prep_f32_kernel(const float *__restrict__ w, int mn, int dim, int nblk,
                                                       const float *__restrict__ centre, f32x4 *__restrict__ frag_f32,
                                                       float *__restrict__ norms_nat)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nblk * 32) return;
    const int blk = p >> 5, row = p & 31;
    const int j = p < mn ? p : -1;
    float v[DP];
    float nrm = 0.f;
#pragma unroll
    for (int d = 0; d < DP; d++) {
        v[d] = (j >= 0 && d < dim) ? __fsub_rn(w[(int64_t)j * dim + d], centre[d]) : 0.f;
        nrm = __fmaf_rn(v[d], v[d], nrm);
    }
    // MFMA 32x32x2 operand order: K step st = d/2 goes to lane row + 32*(d&1), element st&3
#pragma unroll
    for (int q = 0; q < DP / 8; q++) {
        const int64_t u = (((int64_t)blk * (DP / 8) + q) * 64 + row);
        frag_f32[u] = f32x4{v[8 * q], v[8 * q + 2], v[8 * q + 4], v[8 * q + 6]};
        frag_f32[u + 32] = f32x4{v[8 * q + 1], v[8 * q + 3], v[8 * q + 5], v[8 * q + 7]};
    }
    norms_nat[p] = j >= 0 ? nrm : __builtin_inff();
}

// Launch helpers -----------------------------------------------------------------------------------

int64_t exact_blocks(int64_t grid_items)
{
    int64_t blocks = (grid_items + 255) / 256;
    if (blocks < 1) blocks = 1;
    if (blocks > 65535 * 8) blocks = 65535 * 8;
    return blocks;
}

template <int DP>
void launch_exact(int mode, bool need_c2, hipStream_t st, const float *x, int64_t n, int dim, const int64_t *list,
                  const unsigned int *list_count, int64_t grid_items, const float *w, int mn, int default_index,
                  int32_t *c1, int32_t *c2, double *d1, float *xmax_part)
{
    const int64_t blocks = exact_blocks(grid_items);
    dim3 grid((unsigned)blocks), block(256);
#define SOM_EX(M, C)                                                                                            \
    hipLaunchKernelGGL((bmu_exact_kernel<DP, M, C>), grid, block, 0, st, x, n, dim, list, list_count, w, mn,  \
                       default_index, c1, c2, d1, xmax_part)
    if (mode == SOMHIP_RERANK_FP64) {
        if (need_c2) SOM_EX(SOMHIP_RERANK_FP64, true); else SOM_EX(SOMHIP_RERANK_FP64, false);
    } else {
        if (need_c2) SOM_EX(SOMHIP_RERANK_REF32, true); else SOM_EX(SOMHIP_RERANK_REF32, false);
    }
#undef SOM_EX
}

template <int DP>
void launch_exact64(bool need_c2, hipStream_t st, const double *x, int64_t n, int dim, const double *w, int mn,
                    int default_index, int32_t *c1, int32_t *c2, double *d1)
{
    dim3 grid((unsigned)exact_blocks(n)), block(256);
    if (need_c2)
        hipLaunchKernelGGL((bmu_exact_kernel<DP, SOMHIP_RERANK_FP64, true, double>), grid, block, 0, st, x, n, dim,
                           nullptr, nullptr, w, mn, default_index, c1, c2, d1, nullptr);
    else
        hipLaunchKernelGGL((bmu_exact_kernel<DP, SOMHIP_RERANK_FP64, false, double>), grid, block, 0, st, x, n, dim,
                           nullptr, nullptr, w, mn, default_index, c1, c2, d1, nullptr);
}

constexpr int G_FP32 = 2;
// 32-sample groups per wave of the FP32 kernel: one at D = 64, where two would spill
constexpr int fp32_groups(int dpad) { return dpad <= 32 ? G_FP32 : 1; }

__global__ void zero_u32_kernel(unsigned int *p) { *p = 0u; }

template <int DP>
void launch_fp32(hipStream_t st, somhip_model *M, const float *x, int64_t n, int default_index, int32_t *c1,
                 int32_t *c2, double *d1, float *xmax_part)
{
    constexpr int G = fp32_groups(DP);
    const int64_t per_block = (int64_t)BMU_WAVES * G * 32;
    const int64_t blocks = (n + per_block - 1) / per_block;
    hipLaunchKernelGGL((bmu_fp32_kernel<DP, G>), dim3((unsigned)blocks), dim3(BMU_WAVES * WAVE), 0, st, x, n,
                       M->dim, M->centre, (const f32x4 *)M->frag_f32, (const f32x4 *)M->norms_nat, M->nblk, M->mn,
                       default_index, c1, c2, d1, xmax_part);
}

}  // namespace

// ------------------------------------------------------------------------------------------------
// Internal entry points.
// ------------------------------------------------------------------------------------------------
BmuModelDev somhip_model_dev(const somhip_model *M)
{
    BmuModelDev d;
    d.frag = (const f16x8 *)M->frag_h;
    d.rot = M->rot;
    d.plan = M->plan;
    d.perm = M->perm;
    d.centre = M->centre;
    d.wslot = M->wslot;
    d.nblk = M->pblk;
    d.nblk_a = M->pblk_a;
    d.mn = M->mn;
    d.dim = M->dim;
    d.ncol = M->n;
    return d;
}

int somhip_launch_zero_u32(hipStream_t st, unsigned int *p)
{
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, st, p);
    SOM_HIP_TRY(hipGetLastError());
    return SOMHIP_OK;
}

// ------------------------------------------------------------------------------------------------
namespace {

template <int DP, class T>
int prepare_t(somhip_model *M, const T *w, bool rotated)
{
    hipStream_t st = M->ctx->stream;
    const int slots = M->pblk * 32;
    const dim3 grid((slots + WAVE - 1) / WAVE), block(WAVE);
    hipLaunchKernelGGL(prep_centre_kernel<T>, dim3(DP), dim3(256), 0, st, w, M->mn, M->n, M->dim, DP, M->centre, M->plan);
    if (rotated) {
        hipLaunchKernelGGL((prep_basis_kernel<DP, T>), dim3(1), dim3(BASIS_NT), 0, st, w, M->mn, M->dim, M->centre,
                           M->basis, M->rot, M->plan);
        hipLaunchKernelGGL((prep_rotate_kernel<DP, T>), dim3(slots / ROT_SLOTS), dim3(ROT_NT), 0, st, w, M->mn, M->dim, M->pblk, M->centre, M->basis,
                           M->perm, (T *)M->wslot, M->wrot, M->norms, M->plan);
        hipLaunchKernelGGL((prep_frag_kernel<DP, true, T>), grid, block, 0, st, w, M->mn, M->dim, M->pblk, M->centre,
                           M->perm, (T *)M->wslot, M->wrot, M->norms, (f16x8 *)M->frag_h, f16_nk_limit(M, true), M->plan);
    } else {
        hipLaunchKernelGGL((prep_frag_kernel<DP, false, T>), grid, block, 0, st, w, M->mn, M->dim, M->pblk, M->centre,
                           M->perm, (T *)M->wslot, M->wrot, M->norms, (f16x8 *)M->frag_h, f16_nk_limit(M, false), M->plan);
    }
    SOM_HIP_TRY(hipGetLastError());
    return SOMHIP_OK;
}

// Whether a search of n rows rotates: nearly always. It costs two launches after each change of the weights (20, 40
// and 75 us at up to 16, 32 and 64 dims), and saves the wider window of the data's own dimensions, which on trained maps
// fills the candidate lists, and at more than 16 dims K slices. Short searches of small maps do without.
bool rotate(const somhip_model *M, int64_t n)
{
    const int64_t pairs = M->kpad <= 32 ? 1 << 26 : 1 << 25;
    const int large = M->kpad <= 32 ? 6000 : 4000;
    return M->mn >= large || n >= pairs / M->mn;
}

}  // namespace

int somhip_prepare(somhip_model *M, int64_t n)
{
    const bool rotated = rotate(M, n);
    if (M->prepared >= (rotated ? 2 : 1)) return SOMHIP_OK;
    TimerScope ts(M->ctx, TK_PREP);
    int rc;
    if (M->f64)
        rc = M->kpad == 16   ? prepare_t<16>(M, M->w64, rotated)
             : M->kpad == 32 ? prepare_t<32>(M, M->w64, rotated)
                             : prepare_t<64>(M, M->w64, rotated);
    else
        rc = M->kpad == 16   ? prepare_t<16>(M, M->w, rotated)
             : M->kpad == 32 ? prepare_t<32>(M, M->w, rotated)
                             : prepare_t<64>(M, M->w, rotated);
    if (rc) return rc;
    M->prepared = rotated ? 2 : 1;
    return SOMHIP_OK;
}

int somhip_prepare_f32(somhip_model *M)
{
    if (M->prepared_f32) return SOMHIP_OK;
    TimerScope ts(M->ctx, TK_PREP);
    hipStream_t st = M->ctx->stream;
    const dim3 grid((M->nblk * 32 + 255) / 256), block(256);
    if (!M->prepared)  // else the centroid is there, and the plan that this kernel clears is in use (also by a server)
        hipLaunchKernelGGL(prep_centre_kernel<float>, dim3(M->kpad), dim3(256), 0, st, M->w, M->mn, M->n, M->dim, M->kpad,
                           M->centre, M->plan);
#define SOM_PREP(D)                                                                                           \
    hipLaunchKernelGGL(prep_f32_kernel<D>, grid, block, 0, st, M->w, M->mn, M->dim, M->nblk, M->centre,       \
                       (f32x4 *)M->frag_f32, M->norms_nat)
    if (M->dpad == 16) SOM_PREP(16);
    else if (M->dpad == 32) SOM_PREP(32);
    else SOM_PREP(64);
#undef SOM_PREP
    SOM_HIP_TRY(hipGetLastError());
    M->prepared_f32 = true;
    return SOMHIP_OK;
}

// Workspace for the search's fallback list (grow-only, per context).
static int fb_workspace(somhip_ctx *C, int64_t n, int64_t **list, unsigned int **count)
{
    size_t need = sizeof(int64_t) * (size_t)(n > 0 ? n : 1) + 256;
    if (C->scratch_bytes < need) {
        if (C->scratch) SOM_HIP_TRY(hipFree(C->scratch));
        C->scratch = nullptr;
        C->scratch_bytes = 0;
        SOM_HIP_TRY(hipMalloc(&C->scratch, need));
        C->scratch_bytes = need;
    }
    *count = (unsigned int *)C->scratch;
    *list = (int64_t *)((char *)C->scratch + 256);
    return SOMHIP_OK;
}

int64_t somhip_bmu_xmax_rows(int precision, int dpad, int64_t n)
{
    if (n <= 0) return 0;
    if (precision == SOMHIP_PREC_EXACT) return exact_blocks(n) * 4;
    if (precision == SOMHIP_PREC_FP32) {
        const int64_t per_block = (int64_t)BMU_WAVES * fp32_groups(dpad) * 32;
        return (n + per_block - 1) / per_block * BMU_WAVES;
    }
    if (n <= SMALL_ROWS) return (n + NW_SMALL * 32 - 1) / (NW_SMALL * 32) * NW_SMALL;
    if (n <= MEDIUM_ROWS) return (n + NW_F16 * 32 - 1) / (NW_F16 * 32) * NW_F16;
    return (n + SOM_TILE_ROWS - 1) / SOM_TILE_ROWS * NW_F16;
}

int somhip_bmu_precision(const somhip_model *M, int precision)
{
    // Candidate slots are 16-bit in LDS (0xFFFF marks an empty entry). BF16_RERANK promises the exact
    // winners of its rerank arithmetic, which the exact kernel computes directly, so maps with more
    // slots run that kernel.
    if (precision == SOMHIP_PREC_BF16_RERANK && (int64_t)M->pblk * 32 >= 65536) return SOMHIP_PREC_EXACT;
    return precision;
}

namespace {

template <class T>
int search_f16(somhip_model *M, const T *x, int64_t n, int arithmetic, int need_c2, int default_index, int32_t *c1,
               int32_t *c2, double *d1, float *xmax_part, int64_t *fb_list, unsigned int *fb_count,
               const int32_t *prev_c1)
{
    int rc = somhip_prepare(M, n);
    if (rc) return rc;
    if (fb_list) {
        // caller's workspace: cleared by a kernel, so the call holds no memset node under graph capture
        if ((rc = somhip_launch_zero_u32(M->ctx->stream, fb_count))) return rc;
    } else {
        if ((rc = fb_workspace(M->ctx, n, &fb_list, &fb_count))) return rc;
        SOM_HIP_TRY(hipMemsetAsync(fb_count, 0, sizeof(unsigned int), M->ctx->stream));
    }
    if (M->kpad == 16)
        return somhip_search_f16<16, T>(M, x, n, arithmetic, need_c2, default_index, c1, c2, d1, xmax_part, fb_list, fb_count, prev_c1);
    if (M->kpad == 32)
        return somhip_search_f16<32, T>(M, x, n, arithmetic, need_c2, default_index, c1, c2, d1, xmax_part, fb_list, fb_count, prev_c1);
    return somhip_search_f16<64, T>(M, x, n, arithmetic, need_c2, default_index, c1, c2, d1, xmax_part, fb_list, fb_count, prev_c1);
}

}  // namespace

int somhip_launch_bmu(somhip_model *M, const float *x, int64_t n, int precision, int arithmetic, int need_c2,
                      int default_index, int32_t *c1, int32_t *c2, double *d1, float *xmax_part, int64_t *fb_list_ext,
                      unsigned int *fb_count_ext, const int32_t *prev_c1)
{
    if (n <= 0) return SOMHIP_OK;
    precision = somhip_bmu_precision(M, precision);
    hipStream_t st = M->ctx->stream;
    const int dp = M->dpad;
    if (precision == SOMHIP_PREC_EXACT) {
        TimerScope ts(M->ctx, TK_BMU_EXACT);
        switch (dp) {
            case 16: launch_exact<16>(arithmetic, need_c2, st, x, n, M->dim, nullptr, nullptr, n, M->w, M->mn, default_index, c1, c2, d1, xmax_part); break;
            case 32: launch_exact<32>(arithmetic, need_c2, st, x, n, M->dim, nullptr, nullptr, n, M->w, M->mn, default_index, c1, c2, d1, xmax_part); break;
            case 48: launch_exact<48>(arithmetic, need_c2, st, x, n, M->dim, nullptr, nullptr, n, M->w, M->mn, default_index, c1, c2, d1, xmax_part); break;
            case 64: launch_exact<64>(arithmetic, need_c2, st, x, n, M->dim, nullptr, nullptr, n, M->w, M->mn, default_index, c1, c2, d1, xmax_part); break;
            default: somhip_set_error("dim > 64 is not supported"); return SOMHIP_ERR_UNSUPPORTED;
        }
        SOM_HIP_TRY(hipGetLastError());
        return SOMHIP_OK;
    }
    if (dp > 64) {
        somhip_set_error("MFMA precisions support dim <= 64");
        return SOMHIP_ERR_UNSUPPORTED;
    }
    if (precision == SOMHIP_PREC_FP32) {
        const int rc = somhip_prepare_f32(M);
        if (rc) return rc;
        TimerScope ts(M->ctx, TK_BMU_FP32);
        if (dp == 16) launch_fp32<16>(st, M, x, n, default_index, c1, c2, d1, xmax_part);
        else if (dp == 32) launch_fp32<32>(st, M, x, n, default_index, c1, c2, d1, xmax_part);
        else launch_fp32<64>(st, M, x, n, default_index, c1, c2, d1, xmax_part);
        SOM_HIP_TRY(hipGetLastError());
        return SOMHIP_OK;
    }
    if (precision != SOMHIP_PREC_BF16_RERANK) {
        somhip_set_error("unknown precision");
        return SOMHIP_ERR_ARG;
    }
    return search_f16(M, x, n, arithmetic, need_c2, default_index, c1, c2, d1, xmax_part, fb_list_ext, fb_count_ext,
                      prev_c1);
}

int somhip_launch_bmu_f64(somhip_model *M, const double *x, int64_t n, int need_c2, int default_index, int32_t *c1,
                          int32_t *c2, double *d1)
{
    if (n <= 0) return SOMHIP_OK;
    if (somhip_bmu_precision(M, SOMHIP_PREC_BF16_RERANK) == SOMHIP_PREC_BF16_RERANK)
        return search_f16<double>(M, x, n, SOMHIP_RERANK_FP64, need_c2, default_index, c1, c2, d1, nullptr, nullptr,
                                  nullptr, nullptr);
    hipStream_t st = M->ctx->stream;
    TimerScope ts(M->ctx, TK_BMU_EXACT);
    const bool c2n = need_c2 != 0;
    switch ((M->dim + 15) / 16 * 16) {
        case 16: launch_exact64<16>(c2n, st, x, n, M->dim, M->w64, M->mn, default_index, c1, c2, d1); break;
        case 32: launch_exact64<32>(c2n, st, x, n, M->dim, M->w64, M->mn, default_index, c1, c2, d1); break;
        case 48: launch_exact64<48>(c2n, st, x, n, M->dim, M->w64, M->mn, default_index, c1, c2, d1); break;
        case 64: launch_exact64<64>(c2n, st, x, n, M->dim, M->w64, M->mn, default_index, c1, c2, d1); break;
        default: somhip_set_error("dim > 64 is not supported"); return SOMHIP_ERR_UNSUPPORTED;
    }
    SOM_HIP_TRY(hipGetLastError());
    return SOMHIP_OK;
}
