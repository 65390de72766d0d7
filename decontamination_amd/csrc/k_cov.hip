// Weighted covariance of a chunk of samples (Covariance.compute, decontamination/algo/covariance.py:
// _update_welford_cov_sums :30-84 and _finalize_welford_cov :90-119), the pass that initialises a
// SOM_PCA.
//
// The reference runs Welford's update sample by sample on one CPU thread. Here one chunk takes one
// HBM-bound streaming pass with fixed-order reductions (deterministic), after a look at a sample:
//   pass 1: sum w and sum w x over the valid rows of a sample spread over the chunk (short chunks: all rows), whose
//           mean is the shift;
//   pass 2: on d = x - shift, W = sum w, S = sum w d d^T and c = sum w d, from which the host forms
//           M2 = S - c c^T / W and the mean, shift + c / W.
// The correction cancels (shift - mean)^2 against S: where it is more than 1/64 of a column's variance, pass 2 runs
// again with the mean that it found as the shift, which is the corrected two-pass form.
// A row is valid when its weight is finite and > 0 and all its values are finite (the reference's
// rule). Chunks are merged on the host with Chan's update.
//
// Layout: a wave takes 4 rows at a time, lane l holding value (row l/16, column 16b + l%16) of each
// 16-column block b, so one wave load reads 4 consecutive rows of a 16-column block (256 contiguous
// bytes when dim = 16). That is also the operand layout of v_mfma_f64_16x16x4f64 for both A (16 x 4,
// A[i][k] in lane i + 16k) and B (4 x 16, B[k][j] in lane j + 16k), so the 16 x 16 tile
// S_bi,bj += (w d_bi)^T d_bj of 4 rows is one FP64 MFMA; its result sits in lane j + 16q, register
// r, as D[4r + q][j] (rows interleaved across the lane groups, unlike the FP32 16x16 forms).
#include "launch.hpp"

#include <algorithm>
#include <vector>

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int COV_NT = 256;   // threads per workgroup (4 waves)
constexpr int COV_UNROLL = 8; // row quads per wave per step (32 rows, loads in flight together)

template <typename T>
__device__ __forceinline__ bool finite_val(T v)
{
    return __builtin_isfinite(v);
}

// Issues the loads of this lane's values of row `row` (lane column j, blocks 0..NBLK-1) and of the
// row's weight; the tail row and columns beyond dim read a clamped in-bounds address instead.
template <typename T, int NBLK>
__device__ __forceinline__ void load_row(const T *x, const double *rho, int64_t row, int64_t r1, int dim, int j,
                                         T (&v)[NBLK], double &w)
{
    const int64_t rr = row < r1 ? row : r1 - 1;
    w = rho ? rho[rr] : 1.0;
#pragma unroll
    for (int b = 0; b < NBLK; b++) {
        const int col = 16 * b + j;
        v[b] = x[rr * dim + (col < dim ? col : dim - 1)];
    }
}

// The loaded row as FP64 values (0 beyond dim) and its weight, 0 when the row is past r1 or invalid
// (weight not finite or <= 0, or any of its values not finite). Every lane of the wave calls it.
template <typename T, int NBLK>
__device__ __forceinline__ double check_row(const T (&raw)[NBLK], double w, int64_t row, int64_t r1, int dim, int j,
                                            int k, double (&v)[NBLK])
{
    bool fin = true;
#pragma unroll
    for (int b = 0; b < NBLK; b++) {
        const bool in = 16 * b + j < dim;
        fin = fin && (!in || finite_val(raw[b]));
        v[b] = in ? (double)raw[b] : 0.0;
    }
    if (!(row < r1 && __builtin_isfinite(w) && w > 0.0)) w = 0.0;
    const unsigned long long bad = __ballot(!fin);
    if ((bad >> (16 * k)) & 0xFFFFull) w = 0.0;
    return w;
}

// pass 1: per-workgroup partials [sum w, sum w x_col (col < 16*NBLK)] over the first `take` rows of each range
template <typename T, int NBLK>
__global__ __launch_bounds__(COV_NT) void cov_pass1_kernel(const T *x, const double *rho, int64_t n, int dim,
                                                           int64_t rows_per_wg, int64_t take, double *part)
{
    constexpr int DP = 16 * NBLK;
    __shared__ double red[COV_NT / 64][DP + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane & 15, k = lane >> 4;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_wg;
    const int64_t r1 = min(n, r0 + min(rows_per_wg, take));
    double sw = 0.0, sx[NBLK];
#pragma unroll
    for (int b = 0; b < NBLK; b++) sx[b] = 0.0;
    for (int64_t q0 = r0 + 4 * wave; q0 < r1; q0 += 4 * 4 * COV_UNROLL) {
        T raw[COV_UNROLL][NBLK];
        double v[COV_UNROLL][NBLK], w[COV_UNROLL];
        // all loads of the step first, then the checks (their ballots wait for the data)
#pragma unroll
        for (int u = 0; u < COV_UNROLL; u++) load_row<T, NBLK>(x, rho, q0 + 16 * u + k, r1, dim, j, raw[u], w[u]);
#pragma unroll
        for (int u = 0; u < COV_UNROLL; u++) w[u] = check_row<T, NBLK>(raw[u], w[u], q0 + 16 * u + k, r1, dim, j, k, v[u]);
#pragma unroll
        for (int u = 0; u < COV_UNROLL; u++) {
            if (w[u] > 0.0) {
                sw += w[u];
#pragma unroll
                for (int b = 0; b < NBLK; b++) sx[b] += w[u] * v[u][b];
            }
        }
    }
    // lanes j, j+16, j+32, j+48 hold the four row phases of column j
#pragma unroll
    for (int b = 0; b < NBLK; b++) {
        sx[b] += __shfl_xor(sx[b], 16);
        sx[b] += __shfl_xor(sx[b], 32);
    }
    sw += __shfl_xor(sw, 16);
    sw += __shfl_xor(sw, 32);
    if (lane < 16) {
#pragma unroll
        for (int b = 0; b < NBLK; b++) red[wave][1 + 16 * b + j] = sx[b];
        if (lane == 0) red[wave][0] = sw;
    }
    __syncthreads();
    for (int e = threadIdx.x; e <= dim; e += COV_NT) {
        double s = 0.0;
        for (int wv = 0; wv < COV_NT / 64; wv++) s += red[wv][e];
        part[(int64_t)blockIdx.x * (dim + 1) + e] = s;
    }
}

// pass 2: per-workgroup partials [S tiles (T tiles x 256, D[i][j] at 16 i + j), c (16*NBLK), W].
// Bound by issue: an FP64 product and about ten FP64 instructions per 4 rows beside 2.6 TB/s of loads. A step of 8 quads
// whose rows are all valid, tested with one ballot, needs no zeroing: 351 us for 12.6 M weighted rows of 16 dims, 361 us
// with a ballot per quad. Reading all rows for the shift too took another 262 us, a sample of them 14 us.
template <typename T, int NBLK>
__global__ __launch_bounds__(COV_NT) void cov_pass2_kernel(const T *x, const double *rho, int64_t n, int dim,
                                                           int64_t rows_per_wg, const double *sums, double *part)
{
    constexpr int DP = 16 * NBLK;
    constexpr int NT = NBLK * (NBLK + 1) / 2;  // upper-triangle 16x16 tiles
    constexpr int OUT = NT * 256 + DP + 1;
    __shared__ double red[COV_NT / 64][OUT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane & 15, k = lane >> 4;
    const double W = sums[0];
    double sw = 0.0, mean[NBLK];
#pragma unroll
    for (int b = 0; b < NBLK; b++) {
        const int col = 16 * b + j;
        mean[b] = (col < dim && W > 0.0) ? sums[1 + col] / W : 0.0;
    }
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_wg;
    const int64_t r1 = min(n, r0 + rows_per_wg);
    f64x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f64x4{0.0, 0.0, 0.0, 0.0};
    double cs[NBLK];
#pragma unroll
    for (int b = 0; b < NBLK; b++) cs[b] = 0.0;
    for (int64_t q0 = r0 + 4 * wave; q0 < r1; q0 += 4 * 4 * COV_UNROLL) {
        T raw[COV_UNROLL][NBLK];
        double w[COV_UNROLL];
        // all loads of the step first, then the checks (their ballots wait for the data)
#pragma unroll
        for (int u = 0; u < COV_UNROLL; u++) load_row<T, NBLK>(x, rho, q0 + 16 * u + k, r1, dim, j, raw[u], w[u]);
        bool fine = true;  // columns past dim repeat the last one
#pragma unroll
        for (int u = 0; u < COV_UNROLL; u++) {
            if (rho) fine = fine && __builtin_isfinite(w[u]) && w[u] > 0.0;
#pragma unroll
            for (int b = 0; b < NBLK; b++) fine = fine && finite_val(raw[u][b]);
        }
        const bool all = q0 + 16 * (COV_UNROLL - 1) + 4 <= r1 && __ballot(!fine) == 0ull;  // uniform
        if (!all) {
            // invalid rows become rows of the shift with weight 0
#pragma unroll
            for (int u = 0; u < COV_UNROLL; u++) {
                double v[NBLK];
                w[u] = check_row<T, NBLK>(raw[u], w[u], q0 + 16 * u + k, r1, dim, j, k, v);
#pragma unroll
                for (int b = 0; b < NBLK; b++) raw[u][b] = w[u] > 0.0 ? raw[u][b] : (T)0;
            }
        }
#pragma unroll
        for (int u = 0; u < COV_UNROLL; u++) {
            double d[NBLK], wd[NBLK];
            sw += w[u];
#pragma unroll
            for (int b = 0; b < NBLK; b++) {
                // columns past dim: their tile entries are not read
                d[b] = (double)raw[u][b] - mean[b];
                wd[b] = w[u] * d[b];
                cs[b] += wd[b];
            }
            int t = 0;
#pragma unroll
            for (int bi = 0; bi < NBLK; bi++)
#pragma unroll
                for (int bj = bi; bj < NBLK; bj++, t++)
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wd[bi], d[bj], acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int b = 0; b < NBLK; b++) {
        cs[b] += __shfl_xor(cs[b], 16);
        cs[b] += __shfl_xor(cs[b], 32);
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) red[wave][t * 256 + 16 * (4 * r + k) + j] = acc[t][r];
    if (lane < 16)
#pragma unroll
        for (int b = 0; b < NBLK; b++) red[wave][NT * 256 + 16 * b + j] = cs[b];
    sw += __shfl_xor(sw, 16);
    sw += __shfl_xor(sw, 32);
    if (lane == 0) red[wave][OUT - 1] = sw;
    __syncthreads();
    for (int e = threadIdx.x; e < OUT; e += COV_NT) {
        double s = 0.0;
        for (int wv = 0; wv < COV_NT / 64; wv++) s += red[wv][e];
        part[(int64_t)blockIdx.x * OUT + e] = s;
    }
}

// out[e] = sum over p of part[p * width + e]: one workgroup per entry, fixed reduction order
__global__ __launch_bounds__(256) void cov_reduce_kernel(const double *part, int nparts, int width, double *out)
{
    __shared__ double red[4];
    const int e = blockIdx.x;
    double s = 0.0;
    for (int p = threadIdx.x; p < nparts; p += 256) s += part[(int64_t)p * width + e];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[e] = (red[0] + red[1]) + (red[2] + red[3]);
}

template <typename T, int NBLK>
int cov_launch(somhip_ctx *C, const T *x, const double *rho, int64_t n, int dim, double *out_host)
{
    constexpr int NT = NBLK * (NBLK + 1) / 2;
    constexpr int OUT = NT * 256 + 16 * NBLK + 1;
    hipStream_t st = C->stream;
    // one round of resident workgroups, each a contiguous run of whole row quads
    static int per_cu = 0;
    if (!per_cu) {
        int a = 0, b = 0;
        SOM_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, cov_pass1_kernel<T, NBLK>, COV_NT, 0));
        SOM_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, cov_pass2_kernel<T, NBLK>, COV_NT, 0));
        per_cu = std::max(1, std::min(a, b));
    }
    const int64_t groups = std::max<int64_t>(1, std::min<int64_t>((int64_t)C->num_cus * per_cu, (n + 1023) / 1024));
    const int64_t rows_per_wg = std::max<int64_t>(4, ((n + groups - 1) / groups + 3) / 4 * 4);
    const int G = (int)std::max<int64_t>(1, (n + rows_per_wg - 1) / rows_per_wg);
    Workspace &Wk = C->ws;
    int rc;
    if ((rc = Wk.part.ensure(sizeof(double) * (size_t)G * std::max(OUT, dim + 1))) ||
        (rc = Wk.maps.ensure(sizeof(double) * (size_t)(dim + 1 + OUT))))
        return rc;
    double *part = (double *)Wk.part.p;
    double *sums = (double *)Wk.maps.p;
    double *tiles = sums + dim + 1;
    // 128 rows of each of a thousand ranges place the shift within a few thousandths of a deviation
    const int64_t take = n <= 262144 ? rows_per_wg : 128;
    hipLaunchKernelGGL((cov_pass1_kernel<T, NBLK>), dim3(G), dim3(COV_NT), 0, st, x, rho, n, dim, rows_per_wg, take, part);
    SOM_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(cov_reduce_kernel, dim3(dim + 1), dim3(256), 0, st, part, G, dim + 1, sums);
    SOM_HIP_TRY(hipGetLastError());
    std::vector<double> h((size_t)dim + 1 + OUT);
    const double *S = h.data() + dim + 1;
    const double *c = S + NT * 256;
    double W = 0.0;
    for (int pass = 0;; pass++) {
        hipLaunchKernelGGL((cov_pass2_kernel<T, NBLK>), dim3(G), dim3(COV_NT), 0, st, x, rho, n, dim, rows_per_wg, sums,
                           part);
        SOM_HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL(cov_reduce_kernel, dim3(OUT), dim3(256), 0, st, part, G, OUT, tiles);
        SOM_HIP_TRY(hipGetLastError());
        SOM_HIP_TRY(hipMemcpyAsync(h.data(), sums, sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
        SOM_HIP_TRY(hipStreamSynchronize(st));
        W = c[16 * NBLK];
        // the shift's distance to the mean, against the deviation about the mean
        bool near = true;
        for (int a = 0; a < dim; a++) {
            const int t = (a / 16) * NBLK - (a / 16) * (a / 16 - 1) / 2;  // tile (a / 16, a / 16)
            const double off2 = c[a] * c[a] / W, var = S[t * 256 + 17 * (a % 16)] - off2;
            near = near && (off2 == 0.0 || off2 <= var / 64.0);
        }
        if (pass == 1 || near || !(W > 0.0)) break;
        // the mean found so far (sums over W, as the kernel divides them)
        std::vector<double> again((size_t)dim + 1);
        again[0] = W;
        for (int a = 0; a < dim; a++) again[1 + a] = ((h[0] > 0.0 ? h[1 + a] / h[0] : 0.0) + c[a] / W) * W;
        SOM_HIP_TRY(hipMemcpyAsync(sums, again.data(), sizeof(double) * again.size(), hipMemcpyHostToDevice, st));
        SOM_HIP_TRY(hipStreamSynchronize(st));
    }
    // W, the shift (the division pass 2 used), then M2 = S - c c^T / W and the mean, shift + c / W
    out_host[0] = W;
    double *mean = out_host + 1, *m2 = out_host + 1 + dim;
    for (int a = 0; a < dim; a++) mean[a] = W > 0.0 && h[0] > 0.0 ? h[1 + a] / h[0] : 0.0;
    for (int a = 0; a < dim; a++)
        for (int b = 0; b < dim; b++) {
            const int lo = std::min(a, b), hi = std::max(a, b);
            const int bi = lo / 16, bj = hi / 16;
            const int t = bi * NBLK - bi * (bi - 1) / 2 + (bj - bi);  // tile (bi, bj) of the upper triangle
            const double s = S[t * 256 + 16 * (lo % 16) + (hi % 16)];
            m2[a * dim + b] = W > 0.0 ? s - c[lo] * c[hi] / W : 0.0;
        }
    if (W > 0.0)
        for (int a = 0; a < dim; a++) mean[a] += c[a] / W;
    return SOMHIP_OK;
}

}  // namespace

extern "C" int somhip_covariance_chunk(somhip_ctx *C, const void *x, int x_is_f64, const double *rho, int64_t n,
                                       int dim, double *out_host)
{
    if (!C || n < 0 || dim < 1 || dim > 64 || !out_host || (n > 0 && !x)) {
        somhip_set_error("somhip_covariance_chunk: invalid arguments (1 <= dim <= 64)");
        return SOMHIP_ERR_ARG;
    }
    SOM_HIP_TRY(hipSetDevice(C->device));
#define SOM_COV(NB)                                                                                             \
    return x_is_f64 ? cov_launch<double, NB>(C, (const double *)x, rho, n, dim, out_host)                      \
                    : cov_launch<float, NB>(C, (const float *)x, rho, n, dim, out_host)
    switch ((dim + 15) / 16) {
        case 1: SOM_COV(1);
        case 2: SOM_COV(2);
        case 3: SOM_COV(3);
        default: SOM_COV(4);
    }
#undef SOM_COV
}
