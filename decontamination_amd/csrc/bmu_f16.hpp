// Device code of the 16-bit BMU search (k_f16_*.hip instantiate it per padded dimension and row type) and the
// helpers it shares with the other searches.
#pragma once

#include "common.hpp"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int WAVE = 64;
constexpr int BMU_WAVES = 4;                 // waves per workgroup of the MFMA kernels
constexpr float U32 = 5.9604644775390625e-8f;  // 2^-24

// Pointers in the global address space. The search body reads everything through these, so its accesses
// are global loads and stores also when its pointers come from descriptors in memory (the serving form),
// which the compiler would otherwise treat as generic and access with flat instructions.
template <class T>
using gptr = T __attribute__((address_space(1))) *;

// p itself, or p in the global address space (GC); kernels whose pointers are kernel arguments keep
// them as they are, since the compiler already knows where those point and assigns their registers best
template <bool GC, class T>
__device__ __forceinline__ auto aptr(T *p)
{
    if constexpr (GC) return (gptr<T>)p;
    else return p;
}
__device__ __forceinline__ const f32x4 *as_f32x4(const float *p) { return (const f32x4 *)p; }
__device__ __forceinline__ gptr<const f32x4> as_f32x4(gptr<const float> p) { return (gptr<const f32x4>)p; }
// 16-byte units at a float or double address
__device__ __forceinline__ const f32x4 *as_f32x4_any(const float *p) { return (const f32x4 *)p; }
__device__ __forceinline__ const f32x4 *as_f32x4_any(const double *p) { return (const f32x4 *)p; }
__device__ __forceinline__ gptr<const f32x4> as_f32x4_any(gptr<const float> p) { return (gptr<const f32x4>)p; }
__device__ __forceinline__ gptr<const f32x4> as_f32x4_any(gptr<const double> p) { return (gptr<const f32x4>)p; }

// Each lane needs its partner (lane ^ 32) value: both hold the same sample column.
__device__ __forceinline__ float xchg32(float v) { return __shfl_xor(v, 32, WAVE); }
__device__ __forceinline__ int xchg32i(int v) { return __shfl_xor(v, 32, WAVE); }
__device__ __forceinline__ double xchg32d(double v) { return __shfl_xor(v, 32, WAVE); }

// ------------------------------------------------------------------------------------------------
// Per-sample preparation shared by the MFMA kernels: load this lane's 8 dims (per 16-dim chunk) of
// the sample, centre them, and compute the quantities of the error bound.
// ------------------------------------------------------------------------------------------------
// Square root of a maximum held as float bits, rounded up a little.
__device__ __forceinline__ float root(unsigned int bits) { return __builtin_amdgcn_sqrtf(__builtin_bit_cast(float, bits)) * (1.f + 8.f * U32); }

// A row value centred: the difference in the row's type, rounded to FP32.
__device__ __forceinline__ float centred(float v, float c) { return __fsub_rn(v, c); }
__device__ __forceinline__ float centred(double v, float c) { return (float)__dsub_rn(v, (double)c); }

// 16 bytes of a row, at an address that is aligned to its values only
typedef f32x4 f32x4_row __attribute__((aligned(4)));
__device__ __forceinline__ f32x4 load_unit(const float *p) { return *(const f32x4_row *)p; }
__device__ __forceinline__ f32x4 load_unit(const double *p) { return *(const f32x4_row *)p; }
__device__ __forceinline__ f32x4 load_unit(gptr<const float> p) { return *(gptr<const f32x4_row>)p; }
__device__ __forceinline__ f32x4 load_unit(gptr<const double> p) { return *(gptr<const f32x4_row>)p; }

// N values from p[k0] on, zeros past p[dim]: whole 16-byte units in one load each, whatever the row's alignment (a
// load of one value per lane and instruction touches a cache line per lane and costs as much as a unit: at D = 40 the
// rows took two thirds of a short search), the last values of a row one by one.
template <class T, int N, class P>
__device__ __forceinline__ void load_values(P p, int k0, int dim, T (&v)[N])
{
    constexpr int V = 16 / (int)sizeof(T);
#pragma unroll
    for (int i = 0; i < N / V; i++) {
        const int k = k0 + V * i;
        if (k + V <= dim) {
            const f32x4 t = load_unit(p + k);
            if constexpr (V == 4) {
#pragma unroll
                for (int e = 0; e < V; e++) v[V * i + e] = t[e];
            } else {
                typedef double f64x2 __attribute__((ext_vector_type(2)));
                const f64x2 d = __builtin_bit_cast(f64x2, t);
                v[V * i] = d[0];
                v[V * i + 1] = d[1];
            }
        } else {
#pragma unroll
            for (int e = 0; e < V; e++) v[V * i + e] = k + e < dim ? p[k + e] : (T)0;
        }
    }
}

// Maximum over the 32 lanes of a half, in every lane of it: within rows of 16 by DPP, then across the two rows.
__device__ __forceinline__ float half_max(float v)
{
    auto dpp = [](float x, auto ctrl) {
        const int i = __builtin_bit_cast(int, x);
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, decltype(ctrl)::value, 0xF, 0xF, true));
    };
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0xB1>{}));   // quad_perm 1,0,3,2
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x4E>{}));   // quad_perm 2,3,0,1
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x141>{}));  // row_half_mirror
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x140>{}));  // row_mirror
    const unsigned int u = __builtin_bit_cast(unsigned int, v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned int)r[0]), __builtin_bit_cast(float, (unsigned int)r[1]));
}

// Per-wave max of |x| of 8 dimensions per half: lanes l and l^32 hold different dims, the 32 lanes of a half
// hold the same dims for different samples. Writes 16 floats of this wave's row (plain stores), or raises them.
template <int DP>
__device__ __forceinline__ void wave_dim_max(const float (&amax)[8], int kc, bool first, int lane, float *__restrict__ part)
{
    float m[8];
#pragma unroll
    for (int e = 0; e < 8; e++) m[e] = half_max(amax[e]);
    if ((lane & 31) == 0) {
        const int64_t wid = (int64_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
        float *at = part + wid * DP + kc * 16 + 8 * (lane >> 5);
#pragma unroll
        for (int e = 0; e < 8; e++) at[e] = first ? m[e] : fmaxf(m[e], at[e]);
    }
}

// ------------------------------------------------------------------------------------------------
// 16-bit search with a provable candidate window and exact rerank.
//
// What is computed: a_j = |w'_j|^2 - 2 x'.w'_j for every neuron j, approximately, on
// v_mfma_f32_32x32x16_f16, with a bound E on |a_j - exact| per sample; every neuron inside the window
// (second best) + 2E is recorded and reranked with the exact formula.
//
// The K slots. For longer searches x' and w' (centred on the weight centroid) are rotated onto an orthonormal
// basis whose first directions carry most of the map (a trained map is close to a two-dimensional sheet, so
// its extent falls by orders of magnitude within a dozen directions). Each half wave of the B operand holds
// 8 nk slots: its first q3h directions as three products (x_h w_h, x_l w_h, x_h w_l), the following ones as
// x_h w_h alone, the rest left out, and one slot for the norm (its high part in one half, its low part in the
// other, against a power of two). Two or three MFMAs per 32x32 block, mostly whatever the dimension, no norms
// to read and C = 0; a split of every dimension in three products takes 3, 6 and 12 at D = 16, 32 and 64.
// nk and q3h are chosen at preparation from the maxima of the rotated weights.
//
// What bounds it: power. MFMA and VALU work of different waves overlaps almost completely in cycles, but
// the clock falls with it (2.0 GHz with MFMA alone, 1.6-1.8 GHz with both), so each product and each VALU
// instruction in the block loop costs: measured per 32x32 block and SIMD with minima and thresholds but
// without recording, 67 ns at three products, 49 ns at two.
//
// A workgroup of NW waves (NW*G*32 samples, one tile) streams the 32-neuron blocks through LDS in
// chunks of CB blocks, double-buffered: while the waves compute chunk c from one buffer, every thread
// holds its share of chunk c+1 in registers and writes it to the other buffer after its last block of
// chunk c; one barrier per chunk.
// ------------------------------------------------------------------------------------------------
constexpr int NW_F16 = 8;       // waves per workgroup
constexpr int G_F16 = 2;        // 32-sample groups per wave
// Short searches take tiles of one group per wave: at 512 rows a tile, 131,072 rows make one workgroup per CU and
// fewer leave CUs idle. 4 waves a tile as long as all tiles fit the 256 CUs at once (three a CU), then 8 waves:
// errors of 98,000 rows on 64x64 at D = 16 take 119 us in tiles of 4 waves and 145 us in large ones; of 131,000 rows 173
// us in tiles of 4 waves, 130 us in tiles of 8 and 148 us in large ones. Longer ones keep the large tile, whose
// fragment traffic per row is a half: 500,000 rows take 319 us, 352 us in tiles of 8 waves and one group.
constexpr int NW_SMALL = 4;
constexpr int64_t SMALL_ROWS = 3 * 256 * NW_SMALL * 32;
constexpr int64_t MEDIUM_ROWS = 131072;
constexpr int FRAG_UNITS = 1024; // 16-byte units of A fragments per chunk buffer
static_assert(NW_F16 * G_F16 * 32 == SOM_TILE_ROWS, "tile rows must match the search workgroup");

// Candidate lists. Rows of up to 64 bytes: 20 per lane; a lane past that sends its sample to the fallback.
// Wider rows (more neurons closer than the window, on large smooth maps): 16 per lane plus a pool of 128
// shared by the 32-sample group for lanes past that, in the same LDS; only a full pool sends a sample
// to the fallback. The pool's spill test costs a few percent at D = 16, where lists rarely fill.
using lds_u16 = unsigned short __attribute__((address_space(3)));
// LDS byte address of an object in LDS
template <class T>
__device__ __forceinline__ unsigned int lds_addr(T *p)
{
    return (unsigned int)(size_t)(T __attribute__((address_space(3))) *)p;
}
constexpr unsigned short CAND_EMPTY = 0xFFFF;  // slots are < 65535 (checked at launch)

template <int KC>
struct F16Cand {
    static constexpr int CAPL = KC == 1 ? 20 : 16;  // own list per lane
    static constexpr int POOL = KC == 1 ? 0 : 128;  // shared entries per group
};

template <int KC, int NW, int G>
struct F16Smem {
    static constexpr int CAPL = F16Cand<KC>::CAPL;
    u32x4 frag[2][FRAG_UNITS];          // [buf][cb][slice][lane] 16 B
    unsigned short cand[NW][G][CAPL + 1][WAVE];  // last row: writes past a full list
    unsigned int pool[NW][G][F16Cand<KC>::POOL > 0 ? F16Cand<KC>::POOL : 1];  // (lane << 16) | slot
    unsigned short rows[NW][G][32];  // tile row of each (wave, group, column), reloaded for the rerank
};

// Both lanes' values of a pair (lane, lane ^ 32): a from the lower, b from the upper one, in every lane.
__device__ __forceinline__ void pair32(float v, float &a, float &b)
{
    const unsigned int u = __builtin_bit_cast(unsigned int, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    a = __builtin_bit_cast(float, (unsigned int)r[0]);
    b = __builtin_bit_cast(float, (unsigned int)r[1]);
}
__device__ __forceinline__ float sum32(float v)
{
    float a, b;
    pair32(v, a, b);
    return a + b;
}

// Split directions per half the plans choose from: as many as leave the other directions a slot each, up to
// as many as the slots hold.
template <int NK, int HD>
struct F16Split {
    static constexpr int SLOTS = 8 * NK - 1;                                  // without the norm's
    static constexpr int QMIN = SLOTS > HD ? ((SLOTS - HD) / 2 < 7 ? (SLOTS - HD) / 2 : 7) : 0;
    static constexpr int QMAX = SLOTS / 3 < (HD < 7 ? HD : 7) ? SLOTS / 3 : (HD < 7 ? HD : 7);
    // directions held by their high part alone
    static constexpr int q1(int q3) { return HD - q3 < SLOTS - 3 * q3 ? HD - q3 : SLOTS - 3 * q3; }
};

// A half's directions. A vector by value: of an array the variants of build_slots would be merged into one with
// run-time indices, through scratch memory.
template <int HD>
using HalfDirs = float __attribute__((ext_vector_type(HD)));

// One half wave's B slots from its scaled directions: the first Q3 as (high, low, high), then high parts; sums the
// squares of the remainders of the latter (rs).
template <int NK, int HD, int Q3>
__device__ __forceinline__ void build_slots(HalfDirs<HD> xi, float norm_mult, f16x8 (&b)[NK], float &rs)
{
    constexpr int Q1 = F16Split<NK, HD>::q1(Q3);
#pragma unroll
    for (int c = 0; c < NK; c++)
#pragma unroll
        for (int e = 0; e < 8; e++) b[c][e] = (_Float16)0.f;
#pragma unroll
    for (int t = 0; t < Q3; t++) {
        const _Float16 h = (_Float16)xi[t];
        const _Float16 l = (_Float16)(xi[t] - (float)h);
        b[(3 * t) / 8][(3 * t) % 8] = h;
        b[(3 * t + 1) / 8][(3 * t + 1) % 8] = l;
        b[(3 * t + 2) / 8][(3 * t + 2) % 8] = h;
    }
#pragma unroll
    for (int u = 0; u < Q1; u++) {
        constexpr int S0 = 3 * Q3;
        const float v = xi[Q3 + u];
        const _Float16 h = (_Float16)v;
        const float r1 = v - (float)h;
        rs = fmaf(r1, r1, rs);
        b[(S0 + u) / 8][(S0 + u) % 8] = h;
    }
    b[NK - 1][7] = (_Float16)norm_mult;
}
// The same for a plan's q3 (uniform).
template <int NK, int HD, int Q3 = F16Split<NK, HD>::QMIN>
__device__ __forceinline__ void build_slots_q(int q3, HalfDirs<HD> xi, float norm_mult, f16x8 (&b)[NK], float &rs)
{
    if constexpr (Q3 < F16Split<NK, HD>::QMAX) {
        if (q3 != Q3) return build_slots_q<NK, HD, Q3 + 1>(q3, xi, norm_mult, b, rs);
    }
    build_slots<NK, HD, Q3>(xi, norm_mult, b, rs);
}

// Power of two 2^e for |e| <= 126.
__device__ __forceinline__ float exp2i(int e) { return __builtin_bit_cast(float, (unsigned int)(e + 127) << 23); }
// Exponent of a positive finite float (floor(log2 v), subnormals as -127).
__device__ __forceinline__ int expo(float v) { return (int)((__builtin_bit_cast(unsigned int, v) >> 23) & 0xFFu) - 127; }

// 16 values at a 16-byte aligned address as vector loads (float or double; plain or global pointers).
template <class P, class T>
__device__ __forceinline__ void load16(P p, T (&v)[16])
{
    constexpr int V = 16 / (int)sizeof(T);
    const auto q = as_f32x4_any(p);
#pragma unroll
    for (int i = 0; i < 16 / V; i++) {
        const f32x4 t = q[i];
        if constexpr (sizeof(T) == 4) {
            v[4 * i] = t[0]; v[4 * i + 1] = t[1]; v[4 * i + 2] = t[2]; v[4 * i + 3] = t[3];
        } else {
            typedef double f64x2 __attribute__((ext_vector_type(2)));
            const f64x2 d = __builtin_bit_cast(f64x2, t);
            v[2 * i] = d[0]; v[2 * i + 1] = d[1];
        }
    }
}

// r + the squared distance of 16 more dimensions, in sqd_ref32 / sqd_fp64 / sqd_f64 order.
template <int MODE>
__device__ __forceinline__ double sqd_more(double r, const float (&a)[16], const float (&b)[16])
{
#pragma unroll
    for (int k = 0; k < 16; k++) {
        if constexpr (MODE == SOMHIP_RERANK_FP64) {
            const double d = __dsub_rn((double)a[k], (double)b[k]);
            r = __dadd_rn(r, __dmul_rn(d, d));
        } else {
            const float d = __fsub_rn(a[k], b[k]);
            r = __dadd_rn(r, (double)__fmul_rn(d, d));
        }
    }
    return r;
}
template <int MODE>
__device__ __forceinline__ double sqd_more(double r, const double (&a)[16], const double (&b)[16])
{
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const double d = __dsub_rn(a[k], b[k]);
        r = __dadd_rn(r, __dmul_rn(d, d));
    }
    return r;
}

template <int DP, int NK, int NW, int G, int MODE, bool NEED_C2, bool GC, class T>
__device__ __forceinline__ void bmu_f16_body(const BmuModelDev &Md, const T *__restrict__ x_in, int64_t n,
                                             int64_t tile_row0, int default_index, int32_t *__restrict__ c1_out,
                                             int32_t *__restrict__ c2_out, double *__restrict__ d1_out,
                                             int64_t *__restrict__ fb_list_out, unsigned int *__restrict__ fb_count,
                                             int64_t fb_tag, F16Smem<DP / 16, NW, G> &sm, float *__restrict__ xmax_part,
                                             const int32_t *__restrict__ prev_c1)
{
    constexpr int KC = DP / 16;
    constexpr int HD = DP / 2;               // directions per lane half
    constexpr int CB = FRAG_UNITS / (64 * NK);  // blocks per chunk
    constexpr int CU = CB * NK * 64;            // 16-byte units per chunk
    constexpr int CAPL = F16Cand<KC>::CAPL;
    constexpr int POOL = F16Cand<KC>::POOL;
    constexpr int NT = NW * WAVE;           // threads per workgroup
    constexpr int FU = (CU + NT - 1) / NT;  // fragment units per thread
    const auto centre = aptr<GC>(Md.centre);
    const auto rot = aptr<GC>(Md.rot);
    const auto plan = aptr<GC>(Md.plan);
    // loads through a plain vector type: a class type (uint4) cannot be copied from a global-address-space
    // reference in the host compilation pass
    const auto gfrag = aptr<GC>((const u32x4 *)Md.frag);
    const auto perm = aptr<GC>(Md.perm);
    const auto wslot = aptr<GC>((const T *)Md.wslot);
    const auto x = aptr<GC>(x_in);
    const auto c1 = aptr<GC>(c1_out);
    const auto c2 = aptr<GC>(c2_out);
    const auto d1 = aptr<GC>(d1_out);
    const auto fb_list = aptr<GC>(fb_list_out);
    const int nblk = Md.nblk, dim = Md.dim;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = tid / WAVE;
    const int col = lane & 31;
    const int khalf = lane >> 5;
    // rl[g]: the tile row this lane's group g works on. Without earlier BMUs, slot order; with them, the
    // tile's rows counting-sorted by the 8x8 map patch (in Morton order) of their earlier BMU, so a
    // 32-sample group tends to share its nearest neurons and records candidates in fewer blocks. The
    // scratch is the fragment buffer, which the first chunk load overwrites after a barrier.
    constexpr int TR = NW * G * 32;  // rows per tile
    constexpr int NBK = 65;               // 64 patches + rows past the end
    int rl[G];
#pragma unroll
    for (int g = 0; g < G; g++) rl[g] = wave * (G * 32) + g * 32 + col;
    if (prev_c1) {
        unsigned int *bcount = (unsigned int *)&sm.frag[0][0];
        unsigned int *bcur = bcount + NBK;
        unsigned short *ord = (unsigned short *)(bcur + NBK);
        for (int b = tid; b < NBK; b += NT) bcount[b] = 0u;
        __syncthreads();
        const int mcol = max(Md.ncol, 1), mrow = max(Md.mn / mcol, 1);
        int key[(TR + NT - 1) / NT];
#pragma unroll
        for (int u = 0; u < (TR + NT - 1) / NT; u++) {
            const int r = tid + u * NT;
            const int64_t row = tile_row0 + r;
            int k = NBK - 1;
            if (r < TR && row < n) {
                const int c = min(max((int)aptr<GC>(prev_c1)[row], 0), Md.mn - 1);
                const int a = c / mcol, b = c - a * mcol;
                const int pa = a * 8 / mrow, pb = b * 8 / mcol;
                k = 0;
#pragma unroll
                for (int bit = 0; bit < 3; bit++) k |= (((pa >> bit) & 1) << (2 * bit + 1)) | (((pb >> bit) & 1) << (2 * bit));
            }
            key[u] = k;
            if (r < TR) atomicAdd(&bcount[k], 1u);
        }
        __syncthreads();
        if (tid == 0) {
            unsigned int acc = 0u;
            for (int b = 0; b < NBK; b++) {
                bcur[b] = acc;
                acc += bcount[b];
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < (TR + NT - 1) / NT; u++) {
            const int r = tid + u * NT;
            if (r < TR) ord[atomicAdd(&bcur[key[u]], 1u)] = (unsigned short)r;
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G; g++) rl[g] = ord[rl[g]];
    }
    // kept in LDS rather than in registers across the block loop (both lanes of a column write the same)
#pragma unroll
    for (int g = 0; g < G; g++) sm.rows[wave][g][col] = (unsigned short)rl[g];
    unsigned short(*cw)[CAPL + 1][WAVE] = sm.cand[wave];
    const int nchunks = (nblk + CB - 1) / CB;
    const int64_t frag_units_total = (int64_t)nblk * NK * 64;

    // -inf as a value the compiler cannot see, so v_med3(m1, t, -inf) is not folded back into a minimum
    // that needs canonicalising moves in IEEE mode
    float neg_inf = -__builtin_inff();
    asm volatile("" : "+v"(neg_inf));
    f16x8 bx[G][NK];
    float E[G], K[G];
    // |x| maxima of the wave's groups; of wide rows, whose registers are short, each group writes its own
    constexpr bool AMAX_HELD = KC < 4 && sizeof(T) == 4;
    float amax[AMAX_HELD ? KC : 1][8];
#pragma unroll
    for (int kc = 0; kc < (AMAX_HELD ? KC : 1); kc++)
#pragma unroll
        for (int e = 0; e < 8; e++) amax[kc][e] = 0.f;
    {
        const int q3h = plan->q3h, kw = plan->k;
        const float NS = root(plan->ns2), RS = root(plan->rs2), ND = root(plan->nd2), LT = root(plan->lt2),
                    NT3 = root(plan->nt2), RT = root(plan->rt2);
        const float nw_s = root(plan->nw2) * exp2i(kw), rn = __builtin_bit_cast(float, plan->rn);
        const bool rotated = plan->rotated != 0;
        const float xfac = 2.02f * (RS + RT + ND) + (rotated ? 4.f * (DP + 1.f) * U32 * plan->s1 * exp2i(kw) : 0.f) +
                           (2.f * plan->defect + (4.f * 16 * NK + 20.f) * U32) * nw_s;
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int64_t s = tile_row0 + rl[g];
            float xc[KC][8];
            float kk = 0.f;
#pragma unroll
            for (int kc = 0; kc < KC; kc++) {
                const int k0 = kc * 16 + 8 * khalf;
                T v[8];
                load_values(x + s * dim, k0, s < n ? dim : 0, v);
                float av[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    xc[kc][e] = k0 + e < dim ? centred(v[e], centre[k0 + e]) : 0.f;
                    kk = fmaf(xc[kc][e], xc[kc][e], kk);
                    const float a = fabsf((float)v[e]);
                    av[e] = a < __builtin_inff() ? a : 0.f;
                    // FP64 rows take their scales from their FP64 maxima
                    if constexpr (AMAX_HELD) amax[kc][e] = fmaxf(amax[kc][e], av[e]);
                }
                if constexpr (!AMAX_HELD && sizeof(T) == 4)
                    if (xmax_part) wave_dim_max<DP>(av, kc, g == 0, lane, xmax_part);
            }
            kk = sum32(kk);
            // this half's directions: rotated on the FP32 matrix unit (row r of a 32-row A operand is the
            // half's direction 4 (r >> 3) + (r & 3) of half (r >> 2) & 1, so accumulator register t of a lane
            // is its half's direction t), or the lane's own dimensions
            constexpr int NR = (HD + 15) / 16;  // 32-row operands
            HalfDirs<HD> xi;
            if (rotated) {
                f32x16 xr[NR];
#pragma unroll
                for (int q = 0; q < NR; q++)
#pragma unroll
                    for (int r = 0; r < 16; r++) xr[q][r] = 0.f;
#pragma unroll
                for (int kc = 0; kc < KC; kc++) {
                    if (KC == 4 && kc * 16 >= dim) continue;  // uniform: zeros
#pragma unroll
                    for (int q = 0; q < NR; q++) {
                        const auto ra = as_f32x4(rot + ((int64_t)(kc * NR + q) * WAVE + lane) * 8);
                        const f32x4 r0 = ra[0], r1 = ra[1];
#pragma unroll
                        for (int e = 0; e < 8; e++)
                            xr[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(e < 4 ? r0[e & 3] : r1[e & 3], xc[kc][e],
                                                                         xr[q], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int t = 0; t < HD; t++) xi[t] = xr[t / 16][t % 16];
            } else {
#pragma unroll
                for (int t = 0; t < HD; t++) xi[t] = xc[t / 8][t % 8];
            }
            float xm = 0.f;
#pragma unroll
            for (int t = 0; t < HD; t++) xm = fmaxf(xm, fabsf(xi[t]));
            {
                float a, b;
                pair32(xm, a, b);
                xm = fmaxf(a, b);
            }
            // scale: the largest direction to [2^5, 2^6), so high parts and low parts stay normal numbers
            const int ex = min(max(5 - expo(xm), -100), min(100, 11 + kw));
            const int nm = 4 + ex - kw;  // exponent of the norm slots' multiplier
            const float sc = exp2i(ex);
#pragma unroll
            for (int t = 0; t < HD; t++) xi[t] *= sc;
            float rs = 0.f;
            build_slots_q<NK, HD>(q3h, xi, exp2i(max(nm, -14)), bx[g], rs);
            rs = __builtin_amdgcn_sqrtf(sum32(rs));
            // Error bound of a_j, in units of 2^-(kw + ex):
            //   products left out: 2 (|remainder of x| |w| + |x| |remainder of w| + |low x| |low w|) per class
            //   of directions, by Cauchy-Schwarz; directions left out 2 |x| |w|; both in xfac but for the
            //   remainders of x;
            //   rotation of x (FP32, each direction within 2 (D+1) 2^-24 |x|) and its departure from an
            //   orthonormal one; FP32 accumulation of 16 nk products, truncating (twice 2^-24 each), and the
            //   rounding of the rotated weights 2 (16 nk + 5) 2^-24 (|w|^2 + 2|x||w|); remainder of the norm;
            //   centring 4*2^-24 (|x|^2 + |w|^2).
            // 10% on top for the roundings of this arithmetic itself.
            //   Low parts of x are at most 2^-11 of it and its remainders 2^-22, but for 2^-25 a direction where
            //   they are subnormal; the remainders of directions without a low part are summed (rs).
            const float X = __builtin_amdgcn_sqrtf(kk) * (1.f + 4.f * U32) * sc;
            const float lt = 4.9e-4f * X + 2.4e-7f, rt = 2.5e-7f * X + 2.4e-7f;
            const float back = exp2i(min(max(ex - kw, -126), 126));
            const float ns = nw_s * nw_s * back;
            const float kks = X * X * exp2i(min(max(kw - ex, -126), 126));
            float e = 2.02f * (rs * NS + lt * LT + rt * NT3) + X * xfac + rn * back + (2.f * 16 * NK + 14.f) * U32 * ns + 4.f * U32 * kks;
            e = 1.1f * e + 1e-36f * exp2i(min(max(kw + ex, -126), 126));
            // a sample too far out for the norm slots, or not finite, records nothing and goes to the fallback
            E[g] = (nm >= -14 && e < 1e30f) ? e : __builtin_nanf("");
            K[g] = kks * (1.f + (DP + 2) * U32);
        }
    }
    if constexpr (AMAX_HELD)
        if (xmax_part)
#pragma unroll
            for (int kc = 0; kc < KC; kc++) wave_dim_max<DP>(amax[kc], kc, true, lane, xmax_part);

    // chunk streaming ---------------------------------------------------------------------------
    u32x4 pf[FU];
    auto load_chunk = [&](int c) {
        const int64_t fb = (int64_t)c * CU;
#pragma unroll
        for (int u = 0; u < FU; u++) {
            const int i = tid + u * NT;
            pf[u] = i < CU && fb + i < frag_units_total ? gfrag[fb + i] : u32x4{0u, 0u, 0u, 0u};
        }
    };
    auto store_chunk = [&](int buf) {
#pragma unroll
        for (int u = 0; u < FU; u++)
            if (CU % NT == 0 || tid + u * NT < CU) sm.frag[buf][tid + u * NT] = pf[u];
    };
    auto block_acc = [&](int g, const f16x8 (&a)[NK]) {
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
        for (int i = 0; i < NK; i++) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], bx[g][i], acc, 0, 0, 0);
        return acc;
    };
    auto block_min = [](const f32x16 &v) {
        float t = __builtin_inff();
#pragma unroll
        for (int r = 0; r < 16; r += 2) t = fminf(fminf(t, v[r]), v[r + 1]);
        return t;
    };
    // minima of the lane's four row quads (rows 4i..4i+3 are 4 consecutive neurons) and of the block;
    // chains seeded with +inf, as in block_min, compile to v_min3 without canonicalising the inputs
    auto quad_min = [](const f32x16 &v, float (&q)[4]) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            q[i] = fminf(fminf(fminf(fminf(__builtin_inff(), v[4 * i]), v[4 * i + 1]), v[4 * i + 2]), v[4 * i + 3]);
        return fminf(fminf(fminf(q[0], q[1]), q[2]), q[3]);
    };

    // Own top-2 of this lane's half-block minima. The two lanes of a sample cover disjoint neuron
    // sets, so the merged top-2 are approximate distances of two distinct neurons.
    float m1[G], m2[G], thr[G];
#pragma unroll
    for (int g = 0; g < G; g++) m1[g] = m2[g] = __builtin_inff();
    // Threshold from the merged top-2: every neuron whose exact distance can be <= the second-best
    // (best, without NEED_C2) exact distance has D <= T. T only decreases as more blocks are merged.
    auto refresh = [&]() {
#pragma unroll
        for (int g = 0; g < G; g++) {
            float a1, b1, a2, b2;
            pair32(m1[g], a1, b1);
            pair32(m2[g], a2, b2);
            const float A = NEED_C2 ? fminf(fmaxf(a1, b1), fminf(a2, b2)) : fminf(a1, b1);
            const float scale = fmaxf(A + K[g] + E[g], 0.f);
            thr[g] = A + 2.f * E[g] + 6.2f * U32 * scale + 8.f * U32 * fabsf(A);
        }
    };
    auto update = [&](int g, float t) {
        // both as v_med3: a NaN t leaves the pair unchanged, as fminf would, without the
        // canonicalising moves fminf needs in IEEE mode
        if (NEED_C2) m2[g] = __builtin_amdgcn_fmed3f(m1[g], m2[g], t);
        m1[g] = __builtin_amdgcn_fmed3f(m1[g], t, neg_inf);
    };
    // Without a pool (D = 16), lp is the LDS byte address of this lane's next list entry, held at the
    // spare last row once the list is full (a store then costs one add and one min); the spare row
    // starts as CAND_EMPTY, which no slot takes, so a list that overflowed is told apart from one that
    // filled exactly. With a pool (D = 32), cnt counts the lane's candidates (two fewer registers).
    unsigned int lp[G], lcap[G];
    int cnt[G], pool_n[G];  // pool_n: wave-uniform fill of the group's shared pool
    bool lost[G];           // a candidate of this lane found both its list and the pool full (D = 32)
#pragma unroll
    for (int g = 0; g < G; g++) {
        if constexpr (POOL == 0) {
            lp[g] = lds_addr(&cw[g][0][lane]);
            lcap[g] = lds_addr(&cw[g][CAPL][lane]);
            cw[g][CAPL][lane] = CAND_EMPTY;
        } else {
            cnt[g] = 0;
        }
        pool_n[g] = 0;
        lost[g] = false;
    }
    // Appends every row of this lane's half-block with D <= T; the pre-check skips the per-value
    // compares when no lane of the wave has a hit in the block, and a second one per row quad skips
    // the quads without a hit (hits in a block usually fall in one quad).
    // Rows of a quad with a hit cost one wave compare and one scalar test each when none of their lanes
    // hits. Past CAPL a lane's candidates go to its group's shared pool when there is one (slots handed
    // out in lane order from the wave's ballot), else the lane is lost to the fallback. Only the lanes
    // with a hit store (an exec-masked store); candidates past the list land in the spare last row.
    // A block without a hit (about half of them) leaves the running minima alone too: its minima lie above
    // T, hence above the merged minimum that T is made of.
    auto record = [&](int blk, int g, const f32x16 &v, const float (&q)[4], float t, bool merge) {
        if (__builtin_amdgcn_ballot_w64(t <= thr[g]) == 0ull) return;
        if (merge) update(g, t);
        unsigned long long bq[4];
#pragma unroll
        for (int i = 0; i < 4; i++) bq[i] = __builtin_amdgcn_ballot_w64(q[i] <= thr[g]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (bq[i] == 0ull) continue;  // uniform: no hit in this quad
            unsigned long long br[4];
#pragma unroll
            for (int r = 0; r < 4; r++) br[r] = __builtin_amdgcn_ballot_w64(v[4 * i + r] <= thr[g]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (br[r] == 0ull) continue;  // uniform
                const bool hit = __builtin_amdgcn_inverse_ballot_w64(br[r]);
                // opaque here, so that the slots are not computed ahead in every block
                int sbase = blk;
                asm volatile("" : "+s"(sbase));
                const unsigned short slot = (unsigned short)(sbase * 32 + 4 * khalf + 8 * i + r);
                if constexpr (POOL > 0) {
                    const bool spill = hit && cnt[g] >= CAPL;
                    const unsigned long long sp = __builtin_amdgcn_ballot_w64(spill);
                    if (__builtin_expect(sp != 0ull, 0)) {  // uniform, rare
                        const int off = pool_n[g] + (int)__builtin_amdgcn_mbcnt_hi(
                                            (unsigned)(sp >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)sp, 0u));
                        if (spill && off < POOL) sm.pool[wave][g][off] = ((unsigned)lane << 16) | slot;
                        lost[g] = lost[g] || (spill && off >= POOL);
                        pool_n[g] += __builtin_popcountll(sp);
                    }
                }
                if (hit) {
                    if constexpr (POOL == 0) {
                        *(lds_u16 *)(size_t)lp[g] = slot;
                        // orders the address update after the store, so it is made in place (no
                        // move); the empty statement emits no instruction
                        asm volatile("" : "+v"(lp[g]) : : "memory");
                        lp[g] = min(lp[g] + (unsigned)sizeof(cw[g][0]), lcap[g]);
                    } else {
                        cw[g][min(cnt[g], CAPL)][lane] = slot;
                        cnt[g] += 1;
                    }
                }
            }
        }
    };
    // The chunks in the order they are scanned: phase A, the first half of the coarse section, for the minima
    // alone; phase B, every other block (the rest of the coarse section first), recorded against the threshold
    // in force before its own minima are merged, refreshed after every chunk; phase C, phase A's chunks again under
    // the final threshold. The threshold in force at any time is >= the final one, so the recorded set contains
    // every neuron with D <= final T. The next chunk is loaded while the waves compute, one barrier per chunk.
    const int nchunks_a = max(1, ((Md.nblk_a + CB - 1) / CB) / 2);
    const int total = nchunks + nchunks_a;
    int buf = 0;
    __syncthreads();  // the buffers hold the grouping's scratch
    load_chunk(0);
    store_chunk(0);
    __syncthreads();
    for (int q = 0; q < total; q++) {
        const int c = q < nchunks ? q : q - nchunks;
        if (q + 1 < total) load_chunk(q + 1 < nchunks ? q + 1 : q + 1 - nchunks);
        const int b0 = c * CB;
        const int b1 = min(nblk, b0 + CB);
        auto operands = [&](int blk, f16x8 (&a)[NK]) {
#pragma unroll
            for (int i = 0; i < NK; i++)
                a[i] = __builtin_bit_cast(f16x8, sm.frag[buf][((blk - b0) * NK + i) * 64 + lane]);
        };
        if (q < nchunks_a) {
            for (int blk = b0; blk < b1; blk++) {
                f16x8 a[NK];
                operands(blk, a);
                f32x16 acc[G];
#pragma unroll
                for (int g = 0; g < G; g++) acc[g] = block_acc(g, a);
#pragma unroll
                for (int g = 0; g < G; g++) update(g, block_min(acc[g]));
            }
        } else {
            const bool merge = q < nchunks;
            for (int blk = b0; blk < b1; blk++) {
                f16x8 a[NK];
                operands(blk, a);
                f32x16 acc[G];
#pragma unroll
                for (int g = 0; g < G; g++) acc[g] = block_acc(g, a);
#pragma unroll
                for (int g = 0; g < G; g++) {
                    float qm[4];
                    const float t = quad_min(acc[g], qm);
                    record(blk, g, acc[g], qm, t, merge);
                }
            }
        }
        if (q + 1 < total) store_chunk(buf ^ 1);
        __syncthreads();
        buf ^= 1;
        if (q + 1 >= nchunks_a && q < nchunks) refresh();
    }

    // ---------------- exact rerank of the candidate set ----------------
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int64_t s = tile_row0 + sm.rows[wave][g][col];
        const bool valid_s = s < n;
        Top2 tp;
        tp.init();
        int mycnt;
        bool ovf;
        if constexpr (POOL == 0) {
            mycnt = (int)((lp[g] - lds_addr(&cw[g][0][lane])) / (unsigned)sizeof(cw[g][0]));
            ovf = mycnt == CAPL && cw[g][CAPL][lane] != CAND_EMPTY;
        } else {
            mycnt = min(cnt[g], CAPL);
            ovf = lost[g];
        }
        // The two lanes of a sample share its candidates: the pair's lists, the khalf 0 lane's first,
        // are split in two halves, one per lane, so a wave runs as many candidate distances as its most
        // loaded pair's mean, not its longest list. Top-2 insertion is order-independent.
        const int pcnt = xchg32i(mycnt);
        const bool povf = xchg32i(ovf ? 1 : 0) != 0;
        if (valid_s && !ovf && !povf) {
            const int nlo = khalf == 0 ? mycnt : pcnt;  // entries of the khalf 0 lane's list
            const int half = (mycnt + pcnt + 1) / 2;
            const int eb = khalf == 0 ? 0 : half, ee = khalf == 0 ? half : mycnt + pcnt;
            auto slot_of = [&](int e) {
                const bool lo = e < nlo;
                return (int)cw[g][lo ? e : e - nlo][lo ? col : col + 32];
            };
            // 16 values of the sample's row / of a candidate's row of the slot-ordered copy of W (no index
            // indirection before the load), zero padded
            auto x_part = [&](int kc, T (&v)[16]) { load_values(x + s * dim, kc * 16, dim, v); };
            auto w_part = [&](int slot, int kc, T (&v)[16]) { load16(wslot + (int64_t)slot * DP + kc * 16, v); };
            // up to 128 bytes of the sample stay in registers; of wider rows 16 values of each side are
            // read at a time, so the rerank does not set the kernel's register peak (which would halve the
            // waves per SIMD)
            constexpr bool HOLD_X = DP * sizeof(T) <= 128;
            T xr[HOLD_X ? KC : 1][16];
            if constexpr (HOLD_X) {
#pragma unroll
                for (int kc = 0; kc < KC; kc++) x_part(kc, xr[kc]);
            }
            auto distance = [&](int slot) {
                double d = 0.0;
                if constexpr (HOLD_X) {
                    T wr[KC][16];
#pragma unroll
                    for (int kc = 0; kc < KC; kc++) w_part(slot, kc, wr[kc]);
#pragma unroll
                    for (int kc = 0; kc < KC; kc++) {
                        if constexpr (KC > 1) {
                            // keeps the FP64 arithmetic from holding the sample converted to double across
                            // the candidates (64 more registers); the empty statement emits no instruction
#pragma unroll
                            for (int k = 0; k < 16; k++) asm volatile("" : "+v"(xr[kc][k]));
                        }
                        d = sqd_more<MODE>(d, wr[kc], xr[kc]);
                    }
                } else {
#pragma unroll 1
                    for (int kc = 0; kc < KC; kc++) {
                        T wr[16], xv[16];
                        w_part(slot, kc, wr);
                        x_part(kc, xv);
                        d = sqd_more<MODE>(d, wr, xv);
                    }
                }
                return d;
            };
            if constexpr (HOLD_X && KC == 1) {
                // the next candidate's row is loaded while this one is evaluated
                T wn[16];
                int jn = -1;
                if (eb < ee) {
                    const int slot = slot_of(eb);
                    jn = perm[slot];
                    w_part(slot, 0, wn);
                }
                for (int e = eb; e < ee; e++) {
                    T wr[16];
#pragma unroll
                    for (int k = 0; k < 16; k++) wr[k] = wn[k];
                    const int j = jn;
                    if (e + 1 < ee) {
                        const int slot = slot_of(e + 1);
                        jn = perm[slot];
                        w_part(slot, 0, wn);
                    }
                    if (j >= 0) tp.push(sqd_more<MODE>(0.0, wr, xr[0]), j);  // zero-padded dims add exact zeros
                }
            } else {
                for (int e = eb; e < ee; e++) {
                    const int slot = slot_of(e);
                    const int j = perm[slot];
                    const double d = distance(slot);
                    if (j >= 0) tp.push(d, j);
                }
            }
            // the group's spilled candidates: each entry is reranked by the lane that recorded it
            const int np = POOL > 0 ? min(pool_n[g], POOL) : 0;
            for (int e = 0; e < np; e++) {
                const unsigned int ent = sm.pool[wave][g][e];
                if ((int)(ent >> 16) == lane) {
                    const int slot = (int)(ent & 0xFFFFu);
                    const int j = perm[slot];
                    const double d = distance(slot);
                    if (j >= 0) tp.push(d, j);
                }
            }
        }
        // merge with the partner lane
        const double pd1 = xchg32d(tp.d1), pd2 = xchg32d(tp.d2);
        const int pi1 = xchg32i(tp.i1), pi2 = xchg32i(tp.i2);
        if (pi1 >= 0) tp.push(pd1, pi1);
        if (pi2 >= 0) tp.push(pd2, pi2);
        const bool bad = ovf || povf || !(thr[g] < __builtin_inff());  // also a NaN T
        if (lane < 32 && valid_s) {
            if (bad) {
                const unsigned int slot = atomicAdd(fb_count, 1u);
                fb_list[slot] = fb_tag | s;
            } else {
                c1[s] = tp.i1 >= 0 ? tp.i1 : default_index;
                if (c2) c2[s] = tp.i2;
                if (d1) d1[s] = tp.i1 >= 0 ? tp.d1 : __builtin_nan("");
            }
        }
    }
}

// The body for the plan's number of K slices (uniform; the kernel's registers are those of the largest). A plan of
// more slices than the kernel was chosen for can meet it where a captured launch is replayed after the map was
// prepared anew: its rows go to the exact scan.
template <int DP, int NKMAX, int NW, int G, int MODE, bool NEED_C2, bool GC, class T>
__device__ __forceinline__ void bmu_f16_run(const BmuModelDev &Md, const T *x, int64_t n, int64_t tile_row0,
                                            int default_index, int32_t *c1, int32_t *c2, double *d1, int64_t *fb_list,
                                            unsigned int *fb_count, int64_t fb_tag, F16Smem<DP / 16, NW, G> &sm,
                                            float *xmax_part, const int32_t *prev_c1)
{
    const int nk = aptr<GC>(Md.plan)->nk;
    auto run = [&](auto k) {
        bmu_f16_body<DP, decltype(k)::value, NW, G, MODE, NEED_C2, GC, T>(
            Md, x, n, tile_row0, default_index, c1, c2, d1, fb_list, fb_count, fb_tag, sm, xmax_part, prev_c1);
    };
    using std::integral_constant;
    if constexpr (NKMAX < f16_max_nk(DP)) {
        if (nk > NKMAX) {
            for (int r = threadIdx.x; r < NW * G * 32; r += NW * WAVE)
                if (tile_row0 + r < n) aptr<GC>(fb_list)[atomicAdd(fb_count, 1u)] = fb_tag | (tile_row0 + r);
            return;
        }
    }
    if constexpr (NKMAX >= 5) {
        if (nk == 5) return run(integral_constant<int, 5>{});
    }
    if (nk == 3) return run(integral_constant<int, 3>{});
    run(integral_constant<int, 2>{});
}

// 4 waves per SIMD (3 of the small tiles, by their LDS; 6 of those of 8 waves and one group at D = 16)
template <int DP, int NKMAX, int NW, int G, int MODE, bool NEED_C2, class T>
__global__ __launch_bounds__(NW * WAVE, NW == NW_SMALL ? 3 : G == 1 && DP == 16 ? 6 : 4) void bmu_f16_kernel(BmuModelDev Md, const T *__restrict__ x, int64_t n,
                                                                   int default_index, int32_t *__restrict__ c1,
                                                                   int32_t *__restrict__ c2, double *__restrict__ d1,
                                                                   int64_t *__restrict__ fb_list,
                                                                   unsigned int *__restrict__ fb_count,
                                                                   float *__restrict__ xmax_part,
                                                                   const int32_t *__restrict__ prev_c1)
{
    __shared__ F16Smem<DP / 16, NW, G> sm;
    bmu_f16_run<DP, NKMAX, NW, G, MODE, NEED_C2, false, T>(Md, x, n, (int64_t)blockIdx.x * (NW * G * 32), default_index, c1, c2,
                                                    d1, fb_list, fb_count, 0, sm, xmax_part, prev_c1);
}

// Exact top-2 of one sample by one workgroup of FB_THREADS threads: thread t scans the permuted
// slots t, t + FB_THREADS, ... of the slot-ordered weight copy (4 rows in flight per thread), then
// the top-2 lists are merged (butterfly in each wave, then the waves through LDS), lexicographic on
// (distance, neuron index), so the scan order does not matter. Uniform over the workgroup.
constexpr int FB_THREADS = 256;

struct Top2Slot {
    double d1, d2;
    int i1, i2;
};

template <int DP, int MODE, class T>
__device__ __forceinline__ Top2 group_exact_top2(const T *__restrict__ xrow, int dim, const BmuModelDev &Md,
                                                 Top2Slot *red)
{
    constexpr int U = DP * sizeof(T) <= 256 ? 4 : 2;
    const int tid = threadIdx.x;
    T xr[DP / 16][16];
#pragma unroll
    for (int k = 0; k < DP; k++) xr[k / 16][k % 16] = k < dim ? ((gptr<const T>)xrow)[k] : (T)0;
    Top2 tp;
    tp.init();
    const int nslots = Md.nblk * 32;
    const gptr<const T> rows = (gptr<const T>)Md.wslot;
    const gptr<const int> perm = (gptr<const int>)Md.perm;
    for (int p0 = tid; p0 < nslots; p0 += U * FB_THREADS) {
        double d[U];
        int jj[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int p = p0 + u * FB_THREADS;
            jj[u] = p < nslots ? perm[p] : -1;
            d[u] = 0.0;
        }
#pragma unroll
        for (int kc = 0; kc < DP / 16; kc++) {
            T wr[U][16];
#pragma unroll
            for (int u = 0; u < U; u++) load16(rows + (int64_t)min(p0 + u * FB_THREADS, nslots - 1) * DP + kc * 16, wr[u]);
#pragma unroll
            for (int u = 0; u < U; u++) d[u] = sqd_more<MODE>(d[u], wr[u], xr[kc]);  // zero-padded dims add zeros
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (jj[u] >= 0) tp.push(d[u], jj[u]);
    }
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) {
        const double pd1 = __shfl_xor(tp.d1, o, WAVE), pd2 = __shfl_xor(tp.d2, o, WAVE);
        const int pi1 = __shfl_xor(tp.i1, o, WAVE), pi2 = __shfl_xor(tp.i2, o, WAVE);
        if (pi1 >= 0) tp.push(pd1, pi1);
        if (pi2 >= 0) tp.push(pd2, pi2);
    }
    if ((tid & (WAVE - 1)) == 0) red[tid / WAVE] = Top2Slot{tp.d1, tp.d2, tp.i1, tp.i2};
    __syncthreads();
    if (tid == 0)
        for (int v = 1; v < FB_THREADS / WAVE; v++) {
            if (red[v].i1 >= 0) tp.push(red[v].d1, red[v].i1);
            if (red[v].i2 >= 0) tp.push(red[v].d2, red[v].i2);
        }
    __syncthreads();  // red is reused by the next sample
    return tp;        // complete in thread 0
}

// Fallback of the plain form: one workgroup per listed sample, grid-stride over the device-side
// count.
template <int DP, int MODE, class T>
__global__ __launch_bounds__(FB_THREADS) void bmu_exact_group_kernel(BmuModelDev Md, const T *__restrict__ x,
                                                                     const int64_t *__restrict__ list,
                                                                     const unsigned int *__restrict__ list_count,
                                                                     int default_index, int32_t *__restrict__ c1,
                                                                     int32_t *__restrict__ c2,
                                                                     double *__restrict__ d1)
{
    __shared__ Top2Slot red[FB_THREADS / WAVE];
    const int64_t total = (int64_t)(*list_count);
    for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int64_t i = list[t];
        const Top2 tp = group_exact_top2<DP, MODE, T>(x + i * Md.dim, Md.dim, Md, red);
        if (threadIdx.x == 0) {
            c1[i] = tp.i1 >= 0 ? tp.i1 : default_index;
            if (c2) c2[i] = tp.i2;
            if (d1) d1[i] = tp.i1 >= 0 ? tp.d1 : __builtin_nan("");
        }
    }
}

template <int DP, class T>
void launch_exact_group(int mode, hipStream_t st, const BmuModelDev &Md, const T *x, const int64_t *list,
                        const unsigned int *list_count, int64_t blocks, int default_index, int32_t *c1, int32_t *c2,
                        double *d1)
{
    const dim3 grid((unsigned)blocks), block(FB_THREADS);
    if (sizeof(T) == 8 || mode == SOMHIP_RERANK_FP64)
        hipLaunchKernelGGL((bmu_exact_group_kernel<DP, SOMHIP_RERANK_FP64, T>), grid, block, 0, st, Md, x, list,
                           list_count, default_index, c1, c2, d1);
    else if constexpr (sizeof(T) == 4)
        hipLaunchKernelGGL((bmu_exact_group_kernel<DP, SOMHIP_RERANK_REF32, T>), grid, block, 0, st, Md, x, list,
                           list_count, default_index, c1, c2, d1);
}

template <int DP, int NKMAX, int NW, int G, class T>
void launch_f16(int mode, bool need_c2, hipStream_t st, somhip_model *M, const T *x, int64_t n, int default_index,
                int32_t *c1, int32_t *c2, double *d1, int64_t *fb_list, unsigned int *fb_count, float *xmax_part,
                const int32_t *prev_c1)
{
    const int64_t blocks = (n + NW * G * 32 - 1) / (NW * G * 32);
    dim3 grid((unsigned)blocks), block(NW * WAVE);
#define SOM_F16(MO, C)                                                                                              \
    hipLaunchKernelGGL((bmu_f16_kernel<DP, NKMAX, NW, G, MO, C, T>), grid, block, 0, st, somhip_model_dev(M), x, n,         \
                       default_index, c1, c2, d1, fb_list, fb_count, xmax_part, prev_c1)
    if (sizeof(T) == 8 || mode == SOMHIP_RERANK_FP64) {
        if (need_c2) SOM_F16(SOMHIP_RERANK_FP64, true); else SOM_F16(SOMHIP_RERANK_FP64, false);
    } else if constexpr (sizeof(T) == 4) {
        if (need_c2) SOM_F16(SOMHIP_RERANK_REF32, true); else SOM_F16(SOMHIP_RERANK_REF32, false);
    }
#undef SOM_F16
}

}  // namespace

// The 16-bit search and its fallback, for FP32 rows or, on float64 models, FP64 rows.
template <int DP, class T>
int somhip_search_f16(somhip_model *M, const T *x, int64_t n, int arithmetic, int need_c2, int default_index, int32_t *c1,
                  int32_t *c2, double *d1, float *xmax_part, int64_t *fb_list, unsigned int *fb_count,
                  const int32_t *prev_c1)
{
    hipStream_t st = M->ctx->stream;
    {
        TimerScope ts(M->ctx, TK_BMU_BF16);
        auto launch = [&](auto nkmax, auto nw, auto g) {
            launch_f16<DP, decltype(nkmax)::value, decltype(nw)::value, decltype(g)::value, T>(
                arithmetic, need_c2, st, M, x, n, default_index, c1, c2, d1, fb_list, fb_count, xmax_part, prev_c1);
        };
        using std::integral_constant;
        constexpr int NKMAX = f16_max_nk(DP);
        // a plan of at most three slices runs the kernel without the five-slice body, whose registers would
        // spill in it
        const bool three = NKMAX > 3 && f16_nk_limit(M, M->prepared == 2) == 3;
        if (n <= SMALL_ROWS) {
            launch(integral_constant<int, NKMAX>{}, integral_constant<int, NW_SMALL>{}, integral_constant<int, 1>{});
        } else if (n <= MEDIUM_ROWS) {
            launch(integral_constant<int, NKMAX>{}, integral_constant<int, NW_F16>{}, integral_constant<int, 1>{});
        } else if (three) {
            if constexpr (NKMAX > 3)
                launch(integral_constant<int, 3>{}, integral_constant<int, NW_F16>{}, integral_constant<int, G_F16>{});
        } else {
            launch(integral_constant<int, NKMAX>{}, integral_constant<int, NW_F16>{}, integral_constant<int, G_F16>{});
        }
        SOM_HIP_TRY(hipGetLastError());
    }
    TimerScope tf(M->ctx, TK_BMU_FALLBACK);
    // Fallback over the flagged samples: one workgroup per sample, a fixed grid that reads the
    // device-side count (an empty list costs one launch).
    const int64_t fb_blocks = std::max<int64_t>(1, std::min<int64_t>(n, (int64_t)M->ctx->num_cus * 8));
    launch_exact_group<DP, T>(arithmetic, st, somhip_model_dev(M), x, fb_list, fb_count, fb_blocks, default_index, c1, c2,
                              d1);
    SOM_HIP_TRY(hipGetLastError());
    return SOMHIP_OK;
}

