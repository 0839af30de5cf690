// Dense weights (F32, F16, BF16) @ F32 activations -> F32: jam's dense paths (jam/jam-native/src/jam.c:596-660).
//
// Semantics. F32 and F16 weights multiply the f32 activations as they are (f16 -> f32 is exact); BF16 weights
// multiply activations rounded to bf16 (round to nearest even) wherever jam's bf16 kernels take the call on an
// AVX-512-BF16 host (n >= 8 with k even: the packed-panel kernel; k % 32 == 0: the convert-once kernel) and the
// f32 activations otherwise (the convert-and-FMA floor). Every product is exact in f32 (bf16 x bf16, f16 x f32
// and f32 x f32 products are formed exactly by the FMA / the matrix cores); only the f32 summation order
// differs from jam's.
//
// Layout. A device copy keeps the rows row-major, each padded with zeros to a pitch of whole 256 bytes (dense_row_pitch,
// WeightView::G), so every row starts 16-byte aligned and a 16-byte load never crosses into the next row.
//
// Kernels.
//  * dense_gemv2_kernel (n <= 8 while the token tile's activations fit 64 KB of LDS; HBM-bound): activations
//    staged in LDS, each wave streaming 1..4 rows two 16-byte pieces per lane deep; dense_gemv_kernel
//    otherwise: a wave streams 8 rows with 16-byte loads, the activations from L2.
//  * dense_tile_kernel (F32, and BF16 with unrounded activations, past the GEMV): v_mfma_f32_*f32 on exact operands loaded
//    straight from global memory, one tile per workgroup, its waves splitting k.
//  * dense_mma_kernel (F16, and BF16 with rounded activations, past the GEMV): LDS-staged f16 / bf16 matrix cores.
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace jamhip {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// jam's bf16 activation rounding (vcvtne2ps2bf16): round to nearest even on the dropped 16 bits; NaN stays NaN.
JAMHIP_DEV uint32_t bf16_bits(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
JAMHIP_DEV float bf16_round(float x) { return __builtin_bit_cast(float, bf16_bits(x) << 16); }

// 16 weight bytes -> V = 16 / element size f32 values
template <int DT> JAMHIP_DEV void wvals(const uint4 v, float* f) {
    if constexpr (DT == F32) {
        f[0] = __builtin_bit_cast(float, v.x);
        f[1] = __builtin_bit_cast(float, v.y);
        f[2] = __builtin_bit_cast(float, v.z);
        f[3] = __builtin_bit_cast(float, v.w);
    } else {
        const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (DT == F16) {
                f[2 * i] = h2f(u[i] & 0xffffu);
                f[2 * i + 1] = h2f(u[i] >> 16);
            } else {
                f[2 * i] = __builtin_bit_cast(float, u[i] << 16);
                f[2 * i + 1] = __builtin_bit_cast(float, u[i] & 0xffff0000u);
            }
        }
    }
}

JAMHIP_DEV uint4 ld16_nt(const void* p) {
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    const v4u v = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

constexpr int DG_WAVES = 4, DG_RPW = 8;   // GEMV: waves per workgroup, rows per wave

// ------------------------------------------------------------------------------------------ GEMV
template <int DT, int NT>
__global__ void __launch_bounds__(64 * DG_WAVES) dense_gemv_kernel(WeightView w, const float* __restrict__ a, int lda,
                                                                   int k, int m, int n, float* __restrict__ c, int ldc,
                                                                   int rnd, Epi ep) {
    constexpr int ES = block_bytes(DT), V = 16 / ES;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t row0 = ((int64_t) blockIdx.x * DG_WAVES + wave) * DG_RPW;
    if (row0 >= m) return;   // wave-uniform; the kernel has no barrier
    const int t0 = blockIdx.y * NT, ntv = n - t0 < NT ? n - t0 : NT;
    const uint8_t* wr[DG_RPW];
#pragma unroll
    for (int r = 0; r < DG_RPW; r++) {
        const int64_t row = row0 + r < m ? row0 + r : m - 1;
        wr[r] = w.qs + (w.r0 + row) * w.G;
    }
    float acc[DG_RPW][NT];
#pragma unroll
    for (int r = 0; r < DG_RPW; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = 0.0f;
    for (int e0 = lane * V; e0 < k; e0 += 64 * V) {   // e0·ES + 16 <= the pitch: pieces never cross rows
        uint4 raw[DG_RPW];
#pragma unroll
        for (int r = 0; r < DG_RPW; r++) raw[r] = ld16_nt(wr[r] + (int64_t) e0 * ES);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (t >= ntv) break;
            const float* ar = a + (int64_t) (t0 + t) * lda;
            float x[V];
#pragma unroll
            for (int i = 0; i < V; i++) {
                const float v = e0 + i < k ? ar[e0 + i] : 0.0f;
                x[i] = rnd ? bf16_round(v) : v;
            }
#pragma unroll
            for (int r = 0; r < DG_RPW; r++) {
                float f[V];
                wvals<DT>(raw[r], f);
#pragma unroll
                for (int i = 0; i < V; i++) {
                    const float wv = e0 + i < k ? f[i] : 0.0f;   // a pinned row's columns past k may hold anything
                    acc[r][t] = fmaf(wv, x[i], acc[r][t]);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < DG_RPW; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const float v = wave_sum(acc[r][t]);
            const int64_t row = row0 + r;
            if (lane == 0 && t < ntv && row < m) {
                float* dst = c + (int64_t) (t0 + t) * ldc + row;
                *dst = epilogue(ep, v, row, dst);
            }
        }
}

// GEMV with the activations in LDS and the weight stream two steps deep in registers (n <= 8 where the NT-token
// tile's activations fit 64 KB of LDS). A workgroup of 4 waves stages its tile's activations (bf16-rounded
// where jam rounds them; zero past k), each wave streams RPW rows: per step a lane loads one 16-byte piece of
// every row (the wave reads RPW contiguous 1 KB runs), and step j + 1's pieces are in flight while step j
// is multiplied. The loads are unconditional (a step past the row's end re-reads the last piece and adds
// nothing), so the compiler waits for exactly the step it computes. Columns past k inside a row's last
// piece are zeroed before use (a pinned row's may hold anything, NaN included).
constexpr int DG2_LDS_MAX = 64 * 1024, DG2_KSPLIT_ROWS = 256;

// KS (one row per workgroup): the four waves take every fourth step of the row instead of a row each, and their sums
// meet in LDS. A router of 32 rows is 8 workgroups walking 12 dependent steps otherwise (F32 32x2880, one token:
// 4.5 -> 3.5 us, 256x4096: 7.0 -> 4.7, F16 256x4096: 5.6 -> 4.2).
template <int DT, int NT, int RPW, bool KS = false>
__global__ void __launch_bounds__(64 * DG_WAVES) dense_gemv2_kernel(WeightView w, const float* __restrict__ a, int lda,
                                                                    int k, int m, int n, float* __restrict__ c,
                                                                    int ldc, int rnd, int kp, Epi ep) {
    constexpr int ES = block_bytes(DT), V = 16 / ES;
    extern __shared__ __align__(16) float xs[];   // [NT][kp], kp a multiple of 64·V
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t0 = blockIdx.y * NT, ntv = n - t0 < NT ? n - t0 : NT;
    const int64_t row0 = KS ? (int64_t) blockIdx.x : ((int64_t) blockIdx.x * DG_WAVES + wave) * RPW;
    static_assert(!KS || RPW == 1, "a split row is alone in its workgroup");
    constexpr int JS = KS ? DG_WAVES : 1;         // step stride of a wave
    const int S = kp / (64 * V), jw = KS ? wave : 0;   // steps per row, the wave's first one
    const uint8_t* wr[RPW];
#pragma unroll
    for (int r = 0; r < RPW; r++) {
        const int64_t row = row0 + r < m ? row0 + r : m - 1;
        wr[r] = w.qs + (w.r0 + row) * w.G;
    }
    // the last piece holding a column of the row: later steps re-read it (in bounds of the row's pitch)
    const int elast = (k - 1) / V * V;
    auto load = [&](uint4 (&raw)[RPW], int j) {
        const int e0 = min((j * 64 + lane) * V, elast);
#pragma unroll
        for (int r = 0; r < RPW; r++) raw[r] = ld16_nt(wr[r] + (int64_t) e0 * ES);
    };
    uint4 raw[2][RPW];
    load(raw[0], jw);
    load(raw[1], jw + JS);
    // stage the tile's activations: float4 slots of [NT][kp]
    const int q4 = kp / 4;
    for (int i = threadIdx.x; i < NT * q4; i += 64 * DG_WAVES) {
        const int t = i / q4, e = 4 * (i - t * q4);
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float x = t < ntv && e + u < k ? a[(int64_t) (t0 + t) * lda + e + u] : 0.0f;
            v[u] = rnd ? bf16_round(x) : x;
        }
        *reinterpret_cast<float4*>(xs + (int64_t) t * kp + e) = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    if (row0 >= m) return;   // wave-uniform; after the workgroup's only barrier
    float acc[RPW][NT];
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = 0.0f;
    auto step = [&](const uint4 (&rv)[RPW], int j) {
        const int e0 = (j * 64 + lane) * V;
        const bool tail = e0 + V > k;   // the row's last piece (or past it): columns >= k -> 0
        float f[RPW][V];
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            wvals<DT>(rv[r], f[r]);
            if (tail)
#pragma unroll
                for (int i = 0; i < V; i++) f[r][i] = e0 + i < k ? f[r][i] : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (t >= ntv) break;
            float x[V];
#pragma unroll
            for (int i = 0; i < V; i += 4) {
                const float4 v = *reinterpret_cast<const float4*>(xs + (int64_t) t * kp + e0 + i);
                x[i] = v.x, x[i + 1] = v.y, x[i + 2] = v.z, x[i + 3] = v.w;
            }
#pragma unroll
            for (int r = 0; r < RPW; r++)
#pragma unroll
                for (int i = 0; i < V; i++) acc[r][t] = fmaf(f[r][i], x[i], acc[r][t]);
        }
    };
    for (int j = jw; j < S; j += 2 * JS) {
        step(raw[0], j);
        load(raw[0], j + 2 * JS);
        if (j + JS < S) step(raw[1], j + JS);
        load(raw[1], j + 3 * JS);
    }
    if constexpr (KS) {   // every wave reaches this: row0 < m for the whole workgroup
        // the waves' sums [DG_WAVES][NT] take the activations' place: beside a full 64 KB of them a launch would ask for
        // more LDS than it may without raising its kernel's limit
        static_assert(DG_WAVES <= 64 * V, "the sums fit the shortest activation rows");
        __syncthreads();   // every wave is done with the activations
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const float v = wave_sum(acc[0][t]);
            if (lane == 0) xs[wave * NT + t] = v;
        }
        __syncthreads();
        if ((int) threadIdx.x < ntv) {
            const int t = threadIdx.x;
            float* dst = c + (int64_t) (t0 + t) * ldc + row0;
            *dst = epilogue(ep, (xs[t] + xs[NT + t]) + (xs[2 * NT + t] + xs[3 * NT + t]), row0, dst);
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < RPW; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const float v = wave_sum(acc[r][t]);
            const int64_t row = row0 + r;
            if (lane == 0 && t < ntv && row < m) {
                float* dst = c + (int64_t) (t0 + t) * ldc + row;
                *dst = epilogue(ep, v, row, dst);
            }
        }
}

// ------------------------------------------------------------------------------------------ GEMM
// F32 weights, and BF16 weights with unrounded activations (n > 8, or past the GEMV's LDS): f32 MFMA on exact operands.
// One wave per 32 x 64 tile, walking k alone behind its own loads, held 32 rows x 512 tokens (a router) to 8 waves on
// 2 CUs: 296 us at k = 2880. Here a workgroup of 8 waves owns one T x T tile (16 or 32) and its waves take every
// eighth run of k: 64 CUs on that shape, 12.3 us (2.7 us of it the f32 matrix rate of one CU on a 16 x 16 x 2880 tile), and
// more than twice as fast where the tiles fill the chip (F32 4096x4096 n = 512: 556 -> 255 us; 2048x2880 n = 512:
// 391 -> 95). Two or three runs in flight per wave instead of one lose 5 to 30%: the registers cost more waves than the
// distance hides. The waves' sums meet in LDS in a fixed order.
constexpr int DT_WAVES = 8;

template <int DT, int T>
__global__ void __launch_bounds__(64 * DT_WAVES) dense_tile_kernel(WeightView w, const float* __restrict__ a, int lda,
                                                                   int k, int m, int n, float* __restrict__ c, int ldc,
                                                                   int nt, Epi ep) {
    constexpr int Q = 64 / T, RUN = 16 * Q, E = T * T / 64, LD = T + 4;
    constexpr int ES = block_bytes(DT);
    static_assert(DT == F32 || DT == BF16, "F16 takes the staged GEMM");
    typedef float accv __attribute__((ext_vector_type(E)));
    __shared__ __align__(16) float red[DT_WAVES][T * LD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane % T, q = lane / T;
    const int64_t row0 = (int64_t) (blockIdx.x / nt) * T;   // nt token tiles per row tile
    const int t0 = (int) (blockIdx.x % nt) * T;
    const int64_t wrow = row0 + r < m ? row0 + r : m - 1;   // clamped: its products are never stored
    const int trow = t0 + r < n ? t0 + r : n - 1;
    const uint8_t* wp = w.qs + (w.r0 + wrow) * w.G;
    const float* ap = a + (int64_t) trow * lda;
    const int runs = (k + RUN - 1) / RUN;
    // Piece i of a run is 4·Q consecutive k of a row, 4 per lane, so a load instruction reads 16·Q (F32) contiguous bytes
    // of T rows. A run never crosses a row's 256-byte pitch (RUN·ES divides it): weight loads past k stay in the row.
    typedef uint32_t piece __attribute__((ext_vector_type(ES)));   // 4 weights
    // Activation rows start at any 4-byte address (row strides are the caller's): gfx950 loads 16 bytes from there in one
    // instruction, where element-wise loads made odd strides slow (F32 41478x634 n = 190 314 -> 178 us, 42665x1090 n = 255 734 -> 382).
    typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
    auto load = [&](piece (&wv)[4], f32x4u (&xv)[4], int it) {
        const int e0 = it * RUN + 4 * q;
#pragma unroll
        for (int i = 0; i < 4; i++) wv[i] = *reinterpret_cast<const piece*>(wp + (int64_t) (e0 + 4 * Q * i) * ES);
        if ((it + 1) * RUN <= k) {   // wave-uniform
#pragma unroll
            for (int i = 0; i < 4; i++) xv[i] = *reinterpret_cast<const f32x4u*>(ap + e0 + 4 * Q * i);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int e = e0 + 4 * Q * i;
                xv[i] = f32x4u{e < k ? ap[e] : 0.0f, e + 1 < k ? ap[e + 1] : 0.0f, e + 2 < k ? ap[e + 2] : 0.0f,
                               e + 3 < k ? ap[e + 3] : 0.0f};
            }
        }
    };
    accv acc[2] = {accv{}, accv{}};
    auto mul = [&](const piece (&wv)[4], const f32x4u (&xv)[4], int it) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float f[4];
            if constexpr (DT == F32) {
#pragma unroll
                for (int u = 0; u < 4; u++) f[u] = __builtin_bit_cast(float, (uint32_t) wv[i][u]);
            } else {
#pragma unroll
                for (int u = 0; u < 4; u++)
                    f[u] = __builtin_bit_cast(float, u & 1 ? wv[i][u / 2] & 0xffff0000u : wv[i][u / 2] << 16);
            }
            if ((it + 1) * RUN > k) {   // a pinned row's columns past k may hold anything
#pragma unroll
                for (int u = 0; u < 4; u++) f[u] = it * RUN + 4 * q + 4 * Q * i + u < k ? f[u] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if constexpr (T == 16)
                    acc[u & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[u], xv[i][u], acc[u & 1], 0, 0, 0);
                else
                    acc[u & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[u], xv[i][u], acc[u & 1], 0, 0, 0);
            }
        }
    };
    for (int it = wave; it < runs; it += DT_WAVES) {
        piece wv[4];
        f32x4u xv[4];
        load(wv, xv, it);
        mul(wv, xv, it);
    }
    // lane: token r, rows 4q + e (T = 16) or 8·(e / 4) + 4q + e % 4 (T = 32)
    const accv s = acc[0] + acc[1];
#pragma unroll
    for (int g = 0; g < E / 4; g++)
        *reinterpret_cast<float4*>(&red[wave][r * LD + 8 * g + 4 * q]) =
            make_float4(s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]);
    __syncthreads();
    for (int i = threadIdx.x; i < T * T; i += 64 * DT_WAVES) {
        const int row = i % T, t = i / T;
        if (row0 + row >= m || t0 + t >= n) continue;
        float v = red[0][t * LD + row];
#pragma unroll
        for (int u = 1; u < DT_WAVES; u++) v += red[u][t * LD + row];
        float* dst = c + (int64_t) (t0 + t) * ldc + row0 + row;
        *dst = epilogue(ep, v, row0 + row, dst);
    }
}

// ------------------------------------------------------------------------- staged matrix-core GEMM (n >= 9)
// F16 weights and BF16 weights with bf16-rounded activations (k even or k % 32 == 0: jam's bf16 kernels) run
// on the f16 / bf16 matrix cores with LDS-staged operands, the structure of the quantized prefill GEMM
// (mma.hip) without its per-block scales:
//  * dense_prep_kernel writes the activations in the MFMA operand order, planes
//    [Kp/16 K-steps][2 halves][NP slots][8] (half h = elements 8h..8h+7 of the K-step, zero past k): for F16
//    weights the f16 high part and f16 remainder of x·2^-e_t, e_t putting the token's largest |x| in
//    [2^14, 2^15) (hi + lo hold x to about 22 bits), and es[t] = 2^e_t; for BF16 weights jam's bf16(x), es = 1.
//  * dense_mma_kernel: a workgroup of 4 waves owns 128 rows x 64 tokens and walks k in stages of 64 elements.
//    Each stage's operands are copied global -> LDS by the waves (global_load_lds, double-buffered): a wave's
//    own 32 rows as 8 pieces of 32 rows x 16 bytes (lane r of a piece reads row r: the LDS tile is the
//    fragment layout, conflict-free to read), and 1 KB pieces of the activation planes. Per 16-element K-step
//    and 32-token tile one MFMA per plane: f16 weights x hi, then x lo; bf16 x bf16. Products are exact in f32;
//    only the summation order differs from jam's f32 FMA chain, plus for F16 the ~2^-22 relative remainder
//    of x that hi + lo drop. Weight columns past k in the last stage are zeroed in the fragment (a pinned
//    row's may hold anything). Small grids split k like the quantized GEMM (partials summed in slice order).
constexpr int DMM_STAGE = 64;

int dense_mma_planes(int dt, int n, int k);   // below
static int dense_np(int n) { return (n + 63) / 64 * 64; }
static int dense_kp(int k) { return (k + DMM_STAGE - 1) / DMM_STAGE * DMM_STAGE; }

size_t dense_act_bytes(int dt, int n, int k) {
    const int pl = dense_mma_planes(dt, n, k);
    const size_t plane = ((size_t) dense_kp(k) * dense_np(n) * 2 + 255) / 256 * 256;
    return pl * plane + ((size_t) dense_np(n) * 4 + 255) / 256 * 256;
}

// A workgroup of 8 waves takes 8 tokens and one of gridDim.y runs of their rows: each wave first finds its token's largest
// |x| (the whole row, from L2 past the first workgroup), then 8 consecutive threads store one 8-element row of the
// operand for the 8 tokens, a whole 128-byte line. One workgroup per token stored 16 bytes of each line and read its
// row alone: 512 x 4096 15.6 -> 9.2 us.
__global__ void __launch_bounds__(512) dense_prep_kernel(const float* __restrict__ a, int lda, int n, int k, int Kp,
                                                         int NP, int hl, uint16_t* __restrict__ hi,
                                                         uint16_t* __restrict__ lo, float* __restrict__ es) {
    __shared__ float sdown[8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t0 = 8 * blockIdx.x;
    if (t0 >= n) return;   // the whole workgroup: the grid is padded (dense_prep_grid)
    if (hl && t0 + wave < n) {   // a non-finite largest |x| leaves the scale at 1 (the outputs go non-finite)
        const float* x = a + (int64_t) (t0 + wave) * lda;
        float mx = 0.0f;
        if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
            const int k4 = k / 4;
#pragma unroll 8
            for (int e = lane; e < k4; e += 64) {
                const float4 f = reinterpret_cast<const float4*>(x)[e];
                mx = fmaxf(fmaxf(mx, fmaxf(fabsf(f.x), fabsf(f.y))), fmaxf(fabsf(f.z), fabsf(f.w)));
            }
            for (int e = 4 * k4 + lane; e < k; e += 64) mx = fmaxf(mx, fabsf(x[e]));
        } else {
#pragma unroll 8
            for (int e = lane; e < k; e += 64) mx = fmaxf(mx, fabsf(x[e]));
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        int ex = 0;
        if (mx > 0.0f && mx <= 3.40282347e38f) {
            int e2;
            frexpf(mx, &e2);   // mx in [2^(e2-1), 2^e2)
            ex = 15 - e2;
            ex = ex > 126 ? 126 : ex;
        }
        if (lane == 0) {
            sdown[wave] = ldexpf(1.0f, ex);
            if (blockIdx.y == 0) es[t0 + wave] = ldexpf(1.0f, -ex);
        }
    } else if (!hl && blockIdx.y == 0 && lane == 0 && t0 + wave < n) {
        es[t0 + wave] = 1.0f;
    }
    __syncthreads();
    const int t = t0 + (threadIdx.x & 7);
    if (t >= n) return;   // after the only barrier
    const float* x = a + (int64_t) t * lda;
    const float down = hl ? sdown[threadIdx.x & 7] : 1.0f;
    const bool vec = (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    // 8-element runs: run g = elements 8g..8g+7 = K-step g / 2, half g % 2
    const int ng = Kp / 8, per = (ng + (int) gridDim.y - 1) / (int) gridDim.y;
    const int g1 = min(ng, per * ((int) blockIdx.y + 1));
    for (int g = per * (int) blockIdx.y + (threadIdx.x >> 3); g < g1; g += 64) {
        float v[8];
        const int e0 = 8 * g;
        if (vec && e0 + 8 <= k) {
            const float4 f0 = *reinterpret_cast<const float4*>(x + e0), f1 = *reinterpret_cast<const float4*>(x + e0 + 4);
            v[0] = f0.x, v[1] = f0.y, v[2] = f0.z, v[3] = f0.w, v[4] = f1.x, v[5] = f1.y, v[6] = f1.z, v[7] = f1.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = e0 + i < k ? x[e0 + i] : 0.0f;
        }
        uint32_t h[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (hl) {
                const F16Pair p0 = split_f16(v[2 * i] * down), p1 = split_f16(v[2 * i + 1] * down);
                h[i] = (uint32_t) __builtin_bit_cast(uint16_t, p0.hi) | ((uint32_t) __builtin_bit_cast(uint16_t, p1.hi) << 16);
                l[i] = (uint32_t) __builtin_bit_cast(uint16_t, p0.lo) | ((uint32_t) __builtin_bit_cast(uint16_t, p1.lo) << 16);
            } else {
                h[i] = bf16_bits(v[2 * i]) | (bf16_bits(v[2 * i + 1]) << 16);
            }
        }
        const int64_t o = ((int64_t) g * NP + t) * 8;   // (K-step g/2, half g%2) = plane row g
        *reinterpret_cast<uint4*>(hi + o) = make_uint4(h[0], h[1], h[2], h[3]);
        if (hl) *reinterpret_cast<uint4*>(lo + o) = make_uint4(l[0], l[1], l[2], l[3]);
    }
}

// Short rows of few tokens (dense_prep_few): a workgroup per token, which reads its row in whole lines.
__global__ void __launch_bounds__(256) dense_prep_few_kernel(const float* __restrict__ a, int lda, int n, int k, int Kp,
                                                         int NP, int hl, uint16_t* __restrict__ hi,
                                                         uint16_t* __restrict__ lo, float* __restrict__ es) {
    __shared__ float wmax[4];
    const int t = blockIdx.x;
    const float* x = a + (int64_t) t * lda;
    float down = 1.0f;
    if (hl) {   // the token's largest |x|; a non-finite one leaves the scale at 1 (the outputs go non-finite)
        float mx = 0.0f;
        for (int e = threadIdx.x; e < k; e += 256) mx = fmaxf(mx, fabsf(x[e]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
        int ex;
        if (mx > 0.0f && mx <= 3.40282347e38f) {
            int e2;
            frexpf(mx, &e2);   // mx in [2^(e2-1), 2^e2)
            ex = 15 - e2;
            ex = ex > 126 ? 126 : ex;
        } else {
            ex = 0;
        }
        down = ldexpf(1.0f, ex);
        if (threadIdx.x == 0) es[t] = ldexpf(1.0f, -ex);
    } else if (threadIdx.x == 0) {
        es[t] = 1.0f;
    }
    // 8-element runs: run g = elements 8g..8g+7 = K-step g / 2, half g % 2
    for (int g = threadIdx.x; g < Kp / 8; g += 256) {
        float v[8];
        const int e0 = 8 * g;
        if (e0 + 8 <= k && ((reinterpret_cast<uintptr_t>(x + e0) & 15) == 0)) {
            const float4 f0 = *reinterpret_cast<const float4*>(x + e0), f1 = *reinterpret_cast<const float4*>(x + e0 + 4);
            v[0] = f0.x, v[1] = f0.y, v[2] = f0.z, v[3] = f0.w, v[4] = f1.x, v[5] = f1.y, v[6] = f1.z, v[7] = f1.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = e0 + i < k ? x[e0 + i] : 0.0f;
        }
        uint32_t h[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (hl) {
                const F16Pair p0 = split_f16(v[2 * i] * down), p1 = split_f16(v[2 * i + 1] * down);
                h[i] = (uint32_t) __builtin_bit_cast(uint16_t, p0.hi) | ((uint32_t) __builtin_bit_cast(uint16_t, p1.hi) << 16);
                l[i] = (uint32_t) __builtin_bit_cast(uint16_t, p0.lo) | ((uint32_t) __builtin_bit_cast(uint16_t, p1.lo) << 16);
            } else {
                h[i] = bf16_bits(v[2 * i]) | (bf16_bits(v[2 * i + 1]) << 16);
            }
        }
        const int64_t o = ((int64_t) g * NP + t) * 8;   // (K-step g/2, half g%2) = plane row g
        *reinterpret_cast<uint4*>(hi + o) = make_uint4(h[0], h[1], h[2], h[3]);
        if (hl) *reinterpret_cast<uint4*>(lo + o) = make_uint4(l[0], l[1], l[2], l[3]);
    }
}

typedef _Float16 half8d __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void_d;
typedef uint32_t u32x4d __attribute__((ext_vector_type(4)));

template <bool HL>
__global__ void __launch_bounds__(256, 2) dense_mma_kernel(WeightView w, const uint16_t* __restrict__ xh,
                                                           const uint16_t* __restrict__ xl, const float* __restrict__ es,
                                                           int NP, int Kp, int k, int m, int n, float* __restrict__ c,
                                                           int ldc, int nrb, int ncb, int st_per, int64_t c_slice,
                                                           Epi ep) {
    constexpr int PL = HL ? 2 : 1, A_BYTES = 4 * 4096, BYTES = A_BYTES + PL * 8192;
    extern __shared__ __align__(1024) unsigned char dsm[];
    const int total = nrb * ncb, lin = tile_of_block(false, total);
    if (lin >= total) return;
    const int rb = lin / ncb, cb = lin % ncb;
    const int lane = threadIdx.x & 63, r = lane & 31, q = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = (int64_t) rb * 128 + 32 * wave;
    const int n0 = cb * 64;
    const int nstk = Kp / DMM_STAGE;
    const int st0 = st_per > 0 ? st_per * (int) blockIdx.y : 0;
    const int nst = st_per > 0 ? min(nstk, st0 + st_per) : nstk;
    const int64_t crow = row0 + r < m ? row0 + r : m - 1;   // the row this lane copies (clamped to the view)
    const uint8_t* wrow = w.qs + (w.r0 + crow) * w.G + 16 * q;
    const uint16_t* bsrc = xh + ((int64_t) (2 * wave) * NP + n0) * 8 + 8 * lane;
    const int64_t plane_off = xl - xh;
    auto issue = [&](int st, unsigned char* buf) {
        // weights: pieces 2i + q (elements 64·st + 8(2i + q)..) of row r, 4 instructions of 1 KB
#pragma unroll
        for (int i = 0; i < 4; i++)
            __builtin_amdgcn_global_load_lds(wrow + ((int64_t) DMM_STAGE * st + 16 * i) * 2,
                                             (lds_void_d*) (buf + wave * 4096 + i * 1024), 16, 0, 0);
        // activations: plane rows 8·st + 2·wave and + 1 (K-step 4st + wave, halves 0 and 1), 1 KB each
#pragma unroll
        for (int pl = 0; pl < PL; pl++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                __builtin_amdgcn_global_load_lds(bsrc + pl * plane_off + ((int64_t) (8 * st + h)) * NP * 8,
                                                 (lds_void_d*) (buf + A_BYTES + pl * 8192 + (2 * wave + h) * 1024), 16, 0,
                                                 0);
    };
    floatx16 acc[2] = {floatx16{}, floatx16{}};
    issue(st0, dsm + (st0 & 1) * BYTES);   // a K slice may start on an odd stage
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int st = st0; st < nst; st++) {
        unsigned char* buf = dsm + (st & 1) * BYTES;
        uint4 af[4];
        uint4 bf[PL][4][2];
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            af[ks] = *reinterpret_cast<const uint4*>(buf + wave * 4096 + (2 * ks + q) * 512 + 16 * r);
#pragma unroll
            for (int pl = 0; pl < PL; pl++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    bf[pl][ks][j] = *reinterpret_cast<const uint4*>(buf + A_BYTES + pl * 8192 + (2 * ks + q) * 1024 +
                                                                   (32 * j + r) * 16);
        }
        if (DMM_STAGE * (st + 1) > k) {   // the stage holding column k - 1: columns >= k -> 0
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const int e0 = DMM_STAGE * st + 16 * ks + 8 * q;
                uint32_t u[4] = {af[ks].x, af[ks].y, af[ks].z, af[ks].w};
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (e0 + i >= k) u[i >> 1] &= (i & 1) ? 0x0000ffffu : 0xffff0000u;
                af[ks] = make_uint4(u[0], u[1], u[2], u[3]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (st + 1 < nst) issue(st + 1, dsm + ((st + 1) & 1) * BYTES);
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int pl = 0; pl < PL; pl++) {
                    if constexpr (HL)
                        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8d, af[ks]),
                                                                        __builtin_bit_cast(half8d, bf[pl][ks][j]), acc[j], 0, 0, 0);
                    else
                        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[ks]),
                                                                         __builtin_bit_cast(bf16x8, bf[pl][ks][j]), acc[j], 0, 0, 0);
                }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    // lane holds token n0 + 32j + r, rows 8·(e/4) + 4q + e%4 of the wave's 32; a K slice writes its partial
    // result at c + y·c_slice
    if (st_per > 0) c += (int64_t) blockIdx.y * c_slice;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int t = n0 + 32 * j + r;
        if (t >= n) continue;
        const float sc = es[t];
        store_column(c + (int64_t) t * ldc, row0 + 4 * q, m, acc[j], sc, ep, st_per > 0);
    }
}

// Calls with many tokens: the same operands in tiles of 256 rows x 128 tokens, 8 waves of 64 x 64 (4 x 2), k in stages of
// 64. The 128 x 64 kernel above moves 512 bytes (F16) global -> LDS per 128 x 64 outputs and k, and its waves wait for
// those copies (26% MFMA busy); here it is 1024 bytes per 256 x 128, each fragment read from LDS feeds two MFMAs per
// plane, and a stage's copies run during the whole stage before it (two LDS buffers, one workgroup per CU). A stage is 1536
// cycles of LDS reads and 2048 of products on each SIMD (F16): its two waves take turns, one reading while the other
// multiplies. With the prep, 128 x 64 kernel -> this one: F16 14336x4096 n = 512 243 -> 126 us, n = 2048 825 -> 486, BF16 n = 512
// 197 -> 96; it then moves about 8 TB/s global -> LDS. Four buffers of 32 measured slower (140 us: the compiler makes LDS
// reads wait for copies in flight to the other buffers).
// LDS: weights [256 rows][128 B], the row's 16-byte piece p at position p ^ (row % 8), so that a fragment read's 8 lanes
// per cycle fall on different banks (the copy writes lane-linear: the lane picks its source piece instead); activations
// as prepared, [PL][8 8-element rows][128 tokens][16 B].

template <bool HL>
__global__ void __launch_bounds__(512, 1) dense_big_kernel(WeightView w, const uint16_t* __restrict__ xh,
                                                           const uint16_t* __restrict__ xl, const float* __restrict__ es,
                                                           int NP, int Kp, int k, int m, int n, float* __restrict__ c,
                                                           int ldc, int nrb, int ncb, int st_per, int64_t c_slice,
                                                           Epi ep) {
    constexpr int PL = HL ? 2 : 1, A_BYTES = 256 * 128, BYTES = A_BYTES + PL * 16384;
    __shared__ __align__(1024) unsigned char sb0[BYTES], sb1[BYTES];
    const int total = nrb * ncb, lin = tile_of_block(false, total);
    if (lin >= total) return;
    const int rb = lin / ncb, cb = lin % ncb;
    const int lane = threadIdx.x & 63, r = lane & 31, q = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave >> 1, wt = wave & 1;
    const int64_t row0 = (int64_t) rb * 256;
    const int n0 = cb * 128;
    const int nstk = Kp / DMM_STAGE;
    const int st0 = st_per > 0 ? st_per * (int) blockIdx.y : 0;
    const int nst = st_per > 0 ? min(nstk, st0 + st_per) : nstk;
    // weights: the wave copies rows 32·wave.. in four pieces of 8 rows x 128 bytes
    const uint8_t* asrc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int lr = 32 * wave + 8 * i + (lane >> 3);
        const int64_t row = row0 + lr < m ? row0 + lr : m - 1;
        asrc[i] = w.qs + (w.r0 + row) * w.G + 16 * ((lane & 7) ^ (lr & 7));
    }
    // activations: 8-element row `wave` of the stage, tokens 0..63 and 64..127; a last half block re-reads its first slots
    const int t1 = n0 + 64 < NP ? 64 : 0;
    const uint16_t* bsrc = xh + ((int64_t) wave * NP + n0) * 8 + 8 * lane;
    const int64_t plane_off = xl - xh;
    auto issue = [&](int st, unsigned char* buf) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            __builtin_amdgcn_global_load_lds(asrc[i] + (int64_t) st * (DMM_STAGE * 2),
                                             (lds_void_d*) (buf + wave * 4096 + i * 1024), 16, 0, 0);
#pragma unroll
        for (int pl = 0; pl < PL; pl++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                __builtin_amdgcn_global_load_lds(bsrc + pl * plane_off + ((int64_t) (8 * st) * NP + h * t1) * 8,
                                                 (lds_void_d*) (buf + A_BYTES + pl * 16384 + wave * 2048 + h * 1024), 16, 0,
                                                 0);
    };
    floatx16 acc[2][2] = {{floatx16{}, floatx16{}}, {floatx16{}, floatx16{}}};
    u32x4d af[4][2], bf[4][PL][2];   // a stage's fragments [K-step][..]
    auto read = [&](auto U, int st) __attribute__((always_inline)) {
        const unsigned char* buf = decltype(U)::value ? sb1 : sb0;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int lr = 64 * wr + 32 * i + r;
                af[ks][i] = *reinterpret_cast<const u32x4d*>(buf + lr * 128 + (((2 * ks + q) ^ (lr & 7)) * 16));
            }
#pragma unroll
            for (int pl = 0; pl < PL; pl++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    bf[ks][pl][j] = *reinterpret_cast<const u32x4d*>(buf + A_BYTES + pl * 16384 + (2 * ks + q) * 2048 +
                                                                    (64 * wt + 32 * j + r) * 16);
        }
        if (DMM_STAGE * (st + 1) > k) {   // the stage holding column k - 1: columns >= k -> 0 (they may hold anything)
#pragma unroll
            for (int ks = 0; ks < 4; ks++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int e0 = DMM_STAGE * st + 16 * ks + 8 * q;
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (e0 + e >= k) af[ks][i][e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
                }
        }
        __builtin_amdgcn_sched_barrier(0);   // the phases stay apart: reads | copies | products
    };
    auto mul = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int pl = 0; pl < PL; pl++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        if constexpr (HL)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8d, af[ks][i]),
                                                                               __builtin_bit_cast(half8d, bf[ks][pl][j]), acc[i][j], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[ks][i]),
                                                                                __builtin_bit_cast(bf16x8, bf[ks][pl][j]), acc[i][j], 0, 0, 0);
                    }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto copies_in = [&]() { __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); };   // vmcnt(0): this wave's copies
    auto meet = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, 0> b0{};
    constexpr std::integral_constant<int, 1> b1{};
    // Waves 0..3 (one per SIMD) read stage s in half-step 2s and multiply in 2s + 1; waves 4..7 a half-step later. Buffer
    // s % 2 is last read in 2s + 1, refilled with stage s + 2 from 2s + 2 on (each wave its own pieces) and complete, by
    // every wave's wait before the barrier that ends it, with 2s + 3.
    issue(st0, sb0);
    copies_in();
    meet();
    if (wave < 4) {
        auto step = [&](auto U, int st) __attribute__((always_inline)) {
            read(U, st);
            if (st + 1 < nst) issue(st + 1, decltype(U)::value ? sb0 : sb1);
            meet();
            mul();
            copies_in();
            meet();
        };
        for (int st = st0; st < nst; st += 2) {
            step(b0, st);
            if (st + 1 < nst) step(b1, st + 1);
        }
        meet();   // the other waves' last half-step
    } else {
        if (st0 + 1 < nst) issue(st0 + 1, sb1);
        meet();
        auto step = [&](auto U, int st) __attribute__((always_inline)) {
            read(U, st);
            copies_in();
            meet();
            if (st + 2 < nst) issue(st + 2, decltype(U)::value ? sb1 : sb0);
            mul();
            meet();
        };
        for (int st = st0; st < nst; st += 2) {
            step(b0, st);
            if (st + 1 < nst) step(b1, st + 1);
        }
    }
    if (st_per > 0) c += (int64_t) blockIdx.y * c_slice;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int t = n0 + 64 * wt + 32 * j + r;
        if (t >= n) continue;
        const float sc = es[t];
#pragma unroll
        for (int i = 0; i < 2; i++)
            store_column(c + (int64_t) t * ldc, row0 + 64 * wr + 32 * i + 4 * q, m, acc[i][j], sc, ep, st_per > 0);
    }
}

// ----------------------------------------------------------------------------------------- launchers
// jam rounds BF16's activations to bf16 where its bf16 kernels take the call (jam.c:622-652).
static bool bf16_rounds(int n, int k) { return (n >= 8 && k % 2 == 0) || k % 32 == 0; }

template <int DT, int NT, int RPW, bool KS = false>
static void gemv2_go(const WeightView& w, const float* a, int lda, int k, int kp, int m, int n, float* c, int ldc,
                     int rnd, hipStream_t st, const Epi& ep) {
    const int rows_per_wg = KS ? 1 : DG_WAVES * RPW;
    const dim3 grid((unsigned) ((m + rows_per_wg - 1) / rows_per_wg), (unsigned) ((n + NT - 1) / NT));
    dense_gemv2_kernel<DT, NT, RPW, KS><<<grid, 64 * DG_WAVES, (size_t) NT * kp * 4, st>>>(w, a, lda, k, m, n, c, ldc, rnd,
                                                                                       kp, ep);
}

// The NT-token tile of n <= 8 tokens fits the staged GEMV's LDS.
static bool gemv2_fits(int n, int dt, int k) {
    const int nt = n <= 2 ? n : n <= 4 ? 4 : 8, run = 64 * 16 / block_bytes(dt), kp = (k + run - 1) / run * run;
    return (size_t) nt * kp * 4 <= (size_t) DG2_LDS_MAX;
}

template <int DT, int NT>
static void gemv_go(const WeightView& w, const float* a, int lda, int k, int m, int n, float* c, int ldc, int rnd,
                    hipStream_t st, const Epi& ep) {
    constexpr int V = 16 / block_bytes(DT);
    const int kp = (k + 64 * V - 1) / (64 * V) * (64 * V);
    if ((size_t) NT * kp * 4 <= (size_t) DG2_LDS_MAX) {
        // up to a row per CU: a workgroup per row, its waves splitting k (four times as many workgroups; from there
        // on the one-row waves alone fill the CUs)
        if (m <= DG2_KSPLIT_ROWS) return gemv2_go<DT, NT, 1, true>(w, a, lda, k, kp, m, n, c, ldc, rnd, st, ep);
        // rows per wave: about 2048 waves or more over the device, 4 rows a wave at most
        if (m >= 4 * 2048) return gemv2_go<DT, NT, 4>(w, a, lda, k, kp, m, n, c, ldc, rnd, st, ep);
        if (m >= 2 * 2048) return gemv2_go<DT, NT, 2>(w, a, lda, k, kp, m, n, c, ldc, rnd, st, ep);
        return gemv2_go<DT, NT, 1>(w, a, lda, k, kp, m, n, c, ldc, rnd, st, ep);
    }
    const int rows_per_wg = DG_WAVES * DG_RPW;   // one token, k past the staged GEMV's LDS
    const dim3 grid((unsigned) ((m + rows_per_wg - 1) / rows_per_wg), (unsigned) ((n + NT - 1) / NT));
    if constexpr (NT == 1) dense_gemv_kernel<DT, NT><<<grid, 64 * DG_WAVES, 0, st>>>(w, a, lda, k, m, n, c, ldc, rnd, ep);
}

template <int DT>
static hipError_t dense_go(const WeightView& w, const float* a, int lda, int k, int m, int n, float* c, int ldc,
                           hipStream_t st, const Epi& ep) {
    const bool rnd = DT == BF16 && bf16_rounds(n, k);
    if (n == 1 || (n <= 8 && gemv2_fits(n, DT, k))) {
        if (n == 1) gemv_go<DT, 1>(w, a, lda, k, m, n, c, ldc, rnd, st, ep);
        else if (n == 2) gemv_go<DT, 2>(w, a, lda, k, m, n, c, ldc, rnd, st, ep);
        else if (n <= 4) gemv_go<DT, 4>(w, a, lda, k, m, n, c, ldc, rnd, st, ep);
        else gemv_go<DT, 8>(w, a, lda, k, m, n, c, ldc, rnd, st, ep);
        return hipGetLastError();
    }
    // F16 and bf16-rounded BF16 calls of 2 or more tokens past the GEMV took the staged GEMM (dense_mma_planes)
    if constexpr (DT != F16) {
        const int64_t nt32 = (n + 31) / 32, tiles32 = (int64_t) ((m + 31) / 32) * nt32;
        const int64_t nt16 = (n + 15) / 16, tiles16 = (int64_t) ((m + 15) / 16) * nt16;
        if (tiles32 > 0x7fffffff) return hipErrorInvalidValue;   // (16 x 16 tiles: n <= 16 or few)
        if (dense_tile32(m, n))
            dense_tile_kernel<DT, 32><<<(unsigned) tiles32, 64 * DT_WAVES, 0, st>>>(w, a, lda, k, m, n, c, ldc, (int) nt32,
                                                                                    ep);
        else
            dense_tile_kernel<DT, 16><<<(unsigned) tiles16, 64 * DT_WAVES, 0, st>>>(w, a, lda, k, m, n, c, ldc, (int) nt16,
                                                                                    ep);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;
}

// 2 planes (F16: hi, lo), 1 (BF16 with jam's bf16 rounding), 0: the staged GEMM does not take the call. It
// takes n >= DENSE_MMA_MIN_N, and from 2 tokens the calls whose token tile's activations would not fit the
// LDS-staged GEMV (k = 14336 at n = 2: 63 against 95 us for BF16 4096x14336; k = 4096 at n = 8: 63 against
// 128 us for F16 14336x4096). The staged GEMV stays ahead where it fits (F16 14336x4096 n = 4: 46 against 63).
int dense_mma_planes(int dt, int n, int k) {
    if (dt != F16 && !(dt == BF16 && bf16_rounds(n, k))) return 0;
    if (n < DENSE_MMA_MIN_N) {
        if (n < 2) return 0;
        if (gemv2_fits(n, dt, k)) return 0;
    }
    return dt == F16 ? 2 : 1;
}

// K slices, the quantized GEMM's rule over stages of 64
static Split dense_split(int m, int n, int k) { return split_plan(up_div(m, 128) * (dense_np(n) / 64), dense_kp(k) / DMM_STAGE); }

size_t dense_mma_split_floats(int dt, int k, int m, int n) {
    if (!dense_mma_planes(dt, n, k)) return 0;
    const int ns = dense_split(m, n, k).ns;
    return ns > 1 ? (size_t) ns * n * m : 0;
}

hipError_t launch_dense_mma(int dt, const WeightView& w, const float* a, int lda, int k, int m, int n, float* c,
                            int ldc, void* scratch, float* part, hipStream_t st, const Epi& ep) {
    const int pl = dense_mma_planes(dt, n, k);
    if (!pl) return hipErrorNotSupported;
    const int NP = dense_np(n), Kp = dense_kp(k);
    const size_t plane = ((size_t) Kp * NP * 2 + 255) / 256 * 256;
    uint16_t* xh = (uint16_t*) scratch;
    uint16_t* xl = (uint16_t*) ((uint8_t*) scratch + plane);
    float* es = (float*) ((uint8_t*) scratch + pl * plane);
    const PrepGrid pg = dense_prep_grid(n, Kp);
    if (dense_prep_few(dt, k, n))
        dense_prep_few_kernel<<<n, 256, 0, st>>>(a, lda, n, k, Kp, NP, pl == 2, xh, pl == 2 ? xl : xh, es);
    else
        dense_prep_kernel<<<dim3((unsigned) pg.x, (unsigned) pg.y), 512, 0, st>>>(a, lda, n, k, Kp, NP, pl == 2, xh, pl == 2 ? xl : xh, es);
    const Split sp = dense_split(m, n, k);
    const int ns = sp.ns, st_per = sp.per;
    if (ns > 1 && part == nullptr) return hipErrorInvalidValue;
    float* out = ns > 1 ? part : c;
    const int ldo = ns > 1 ? m : ldc;
    const int64_t slice = (int64_t) n * m;
    const Epi epo = ns > 1 ? Epi{} : ep;
    if (dense_big(dt, Kp / DMM_STAGE, m, n, sp, device_cus())) {
        const int brb = (m + 255) / 256, bcb = (NP + 127) / 128;
        const dim3 grid((unsigned) tile_grid(false, brb * bcb), (unsigned) ns);
        if (pl == 2)
            dense_big_kernel<true><<<grid, 512, 0, st>>>(w, xh, xl, es, NP, Kp, k, m, n, out, ldo, brb, bcb, st_per, slice, epo);
        else
            dense_big_kernel<false><<<grid, 512, 0, st>>>(w, xh, xh, es, NP, Kp, k, m, n, out, ldo, brb, bcb, st_per, slice, epo);
    } else {
        const int nrb = (m + 127) / 128, ncb = NP / 64;
        const dim3 grid((unsigned) tile_grid(false, nrb * ncb), (unsigned) ns);
        const size_t lds = 2 * (size_t) (4 * 4096 + pl * 8192);
        if (pl == 2)
            dense_mma_kernel<true><<<grid, 256, lds, st>>>(w, xh, xl, es, NP, Kp, k, m, n, out, ldo, nrb, ncb, st_per, slice, epo);
        else
            dense_mma_kernel<false><<<grid, 256, lds, st>>>(w, xh, xh, es, NP, Kp, k, m, n, out, ldo, nrb, ncb, st_per, slice, epo);
    }
    if (ns > 1) return launch_split_reduce(part, ns, slice, m, n, c, ldc, st, ep);
    return hipGetLastError();
}

hipError_t launch_dense(int dt, const WeightView& w, const float* a, int lda, int k, int m, int n, float* c, int ldc,
                        hipStream_t st, const Epi& ep) {
    switch (dt) {
    case F32: return dense_go<F32>(w, a, lda, k, m, n, c, ldc, st, ep);
    case F16: return dense_go<F16>(w, a, lda, k, m, n, c, ldc, st, ep);
    case BF16: return dense_go<BF16>(w, a, lda, k, m, n, c, ldc, st, ep);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace jamhip
