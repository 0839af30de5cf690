// Matrix-core prefill GEMM for MXFP4 weights in jam's semantics (n >= 8: F2 int8 activations, one f32 scale per 32-element
// block; F1 codes for a grouped expert of 1..7 rows): C[n][m] = W[m][k] · A[n][k]^T, activations from launch_gemm_prep.
//
// Arithmetic. One v_mfma_scale_f32_32x32x64_f8f6f4 is a whole 32-element block of a 32 x 32 tile, exactly. Its 64 K
// positions hold the block twice: K 0..31 and K 32..63 are the same 32 e2m1 weight codes as stored (A, fp4; both
// lane halves read the same 16 bytes, nothing is decoded), against the activation code q split into sign and two
// digits, |q| = 16·h + l with h in 0..8 and l in 0..15 (B, fp6 e2m3, whose codes 0..15 are the integers 0..15 over 8):
// the high digits under the block scale 2^7, the low ones under 2^3. With A's block scale the stored exponent e, the
// result is 2^(e - 128)·Σ kv·q (kv jam's doubled codes, jam_mxfp4.h:14-24), which f32 holds exactly: |Σ kv·q| < 2^16.
// Checked on the device against integer sums for random and extreme codes and every exponent up to 238 (subnormal
// results included); the repack keeps tensors with larger ones, whose products could overflow, off this kernel. One f32
// FMA per output then applies the block's activation scale, in groups of 8 blocks summed into the total. While every partial
// sum is a normal, finite f32 the results are bit-identical to the f16 form this replaces, which summed a group in units of its
// largest exponent and applied that once. Below, each block's FMA rounds at 2^-149 where that form rounded once a group;
// and a block term past f32's largest is infinite before a later one could cancel it. jam applies every block's scale by
// itself too, so its own sums round and overflow there.
//
// What bounds it. Nothing but that FMA is left per output and block (16 VALU instructions, 64 cycles of a SIMD, per
// instruction of 33 cycles on the matrix cores, where the f16 form took two MFMAs and 8 conversions per 8 weights), so
// the VALU issue rate is the ceiling, and LDS traffic is next: a wave of 32 x 64 outputs reads 32 cycles of fragments
// per 32 cycles of its share of the FMAs. A wave therefore owns 64 rows x 64 tokens (RT = 2: the token fragments serve two
// row tiles). It is not at that ceiling: 14336x4096 n = 512 has the VALU busy 53% of the time and the matrix cores 19%, and its
// waves wait for a stage's copies or the barrier 21% of theirs (grouped: 43%, 15%, 37%). With the prep, f16 kernel -> this one: 14336x4096 n = 512 103 -> 73 us, n = 2048 373 -> 240 us; the two
// grouped products of a 32-expert 2 x 5760 / 2880 block at 512 tokens, top-4, 166 + 94 -> 117 + 72 us (of a wave's
// cycles there 37% wait on copies and barriers, its weights being read once at 3.2 TB/s).
//
// Tiling. 4 waves, wave w row tiles w·RT.. of the workgroup's 4·RT, 64 tokens; k in stages of 128 (4 blocks), two LDS
// buffers, every operand copied global -> LDS by the waves; two workgroups per CU. The buffers are separate LDS objects
// and all copies in flight go to the other one, so the compiler's waits before LDS reads cover no copy in flight. Weights
// two stages ahead in three buffers measured no faster (MoE block 282 against 277 us, 14336x4096 n = 512 76 against 73).
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace jamhip {

namespace mx4 {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int WAVES = 4;
// stage buffer: weights [4·RT tiles][4 blocks][32 rows][16 B], exponents [4·RT][32 rows][4 B], digits' first 16 bytes
// [4 blocks][2 digits][64 tokens][16 B], their last 8 bytes likewise, block scales [64 tokens][4 blocks] f32
template <int RT> struct Stage {
    static constexpr int A = 0, H = A + WAVES * RT * 2048, B16 = H + WAVES * 256, B8 = B16 + 8192, DX = B8 + 4096,
                         BYTES = DX + 1024;
};

JAMHIP_DEV void copy16(const void* g, void* l) { __builtin_amdgcn_global_load_lds(g, (lds_void*) l, 16, 0, 0); }
JAMHIP_DEV void copy4(const void* g, void* l) { __builtin_amdgcn_global_load_lds(g, (lds_void*) l, 4, 0, 0); }

}  // namespace mx4

template <int RT>
__global__ void __launch_bounds__(64 * mx4::WAVES, 2) mx4_gemm_kernel(WeightView w, GemmAct A, int m, int n,
                                                                      float* __restrict__ c, int ldc, int nrb, int ncb,
                                                                      int64_t tiles, Groups gp, int sb_per,
                                                                      int64_t c_slice, Epi ep, int xsplit) {
    using namespace mx4;
    using S = Stage<RT>;
    constexpr int TW = WAVES * RT;
    __shared__ __align__(1024) unsigned char sb0[S::BYTES], sb1[S::BYTES];
    // workgroup -> tile as in kq_gemm_kernel (XCD runs; xsplit: half tiles in the last round; expert-major when grouped)
    const int total = nrb * ncb;
    int lin, sub = -1;
    if (xsplit > 0) {
        const int T8 = (total + 7) / 8, x = (int) blockIdx.x % 8, i = (int) blockIdx.x / 8, nf = T8 - xsplit;
        lin = x * T8 + (i < nf ? i : nf + (i - nf) / 2);
        if (i >= nf) sub = (i - nf) & 1;
    } else {
        lin = tile_of_block(gp.map64 != nullptr, total);
    }
    if (lin >= total) return;
    int rb = lin / ncb, cb = lin % ncb;
    if (gp.map64 != nullptr && grouped_tile(gp, lin, nrb, &rb, &cb) < 0) return;   // before any barrier
    const int64_t T0 = (int64_t) rb * TW;
    const int n0 = cb * 64 + (sub > 0 ? 32 : 0);
    const int lane = threadIdx.x & 63, r = lane & 31, q = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = (int) w.G, nsb = A.Kp / 256;
    const int st0 = sb_per > 0 ? 2 * sb_per * (int) blockIdx.y : 0;
    const int nstk = min(2 * nsb, (A.K / 32 + 3) / 4);   // stages that hold at least one block of k
    const int nst = sb_per > 0 ? min(nstk, st0 + 2 * sb_per) : nstk;
    int64_t r0t = w.r0 >> 5;
    int slot0 = 0, crow0 = 0, nvalid = n;
    if (gp.map64 != nullptr) {   // grouped: this slot block's expert
        const int e = __builtin_amdgcn_readfirstlane(gp.map64[cb]);
        if (e < 0) return;
        r0t = (w.r0 + (int64_t) e * gp.gm) >> 5;
        tiles = gp.gm / 32;
        m = gp.gm;
        slot0 = __builtin_amdgcn_readfirstlane(gp.poff64[e]);
        crow0 = __builtin_amdgcn_readfirstlane(gp.off[e]);
        nvalid = __builtin_amdgcn_readfirstlane(gp.off[e + 1]) - crow0;
        if (gp.bias != nullptr) ep.bias = gp.bias + (int64_t) e * gp.gm;
    }
    // all valid tokens in the block's first 32 slots, or one half of a split tile: the second token tile is neither
    // copied nor computed nor stored
    const bool half = sub >= 0 || nvalid - (n0 - slot0) <= 32;
    const int64_t TL = T0 + wave * RT;             // the wave's first row tile
    const bool live = TL < tiles;                  // else it copies and waits with the others, and computes nothing

    // ---- one stage's copies: 1 KB pieces with fixed owners
    constexpr int NC = group_chunks(MXFP4);
    auto tile = [&](int64_t T) { return r0t + (T < tiles ? T : tiles - 1); };
    const uint8_t* a_src[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) a_src[i] = w.qs + tile(TL + i) * G * (NC * CHUNK_STRIDE) + 16 * lane;
    const uint8_t* h_src = w.sc + (tile(TL + (RT == 2 ? q : 0)) * G * 32 + r) * 16;
    const uint8_t* b16_src = reinterpret_cast<const uint8_t*>(A.b) + ((int64_t) (2 * wave) * A.NP + n0 + lane) * 16;
    const uint8_t* b8_src = reinterpret_cast<const uint8_t*>(A.b) + (int64_t) A.Kp * A.NP + ((int64_t) (2 * wave + q) * A.NP + n0) * 8 + 16 * r;
    const float* dx_src = A.dx + ((int64_t) n0 + lane) * 4;
    const int64_t np = A.NP;
    auto issue = [&](int st, unsigned char* buf) {
        const int g = st >> 1, h2 = st & 1;
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int p = 0; p < 2; p++)
                copy16(a_src[i] + (int64_t) g * (NC * CHUNK_STRIDE) + (4 * h2 + 2 * p) * CHUNK_STRIDE,
                       buf + S::A + (wave * RT + i) * 2048 + p * 1024);
        if (RT == 2 || lane < 32) copy4(h_src + (int64_t) g * 512 + 4 * h2, buf + S::H + wave * 256);
        // digits: block `wave` of the stage
        if (!half || lane < 32) {
#pragma unroll
            for (int d = 0; d < 2; d++)
                copy16(b16_src + ((int64_t) (8 * st) + d) * np * 16, buf + S::B16 + (2 * wave + d) * 1024);
        }
        if (!half || r < 16) copy16(b8_src + (int64_t) (8 * st) * np * 8, buf + S::B8 + wave * 1024);
        if (wave == (st & 3) && (!half || lane < 32)) copy16(dx_src + (int64_t) st * np * 4, buf + S::DX);
    };

    const int sb = q ? 130 : 134;   // B's block scales: 2^3 under the low digits (lane half 1), 2^7 under the high ones
    floatx16 acc[RT][2], accs[RT][2];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = accs[i][j] = floatx16{};

    auto stage = [&](auto ca, auto U, int st) {
        constexpr int CA = decltype(ca)::value, u = decltype(U)::value, NSTEP = RT * CA;   // products per block
        const unsigned char* buf = u ? sb1 : sb0;
        // this stage's own copies are in; then every wave's are, and every wave is done reading the other buffer
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));   // vmcnt(0)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (st + 1 < nst) issue(st + 1, u ? sb0 : sb1);
        if (live) {
            uint32_t hx[RT];
            f32x4 dx[CA];
#pragma unroll
            for (int i = 0; i < RT; i++) hx[i] = *reinterpret_cast<const uint32_t*>(buf + S::H + wave * 256 + i * 128 + 4 * r);
#pragma unroll
            for (int j = 0; j < CA; j++) dx[j] = *reinterpret_cast<const f32x4*>(buf + S::DX + (32 * j + r) * 16);
            u32x4 av[2][RT];
            u32x4 b16[2][CA];
            u32x2 b8[2][CA];
            auto read = [&](int b) {
#pragma unroll
                for (int i = 0; i < RT; i++)
                    av[b & 1][i] = *reinterpret_cast<const u32x4*>(buf + S::A + ((wave * RT + i) * 4 + b) * 512 + 16 * r);
#pragma unroll
                for (int j = 0; j < CA; j++) {
                    b16[b & 1][j] = *reinterpret_cast<const u32x4*>(buf + S::B16 + ((2 * b + q) * 64 + 32 * j + r) * 16);
                    b8[b & 1][j] = *reinterpret_cast<const u32x2*>(buf + S::B8 + ((2 * b + q) * 64 + 32 * j + r) * 8);
                }
            };
            read(0);
            // product t + 1 goes out on the matrix cores before product t's FMAs, block b + 1's reads before block b's products
            floatx16 P[2];
            auto mul = [&](auto T) {
                constexpr int t = decltype(T)::value, b = t / NSTEP, i = (t % NSTEP) / CA, j = t % CA;
                if constexpr (t % NSTEP == 0 && b < 3) read(b + 1);
                const u32x4 x = av[b & 1][i], y = b16[b & 1][j];
                const u32x2 z = b8[b & 1][j];
                const v8i a8 = {(int) x[0], (int) x[1], (int) x[2], (int) x[3], 0, 0, 0, 0};
                const v8i bb = {(int) y[0], (int) y[1], (int) y[2], (int) y[3], (int) z[0], (int) z[1], 0, 0};
                P[t & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a8, bb, floatx16{}, 4, 2, b, (int) hx[i], 0, sb);
            };
            auto add = [&](auto T) {
                constexpr int t = decltype(T)::value, b = t / NSTEP, i = (t % NSTEP) / CA, j = t % CA;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    if constexpr (u == 0 && b == 0) accs[i][j][e] = P[t & 1][e] * dx[j][b];   // the group's first block
                    else accs[i][j][e] = fmaf(P[t & 1][e], dx[j][b], accs[i][j][e]);
                }
            };
            mul(std::integral_constant<int, 0>{});
            unroll<0, 4 * NSTEP>([&](auto T) {
                if constexpr (decltype(T)::value + 1 < 4 * NSTEP) mul(std::integral_constant<int, decltype(T)::value + 1>{});
                add(T);
            });
            if (u == 1 || st + 1 == nst) {   // the group's end
#pragma unroll
                for (int i = 0; i < RT; i++)
#pragma unroll
                    for (int j = 0; j < CA; j++) acc[i][j] += accs[i][j];
            }
        }
    };
    issue(st0, sb0);   // a K slice starts on a whole group
    auto run = [&](auto ca) {
        for (int st = st0; st < nst; st += 2) {
            stage(ca, std::integral_constant<int, 0>{}, st);
            if (st + 1 < nst) stage(ca, std::integral_constant<int, 1>{}, st + 1);
        }
    };
    if (half) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});

    // lane: token n0 + 32j + r, rows 8·(e / 4) + 4q + e % 4 of each tile
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int t = n0 + 32 * j + r, tl = t - slot0;
        if (tl >= nvalid || (half && j > 0)) continue;
        float* ct = c + (int64_t) blockIdx.y * c_slice + (int64_t) (crow0 + tl) * ldc;
#pragma unroll
        for (int i = 0; i < RT; i++)   // split K: the reduce applies the epilogue
            store_column(ct, (TL + i) * 32 + 4 * q, m, acc[i][j], 1.0f, ep, sb_per > 0);
    }
}

hipError_t launch_mx4_gemm(const WeightView& w, const GemmAct& A, int m, int n, float* c, int ldc, hipStream_t st,
                           const Groups& gp, int rt, int ns, int sb_per, int xsplit, int64_t c_slice, const Epi& ep) {
    const int nrb = (m + 128 * rt - 1) / (128 * rt), ncb = A.NP / 64;
    const int64_t tiles = (w.r0 + tiled_rows(m)) / 32 - w.r0 / 32;
    const dim3 grid((unsigned) (tile_grid(gp.map64 != nullptr, nrb * ncb) + 8 * xsplit), (unsigned) ns);
    if (rt == 2)
        mx4_gemm_kernel<2><<<grid, 64 * mx4::WAVES, 0, st>>>(w, A, m, n, c, ldc, nrb, ncb, tiles, gp, sb_per, c_slice, ep, xsplit);
    else
        mx4_gemm_kernel<1><<<grid, 64 * mx4::WAVES, 0, st>>>(w, A, m, n, c, ldc, nrb, ncb, tiles, gp, sb_per, c_slice, ep, xsplit);
    return hipGetLastError();
}

}  // namespace jamhip
