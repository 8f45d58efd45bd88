// Quantized GEMV on gfx950 MFMA: the reference's matmul_gemv (src/kernels.rs:590-635, decode
// 550-576), Y[M,N] = A[M,K] f16 . deq(W[N,K])^T with the weights dequantized in f32 and f32
// accumulation.  It serves the short question suffix (M <= 20, the reference's GEMV rows,
// src/engine.rs:419-425) and every matrix the tiled kernels do not take: non-default formats
// (int2/int3, asymmetric, group > 32) and N % 64 != 0 (src/engine.rs:434-442), at any M: k_gemv for few rows,
// k_gemm_fmt for many.
//
// Design (HBM/latency-bound weight streaming):
//  * v_mfma_f32_16x16x32_f16 with the weights as the row operand (16 output columns) and the
//    activations as the column operand (16 input rows): D[n][m].  The f32 dequantized value v is
//    split into hi = f16(v) and lo = f16(v - hi) and both go through the MFMA with the same
//    activations; for symmetric formats hi + lo is v exactly (the residual has at most 5 significant
//    bits), so the product is the reference's f32 dequant at f32 accumulation;
//  * a macro step is 128 k (4 quant blocks): lane (i = l % 16, g = l / 16) loads block g of column i
//    (16 bytes for int4) and the 64 bytes of input row i at those 32 k; MFMA k-slice q takes
//    element group q of both, so the operands need no permutation;
//  * a workgroup is 4 waves that split its k range (wave w takes macro steps w, w + 4, ...) and sum
//    their accumulators through LDS at the end, in a fixed order; every wave keeps 4 macro steps of
//    loads in flight (for K = 2048 that is all of them), with explicit vmcnt waits;
//  * workgroups split the columns in tiles of 16 x NCT; with f32 partial outputs the k range is also
//    split over ks workgroups (the consumer sums the slots in order, as for the tiled kernels);
//  * the gate_up of the short path (rows interleaved in groups of 16) can apply SiLU * mul in the
//    epilogue: a wave's two column tiles are then 16 gate and the 16 matching up columns;
//  * every load is a raw buffer load: columns past N, rows past M and k past K read zeros.
//
// Weight layouts: TILED is the engine's int4 group-32 layout (tile_w4, words in the engine nibble
// order of repack_w4); otherwise the reference's plain layout, [N][K/32] blocks of 4*bits bytes in
// the reference's bit order, scales (and asymmetric biases) [N][K/group] f16.
#include <hip/hip_ext.h>

#include "common.h"
#include "device.h"

namespace sd {
namespace {

constexpr int GV_PD = 4;  // macro steps (128 k) in flight per wave

template <int B>
struct BlkT;
template <>
struct BlkT<4> {
    typedef u32x4 T;
};
template <>
struct BlkT<3> {
    typedef u32x3 T;
};
template <>
struct BlkT<2> {
    typedef u32x2 T;
};

template <int B>
__device__ __forceinline__ typename BlkT<B>::T load_blk(Rsrc r, uint32_t off) {
    if constexpr (B == 4) return buf_b128(r, off, 0);
    else if constexpr (B == 3) return buf_b96(r, off, 0);
    else return buf_b64(r, off, 0);
}

// Elements 8q .. 8q + 7 of a quant block as f16 hi and lo parts of their f32 values.
// TILED: int4 in the engine nibble order (nib_pairs), v = (q - 8) sc with hi = f16 product and lo
// the exact residual (one f16 fma).  Plain: the reference's bit order (src/kernels.rs:550-576),
// v = (q - 2^(bits-1)) sc or fma(q, sc, bi) in f32.
template <int BITS, bool ASYM, bool TILED>
__device__ __forceinline__ void deq8(const typename BlkT<BITS>::T& w, uint32_t sc_bits, uint32_t bi_bits, int q,
                                     f16x8& hi, f16x8& lo) {
    const f16 sc = __builtin_bit_cast(f16, (uint16_t)sc_bits);
    if constexpr (TILED) {
        const f16x2 sc2 = f16x2{sc, sc};
        f16x2 p0, p1, p2, p3;
        nib_pairs(w[q], p0, p1, p2, p3);
        const f16x2 h0 = p0 * sc2, h1 = p1 * sc2, h2 = p2 * sc2, h3 = p3 * sc2;
        hi = cat4(h0, h1, h2, h3);
        lo = cat4(__builtin_elementwise_fma(p0, sc2, -h0), __builtin_elementwise_fma(p1, sc2, -h1),
                  __builtin_elementwise_fma(p2, sc2, -h2), __builtin_elementwise_fma(p3, sc2, -h3));
    } else {
        const float s = (float)sc;
        const float bi = ASYM ? (float)__builtin_bit_cast(f16, (uint16_t)bi_bits) : 0.f;
        uint32_t codes[8];
        if constexpr (BITS == 4) {
#pragma unroll
            for (int u = 0; u < 8; u++) codes[u] = (w[q] >> (4 * u)) & 15u;
        } else {
            const uint32_t lw = w[q >> 1] >> (16 * (q & 1));
#pragma unroll
            for (int u = 0; u < 8; u++) codes[u] = (lw >> (2 * u)) & 3u;
            if constexpr (BITS == 3) {
                const uint32_t hw = w[2] >> (8 * q);
#pragma unroll
                for (int u = 0; u < 8; u++) codes[u] |= ((hw >> u) & 1u) << 2;
            }
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const float c = (float)codes[u];
            const float v = ASYM ? __builtin_fmaf(c, s, bi) : (c - (float)(1 << (BITS - 1))) * s;
            const f16 h = (f16)v;
            hi[u] = h;
            lo[u] = (f16)(v - (float)h);
        }
    }
}

// OUT: 0 = f16 Y [M][N]; 1 = f32 slot z of the split-K partials [ks][M][N]; 2 = f16 mid [M][N/2] =
// silu(gate) * up of gate_up rows interleaved in groups of 16 (NCT even: tile 2p is 16 gate columns,
// tile 2p + 1 the matching up columns), gate and up rounded to f16 first as the reference stores them.
template <int BITS, bool ASYM, bool TILED, int NCT, int MT, int OUT>
__global__ __launch_bounds__(256) void k_gemv(const f16* __restrict__ A, const uint32_t* __restrict__ W,
                                              const f16* __restrict__ S, const f16* __restrict__ Bi,
                                              void* __restrict__ Y, int M, int N, int K, int gdiv, int ks) {
    typedef typename BlkT<BITS>::T Blk;
    constexpr int BB = 4 * BITS;                            // bytes per quant block
    constexpr int LPS = NCT * (ASYM ? 3 : 2) + 4 * MT;      // loads a lane issues per macro step
    constexpr int WAIT = vmcnt_imm((GV_PD - 1) * LPS);      // all but the oldest step's loads
    static_assert((GV_PD - 1) * LPS <= 63, "vmcnt holds at most 63");
    static_assert(!TILED || (BITS == 4 && !ASYM), "the tiled layout is int4 group 32 symmetric");
    static_assert(OUT != 2 || NCT % 2 == 0, "SiLU pairs gate and up column tiles");
    __shared__ f32x4 red[4][NCT][MT][64];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * NCT * 16, m0 = blockIdx.y * MT * 16, z = blockIdx.z;
    const int KB = K >> 5, SM = (KB + 3) >> 2, SZ = (SM + ks - 1) / ks;
    const int sb = z * SZ, se = min(SM, sb + SZ);
    const int nst = se > sb + wave ? (se - sb - wave + 3) >> 2 : 0;  // this wave's steps: sb + wave + 4t
    const int KG = KB / gdiv;                                         // scale groups per column (plain)

    const Rsrc rw = make_rsrc(W, (uint32_t)N * KB * BB), rs = make_rsrc(S, (uint32_t)N * (TILED ? KB : KG) * 2),
               rb = make_rsrc(ASYM ? Bi : S, (uint32_t)N * KG * 2), ra = make_rsrc(A, (uint32_t)M * K * 2);

    Blk wr[GV_PD][NCT];
    uint32_t sr[GV_PD][NCT], br[GV_PD][NCT];
    u32x4 ar[GV_PD][MT][4];
    f32x4 acc[NCT][MT];
#pragma unroll
    for (int ct = 0; ct < NCT; ct++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[ct][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Loads of this wave's step t into ring slot `slot`: block b = 4 s + g of each column tile and
    // the matching 32 k of each input row (zeros past the wave's steps, N, M and K).
    auto issue = [&](int t, int slot) {
        const int b = 4 * (sb + wave + 4 * t) + g;
        const bool bok = t < nst && b < KB;
#pragma unroll
        for (int ct = 0; ct < NCT; ct++) {
            const int n = n0 + 16 * ct + i;
            uint32_t wo = OOB, so = OOB, bo = OOB;
            if (bok && n < N) {
                if constexpr (TILED) {
                    const uint32_t idx = ((uint32_t)(n >> 5) * (uint32_t)(KB >> 1) + (uint32_t)(b >> 1)) * 64u +
                                         (uint32_t)(n & 31) * 2u + (uint32_t)(b & 1);
                    wo = idx * 16u;
                    so = idx * 2u;
                } else {
                    wo = ((uint32_t)n * KB + b) * BB;
                    so = bo = ((uint32_t)n * KG + (uint32_t)(b / gdiv)) * 2u;
                }
            }
            wr[slot][ct] = load_blk<BITS>(rw, wo);
            sr[slot][ct] = buf_b16(rs, so, 0);
            if constexpr (ASYM) br[slot][ct] = buf_b16(rb, bo, 0);
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int m = m0 + 16 * mt + i;
            const uint32_t ao = bok && m < M ? ((uint32_t)m * K + 32u * b) * 2u : OOB;
#pragma unroll
            for (int q = 0; q < 4; q++) ar[slot][mt][q] = buf_b128(ra, ao + 16u * q, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // each step's loads stay together and in step order
    };
    auto compute = [&](int slot) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            f16x8 hi[NCT], lo[NCT];
#pragma unroll
            for (int ct = 0; ct < NCT; ct++)
                deq8<BITS, ASYM, TILED>(wr[slot][ct], sr[slot][ct], ASYM ? br[slot][ct] : 0u, q, hi[ct], lo[ct]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const f16x8 av = __builtin_bit_cast(f16x8, ar[slot][mt][q]);
#pragma unroll
                for (int ct = 0; ct < NCT; ct++) {
                    acc[ct][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[ct], av, acc[ct][mt], 0, 0, 0);
                    acc[ct][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[ct], av, acc[ct][mt], 0, 0, 0);
                }
            }
        }
    };

    // Ring of GV_PD steps: wait for the oldest, use it, refill its slot with the step GV_PD later
    // (steps past this wave's count load nothing, so the wait counts stay exact).
    issue(0, 0);
    issue(1, 1);
    issue(2, 2);
    issue(3, 3);
    for (int t = 0; t < nst; t += GV_PD) {
        wait_loads<WAIT>();
        compute(0);
        issue(t + 4, 0);
        wait_loads<WAIT>();
        compute(1);
        issue(t + 5, 1);
        wait_loads<WAIT>();
        compute(2);
        issue(t + 6, 2);
        wait_loads<WAIT>();
        compute(3);
        issue(t + 7, 3);
    }
    wait_loads<vmcnt_imm(0)>();

    // The 4 waves' sums, added in wave order.  Lane l of tile (ct, mt) holds D[4 (l / 16) + r][l % 16]:
    // output column n0 + 16 ct + 4 (l / 16) + r of input row m0 + 16 mt + l % 16.
#pragma unroll
    for (int ct = 0; ct < NCT; ct++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) red[wave][ct][mt][lane] = acc[ct][mt];
    __syncthreads();
    auto total = [&](int ct, int mt, int l) {
        f32x4 v = red[0][ct][mt][l];
#pragma unroll
        for (int w = 1; w < 4; w++) {
            const f32x4 x = red[w][ct][mt][l];
            v[0] += x[0], v[1] += x[1], v[2] += x[2], v[3] += x[3];
        }
        return v;
    };
    if constexpr (OUT == 2) {
        f16* mid = static_cast<f16*>(Y);
        const int half = N >> 1;
        for (int it = tid; it < (NCT / 2) * MT * 64; it += 256) {
            const int l = it & 63, mt = (it >> 6) % MT, p = (it >> 6) / MT;
            const int m = m0 + 16 * mt + (l & 15);
            const int j = (n0 >> 1) + 16 * p + 4 * (l >> 4);
            if (m >= M || j >= half) continue;
            const f32x4 gv = total(2 * p, mt, l), uv = total(2 * p + 1, mt, l);
            f16x4 o;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float gg = (float)(f16)gv[r], uu = (float)(f16)uv[r];
                o[r] = (f16)silu_mul(gg, uu);
            }
            *reinterpret_cast<f16x4*>(mid + (size_t)m * half + j) = o;
        }
        return;
    }
    const bool vec = (N & 3) == 0;
    for (int it = tid; it < NCT * MT * 64; it += 256) {
        const int l = it & 63, mt = (it >> 6) % MT, ct = (it >> 6) / MT;
        const int m = m0 + 16 * mt + (l & 15), n = n0 + 16 * ct + 4 * (l >> 4);
        if (m >= M || n >= N) continue;
        const f32x4 v = total(ct, mt, l);
        if constexpr (OUT == 0) {
            f16* y = static_cast<f16*>(Y) + (size_t)m * N + n;
            if (vec) {
                *reinterpret_cast<f16x4*>(y) = f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (n + r < N) y[r] = (f16)v[r];
            }
        } else {
            float* y = static_cast<float*>(Y) + ((size_t)z * M + m) * N + n;
            if (vec) {
                __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(y));
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (n + r < N) y[r] = v[r];
            }
        }
    }
}

// The same product for many rows of the plain formats.  k_gemv dequantizes every weight again for each 32
// rows and reads A once per 16 columns, which for a 2048 x 2048 matrix at 300 rows is ten dequants and 157 MB
// of A: 32.8 us.  Here a workgroup takes BM = 16 MT rows x 64 columns (4 waves side by side, 16 columns
// each), so a weight is dequantized once per BM rows:
//  * A's step (BM rows x 128 k) goes straight to a ring of 4 LDS stages shared by the waves, the weights and
//    scales to a ring of 4 register stages, both three steps ahead (the scheme of the int4 kernel with
//    pipelined loads: 16-byte chunk q of a stage holds row q / 16, k-chunk (q % 16) ^ (row % 16); steps past
//    the range load zeros, so the waits are exact);
//  * lane (j, g) dequantizes block g of its column j to the f32 values that k_gemv does, split into the same
//    f16 hi + lo, in packed steps: 8 codes become 4 f16 pairs 1024 + q by masks; symmetric formats multiply
//    (q - zero) by the scale in f16 (hi, rounded once) and take the residual with an f16 fma (lo, exact, as the
//    product is); asymmetric ones take q s + b in f32 (one v_fma_mix_f32 each) and its residual likewise;
//  * KH = 2: 8 waves, two k parts with their own rings, whose sums meet in LDS (a workgroup's chain of steps,
//    which a short grid waits for, halves);
//  * bound by each wave's chain of dequant (int3 asymmetric: about 190 VALU a step), fragment reads (every wave
//    reads the whole A tile) and MFMAs, one after the other: 15.0 us for the 2048 x 2048 matrix at 300 rows, of
//    whose CUs' cycles counters show the MFMAs busy for 24%, 2056 VALU instructions a wave (two waves a SIMD: about
//    half of the issue), and one bank-conflict cycle for two of the fragment reads'.  Pinning the dequant among the
//    MFMAs with scheduling groups made it 21; 128 rows per workgroup 26.
template <int BITS>
__device__ __forceinline__ void code_pairs(const typename BlkT<BITS>::T& w, int q, uint32_t (&p)[4]) {
    constexpr uint32_t EXP = 0x64006400u;  // f16 1024 in both halves: | q gives 1024 + q
    if constexpr (BITS == 4) {             // element e at bits 4e: x holds 4 of them, the odd ones 16 bits above
        const uint32_t lo = w[q] & 0xFFFFu, hi = w[q] >> 16, x = lo | (lo << 12), y = hi | (hi << 12);
        p[0] = and_or(x, 0x000F000Fu, EXP);
        p[1] = and_or(x >> 8, 0x000F000Fu, EXP);
        p[2] = and_or(y, 0x000F000Fu, EXP);
        p[3] = and_or(y >> 8, 0x000F000Fu, EXP);
    } else {  // element e of the 8 at bits 2e (the low two bits), and for int3 bit e of a byte of w[2]
        const uint32_t lw = (w[q >> 1] >> (16 * (q & 1))) & 0xFFFFu, x = lw | (lw << 14);
        uint32_t h = 0;
        if constexpr (BITS == 3) {
            const uint32_t hw = (w[2] >> (8 * q)) & 0xFFu;
            h = (hw << 2) | (hw << 17);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            p[k] = and_or(x >> (4 * k), 0x00030003u, EXP);
            if constexpr (BITS == 3) {
                OPAQUE_V(p[k]);  // (not merged into two ands and a three-way or)
                p[k] |= (h >> (2 * k)) & 0x00040004u;
            }
        }
    }
}

template <int BITS, bool ASYM, int MT, bool PARTIAL, int KH>
__global__ __launch_bounds__(256 * KH) void k_gemm_fmt(const f16* __restrict__ A, const uint32_t* __restrict__ W,
                                                  const f16* __restrict__ S, const f16* __restrict__ Bi,
                                                  void* __restrict__ Y, int M, int N, int K, int gdiv, int ks) {
    typedef typename BlkT<BITS>::T Blk;
    constexpr int BB = 4 * BITS;             // bytes per quant block
    constexpr int BM = 16 * MT, BN = 64;
    constexpr int STAGE = BM * 256;          // bytes of one A stage (128 k of BM rows)
    constexpr int PER = MT + (ASYM ? 3 : 2);  // vector-memory loads a thread issues per step
    static_assert(2 * PER <= 63, "vmcnt holds at most 63");
    static_assert((KH - 1) * MT * 4096 <= KH * STAGE, "the parts' sums fit one stage array");
    __shared__ __align__(1024) uint8_t As0[KH * STAGE], As1[KH * STAGE], As2[KH * STAGE], As3[KH * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wall = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kh = wall >> 2, wave = wall & 3;  // k part, wave within it
    uint8_t *const R0 = As0 + kh * STAGE, *const R1 = As1 + kh * STAGE, *const R2 = As2 + kh * STAGE,
            *const R3 = As3 + kh * STAGE;
    const int j = lane & 15, g = lane >> 4;
    int bx, by, bz;
    xcd_tile(blockIdx.x + (N + BN - 1) / BN * (blockIdx.y + (M + BM - 1) / BM * blockIdx.z), (N + BN - 1) / BN,
             (M + BM - 1) / BM, ks, bx, by, bz);
    const int m0 = by * BM, n0 = bx * BN;
    // K is a multiple of 128; part kh of split bz takes `steps` steps from sb (the last ones perhaps fewer, or
    // none: their loads are then out of range), `trips` of them run in every part
    const int KB = K >> 5, SM = K >> 7, SZ = (SM + ks - 1) / ks, trips = (SZ + KH - 1) / KH;
    const int s1 = min(SM, (bz + 1) * SZ), sb = min(bz * SZ + kh * trips, s1), steps = min(trips, s1 - sb);
    const int KG = KB / gdiv;
    const Rsrc ra = make_rsrc(A, (uint32_t)M * K * 2), rw = make_rsrc(W, (uint32_t)N * KB * BB),
               rs = make_rsrc(S, (uint32_t)N * KG * 2), rb = make_rsrc(ASYM ? Bi : S, (uint32_t)N * KG * 2);
    uint32_t aoff[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int q = (i * 4 + wave) * 64 + lane, row = q >> 4, c = (q & 15) ^ (row & 15);
        aoff[i] = (uint32_t)(min(m0 + row, M - 1) * K + c * 8) * 2u;
    }
    const int n = n0 + wave * 16 + j;
    // fragment read of row tile a, slice s: row 16a + j, k-chunk 4g + s
    uint32_t foff[4];
#pragma unroll
    for (int s = 0; s < 4; s++) foff[s] = j * 256 + (((4 * g + s) ^ j) << 4);

    f32x4 acc[MT];
#pragma unroll
    for (int a = 0; a < MT; a++) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    Blk bw[4];
    uint32_t bs[4], bb[4];
    auto issue = [&](int it, uint8_t* dst, int slot) {
        const bool in = it < steps;
        const uint32_t ka = in ? (uint32_t)(sb + it) * 256u : OOB;
        const int b = 4 * (sb + it) + g;
        const bool ok = in && n < N;
        const uint32_t wo = ok ? ((uint32_t)n * KB + b) * BB : OOB;
        const uint32_t so = ok ? ((uint32_t)n * KG + (uint32_t)(b / gdiv)) * 2u : OOB;
#pragma unroll
        for (int i = 0; i < MT; i++) buf_lds16(ra, aoff[i], ka, dst + (i * 4 + wave) * 1024);
        bw[slot] = load_blk<BITS>(rw, wo);
        bs[slot] = buf_b16(rs, so, 0);
        if constexpr (ASYM) bb[slot] = buf_b16(rb, so, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto deq = [&](int slot, int q, f16x8& hi, f16x8& lo) {
        const f16 sc = __builtin_bit_cast(f16, (uint16_t)bs[slot]);
        uint32_t p[4];
        code_pairs<BITS>(bw[slot], q, p);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            f16x2 h, l;
            if constexpr (ASYM) {
                const float s32 = (float)sc, b32 = (float)__builtin_bit_cast(f16, (uint16_t)bb[slot]);
                const f16x2 c = __builtin_bit_cast(f16x2, p[k]) - f16x2{(f16)1024.f, (f16)1024.f};
                const float v0 = mul_add_f16(c[0], s32, b32), v1 = mul_add_f16(c[1], s32, b32);
                split2(v0, v1, h, l);
            } else {
                constexpr float Z = 1024.f + (float)(1 << (BITS - 1));
                const f16x2 c = __builtin_bit_cast(f16x2, p[k]) - f16x2{(f16)Z, (f16)Z}, sc2 = f16x2{sc, sc};
                h = c * sc2;
                l = __builtin_elementwise_fma(c, sc2, -h);
            }
            hi[2 * k] = h[0], hi[2 * k + 1] = h[1];
            lo[2 * k] = l[0], lo[2 * k + 1] = l[1];
        }
    };
    auto step = [&](const uint8_t* cur, uint8_t* fill, int slot, int it) {
        issue(it + 3, fill, (slot + 3) & 3);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            f16x8 hi, lo, af[MT];
#pragma unroll
            for (int a = 0; a < MT; a++) af[a] = *reinterpret_cast<const f16x8*>(cur + a * 4096 + foff[s]);
            deq(slot, s, hi, lo);
#pragma unroll
            for (int a = 0; a < MT; a++) acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[a], hi, acc[a], 0, 0, 0);
#pragma unroll
            for (int a = 0; a < MT; a++) acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[a], lo, acc[a], 0, 0, 0);
        }
        wait_loads<vmcnt_imm(2 * PER)>();  // the loads of steps it + 2, it + 3 may still be in flight
        bar_noflush();
    };
    issue(0, R0, 0);
    issue(1, R1, 1);
    issue(2, R2, 2);
    wait_loads<vmcnt_imm(2 * PER)>();
    bar_noflush();
    int it = 0;
    do {
        step(R0, R3, 0, it);
        step(R1, R0, 1, it + 1);
        step(R2, R1, 2, it + 2);
        step(R3, R2, 3, it + 3);
        it += 4;
    } while (it < trips);
    wait_loads<vmcnt_imm(0)>();  // the trailing out-of-range loads, before the ring is reused
    if constexpr (KH > 1) {
        // the parts' sums, added in k order through the ring: wave w's tile a of part kh at stage a
        lds_barrier();
        f32x4* const x = reinterpret_cast<f32x4*>(As0);
        if (kh)
#pragma unroll
            for (int a = 0; a < MT; a++) x[(((kh - 1) * MT + a) * 4 + wave) * 64 + lane] = acc[a];
        lds_barrier();
        if (kh) return;
#pragma unroll
        for (int p = 1; p < KH; p++)
#pragma unroll
            for (int a = 0; a < MT; a++) {
                const f32x4 v = x[(((p - 1) * MT + a) * 4 + wave) * 64 + lane];
                acc[a][0] += v[0], acc[a][1] += v[1], acc[a][2] += v[2], acc[a][3] += v[3];
            }
    }
    if (n >= N) return;
    // acc[a][r] is row m0 + 16a + 4g + r of column n
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = m0 + a * 16 + g * 4 + r;
            if (m >= M) continue;
            if constexpr (PARTIAL)
                __builtin_nontemporal_store(acc[a][r], static_cast<float*>(Y) + ((size_t)bz * M + m) * N + n);
            else
                static_cast<f16*>(Y)[(size_t)m * N + n] = (f16)acc[a][r];
        }
}

typedef void (*GemvFn)(const f16*, const uint32_t*, const f16*, const f16*, void*, int, int, int, int, int);

template <int BITS, bool ASYM, bool TILED, int NCT>
GemvFn pick_mt(int mt, int out) {
    if (mt == 1) {
        if (out == 0) return k_gemv<BITS, ASYM, TILED, NCT, 1, 0>;
        if (out == 1) return k_gemv<BITS, ASYM, TILED, NCT, 1, 1>;
        if constexpr (NCT % 2 == 0) return k_gemv<BITS, ASYM, TILED, NCT, 1, 2>;
    } else {
        if (out == 0) return k_gemv<BITS, ASYM, TILED, NCT, 2, 0>;
        if (out == 1) return k_gemv<BITS, ASYM, TILED, NCT, 2, 1>;
        if constexpr (NCT % 2 == 0) return k_gemv<BITS, ASYM, TILED, NCT, 2, 2>;
    }
    return nullptr;
}

GemvFn pick_gemv(int bits, bool asym, bool tiled, int nct, int mt, int out) {
    if (tiled) return nct == 2 ? pick_mt<4, false, true, 2>(mt, out) : pick_mt<4, false, true, 1>(mt, out);
    if (out == 2) return nullptr;
    switch (bits * 2 + (asym ? 1 : 0)) {
        case 8: return pick_mt<4, false, false, 1>(mt, out);
        case 9: return pick_mt<4, true, false, 1>(mt, out);
        case 6: return pick_mt<3, false, false, 1>(mt, out);
        case 7: return pick_mt<3, true, false, 1>(mt, out);
        case 4: return pick_mt<2, false, false, 1>(mt, out);
        case 5: return pick_mt<2, true, false, 1>(mt, out);
        default: return nullptr;
    }
}

// k_gemm_fmt for a plain format
template <int MT, int KH, bool PARTIAL>
GemvFn pick_fmt(int bits, bool asym) {
    switch (bits * 2 + (asym ? 1 : 0)) {
        case 8: return k_gemm_fmt<4, false, MT, PARTIAL, KH>;
        case 9: return k_gemm_fmt<4, true, MT, PARTIAL, KH>;
        case 6: return k_gemm_fmt<3, false, MT, PARTIAL, KH>;
        case 7: return k_gemm_fmt<3, true, MT, PARTIAL, KH>;
        case 4: return k_gemm_fmt<2, false, MT, PARTIAL, KH>;
        case 5: return k_gemm_fmt<2, true, MT, PARTIAL, KH>;
        default: return nullptr;
    }
}

}  // namespace

GemvPlan gemv_plan(int M, int N, int K, bool tiled, int out, size_t max_part_elems) {
    GemvPlan p;
    p.mt = M <= 16 ? 1 : 2;
    const int rb = (M + 16 * p.mt - 1) / (16 * p.mt);
    // Plain formats whose k_gemv grid (16 columns x 32 rows each) is more than one workgroup per CU: the kernel
    // that dequantizes a weight once per 32 or 64 rows.  In its grid (64 columns each) two k parts per workgroup
    // while that is at most one workgroup per CU, 32 rows before 64.  us on MI355X, int3 asymmetric group 64,
    // k_gemv | 32 rows, 2 parts | 64 rows, 2 parts | 64 rows, 1 part:
    //   2048 x 2048  64 rows  8.7 | 11.8 | 14.9 | 16.5    96 rows 14.8 | 12.0 | 15.1 | 16.6
    //               300 rows 32.9 | 20.8 | 15.5 | 17.1   600 rows 64.8 | 31.6 | 30.8 | 27.0   1500: 146 | 63 | 53 | 46
    //    512 x 2048 200 rows  8.6 | 11.9 | 14.9 | 16.4   300 rows 14.6 | 12.1 | 14.9 | 16.6
    //   2048 x 6144  64 rows 18.6 | 27.8 | 35.6 | 43.1   300 rows 80.5 | 48.5 | 36.3 | 43.2   1500: 372 | 155 | 121 | 113
    // Up to 16 rows most of its 32 are padding, for k_gemv half of 32: more than two workgroups per CU, and 8 rows.
    // Six formats of int2 to int4, K = 2048, k_gemv's time over this kernel's (least, most):
    //   N = 5120: 8 rows 0.76, 0.99  16 rows 0.87, 1.11  17 rows 1.02, 1.36  33 rows 1.32, 1.71
    //   N = 8256: 4 rows 0.96, 1.29   8 rows 1.04, 1.34  17 rows 1.44, 1.85;  N = 12288: 4 rows 0.99, 1.32  8 rows 1.06, 1.35
    // A single step (K = 128), half of whose two parts idle, from two workgroups per CU: 4096 columns, int4
    // asymmetric, 64 rows 6.77 | 6.94, 65 rows (768) 9.86 | 7.01.
    const size_t blocks = (size_t)((N + 15) / 16) * rb;
    if (!tiled && out != 2 && K % 128 == 0 && blocks > 256 && (blocks > 512 ? M >= 8 : M > 16 && K > 128)) {
        const size_t cols = (N + 63) / 64, g2 = cols * ((M + 31) / 32), g4 = cols * ((M + 63) / 64);
        p.rows = g2 <= 256 ? 2 : 4;
        p.kh = p.rows == 2 || g4 <= 256 ? 2 : 1;
        if (out == 1)  // slots for the consumer to add: until the grid covers the chip, parts of at least 4 steps
            while (p.ks < 8 && (p.rows == 2 ? g2 : g4) * p.ks * 2 <= 256 && K / 128 / (p.ks * 2 * p.kh) >= 4 &&
                   (size_t)(p.ks * 2) * M * N <= max_part_elems)
                p.ks *= 2;
        return p;
    }
    // f16 outputs own their whole k range; two column tiles per workgroup where that still gives
    // about one workgroup per CU (or more), one otherwise
    p.nct = tiled && (out == 2 || (size_t)((N + 31) / 32) * rb >= 240) ? 2 : 1;
    p.ks = 1;
    if (out == 1) {
        // partials: split k until the grid covers the chip (each wave keeps >= 1 macro step)
        const int groups = ((N + 16 * p.nct - 1) / (16 * p.nct)) * rb;
        const int SM = (K / 32 + 3) / 4;
        while (p.ks < 8 && groups * p.ks < 256 && SM / (p.ks * 2) >= 4 &&
               (size_t)(p.ks * 2) * M * N <= max_part_elems)
            p.ks *= 2;
    }
    return p;
}

void gemv(const f16* A, const uint32_t* W, const f16* S, const f16* Bi, void* Y, int out, int M, int N, int K, int bits,
          int group, bool asym, bool tiled, const GemvPlan& plan, hipStream_t st) {
    GemvPlan p = plan;
    if (p.rows && reinterpret_cast<uintptr_t>(A) % 16) {
        // k_gemm_fmt moves A's 16-byte pieces straight to LDS: an A that does not start on one keeps k_gemv,
        // which loads it to registers, with the same k splits
        p.nct = 1;
        p.mt = M <= 16 ? 1 : 2;
        p.rows = 0;
        p.kh = 1;
    }
    SD_CHECK(M >= 1 && N >= 1 && K >= 32 && K % 32 == 0, "gemv: need M, N >= 1 and K a multiple of 32");
    SD_CHECK(bits == 2 || bits == 3 || bits == 4, "gemv: weights must be int2, int3 or int4");
    SD_CHECK(group >= 32 && group % 32 == 0 && K % group == 0, "gemv: the group must be a multiple of 32 dividing K");
    SD_CHECK(!tiled || (bits == 4 && group == 32 && !asym && w4_tileable(N, K)),
             "gemv: the tiled layout is int4 group 32 symmetric with N a multiple of 32");
    SD_CHECK(out != 2 || (tiled && p.nct == 2 && N % 32 == 0), "gemv: SiLU * mul needs the tiled gate_up in pairs");
    SD_CHECK(p.ks >= 1 && (out == 1 || p.ks == 1), "gemv: only partial outputs split k");
    SD_CHECK((size_t)N * (K / 32) * 4 * bits < 0x80000000u && (size_t)M * K * 2 < 0x80000000u,
             "gemv: operands must be below 2 GiB");
    GemvFn f = nullptr;
    if (p.rows) {
        SD_CHECK(!tiled && out != 2 && K % 128 == 0 && ((p.rows == 2 && p.kh == 2) || (p.rows == 4 && p.kh <= 2)),
                 "gemv: no such row tile");
        if (p.rows == 2) f = out ? pick_fmt<2, 2, true>(bits, asym) : pick_fmt<2, 2, false>(bits, asym);
        else if (p.kh == 2) f = out ? pick_fmt<4, 2, true>(bits, asym) : pick_fmt<4, 2, false>(bits, asym);
        else f = out ? pick_fmt<4, 1, true>(bits, asym) : pick_fmt<4, 1, false>(bits, asym);
    } else {
        f = pick_gemv(bits, asym, tiled, p.nct, p.mt, out);
    }
    SD_CHECK(f, "gemv: no kernel for this format and output");
    const dim3 grid = p.rows ? dim3((N + 63) / 64, (M + 16 * p.rows - 1) / (16 * p.rows), p.ks) : dim3((N + 16 * p.nct - 1) / (16 * p.nct), (M + 16 * p.mt - 1) / (16 * p.mt), p.ks);
    const int gdiv = group / 32;
    KernelEvents* ke = kernel_events();
    if (ke && ke->launches == 0) {
        hipExtLaunchKernelGGL(f, grid, dim3(256 * p.kh), 0, st, ke->start, ke->stop, 0u, A, W, S, Bi, Y, M, N, K, gdiv, p.ks);
        ke->launches++;
    } else {
        hipLaunchKernelGGL(f, grid, dim3(256 * p.kh), 0, st, A, W, S, Bi, Y, M, N, K, gdiv, p.ks);
    }
    launched("gemv");
}

}  // namespace sd
