// Full-attention sublayer on gfx950: q/k RMSNorm + partial rotate-half RoPE with the K/V cache
// write (reference: src/kernels.rs:400-448), and causal GQA attention with a sigmoid output gate
// (reference: src/kernels.rs:453-541).
//
// Attention runs on MFMA: k_attn for few rows, k_attn_rows for many (attn_plan).  When the query
// blocks alone cannot fill the GPU (the short question suffix over a long cached prefix), the key range
// is also split over workgroups and a combine kernel merges the partial (max, sum, acc).  As in the
// reference, q is pre-scaled by 1/sqrt(hd) and rounded to f16 before the dot products.  The cache is kept in blocks of 32
// keys, so that the fragment loads of a key block touch whole cache lines: K as [hk][ctx / 32]
// [hd / 32][32 keys][32 dims] (a load of 16 keys x 8 dims reads pairs of consecutive keys' 64 bytes),
// V transposed as [hk][ctx / 32][hd][32 keys] (a block's V^T is 16 KB of consecutive bytes).
#include <climits>
#include <cmath>

#include "common.h"
#include "device.h"

namespace sd {
namespace {

constexpr int BQ = 16;  // queries per workgroup
constexpr int ATTN_KS_MAX = 8;  // key splits the workspace and k_attn_combine provide for

// Kernel arguments: what the prologue needs first, and the head shape as ints, lead (the first 16
// dwords are preloaded into SGPRs, up to the first struct argument).
template <int HD>
__global__ __launch_bounds__(256) void k_qk_prep(const f16* __restrict__ big, const uint32_t* __restrict__ lu, int L,
                                                 int HQ, int HK, int RD, int stride, int ctx,
                                                 const uint32_t* __restrict__ rowt, const float* __restrict__ qw,
                                                 const float* __restrict__ kw, const float* __restrict__ rope,
                                                 f16* __restrict__ Q, f16* __restrict__ Kc, f16* __restrict__ Vc) {
    const AttnShape s{HQ, HK, HD, RD, stride, ctx};
    // Workgroup (4 rows, one q or kv head): wave w takes row w, lane l the 4 dimensions 4l..4l+3
    // (8-byte loads and stores, the norm a wave reduction).  A kv head also writes the 4 rows of
    // V^T, dimension by dimension: 8 contiguous bytes per dimension.
    static_assert(HD == 256, "qk_prep is written for 256-wide heads");
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // without Q the grid covers the kv heads only (the attention kernel computes its queries itself)
    const int t0 = blockIdx.x * 4, slot = Q ? (int)blockIdx.y : s.HQ + (int)blockIdx.y;
    const int P = (int)lu[1];
    const bool isq = slot < s.HQ;
    const int k_off = 2 * s.HQ * HD, v_off = k_off + s.HK * HD;
    const int nt = min(4, L - t0);
    if (!isq) {  // V^T in 32-key blocks, [hk][ctx / 32][hd][32]: thread d writes rows t0 .. t0+3
        const int kh = slot - s.HQ, d = tid;
        f16 v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = i < nt ? big[(size_t)(t0 + i) * s.stride + v_off + kh * HD + d] : (f16)0.f;
        auto at = [&](int pos) { return Vc + (((size_t)kh * (s.ctx / 32) + pos / 32) * HD + d) * 32 + pos % 32; };
        if (nt == 4 && ((P + t0) & 3) == 0) {  // the 4 rows lie in one block
            *reinterpret_cast<f16x4*>(at(P + t0)) = f16x4{v[0], v[1], v[2], v[3]};
        } else {
            for (int i = 0; i < nt; i++) *at(P + t0 + i) = v[i];
        }
    }
    __shared__ __align__(16) float nrow[4][HD];  // a wave's normalized row (rotary dims not a multiple of 8)
    const float* nw = isq ? qw : kw;
    const float4 w4 = *reinterpret_cast<const float4*>(nw + 4 * lane);
    const int rd2 = s.RD / 2;
    if (wv < nt) {
        const int t = t0 + wv;
        const int pos = P + t;                                        // cache row
        const int rpos = P + (rowt ? (int)(rowt[t] & 0xFFFFu) : t);  // RoPE position
        const f16* src = big + (size_t)t * s.stride + (isq ? slot * 2 * HD : k_off + (slot - s.HQ) * HD) + 4 * lane;
        const f16x4 x4 = *reinterpret_cast<const f16x4*>(src);
        float x[4] = {(float)x4[0], (float)x4[1], (float)x4[2], (float)x4[3]};
        float ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
        const float inv = 1.0f / sqrtf(ss / (float)HD + 1e-6f);
        const float wv4[4] = {w4.x, w4.y, w4.z, w4.w};
        float n[4];
#pragma unroll
        for (int u = 0; u < 4; u++) n[u] = x[u] * inv * wv4[u];
        // rotate-half RoPE on dims < RD: the partner of dim d is d +- RD/2.  With RD a multiple of 8
        // it is element u of lane l +- RD/8 (a lane shuffle); otherwise it is read back from the
        // wave's row in LDS (the wave's own stores: LDS operations of one wave complete in order).
        float pn[4];
        if (rd2 % 4 == 0) {
            const int sh = rd2 / 4;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float up = __shfl(n[u], (lane + sh) & 63), dn = __shfl(n[u], (lane - sh) & 63);
                pn[u] = 4 * lane < rd2 ? up : dn;
            }
        } else {
            *reinterpret_cast<float4*>(&nrow[wv][4 * lane]) = float4{n[0], n[1], n[2], n[3]};
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int d = 4 * lane + u;
                pn[u] = d < s.RD ? nrow[wv][d < rd2 ? d + rd2 : d - rd2] : 0.f;
            }
        }
        f16x4 r4;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int d = 4 * lane + u;
            float r = n[u];
            if (d < s.RD) {
                const int j = d % rd2;
                const float c = rope[((size_t)rpos * rd2 + j) * 2], sn = rope[((size_t)rpos * rd2 + j) * 2 + 1];
                r = d < rd2 ? n[u] * c - pn[u] * sn : n[u] * c + pn[u] * sn;
            }
            r4[u] = (f16)r;
        }
        if (isq) *reinterpret_cast<f16x4*>(Q + ((size_t)slot * L + t) * HD + 4 * lane) = r4;
        else
            *reinterpret_cast<f16x4*>(Kc + (((size_t)(slot - s.HQ) * (s.ctx / 32) + pos / 32) * (HD / 32) + lane / 8) * 1024 +
                                      (pos % 32) * 32 + 4 * (lane % 8)) = r4;
    }
}

// The online softmax runs in base 2: scores are scaled by log2(e) and exponentiated with
// v_exp_f32, exp(s - m) = 2^(s log2 e - m log2 e); max and sum states (also those the combine kernel
// merges) are in these units.
constexpr float LOG2E = 1.4426950408889634f;
__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float wave_max16(float v) {  // max over lanes {l, l^16, l^32, l^48}
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float wave_sum16(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

// Causal GQA attention on MFMA.  A workgroup takes 16 queries of one q head; its 4 waves split the
// key range in blocks of 32 keys (wave w takes blocks w, w+4, ...) and merge their online-softmax
// states in LDS at the end.  Per 32-key block a wave computes S^T = K Q^T (keys x queries, 2 x 8
// v_mfma_f32_16x16x32_f16 over the 256 dims), the online softmax per query (column), then
// O^T += V^T P^T (256 dims x 16 queries); with S^T in the MFMA output layout, P^T is already in
// the B-operand layout (lane = query, 8 keys), and the V cache is stored transposed so V^T
// fragments are contiguous (the keys of a block are permuted so that they are 8 consecutive).  P is
// split into f16 hi + lo (two MFMAs) so that the product keeps the reference's f32 P.V to about 22
// bits.  With ks > 1 the workgroups along z also split the keys
// and write unnormalised (acc, max, sum) for k_attn_combine.
template <int HD, int QRD>
__global__ __launch_bounds__(256) void k_attn(const f16* __restrict__ Q, const f16* __restrict__ Kc,
                                              const f16* __restrict__ Vt, const uint32_t* __restrict__ lu, int L,
                                              int HQ, int HK, int stride, int ctx, int ks,
                                              const uint32_t* __restrict__ rowt, const f16* __restrict__ big,
                                              f16* __restrict__ out, float* __restrict__ pacc, float* __restrict__ pml,
                                              const float* __restrict__ qw, const float* __restrict__ rope, int RD) {
    const AttnShape s{HQ, HK, HD, 0, stride, ctx};
    static_assert(HD == 256, "attention is written for 256-wide heads");
    constexpr int ND = HD / 16;   // 16 output dimension tiles
    constexpr int NS = HD / 32;   // 8 k steps over the head dimension
    constexpr int KB = 32;        // keys per block
    __shared__ float Om[4][16][HD + 4];  // per-wave unnormalised outputs [query][dim]
    __shared__ float Mm[4][16], Lm[4][16];
    __shared__ __align__(16) f16 Qs[16][HD + 8];  // the workgroup's queries, scaled (row padding: no bank conflicts on the fragment reads)
    // wv is wave-uniform (readfirstlane): the key loop below is then a scalar loop, not a divergent one
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fq = lane & 15, fg = lane >> 4;
    // cache rows below Pv are every sequence's shared prefix: the cached prefix (P) and, in a forward
    // whose sequences continue one state sequence (lu[6] > 0), that state's rows too
    const int P = (int)lu[1], Pv = P + (int)lu[6];
    SGPR_BATCH("s"(P), "s"(Pv), "s"(rowt), "s"(big), "s"(out), "s"(pacc), "s"(pml));
    const int t0 = blockIdx.x * 16, h = blockIdx.y, z = blockIdx.z;
    const int kh = h / (s.HQ / s.HK);
    const int nq = min(16, L - t0);
    const int nkeys = P + t0 + nq;  // keys 0 .. P + t0 + nq - 1 can be attended
    const int span = ((nkeys + ks - 1) / ks + KB - 1) / KB * KB;
    const int kbeg = z * span, kend = min(nkeys, kbeg + span);
    const float scale = 1.0f / sqrtf((float)HD);
    const int qpos = P + t0 + fq;  // cache row of this lane's query
    const bool qok = fq < nq;
    // keys below jend can be attended by this lane's query (none past nq): the causal limit and the
    // split's end
    const int jend = qok ? min(kend, qpos + 1) : INT_MIN;
    // The row table words of this lane's query and of the tile's first row: buffer loads, issued
    // together and without a branch (a null table is a 0-byte buffer, whose loads read 0).
    const Rsrc rr = make_rsrc(rowt, rowt ? (uint32_t)L * 4u : 0u);
    const uint32_t rwq = buf_b32(rr, (uint32_t)(t0 + min(fq, nq - 1)) * 4u, 0);
    const uint32_t rw0 = buf_b32(rr, (uint32_t)t0 * 4u, 0);
    // and, for the fused query norm and RoPE, that of query 4 wv + lane / 16 (read for its position)
    const uint32_t rwp = QRD ? buf_b32(rr, (uint32_t)(t0 + min(4 * wv + (lane >> 4), nq - 1)) * 4u, 0) : 0u;
    // first cache row of the query's own sequence: rows [Pv, qlo) belong to other sequences
    const int qlo = P + (int)(rwq >> 16);
    // the tile's first row starts the earliest sequence among its queries: a key block inside
    // [Pv, qlo0) belongs to other sequences for every query, is wholly masked and is skipped (its
    // softmax update would leave the running max, sum and output unchanged)
    const int qlo0 = P + (int)(rw0 >> 16);

    // Q^T fragments (B operand), filled after the first key block's loads are issued
    f16x8 qf[NS];
    // The epilogue gives thread tid query qe = tid / 16 and the 16 dimensions d0 .. d0 + 15: its
    // output gates are loaded here (two 16-byte loads, unconditionally: queries past nq read the
    // last one's), while the keys are processed.
    const int qe = tid >> 4, d0 = (tid & 15) * 16;
    f16x8 gv[2];
    {
        const f16* gp = big + (size_t)(t0 + min(qe, nq - 1)) * s.stride + h * 2 * HD + HD + d0;
        gv[0] = *reinterpret_cast<const f16x8*>(gp);
        gv[1] = *reinterpret_cast<const f16x8*>(gp + 8);
    }
    f32x4 acc[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    const f16* Kb = Kc + (size_t)kh * s.ctx * HD;
    const f16* Vb = Vt + (size_t)kh * HD * s.ctx;

    // The wave's key blocks are kbeg + 32 wv + 128 n below kend; those wholly inside [Pv, qlo0) are
    // skipped.  A block's K and V fragments are loaded one block ahead, into the other of two
    // register sets, while the current block's MFMAs and softmax run (one wave per SIMD: no other
    // wave hides a block's load latency).  Every step issues the same 32 loads (past the end they
    // re-read the last block, never used), so the explicit vmcnt wait is exact.
    auto next_block = [&](int j) {
        if (j >= Pv && j + KB <= qlo0) j += ((qlo0 - KB - j) / (4 * KB) + 1) * (4 * KB);
        return j;
    };
    // Keys are ordered inside the 32-key block so that lane (query fq, group fg) ends up with the
    // probabilities of keys j0 + 8fg .. +7: row i of S^T tile tt is key j0 + 8(i/4) + 4tt + i%4.
    // Then the V^T fragment of lane (dim fq, group fg) is those 8 keys, one 16-byte load.
    // The loads of a block stay where they are issued, ahead of the block in flight: the compiler
    // would otherwise sink them to their first use, a block later.  A memory clobber alone does not
    // hold them (the cache pointers are restrict: no asm without them could write their memory), so
    // the clobbering asm takes both pointers as operands.
    const Rsrc rk = make_rsrc(Kb, (uint32_t)s.ctx * HD * 2u), rv = make_rsrc(Vb, (uint32_t)s.ctx * HD * 2u);
    // A block's K fragments (2 NS loads) and V fragments (ND loads).  Past the end they re-read the
    // last block (never used), so every block issues the same loads and the explicit vmcnt waits
    // below are exact.
    auto koff = [&](int j, int tt) {
        const int key = min(min(j, kend - 1) + 8 * (fq >> 2) + 4 * tt + (fq & 3), kend - 1);
        return (uint32_t)((key >> 5) * (HD * 32) + (key & 31) * 32 + fg * 8) * 2u;
    };
    auto voff = [&](int j) { return (uint32_t)((min(j, kend - 1) >> 5) * (HD * 32) + fq * 32 + fg * 8) * 2u; };
    // (the clobbering asm takes both pointers, so the loads before it stay before it)
    auto pin = [&]() {
        asm volatile("" ::"s"(Kb), "s"(Vb) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // Block j0 with the fragments kf, vf, and block jn's loads into kfn, vfn, issued among block
    // j0's MFMAs (K among S = K Q^T, V among O += V^T P^T): the CU's vector memory path takes 64
    // bytes a clock, so a burst of a block's 32 KB per wave held up the wave's issue instead of
    // running beside its MFMAs.  A block's K is waited for before its S, its V before its P V.
    auto process = [&](int j0, const f16x8 (&kf)[2][NS], const f16x8 (&vf)[ND], int jn, f16x8 (&kfn)[2][NS],
                       f16x8 (&vfn)[ND]) {
        wait_loads<vmcnt_imm(ND)>();  // block j0's K has arrived (its V may still be in flight)
        f32x4 st2[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        const uint32_t kn0 = koff(jn, 0), kn1 = koff(jn, 1);
#pragma unroll
        for (int st = 0; st < NS; st++) {
#pragma unroll
            for (int tt = 0; tt < 2; tt++) {
                st2[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[tt][st], qf[st], st2[tt], 0, 0, 0);
                kfn[tt][st] = __builtin_bit_cast(f16x8, buf_b128(rk, tt ? kn1 : kn0, (uint32_t)st * 2048u));
            }
        }
#pragma unroll
        for (int i = 0; i < 2 * NS; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one load
        }
        pin();
        float sv[8];
        float tmax = -INFINITY;
        // a block before every query of the workgroup (and, with several sequences, inside the
        // shared prefix) needs no mask; the rows of queries past nq are computed but never stored
        const bool open = j0 + KB <= kend && j0 + KB <= P + t0 + 1 && (!rowt || j0 + KB <= Pv);
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                // kept: below the lane's end and outside other sequences' rows (bitwise, not
                // short-circuit operators: the short-circuit form compiled to a branch per key)
                const int j = j0 + 8 * fg + 4 * tt + r;
                const bool keep = open | ((j < jend) & ((j < Pv) | (j >= qlo)));
                const float v = keep ? st2[tt][r] * LOG2E : -INFINITY;
                sv[tt * 4 + r] = v;
                tmax = fmaxf(tmax, v);
            }
        tmax = wave_max16(tmax);
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = m_run == -INFINITY ? 0.f : exp2_fast(m_run - m_new);
        const float m_sub = m_new == -INFINITY ? 0.f : m_new;  // every key masked so far: p = 2^-inf = 0
        float psum = 0.f;
        f16x8 ph, pl;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float pv = exp2_fast(sv[e] - m_sub);
            psum += pv;
            const f16 hi = (f16)pv;
            ph[e] = hi;
            pl[e] = (f16)(pv - (float)hi);
        }
        l_run = l_run * alpha + wave_sum16(psum);
        m_run = m_new;
        // O^T += V^T P^T
        wait_loads<vmcnt_imm(2 * NS)>();  // block j0's V has arrived (block jn's K may still be in flight)
        const uint32_t vn = voff(jn);
#pragma unroll
        for (int dt = 0; dt < ND; dt++) {
            f32x4 a = acc[dt];
            a[0] *= alpha, a[1] *= alpha, a[2] *= alpha, a[3] *= alpha;
            a = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[dt], ph, a, 0, 0, 0);
            acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[dt], pl, a, 0, 0, 0);
            vfn[dt] = __builtin_bit_cast(f16x8, buf_b128(rv, vn, (uint32_t)dt * 1024u));
        }
#pragma unroll
        for (int i = 0; i < ND; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // two MFMAs
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one load
        }
        pin();
    };
    f16x8 kA[2][NS], vA[ND], kB[2][NS], vB[ND];
    // Q^T fragments: lane (query fq, group fg) holds Q[fq][32s + 8fg .. +8], pre-scaled by 1/sqrt(hd)
    // and rounded to f16 as the reference does.  The 4 waves prepare them together: wave w takes
    // queries 4w .. 4w + 3, lane (query qq, part kq) two 8-dim chunks c0, c1 of query qq, and writes
    // them to LDS, from where every wave reads its fragments.  Their loads are issued before the
    // first key block's and waited for alone (they are the older ones), so that the computation
    // runs while the block is in flight.
    //
    // QRD = RD: the query's RMSNorm and rotate-half RoPE are done here (the reference's qk_prep for
    // q, src/kernels.rs:400-448): q = x rsqrt(mean(x^2) + 1e-6) w, dims d < RD rotated at the row's
    // RoPE position, rounded to f16, then scaled.  Chunk c (dims 8c .. 8c + 7) of a rotated half
    // pairs with chunk c + NR: part kq < NR takes chunks kq and kq + NR (one cos/sin row for both),
    // part kq >= NR the unrotated chunks 2kq and 2kq + 1 (with QRD = 0 every part: dims 16kq ..
    // 16kq + 15 of the Q row).  The sum of squares is the 16 parts' (lanes 16 apart never mix).
    constexpr int RD2 = QRD / 2, NR = RD2 / 8;
    static_assert(QRD % 16 == 0 && QRD <= HD, "the fused query needs rotary_dim a multiple of 16");
    const int qq = 4 * wv + (lane >> 4), kq = lane & 15;
    const int tq = t0 + min(qq, nq - 1);
    const bool rot = kq < NR;
    const int c0 = rot ? kq : 2 * kq, c1 = rot ? kq + NR : 2 * kq + 1;
    f16x8 xv[2];
    float4 wq[2][2], cs4[4];
    if constexpr (QRD == 0) {
        const f16* qrow = Q + ((size_t)h * L + tq) * HD;
        xv[0] = *reinterpret_cast<const f16x8*>(qrow + 8 * c0);
        xv[1] = *reinterpret_cast<const f16x8*>(qrow + 8 * c1);
        // (the clobber holds the loads here: it takes the pointer, so it may write their memory)
        asm volatile("" ::"s"(Q) : "memory");
    } else {
        const f16* xrow = big + (size_t)tq * s.stride + h * 2 * HD;
        // unrotated parts read a rotated part's cos/sin row and do not use it
        xv[0] = *reinterpret_cast<const f16x8*>(xrow + 8 * c0);
        xv[1] = *reinterpret_cast<const f16x8*>(xrow + 8 * c1);
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int u = 0; u < 2; u++) wq[c][u] = *reinterpret_cast<const float4*>(qw + 8 * (c ? c1 : c0) + 4 * u);
        const int rpos = P + (rowt ? (int)(rwp & 0xFFFFu) : tq);
        const float* rp = rope + ((size_t)rpos * RD2 + 8 * (kq % NR)) * 2;
#pragma unroll
        for (int u = 0; u < 4; u++) cs4[u] = *reinterpret_cast<const float4*>(rp + 4 * u);
        asm volatile("" ::"s"(big), "s"(qw), "s"(rope) : "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
    int j = next_block(kbeg + wv * KB);
    {
        // the first block's K, then V (the order process() waits in)
        const uint32_t k0 = koff(j, 0), k1 = koff(j, 1), v0 = voff(j);
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int st = 0; st < NS; st++)
                kA[tt][st] = __builtin_bit_cast(f16x8, buf_b128(rk, tt ? k1 : k0, (uint32_t)st * 2048u));
#pragma unroll
        for (int dt = 0; dt < ND; dt++) vA[dt] = __builtin_bit_cast(f16x8, buf_b128(rv, v0, (uint32_t)dt * 1024u));
        pin();
    }
    {
        f16x8 q8[2];
        if constexpr (QRD == 0) {
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int e = 0; e < 8; e++) q8[c][e] = (f16)((float)xv[c][e] * scale);
        } else {
            float x[2][8], sp[2] = {0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    x[c][e] = (float)xv[c][e];
                    sp[c] += x[c][e] * x[c][e];
                }
            float ss = sp[0] + sp[1];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) ss += __shfl_xor(ss, o);
            const float inv = 1.0f / sqrtf(ss / (float)HD + 1e-6f);
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const float w8[8] = {wq[c][0].x, wq[c][0].y, wq[c][0].z, wq[c][0].w,
                                     wq[c][1].x, wq[c][1].y, wq[c][1].z, wq[c][1].w};
#pragma unroll
                for (int e = 0; e < 8; e++) x[c][e] = x[c][e] * inv * w8[e];
            }
            const float cs[16] = {cs4[0].x, cs4[0].y, cs4[0].z, cs4[0].w, cs4[1].x, cs4[1].y, cs4[1].z, cs4[1].w,
                                  cs4[2].x, cs4[2].y, cs4[2].z, cs4[2].w, cs4[3].x, cs4[3].y, cs4[3].z, cs4[3].w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float c = cs[2 * e], sn = cs[2 * e + 1], a = x[0][e], bb = x[1][e];
                const float lo = rot ? a * c - bb * sn : a, hi = rot ? bb * c + a * sn : bb;
                q8[0][e] = (f16)((float)(f16)lo * scale);
                q8[1][e] = (f16)((float)(f16)hi * scale);
            }
        }
        *reinterpret_cast<f16x8*>(&Qs[qq][8 * c0]) = q8[0];
        *reinterpret_cast<f16x8*>(&Qs[qq][8 * c1]) = q8[1];
    }
    __syncthreads();
#pragma unroll
    for (int st = 0; st < NS; st++) qf[st] = *reinterpret_cast<const f16x8*>(&Qs[fq][st * 32 + fg * 8]);
    while (j < kend) {
        int jn = next_block(j + 4 * KB);
        process(j, kA, vA, jn, kB, vB);
        j = jn;
        if (j >= kend) break;
        jn = next_block(j + 4 * KB);
        process(j, kB, vB, jn, kA, vA);
        j = jn;
    }
    // merge the 4 waves: acc[dt][r] is O[query fq][dim 16dt + 4fg + r]
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int r = 0; r < 4; r++) Om[wv][fq][dt * 16 + fg * 4 + r] = acc[dt][r];
    if (fg == 0) {
        Mm[wv][fq] = m_run;
        Lm[wv][fq] = l_run;
    }
    __syncthreads();
    // per query (thread q): the merged max, the weight of each wave's state, the merged sum
    __shared__ float Fw[16][4], Ml[16][2];
    if (tid < nq) {
        const int q = tid;
        float m = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; w++)
            if (Lm[w][q] > 0.f) m = fmaxf(m, Mm[w][q]);
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float f = Lm[w][q] > 0.f ? exp2_fast(Mm[w][q] - m) : 0.f;
            l += Lm[w][q] * f;
            Fw[q][w] = f;
        }
        Ml[q][0] = m;
        Ml[q][1] = l;
    }
    __syncthreads();
    // Thread (qe, d0): the 4 waves' partial outputs of query qe at dimensions d0 .. d0 + 15, summed
    // in wave order (16-byte LDS reads), then 16-byte stores.  Every LDS read comes first (a store
    // through a generic pointer keeps the compiler from moving LDS reads past it).
    float av[16];
#pragma unroll
    for (int u = 0; u < 16; u++) av[u] = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float f = Fw[qe][w];
#pragma unroll
        for (int u4 = 0; u4 < 4; u4++) {
            const float4 v = *reinterpret_cast<const float4*>(&Om[w][qe][d0 + 4 * u4]);
            av[4 * u4] += v.x * f;
            av[4 * u4 + 1] += v.y * f;
            av[4 * u4 + 2] += v.z * f;
            av[4 * u4 + 3] += v.w * f;
        }
    }
    const float mq = Ml[qe][0], lq = Ml[qe][1];
    if (qe >= nq) return;
    const int t = t0 + qe;
    if (ks == 1) {
        // out = acc / l * sigmoid(gate), the sigmoid on the hardware exp2 and reciprocal (within about
        // 1 ulp in f32, rounded to f16)
        const float inv_l = 1.0f / lq;
        f16x8 o8[2];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const float g = (float)gv[u >> 3][u & 7];
            const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -LOG2E));
            o8[u >> 3][u & 7] = (f16)(av[u] * inv_l * sg);
        }
        f16* op = out + (size_t)t * s.HQ * HD + h * HD + d0;
        *reinterpret_cast<f16x8*>(op) = o8[0];
        *reinterpret_cast<f16x8*>(op + 8) = o8[1];
    } else {
        const size_t r = ((size_t)z * L + t) * s.HQ + h;
        float4* pp = reinterpret_cast<float4*>(pacc + r * HD + d0);
#pragma unroll
        for (int u4 = 0; u4 < 4; u4++) pp[u4] = float4{av[4 * u4], av[4 * u4 + 1], av[4 * u4 + 2], av[4 * u4 + 3]};
        if (d0 == 0) {
            pml[r * 2] = mq;
            pml[r * 2 + 1] = lq;
        }
    }
}

// The same attention over 32 (query, head) rows per workgroup: NQ = 32 / G queries of all G query
// heads of one kv head (G = HQ / HK, a power of two), so that a key block feeds 32 rows on
// v_mfma_f32_32x32x16_f16 where k_attn's feeds 16.  k_attn is bound by the CU's vector memory path (a
// block is 32 KB per wave, 64 bytes a clock per CU) and by one wave per SIMD waiting in turn for its
// loads, its softmax and its MFMAs.  This kernel is bound by that path too (2048 clocks for the four
// waves' blocks, measured 2340 per block beside 1536 of MFMA, which counters at 2048 rows show busy for 34%
// of the CUs' cycles), for twice the rows, plus about 15 thousand clocks per workgroup of prologue and merge.  On MI355X, 8 query and 2 kv heads: 38.8 us at 2048 rows where
// k_attn takes 104 us, 18.1 against 39 at 1024, 14.6 against 22.7 at 632; 440 TFLOP/s at 2048.
//  * Row c of the workgroup is query c % NQ of head kh G + c / NQ; the 4 waves split the keys in blocks
//    of 32 as in k_attn and merge their states in LDS at the end.
//  * A wave's block goes straight to LDS (buffer_load_dwordx4 lds, whole cache lines: the 16 KB of K
//    and of V^T are contiguous in the cache) into a place of the wave's own, so the key loop has no
//    barrier.  The place holds one block, as 4 + 4 quarters of 4 KB: a quarter is refilled with the next
//    block's as soon as its fragments have been read.  Rows of 64 bytes (a key's 32 dims of K, a dim's
//    32 keys of V^T) have their 16-byte pieces at p ^ (row / 4) % 4, so a fragment read (32 rows, two
//    pieces) meets no bank twice.
//  * Per block: S^T = K Q^T (keys x rows, 16 MFMAs over the 256 dims in one chain), the softmax per
//    column, O^T += V^T P^T (8 dim tiles x 2 key slices, P as f16 hi + lo).  The rows of S^T are permuted
//    so that lane (column, half g) holds keys 16 s + 8 g .. + 7 in registers 8 s ..: P^T's B operand of
//    slice s as it is.  Block n + 1's S MFMAs run among block n's exponentials.
//  * The running maximum a row's exponentials are relative to is raised (and O, l rescaled) only when a
//    block's maximum exceeds it by more than 8: the probabilities then reach at most e^8 = 2981, well inside
//    f16 (hi + lo keep their relative precision), and the factor cancels in acc / l.  Most blocks skip the rescale.
//  * Heavy workgroups first: tiles are taken from the last query block down, so the short ones fill the
//    end; blockIdx.x is the kv head, so with 2 kv heads an XCD's L2 sees one head's keys.
// Vector-memory accounting (every block issues the same DMAs; past the wave's last block they carry
// out-of-range offsets, read nothing and write zeros): in the loop the DMAs in flight are block n + 1's
// K (16), then block n's V (16); reading quarter q leaves the 28 after it, also while the quarters
// before it are refilled.
template <int HD, int QRD>
__global__ __launch_bounds__(256, 1) void k_attn_rows(const f16* __restrict__ Q, const f16* __restrict__ Kc,
                                                      const f16* __restrict__ Vt, const uint32_t* __restrict__ lu,
                                                      int L, int HQ, int HK, int stride, int ctx, int ks,
                                                      const uint32_t* __restrict__ rowt, const f16* __restrict__ big,
                                                      f16* __restrict__ out, float* __restrict__ pacc,
                                                      float* __restrict__ pml, const float* __restrict__ qw,
                                                      const float* __restrict__ rope, int lgq) {
    static_assert(HD == 256, "attention is written for 256-wide heads");
    constexpr int NS = HD / 16;   // 16 k steps over the head dimension
    constexpr int ND = HD / 32;   // 8 output dimension tiles
    constexpr int KB = 32;        // keys per block
    constexpr int QB = 4096;      // bytes of a quarter of a wave's K or V^T block
    constexpr float RAISE = 8.0f;  // the slack of the running maximum
    // One array per quarter (all 4 waves'), so that the compiler sees that the DMAs into one never alias
    // the reads of another.  At the end array dt holds the waves' outputs of dim tile dt.
    __shared__ __align__(1024) uint8_t B0[4 * QB], B1[4 * QB], B2[4 * QB], B3[4 * QB], B4[4 * QB], B5[4 * QB], B6[4 * QB], B7[4 * QB];
    __shared__ __align__(16) f16 Qs[32][HD + 8];  // the rows' queries, scaled
    __shared__ float Mm[4][32], Lm[4][32];
    auto arr = [&](int i) {
        return i == 0 ? B0 : i == 1 ? B1 : i == 2 ? B2 : i == 3 ? B3 : i == 4 ? B4 : i == 5 ? B5 : i == 6 ? B6 : B7;
    };
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;
    const int NQ = 1 << lgq;
    const int kh = blockIdx.x, z = blockIdx.z;
    const int t0 = (((L + NQ - 1) >> lgq) - 1 - (int)blockIdx.y) * NQ;
    const int h0 = kh << (5 - lgq);
    const int nq = min(NQ, L - t0);
    // The rows' inputs first (they depend on no load): wave w prepares rows 8w .. 8w + 7 in two passes of
    // 4 (see k_attn), lane (row, part kq) two 8-dim chunks c0, c1; then the epilogue's thread (row ce,
    // dims 32 dt + 4 ke .. + 3) its output gates.
    constexpr int RD2 = QRD / 2, NR = RD2 / 8;
    const int kq = lane & 15;
    const bool rot = kq < NR;
    const int c0 = rot ? kq : 2 * kq, c1 = rot ? kq + NR : 2 * kq + 1;
    int tq[2];
    f16x8 xv[2][2];
    float4 wq[2][2], cs4[2][4];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int row = 8 * wv + 4 * u + (lane >> 4);
        tq[u] = t0 + min(row & (NQ - 1), nq - 1);
        const int hq = h0 + (row >> lgq);
        const f16* xrow = QRD ? big + (size_t)tq[u] * stride + hq * 2 * HD : Q + ((size_t)hq * L + tq[u]) * HD;
        xv[u][0] = *reinterpret_cast<const f16x8*>(xrow + 8 * c0);
        xv[u][1] = *reinterpret_cast<const f16x8*>(xrow + 8 * c1);
    }
    if constexpr (QRD != 0) {
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int u = 0; u < 2; u++) wq[k][u] = *reinterpret_cast<const float4*>(qw + 8 * (k ? c1 : c0) + 4 * u);
    }
    // (a row past the last query is the last query's again, also in the output, which it writes a second time
    // with the same values: with those rows' lanes switched off instead, a tile of one query, 8 lanes of each
    // wave, ran its last instructions at a third of the rate, 600 against 168 clocks per dim tile, and 257 rows
    // took 19.2 us where 258 took 17.0)
    const int cx = tid >> 3, ke = tid & 7;
    const int ce = (cx & ~(NQ - 1)) | min(cx & (NQ - 1), nq - 1), te = t0 + (ce & (NQ - 1)), he = h0 + (ce >> lgq);
    f16x4 gv[ND];
    {
        const f16* gp = big + (size_t)te * stride + he * 2 * HD + HD + 4 * ke;
#pragma unroll
        for (int u = 0; u < ND; u++) gv[u] = *reinterpret_cast<const f16x4*>(gp + 32 * u);
    }
    // row table words, as in k_attn: this lane's query, the tile's first row, and (for the RoPE position)
    // the queries whose chunks this lane normalizes
    // (a forward without a table takes a branch of its own: its RoPE rows then wait for no load)
    const int qi = c & (NQ - 1);
    uint32_t rwq = 0, rw0 = 0, rpos[2] = {(uint32_t)tq[0], (uint32_t)tq[1]};
    asm volatile("" ::"s"(big), "s"(qw), "s"(rowt), "s"(Q) : "memory");
    if (rowt) {
        const Rsrc rr = make_rsrc(rowt, (uint32_t)L * 4u);
        rwq = buf_b32(rr, (uint32_t)(t0 + min(qi, nq - 1)) * 4u, 0);
        rw0 = buf_b32(rr, (uint32_t)t0 * 4u, 0);
        if constexpr (QRD != 0) {
#pragma unroll
            for (int u = 0; u < 2; u++) rpos[u] = buf_b32(rr, (uint32_t)tq[u] * 4u, 0) & 0xFFFFu;
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    const int P = (int)lu[1], Pv = P + (int)lu[6];
    SGPR_BATCH("s"(P), "s"(Pv), "s"(out), "s"(pacc), "s"(pml));
    const int nkeys = P + t0 + nq;
    const int span = ((nkeys + ks - 1) / ks + KB - 1) / KB * KB;
    const int kbeg = z * span, kend = min(nkeys, kbeg + span);
    const float scale = 1.0f / sqrtf((float)HD);
    const int jend = qi < nq ? min(kend, P + t0 + qi + 1) : INT_MIN;
    if constexpr (QRD != 0) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const float* rp = rope + ((size_t)(P + (int)rpos[u]) * RD2 + 8 * (kq % NR)) * 2;
#pragma unroll
            for (int v = 0; v < 4; v++) cs4[u][v] = *reinterpret_cast<const float4*>(rp + 4 * v);
        }
        asm volatile("" ::"s"(rope) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    const int qlo = P + (int)(rwq >> 16), qlo0 = P + (int)(rw0 >> 16);

    const Rsrc rk = make_rsrc(Kc + (size_t)kh * ctx * HD, (uint32_t)ctx * HD * 2u),
               rv = make_rsrc(Vt + (size_t)kh * HD * ctx, (uint32_t)ctx * HD * 2u);
    auto next_block = [&](int j) {
        if (j >= Pv && j + KB <= qlo0) j += ((qlo0 - KB - j) / (4 * KB) + 1) * (4 * KB);
        return __builtin_amdgcn_readfirstlane(j);
    };
    // quarter q of a 16 KB block at byte boff of the cache, 4 KB: lane's 16 bytes of each KB
    const uint32_t dlane = (uint32_t)((lane >> 2) * 64 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4));
    auto boff = [&](int j) { return j < kend ? (uint32_t)(j >> 5) * (HD * 64u) : OOB; };
    auto dma = [&](Rsrc r, int i, uint32_t off) {  // array i: quarter i & 3
        uint8_t* const dst = arr(i) + wv * QB;
        buf_lds64(r, dlane, off + (uint32_t)((i & 3) * QB), dst);
    };
    // fragment st of K (dims 16 st + 8 g of key kperm of row c), fragment (dt, s) of V^T (keys 16 s + 8 g
    // of dim 32 dt + c)
    const int kperm = 16 * (c >> 4) + 8 * ((c >> 2) & 1) + 4 * ((c >> 3) & 1) + (c & 3);
    const int kfo = kperm * 64 + ((g ^ ((kperm >> 2) & 3)) << 4), vfo = c * 64 + ((g ^ ((c >> 2) & 3)) << 4);
    auto kfrag = [&](int st) {
        return *reinterpret_cast<const f16x8*>(arr(st >> 2) + wv * QB + ((st >> 1) & 1) * 2048 + (kfo ^ ((st & 1) << 5)));
    };
    auto vfrag = [&](int dt, int k) {
        return *reinterpret_cast<const f16x8*>(arr(4 + (dt >> 1)) + wv * QB + (dt & 1) * 2048 + (vfo ^ (k << 5)));
    };
    f16x8 qf[NS];
    f32x16 acc[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[dt][i] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    int j = next_block(kbeg + wv * KB);
    {
        const uint32_t b = boff(j);
#pragma unroll
        for (int q = 0; q < 4; q++) dma(rk, q, b);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        f16x8 q8[2];
        if constexpr (QRD == 0) {
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int e = 0; e < 8; e++) q8[k][e] = (f16)((float)xv[u][k][e] * scale);
        } else {
            float x[2][8], sp[2] = {0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    x[k][e] = (float)xv[u][k][e];
                    sp[k] += x[k][e] * x[k][e];
                }
            float ss = sp[0] + sp[1];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) ss += __shfl_xor(ss, o);
            const float inv = 1.0f / sqrtf(ss / (float)HD + 1e-6f);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float w8[8] = {wq[k][0].x, wq[k][0].y, wq[k][0].z, wq[k][0].w,
                                     wq[k][1].x, wq[k][1].y, wq[k][1].z, wq[k][1].w};
#pragma unroll
                for (int e = 0; e < 8; e++) x[k][e] = x[k][e] * inv * w8[e];
            }
            const float cs[16] = {cs4[u][0].x, cs4[u][0].y, cs4[u][0].z, cs4[u][0].w, cs4[u][1].x, cs4[u][1].y,
                                  cs4[u][1].z, cs4[u][1].w, cs4[u][2].x, cs4[u][2].y, cs4[u][2].z, cs4[u][2].w,
                                  cs4[u][3].x, cs4[u][3].y, cs4[u][3].z, cs4[u][3].w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float cc = cs[2 * e], sn = cs[2 * e + 1], a = x[0][e], bb = x[1][e];
                const float lo = rot ? a * cc - bb * sn : a, hi = rot ? bb * cc + a * sn : bb;
                q8[0][e] = (f16)((float)(f16)lo * scale);
                q8[1][e] = (f16)((float)(f16)hi * scale);
            }
        }
        const int row = 8 * wv + 4 * u + (lane >> 4);
        *reinterpret_cast<f16x8*>(&Qs[row][8 * c0]) = q8[0];
        *reinterpret_cast<f16x8*>(&Qs[row][8 * c1]) = q8[1];
    }
    lds_barrier();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        qf[s] = *reinterpret_cast<const f16x8*>(&Qs[c][s * 16 + g * 8]);
        asm("" : "+a"(qf[s]));  // kept in AGPRs, which an MFMA reads as it reads VGPRs
    }

    // masked scores (unscaled, natural units) and their column maximum over both lane halves
    auto mask_max = [&](f32x16& s, int j0) {
        const bool open = j0 + KB <= kend && j0 + KB <= P + t0 + 1 && (!rowt || j0 + KB <= Pv);
        if (!open) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int key = j0 + 16 * (i >> 3) + 8 * g + (i & 7);
                const bool keep = (key < jend) & ((key < Pv) | (key >= qlo));
                s[i] = keep ? s[i] : -INFINITY;
            }
        }
        float t = s[0];
#pragma unroll
        for (int i = 1; i < 16; i++) t = fmaxf(t, s[i]);
        // (the swap's halves through scalars: a bit cast of a vector's element reads element 0)
        const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, t), __builtin_bit_cast(uint32_t, t), false, false);
        const uint32_t lo = sw[0], hi = sw[1];
        return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
    };
    // The block's probabilities 2^(s log2 e + nm) and their split into f16 hi + lo, pair by pair: pexp
    // exponentiates elements 2u, 2u + 1, psplit adds them to the row sum and packs them.
    f16x8 ph[2], pl[2];
    float pe[16];
    auto pexp = [&](const f32x16& s, int u, float nm) {
        pe[2 * u] = exp2_fast(__builtin_fmaf(s[2 * u], LOG2E, nm));
        pe[2 * u + 1] = exp2_fast(__builtin_fmaf(s[2 * u + 1], LOG2E, nm));
    };
    auto psplit = [&](int u) {
        const float p0 = pe[2 * u], p1 = pe[2 * u + 1];
        f16x2 hi, lo;
        split2(p0, p1, hi, lo);
        l_run += p0;
        l_run += p1;
        ph[u >> 2][(2 * u) & 7] = hi[0];
        ph[u >> 2][(2 * u + 1) & 7] = hi[1];
        pl[u >> 2][(2 * u) & 7] = lo[0];
        pl[u >> 2][(2 * u + 1) & 7] = lo[1];
    };
    auto raise = [&](float tmax) {
        if (!__any(tmax > m_run + RAISE)) return;
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = m_run == -INFINITY ? 0.f : exp2_fast((m_run - m_new) * LOG2E);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < ND; dt++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[dt][i] *= alpha;
    };
    // The loop's unit is a quarter: its fragments were read during the quarter before, and while its MFMAs
    // run the next quarter's are (once its DMAs have landed: WAIT leaves the DMAs after it in flight); then
    // the quarter itself is refilled.  `mid(e)` is VALU work beside MFMA e.
    f16x8 fr[2][4];
    auto read_k = [&](int q) {
#pragma unroll
        for (int e = 0; e < 4; e++) fr[q & 1][e] = kfrag(4 * q + e);
    };
    auto read_v = [&](int q) {
#pragma unroll
        for (int e = 0; e < 4; e++) fr[q & 1][e] = vfrag(2 * q + (e & 1), e >> 1);
    };
    auto k_quarter = [&](f32x16& s, int q, auto mid) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[q & 1][e], qf[4 * q + e], s, 0, 0, 0);
            mid(4 * q + e);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto v_quarter = [&](int q) {
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
#pragma unroll
            for (int d = 0; d < 2; d++)
                acc[2 * q + d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[q & 1][e + d], ph[e >> 1], acc[2 * q + d], 0, 0, 0);
#pragma unroll
            for (int d = 0; d < 2; d++)
                acc[2 * q + d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[q & 1][e + d], pl[e >> 1], acc[2 * q + d], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int W24 = vmcnt_imm(24), W12 = vmcnt_imm(12), W8 = vmcnt_imm(8), W4 = vmcnt_imm(4), W0 = vmcnt_imm(0);
    if (j < kend) {
        int jn = next_block(j + 4 * KB);
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
        {
            // the first block: its K alone is in flight, then block jn's behind it, then its own V
            const uint32_t kn = boff(jn), b = boff(j);
            wait_loads<W12>();
            read_k(0);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (q < 3) {
                    wait_loads<W8>();
                    read_k(q + 1);
                }
                k_quarter(s, q, [](int) {});
                dma(rk, q, kn);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) dma(rv, 4 + q, b);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (jn < kend) {
            wait_loads<vmcnt_imm(28)>();
            read_k(0);
        }
        float tmax = mask_max(s, j);
        while (jn < kend) {
            raise(tmax);
            const int j2 = next_block(jn + 4 * KB);
            const uint32_t kn = boff(j2), vn = boff(jn);
            const float nm = m_run == -INFINITY ? 0.f : m_run * -LOG2E;
            f32x16 s2;
#pragma unroll
            for (int i = 0; i < 16; i++) s2[i] = 0.f;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                wait_loads<W24>();
                if (q < 3) read_k(q + 1);
                else read_v(0);
                k_quarter(s2, q, [&](int st) {
                    if (st % 2 == 0) pexp(s, st >> 1, nm);
                    else psplit(st >> 1);
                });
                dma(rk, q, kn);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                wait_loads<W24>();
                if (q < 3) read_v(q + 1);
                else read_k(0);  // block j2's; past the wave's last block it reads zeros, for nothing
                v_quarter(q);
                dma(rv, 4 + q, vn);
                __builtin_amdgcn_sched_barrier(0);
            }
            s = s2;
            tmax = mask_max(s, jn);
            j = jn;
            jn = j2;
        }
        // the last block: its V alone is to be waited for
        wait_loads<W12>();
        read_v(0);
        raise(tmax);
        const float nm = m_run == -INFINITY ? 0.f : m_run * -LOG2E;
#pragma unroll
        for (int u = 0; u < 8; u++) pexp(s, u, nm);
#pragma unroll
        for (int u = 0; u < 8; u++) psplit(u);
        wait_loads<W8>();
        read_v(1);
        v_quarter(0);
        wait_loads<W4>();
        read_v(2);
        v_quarter(1);
        wait_loads<W0>();
        read_v(3);
        v_quarter(2);
        v_quarter(3);
    }
    wait_loads<vmcnt_imm(0)>();  // every DMA has landed before the arrays take the outputs
    l_run += __shfl_xor(l_run, 32);
    // merge the 4 waves: acc[dt][i] is O[row c][dim 32 dt + 8 (i / 4) + 4 g + i % 4]; array dt, wave w's
    // part: rows of 128 bytes, 16-byte chunk k (dims 4k .. 4k + 3 of the tile) at k ^ row % 8
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            *reinterpret_cast<f32x4*>(arr(dt) + wv * QB + c * 128 + (((2 * q + g) ^ (c & 7)) << 4)) =
                f32x4{acc[dt][4 * q], acc[dt][4 * q + 1], acc[dt][4 * q + 2], acc[dt][4 * q + 3]};
    if (g == 0) {
        Mm[wv][c] = m_run * LOG2E;
        Lm[wv][c] = l_run;
    }
    lds_barrier();
    // every thread merges its row's states itself (8 LDS words, no second barrier)
    float mq = -INFINITY, lq = 0.f, fw[4];
    {
        float mw[4], lw[4];
#pragma unroll
        for (int w = 0; w < 4; w++) mw[w] = Mm[w][ce], lw[w] = Lm[w][ce];
#pragma unroll
        for (int w = 0; w < 4; w++) mq = lw[w] > 0.f ? fmaxf(mq, mw[w]) : mq;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            fw[w] = lw[w] > 0.f ? exp2_fast(mw[w] - mq) : 0.f;
            lq += lw[w] * fw[w];
        }
    }
    // thread (ce, ke): the 4 waves' outputs summed in wave order
    f32x4 av[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++) av[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float f = fw[w];
#pragma unroll
        for (int dt = 0; dt < ND; dt++) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(arr(dt) + w * QB + ce * 128 + ((ke ^ (ce & 7)) << 4));
#pragma unroll
            for (int e = 0; e < 4; e++) av[dt][e] += v[e] * f;
        }
    }
    if (ks == 1) {
        const float inv_l = 1.0f / lq;
        f16* op = out + (size_t)te * HQ * HD + he * HD + 4 * ke;
#pragma unroll
        for (int dt = 0; dt < ND; dt++) {
            f16x4 o4;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f((float)gv[dt][e] * -LOG2E));
                o4[e] = (f16)(av[dt][e] * inv_l * sg);
            }
            *reinterpret_cast<f16x4*>(op + 32 * dt) = o4;
        }
    } else {
        const size_t r = ((size_t)z * L + te) * HQ + he;
#pragma unroll
        for (int dt = 0; dt < ND; dt++) *reinterpret_cast<f32x4*>(pacc + r * HD + 32 * dt + 4 * ke) = av[dt];
        if (ke == 0) {
            pml[r * 2] = mq;
            pml[r * 2 + 1] = lq;
        }
    }
}

template <int HD>
__global__ __launch_bounds__(HD) void k_attn_combine(const float* __restrict__ pacc, const float* __restrict__ pml,
                                                     const f16* __restrict__ big, f16* __restrict__ out, int L, int ks,
                                                     int HQ, int stride) {
    const AttnShape s{HQ, 0, HD, 0, stride, 0};
    const int t = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
    // Every load is issued up front and unconditionally (splits past ks re-read the last one and are
    // then skipped), so none waits behind a branch or another load; the sums run in split order.
    float mz[ATTN_KS_MAX], lz[ATTN_KS_MAX], az[ATTN_KS_MAX];
#pragma unroll
    for (int z = 0; z < ATTN_KS_MAX; z++) {
        const size_t r = ((size_t)min(z, ks - 1) * L + t) * s.HQ + h;
        mz[z] = pml[r * 2];
        lz[z] = pml[r * 2 + 1];
        az[z] = pacc[r * HD + d];
    }
    const float g = (float)big[(size_t)t * s.stride + h * 2 * HD + HD + d];
    float m = -INFINITY;
#pragma unroll
    for (int z = 0; z < ATTN_KS_MAX; z++)
        if (z < ks && lz[z] > 0.f) m = fmaxf(m, mz[z]);
    float l = 0.f, a = 0.f;
#pragma unroll
    for (int z = 0; z < ATTN_KS_MAX; z++)
        if (z < ks && lz[z] > 0.f) {
            const float f = exp2_fast(mz[z] - m);
            l += lz[z] * f;
            a += az[z] * f;
        }
    // as k_attn's unsplit epilogue: acc / l * sigmoid(gate), the sigmoid on exp2 and the reciprocal
    out[(size_t)t * s.HQ * HD + h * HD + d] =
        (f16)(a * (1.0f / l) * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -LOG2E)));
}

}  // namespace

void qk_prep(const f16* big, const AttnShape& s, const float* qw, const float* kw, const float* rope, int L,
             const uint32_t* lu, const Segs& sg, f16* Q, f16* Kc, f16* Vc, hipStream_t st) {
    SD_CHECK(s.HD == 256, "attention: only head_dim 256 is supported");
    SD_CHECK(s.RD % 2 == 0 && s.RD <= s.HD, "attention: bad rotary_dim");
    SD_CHECK(s.stride % 4 == 0, "attention: the row stride must be a multiple of 4");
    SD_CHECK(s.ctx % 32 == 0, "attention: the cache length must be a multiple of 32");
    hipLaunchKernelGGL(k_qk_prep<256>, dim3((L + 3) / 4, Q ? s.HQ + s.HK : s.HK), dim3(256), 0, st, big, lu, L, s.HQ,
                       s.HK, s.RD, s.stride, s.ctx, sg.row, qw, kw, rope, Q, Kc, Vc);
    launched("qk_prep");
}

// Workspace (floats) the key-split path needs for up to `rows` query rows.
size_t attn_ws_floats(int rows, const AttnShape& s) { return (size_t)ATTN_KS_MAX * rows * s.HQ * (s.HD + 2); }

// Which kernel, and how many key splits, for L rows (prefix: the keys include a cached prefix; without one
// they are the rows themselves).  The splits are fixed when a plan is captured, whatever the prefix's length.
// qk_prep + attention + combine on MI355X at 8 query and 2 kv heads, us, k_attn against k_attn_rows:
//   rows + prefix   64 + 512   120 + 512   200 + 512   250 + 2048   512 + 0   1024 + 0   2048 + 0
//   k_attn          17.0       18.7        27.8        32.3         20.2      47.9       119
//   k_attn_rows     18.4       19.3-20.6   22.3        29.4         19.0      26.7       51.1
// A tile of 32 (query, head) rows has half as many workgroups as k_attn's 16 queries of a head, so up to 128
// rows the latter's shorter chains win.  From 129 to 256 rows they also do (us, k_attn | k_attn_rows):
//  * with few heads over a prefix, where 8 splits of k_attn are at most one workgroup per CU (32 tiles): 2
//    query and 2 kv heads, 160 + 512: 16.2 in 8 splits | 17.3 in 4, 16.9 in 8; + 2048 19.8 | 20.7; 250 + 512:
//    17.8 | 18.2.  From 36 tiles on k_attn has 4: 4 and 1 heads, 129 + 2048 22.6 | 21.2, + 3800 29.0 | 25.9;
//  * without a prefix, the keys being the rows, unsplit and within one workgroup per CU: 8 and 2 heads, 129
//    rows 14.1 | 15.4, 250 15.3 | 16.1; 16 and 1 heads, 250 rows 15.8 | 16.6 (32 and 8, 288 tiles: 21.0 | 17.3).
// Where k_attn runs up to 128 rows, or over a prefix:
//  * it splits the keys while its grid stays within one workgroup per CU (70 rows: 18.2 us in 4 splits, 21.0
//    in 8).
//  * k_attn_rows up to 256 rows splits them only over a prefix, in 4 up to 48 tiles (200 + 2048: 25.2 us in 4
//    splits, 28.3 in 2, 33.0 in 1; 128 + 512: 19.3 / 19.5 / 18.3) and in 2 up to 64 (250 + 512: 24.1 / 23.2 /
//    20.5, + 2048: 26.7 / 29.4 / 33.4).
AttnPlan attn_plan(int L, const AttnShape& s, bool prefix) {
    const int G = s.HQ / s.HK;
    AttnPlan p;
    const int tiles16 = (L + BQ - 1) / BQ * s.HQ;  // of k_attn
    const bool few = L <= ATTN_SPLIT_ROWS && tiles16 * (prefix ? ATTN_KS_MAX : 1) <= 256;
    p.rows = L > 128 && !few && G <= 32 && (G & (G - 1)) == 0;
    if (L > ATTN_SPLIT_ROWS || (L > 128 && !prefix)) return p;
    if (p.rows) {
        const int tiles = (L * G + 31) / 32 * s.HK;
        p.ks = tiles > 64 ? 1 : tiles > 48 ? 2 : 4;
    } else {
        while (p.ks < ATTN_KS_MAX && tiles16 * p.ks * 2 <= 256) p.ks *= 2;
    }
    return p;
}

void attention_split(const f16* Q, const f16* Kc, const f16* Vc, const f16* big, const AttnShape& s, int L,
                     const uint32_t* lu, const Segs& sg, const AttnPlan& p, float* ws, f16* out, hipStream_t st,
                     const float* qw, const float* rope) {
    SD_CHECK(s.HD == 256 && s.HQ % s.HK == 0, "attention: unsupported head shape");
    SD_CHECK(Q || (qw && rope && s.RD == 64), "attention: the fused query norm and RoPE take rotary_dim 64");
    SD_CHECK(p.ks >= 1 && p.ks <= ATTN_KS_MAX, "attention: 1 to 8 key splits");
    float* pacc = ws;
    float* pml = ws + (size_t)p.ks * L * s.HQ * s.HD;
    const int G = s.HQ / s.HK;
    // k_attn_rows moves the cache's 16-byte pieces straight to LDS: a cache that does not start on one keeps
    // k_attn, which loads them to registers (with the same key splits)
    const bool pieces = (reinterpret_cast<uintptr_t>(Kc) | reinterpret_cast<uintptr_t>(Vc)) % 16 == 0;
    if (p.rows && pieces) {
        SD_CHECK(G <= 32 && (G & (G - 1)) == 0, "attention: a tile of 32 rows takes a power of two of query heads");
        const auto f = Q ? k_attn_rows<256, 0> : k_attn_rows<256, 64>;
        hipLaunchKernelGGL(f, dim3(s.HK, (L * G + 31) / 32, p.ks), dim3(256), 0, st, Q, Kc, Vc, lu, L, s.HQ, s.HK, s.stride,
                           s.ctx, p.ks, sg.row, big, out, pacc, pml, qw, rope, 5 - __builtin_ctz((unsigned)G));
    } else {
        const auto f = Q ? k_attn<256, 0> : k_attn<256, 64>;
        hipLaunchKernelGGL(f, dim3((L + BQ - 1) / BQ, s.HQ, p.ks), dim3(256), 0, st, Q, Kc, Vc, lu, L, s.HQ, s.HK, s.stride,
                           s.ctx, p.ks, sg.row, big, out, pacc, pml, qw, rope, s.RD);
    }
    launched("attn");
    if (p.ks > 1) {
        hipLaunchKernelGGL(k_attn_combine<256>, dim3(L, s.HQ), dim3(256), 0, st, pacc, pml, big, out, L, p.ks, s.HQ,
                           s.stride);
        launched("attn_combine");
    }
}

}  // namespace sd
