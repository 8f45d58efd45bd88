// Device-side helpers shared by the quantized GEMM and GEMV kernels: raw buffer loads (with their
// zero-filling range check), explicit vector-memory waits and barriers, and the int4 nibble dequant.
#pragma once

#include "common.h"

namespace sd {
namespace {

// Inline asm holds no vector instruction anywhere in these files: the compiler keeps the wait states
// between an MFMA and a vector write of the registers it still reads as SrcC for its own instructions
// only, not for those inside an asm.  Where it has to be led to one instruction, a constant or the
// instruction's result goes through an empty asm that it cannot see through.
#if defined(__HIP_DEVICE_COMPILE__)
#define OPAQUE_V(x) asm("" : "+v"(x))
#define OPAQUE_S(x) asm("" : "+s"(x))
#else
#define OPAQUE_V(x) (void)(x)
#define OPAQUE_S(x) (void)(x)
#endif

// (a & m) | c in one v_and_or_b32 (with constants that it sees, the compiler emits separate and/or here).
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t c) {
    OPAQUE_V(m);
    OPAQUE_S(c);
    return (a & m) | c;
}

// (v0, v1) = hi + lo as f16 pairs, hi rounded and lo the rounded rest: a packed convert for hi, the rest
// v - hi (exact in f32) by one v_fma_mix_f32 on each half of hi's register, a packed convert for lo.  (A
// subtraction, or a product with a -1 that the compiler sees, makes it convert each half on its own.)
__device__ __forceinline__ void split2(float v0, float v1, f16x2& hi, f16x2& lo) {
    uint32_t hb = __builtin_bit_cast(uint32_t, f16x2{(f16)v0, (f16)v1});
    OPAQUE_V(hb);
    hi = __builtin_bit_cast(f16x2, hb);
    float m = -1.0f;
    OPAQUE_S(m);
    float r0 = __builtin_fmaf((float)hi[0], m, v0), r1 = __builtin_fmaf((float)hi[1], m, v1);
    OPAQUE_V(r0);
    OPAQUE_V(r1);
    lo = f16x2{(f16)r0, (f16)r1};
}

// h s + b in f32 by one v_fma_mix_f32 on h's half of its register.
__device__ __forceinline__ float mul_add_f16(f16 h, float s, float b) {
    float r = __builtin_fmaf((float)h, s, b);
    OPAQUE_V(r);
    return r;
}

// The 8 nibbles of a weight word in the engine nibble order (see k_repack_w4) as 4 f16 pairs q - 8
// (exact) for k = (0,1), (2,3), (4,5), (6,7): the nibble at bits 4p lands in the f16 mantissa as
// 1024 + q for p = 0, 2 (and 4, 6 in the high half), as 1024 + 16 q for the others, so two masks per
// 8-bit shift give all four pairs.
__device__ __forceinline__ void nib_pairs(uint32_t w, f16x2& p0, f16x2& p1, f16x2& p2, f16x2& p3) {
    const uint32_t w8 = w >> 8;
    const f16x2 x0 = __builtin_bit_cast(f16x2, and_or(w, 0x000F000Fu, 0x64006400u));
    const f16x2 x1 = __builtin_bit_cast(f16x2, and_or(w, 0x00F000F0u, 0x64006400u));
    const f16x2 x2 = __builtin_bit_cast(f16x2, and_or(w8, 0x000F000Fu, 0x64006400u));
    const f16x2 x3 = __builtin_bit_cast(f16x2, and_or(w8, 0x00F000F0u, 0x64006400u));
    const f16x2 c1032 = {(f16)1032.0f, (f16)1032.0f}, c16 = {(f16)0.0625f, (f16)0.0625f}, c72 = {(f16)-72.0f, (f16)-72.0f};
    p0 = x0 - c1032;
    p1 = __builtin_elementwise_fma(x1, c16, c72);
    p2 = x2 - c1032;
    p3 = __builtin_elementwise_fma(x3, c16, c72);
}

// Raw buffer access (MUBUF): a 128-bit resource of base address and byte size, per-lane 32-bit
// offsets (VGPR) plus a uniform one (SGPR); an offset at or past the size reads zeros and touches no
// memory.  The host pass of hipcc does not see the builtins.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
// 16 bytes per lane straight into LDS at lds + 16 lane (lds wave-uniform).
__device__ __forceinline__ void buf_lds16(Rsrc r, uint32_t voff, uint32_t soff, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 0, 0);
}
// Four of them, 1 KB apart on both sides (the instruction's immediate offset moves the buffer and the LDS
// address alike, so they share one scalar offset and one LDS base).
__device__ __forceinline__ void buf_lds64(Rsrc r, uint32_t voff, uint32_t soff, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 1024, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 2048, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, voff, soff, 3072, 0);
}
__device__ __forceinline__ u32x4 buf_b128(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ uint32_t buf_b16(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0);
}
__device__ __forceinline__ u32x3 buf_b96(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(r, voff, soff, 0));
}
__device__ __forceinline__ u32x2 buf_b64(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ uint32_t buf_b32(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
// A 32-bit store; an offset at or past the resource's size writes nothing.
__device__ __forceinline__ void buf_st32(Rsrc r, uint32_t voff, uint32_t soff, uint32_t v) {
    __builtin_amdgcn_raw_buffer_store_b32(v, r, voff, soff, 0);
}
#else
struct Rsrc {};
__device__ inline Rsrc make_rsrc(const void*, uint32_t) { return {}; }
__device__ inline void buf_lds16(Rsrc, uint32_t, uint32_t, void*) {}
__device__ inline void buf_lds64(Rsrc, uint32_t, uint32_t, void*) {}
__device__ inline u32x4 buf_b128(Rsrc, uint32_t, uint32_t) { return u32x4{}; }
__device__ inline uint32_t buf_b16(Rsrc, uint32_t, uint32_t) { return 0; }
__device__ inline u32x3 buf_b96(Rsrc, uint32_t, uint32_t) { return u32x3{}; }
__device__ inline u32x2 buf_b64(Rsrc, uint32_t, uint32_t) { return u32x2{}; }
__device__ inline uint32_t buf_b32(Rsrc, uint32_t, uint32_t) { return 0; }
__device__ inline void buf_st32(Rsrc, uint32_t, uint32_t, uint32_t) {}
#endif

// A per-lane buffer offset that is out of range for every buffer here: the load returns zeros and
// touches no memory.
constexpr uint32_t OOB = 0x80000000u;

// s_waitcnt immediate for vmcnt(v) with the lgkm and exp counters left unconstrained.
constexpr int vmcnt_imm(int v) { return 0x0F70 | (v & 15) | ((v >> 4) << 14); }

// s_waitcnt with a vmcnt that counts this thread's loads in issue order: scheduling barriers on
// both sides keep the compiler from moving loads across it, which would change what it counts.
template <int IMM>
__device__ __forceinline__ void wait_loads() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(IMM);
    __builtin_amdgcn_sched_barrier(0);
}

// Workgroup barrier without the release fence of __syncthreads, whose wait for every outstanding
// vector-memory load would drain the loads issued for later steps.  The caller waits (vmcnt) for
// the loads the other waves need; the "memory" clobber keeps the compiler from moving LDS
// accesses across.
__device__ __forceinline__ void bar_noflush() { asm volatile("s_barrier" ::: "memory"); }

// Workgroup barrier after this wave's LDS accesses have completed (outstanding global stores are
// not waited for, unlike __syncthreads).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// SGPR_BATCH("s"(x), "s"(y), ...): x, y, ... are in SGPRs at this point.  The scalar loads that
// produce them (kernel arguments past the preloaded ones, lu fields, table entries) are then issued
// as one batch and waited for together, one memory round trip, where the compiler would sink each
// load to its first use, behind branches, and wait for each in turn (scalar loads return out of
// order, so every wait is for all of them).
#define SGPR_BATCH(...) asm volatile("" ::__VA_ARGS__)

// XCD-aware tile order of a (gx column blocks, gy row blocks, gz K splits) grid: the hardware gives
// workgroup b to XCD b % 8, and each XCD has its own L2.  With a K split (gz in {2, 4, 8}) XCD x
// takes split x % gz and a contiguous run of the column-block-major (column, row) tiles, so it reads
// only that split's K range of the activations and of the weights.  Otherwise XCD x takes a
// contiguous run of the tiles in column-block-major order (every row block of a column block
// together), so a column block's weights reach one L2 only.
__device__ __forceinline__ void xcd_tile(int b, int gx, int gy, int gz, int& bx, int& by, int& bz) {
    const int G = gx * gy * gz, q8 = G >> 3;
    if (gz > 1 && 8 % gz == 0 && (G & 7) == 0) {
        const int x = b & 7, t = (x / gz) * q8 + (b >> 3);
        bz = x % gz;
        bx = t / gy;
        by = t % gy;
        return;
    }
    const int tile = b < 8 * q8 ? (b & 7) * q8 + (b >> 3) : b;
    const int gyz = gy * gz;
    bx = tile / gyz;
    by = (tile % gyz) % gy;
    bz = (tile % gyz) / gy;
}

// silu(g) * u = g / (1 + e^-g) * u on the hardware exp2 (v_exp_f32) and reciprocal (v_rcp_f32), each
// within about 1 ulp in f32, where libm's expf and an IEEE divide take ~25 VALU instructions; the
// result is rounded to f16 by the caller, as the reference stores mid (src/kernels.rs:123-135).
// The limits hold: e^-g overflows to inf for g -> -inf and the reciprocal gives 0.
__device__ __forceinline__ float silu_mul(float g, float u) {
#if defined(__HIP_DEVICE_COMPILE__)
    const float e = __builtin_amdgcn_exp2f(g * -1.44269504088896341f);
    return g * __builtin_amdgcn_rcpf(1.0f + e) * u;
#else
    return g * u;
#endif
}

// silu(x) = x / (1 + e^-x) the same way, kept in f32 (the conv output of the chunked delta rule;
// the reference's WGSL exp is no more exact than v_exp_f32).
__device__ __forceinline__ float silu(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.44269504088896341f));
#else
    return x;
#endif
}

__device__ __forceinline__ f16x8 cat4(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
    return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

}  // namespace
}  // namespace sd
