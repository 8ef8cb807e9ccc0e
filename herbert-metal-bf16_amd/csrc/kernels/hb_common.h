// hb_common.h -- shared device helpers of the HIP kernel sources.  These
// sources are compiled by hiprtc at load for gfx950 with every shape baked in
// as -D constants (the role the reference's MSL emission at load plays,
// src/msl/mod.rs:1-27); the build embeds them in libherbert_hip.so.
#pragma once

typedef unsigned int u32;
typedef unsigned short u16;
typedef unsigned long long u64;
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

#define HB_DEV __device__ __attribute__((always_inline)) inline

// src/core/bf16.rs:7-9: exact widening.
HB_DEV float bf16_to_f32(u32 h) { return __builtin_bit_cast(float, h << 16); }
HB_DEV float bf16_lo(u32 w) { return __builtin_bit_cast(float, w << 16); }
HB_DEV float bf16_hi(u32 w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// src/core/bf16.rs:13-23, src/msl/mod.rs:1333-1347: (bits + 0x7fff + lsb) >> 16.
HB_DEV u32 f32_to_bf16(float f) {
    u32 b = __builtin_bit_cast(u32, f);
    return (b + 0x7fffu + ((b >> 16) & 1u)) >> 16;
}
// The same rounding of arithmetic results by gfx950's v_cvt_pk_bf16_f32: one
// instruction a pair against ten.  It equals the integer form on every value
// that is not a NaN, and on the NaNs that arithmetic on bf16 operands gives
// (quiet, their low 16 bits zero).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
HB_DEV u32 pack_bf16x2(float lo, float hi) { return __builtin_bit_cast(u32, bf16x2{(__bf16)lo, (__bf16)hi}); }
HB_DEV float round_bf16(float f) { return bf16_to_f32(__builtin_bit_cast(u16, (__bf16)f)); }

// exp of f32: Cody-Waite reduction by ln 2 and the minimax polynomial of
// Moshier's Cephes expf, every step an explicit fma, so that the CPU oracle
// built with the same steps gives the same bits.  The scaling by 2^n is one
// v_ldexp_f32 (one rounding, as the two exact-then-rounded multiplies that the
// oracle does: equal on all 2^32 inputs) and the range ends are selects.
HB_DEV float exp_core(float x) {
    float n = __builtin_floorf(__builtin_fmaf(x, 1.44269504088896341f, 0.5f));
    float r = __builtin_fmaf(n, -0.693359375f, x);
    r = __builtin_fmaf(n, 2.12194440e-4f, r);
    float z = r * r;
    float p = 1.9875691500e-4f;
    p = __builtin_fmaf(p, r, 1.3981999507e-3f);
    p = __builtin_fmaf(p, r, 8.3334519073e-3f);
    p = __builtin_fmaf(p, r, 4.1665795894e-2f);
    p = __builtin_fmaf(p, r, 1.6666665459e-1f);
    p = __builtin_fmaf(p, r, 5.0000001201e-1f);
    p = __builtin_fmaf(p, z, r);
    p = p + 1.0f;
    return __builtin_ldexpf(p, (int)n);
}
HB_DEV float hb_expf(float x) {
    float y = exp_core(x);
    y = x > 88.72283905206835f ? __builtin_inff() : y;
    y = x < -103.278929903431851103f ? 0.0f : y;
    return x != x ? x : y;
}

// src/msl/mod.rs:885-890: 1 / (1 + e^-x), an IEEE division.
HB_DEV float hb_sigmoid(float x) { return 1.0f / (1.0f + hb_expf(-x)); }

// (g * sigmoid(g)) * u.  A NaN gate gives sigmoid's NaN (-g, quiet), which
// with two NaN factors would be the compiler's choice of their order.
HB_DEV float swiglu_f(float g, float u) {
    const float s = hb_sigmoid(g);
    return g != g ? s : (g * s) * u;
}

// swiglu_f of n bf16-valued gates: its bits on all 65536 of them, in 24
// instructions an output against 40 (a 256 x 288 tile's SwiGLU took 7 us of
// VALU issue).  While every gate is within +-87, e^-g is within 2^-126 and
// 2^126 and needs no range checks, and the division is v_rcp_f32 with one
// Newton step by fma (Markstein), which equals the IEEE quotient for every
// float d from 1 to 2^126 (all 1.06e9 compared).  One test covers the n
// gates; a NaN is not within the range.
template <u32 n>
HB_DEV void swiglu_n(const float* g, const float* u, float* h) {
    bool near = true;
#pragma unroll
    for (u32 i = 0; i < n; i++) near &= __builtin_fabsf(g[i]) <= 87.0f;
    if (!near) {
#pragma unroll 1
        for (u32 i = 0; i < n; i++) h[i] = swiglu_f(g[i], u[i]);
        return;
    }
#pragma unroll
    for (u32 i = 0; i < n; i++) {
        const float d = 1.0f + exp_core(-g[i]);
        const float r = __builtin_amdgcn_rcpf(d);
        h[i] = (g[i] * __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r)) * u[i];
    }
}

// swiglu_n on 8 gates and 8 ups held as bf16 pairs, rounded to bf16 pairs.
HB_DEV u32x4 swiglu_pairs(u32x4 gv, u32x4 uv) {
    float g[8], u[8], h[8];
#pragma unroll
    for (u32 e = 0; e < 4; e++) {
        g[2 * e] = bf16_lo(gv[e]);
        g[2 * e + 1] = bf16_hi(gv[e]);
        u[2 * e] = bf16_lo(uv[e]);
        u[2 * e + 1] = bf16_hi(uv[e]);
    }
    swiglu_n<8>(g, u, h);
    u32x4 o;
#pragma unroll
    for (u32 e = 0; e < 4; e++) o[e] = pack_bf16x2(h[2 * e], h[2 * e + 1]);
    return o;
}

// The 64 lanes' sum in the xor butterfly's association (lanes 32 apart
// first, then 16, 8, 4, 2, 1), every lane with the same bits: the halves and
// the 16-lane rows by lane swaps, then rotations within 16 lanes (once lanes
// 8 apart agree, a rotation by 4 holds what lane l ^ 4 does) and quads.  Six
// __shfl_xor give the same value in six LDS-crossbar round trips.
HB_DEV float butterfly_sum(float v) {
    // Words by value: this compiler's __builtin_bit_cast of a vector's
    // element takes element 0 whatever the index.
    auto f32 = [](u32 w) { return __builtin_bit_cast(float, w); };
    u32 b = __builtin_bit_cast(u32, v);
    const auto h = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    v = f32(h[0]) + f32(h[1]);
    b = __builtin_bit_cast(u32, v);
    const auto q = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    v = f32(q[0]) + f32(q[1]);
#define HB_DPP_ADD(ctrl)                                                                             \
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, \
                                                               0xf, 0xf, true))
    HB_DPP_ADD(0x128);  // row_ror:8
    HB_DPP_ADD(0x124);  // row_ror:4
    HB_DPP_ADD(0x4E);   // quad_perm [2,3,0,1]
    HB_DPP_ADD(0xB1);   // quad_perm [1,0,3,2]
#undef HB_DPP_ADD
    return v;
}

// The row count of a block: state[3] as the reference's kernels read it
// (src/metal/kernels.rs:15, prefill.rs:21-24), never more than the rows the
// launch was sized for.
#define STATE_ROWS 3
HB_DEV u32 rows_of_state(const u32* state, u32 m_launch) {
    u32 m = state[STATE_ROWS];
    return m < m_launch ? m : m_launch;
}

// The workgroups a launch of `groups` spreads over the 8 XCDs round robin
// (workgroup g runs on XCD g % 8): the logical index that gives each XCD a
// contiguous range of tiles, so that tiles sharing a panel of W or X share
// that XCD's L2.
HB_DEV u32 xcd_remap(u32 g, u32 groups) {
    const u32 x = g & 7u, i = g >> 3;
    const u32 q = groups >> 3, r = groups & 7u;
    return x * q + (x < r ? x : r) + i;
}

// The kernel's symbol: the emitted name (gemm_mma_2560x4608_..., set with
// -DHB_NAME by the library), so profiles tell the variants apart.
#ifndef HB_NAME
#define HB_NAME hb_kernel
#endif
