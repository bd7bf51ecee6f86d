// The cascade networks' trained weights as compile-time constants, for kernels that carry
// them as literal operands: read by the compiler from the same model bytes that the
// library embeds (ccnn_model_bytes.h, written by build.py), in the field order that
// load_model reads (model format 1.0 - 1.1).
//
// Why literals: on gfx950 a SIMD issues a float multiply or add every 2 clocks when its
// operands are registers or literals, but every 4 clocks when one is an SGPR (measured
// with 8 waves per SIMD: 0.44 instructions a clock against 0.23; half of the stream with
// an SGPR operand still runs at 0.43, two thirds at 0.31), and weights in LDS cost an LDS
// read per operand. A literal costs four bytes of code.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "ccnn_internal.h"
#include "ccnn_model_bytes.h"

namespace ccnn {

// The weights up to the hidden layer's, laid out as NetShape's offsets say (the output
// layer depends on the detector's index_output and stays in memory).
template <class N>
struct ConstNet {
    float w[N::oOW] = {};
    bool ok = false;
};

namespace detail {
struct ConstReader {
    const unsigned char* p;
    size_t n, at = 0;
    constexpr int i8() { return at < n ? p[at++] : -1; }
    constexpr unsigned u32()
    {
        unsigned v = 0;
        for (int k = 0; k < 4; ++k) v |= (unsigned)(at + k < n ? p[at + k] : 0) << (8 * k);
        at += 4;
        return v;
    }
    constexpr int i32() { return (int)u32(); }
    constexpr float f32() { return __builtin_bit_cast(float, u32()); }
};
}  // namespace detail

template <class N, size_t BYTES>
constexpr ConstNet<N> const_net(const unsigned char (&bytes)[BYTES])
{
    ConstNet<N> r;
    detail::ConstReader in{bytes, BYTES};
    in.f32();                                                    // version
    in.i8();                                                     // max-pooling
    in.i32();
    in.i32();                                                    // window
    if (in.i32() != 3) return r;
    if (in.i32() != N::M1 || in.i32() != N::M2 || in.i32() != N::M3) return r;
    const int kw[3] = {N::K1, 3, N::K3W}, kh[3] = {N::K1, 3, N::K3H}, maps[3] = {N::M1, N::M2, N::M3};
    const int ok[3] = {N::oK1, N::oK2, N::oK3}, ob[3] = {N::oB1, N::oB2, N::oB3};
    for (int l = 0; l < 3; ++l) {
        if (in.i32() != kw[l] || in.i32() != kh[l]) return r;
        for (int k = 0; k < maps[l] * kw[l] * kh[l]; ++k) r.w[ok[l] + k] = in.f32();
    }
    in.f32();                                                    // af_scale
    for (int l = 0; l < 3; ++l)
        for (int m = 0; m < maps[l]; ++m) {
            r.w[ob[l] + m] = in.f32();                           // conv_b
            r.w[ob[l] + maps[l] + m] = in.f32();                 // lrelu_w1
            r.w[ob[l] + 2 * maps[l] + m] = in.f32();             // lrelu_w2
            in.f32();                                            // bn_w (folded into w1 / w2)
            r.w[ob[l] + 3 * maps[l] + m] = in.f32();             // bn_b
        }
    const int full = in.i8();
    if (in.i32() != N::HL || in.i32() != N::HLN || in.i32() != N::HLS) return r;
    const int nin = full ? N::M3 : N::HLN;
    for (int u = 0; u < N::HL; ++u)
        for (int j = 0; j < nin; ++j) {
            const float v = in.f32();
            if (j < N::HLN) r.w[N::oHW + u * N::HLN + j] = v;
        }
    for (int u = 0; u < N::HL; ++u) r.w[N::oHB + u] = in.f32();
    for (int g = 0; g < N::HLG; ++g) r.w[N::oHT + g] = in.f32();
    for (int t = 0; t < N::HLS; ++t) {
        r.w[N::oHBW + t] = in.f32();
        r.w[N::oHBB + t] = in.f32();
    }
    r.ok = in.at <= BYTES;
    return r;
}

template <class N>
struct ConstNetOf;
template <>
struct ConstNetOf<Stage1> {
    static constexpr ConstNet<Stage1> net = const_net<Stage1>(k_model0);
};
template <>
struct ConstNetOf<Stage2> {
    static constexpr ConstNet<Stage2> net = const_net<Stage2>(k_model1);
};
template <>
struct ConstNetOf<Stage3> {
    static constexpr ConstNet<Stage3> net = const_net<Stage3>(k_model2);
};
static_assert(ConstNetOf<Stage1>::net.ok && ConstNetOf<Stage2>::net.ok && ConstNetOf<Stage3>::net.ok,
              "the embedded models have the cascade's network shapes");

// the weight at offset O of network N
template <class N, int O>
constexpr float weight_v = ConstNetOf<N>::net.w[O];
template <class N, int O>
constexpr int weight_bits = __builtin_bit_cast(int, ConstNetOf<N>::net.w[O]);

// f(0), .., f(COUNT - 1) with the index as a compile-time constant
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int COUNT, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_seq(f, std::make_integer_sequence<int, COUNT>{});
}

// A map's convolution at the four positions of a 2x2 pooling quad, its activation with
// batch norm (lrelu_bn) and the max-pool, with every weight a literal. Written in assembly
// because the compiler keeps a constant that is used more than once in an SGPR; as one
// block because it puts an s_nop between an assembly block's result and its next use
// (242 of 873 instructions of the L1 loop with a block per operation). The four chains
// are interleaved, each multiply and add rounded by itself in the order of the scalar code.
//
// When both slopes of the map's activation have the same sign, every rounded step from the
// convolution on is monotone (rising for positive slopes, falling for negative ones), so
// the pool of the activations is the activation of the largest (smallest) convolution, bit
// for bit, NaNs included (the maximum and the minimum both skip them); bn_b is not zero,
// so no sign of a zero is lost. Three of four activations fall away. Slopes of opposite
// sign have no such order (the rounded sum is not monotone between neighbouring floats).
// tap KK at window samples W0..W3 of the quad: first one, then the others
#define CCNN_TAP0(KK, W0, W1, W2, W3)                                                               \
    "v_mul_f32_e32 %[a0], %[" #KK "], %[" #W0 "]\n v_mul_f32_e32 %[a1], %[" #KK "], %[" #W1 "]\n"   \
    "v_mul_f32_e32 %[a2], %[" #KK "], %[" #W2 "]\n v_mul_f32_e32 %[a3], %[" #KK "], %[" #W3 "]\n"
#define CCNN_TAP(KK, W0, W1, W2, W3)                                                                \
    "v_mul_f32_e32 %[t0], %[" #KK "], %[" #W0 "]\n v_mul_f32_e32 %[t1], %[" #KK "], %[" #W1 "]\n"   \
    "v_mul_f32_e32 %[t2], %[" #KK "], %[" #W2 "]\n v_mul_f32_e32 %[t3], %[" #KK "], %[" #W3 "]\n"   \
    "v_add_f32_e32 %[a0], %[a0], %[t0]\n v_add_f32_e32 %[a1], %[a1], %[t1]\n"                       \
    "v_add_f32_e32 %[a2], %[a2], %[t2]\n v_add_f32_e32 %[a3], %[a3], %[t3]\n"
// a of each position: (w2 * max(0, c) + bn_b) + w1 * c with c = a + conv_b
#define CCNN_ACT4                                                                                   \
    "v_add_f32_e32 %[a0], %[cb], %[a0]\n v_add_f32_e32 %[a1], %[cb], %[a1]\n"                       \
    "v_add_f32_e32 %[a2], %[cb], %[a2]\n v_add_f32_e32 %[a3], %[cb], %[a3]\n"                       \
    "v_max_f32_e32 %[t0], 0, %[a0]\n v_mul_f32_e32 %[a0], %[w1], %[a0]\n"                           \
    "v_max_f32_e32 %[t1], 0, %[a1]\n v_mul_f32_e32 %[a1], %[w1], %[a1]\n"                           \
    "v_max_f32_e32 %[t2], 0, %[a2]\n v_mul_f32_e32 %[a2], %[w1], %[a2]\n"                           \
    "v_max_f32_e32 %[t3], 0, %[a3]\n v_mul_f32_e32 %[a3], %[w1], %[a3]\n"                           \
    "v_mul_f32_e32 %[t0], %[w2], %[t0]\n v_mul_f32_e32 %[t1], %[w2], %[t1]\n"                       \
    "v_mul_f32_e32 %[t2], %[w2], %[t2]\n v_mul_f32_e32 %[t3], %[w2], %[t3]\n"                       \
    "v_add_f32_e32 %[t0], %[bb], %[t0]\n v_add_f32_e32 %[t1], %[bb], %[t1]\n"                       \
    "v_add_f32_e32 %[t2], %[bb], %[t2]\n v_add_f32_e32 %[t3], %[bb], %[t3]\n"                       \
    "v_add_f32_e32 %[a0], %[t0], %[a0]\n v_add_f32_e32 %[a1], %[t1], %[a1]\n"                       \
    "v_add_f32_e32 %[a2], %[t2], %[a2]\n v_add_f32_e32 %[a3], %[t3], %[a3]\n"
#define CCNN_MAX4 "v_max_f32_e32 %[a0], %[a0], %[a1]\n v_max3_f32 %[a0], %[a0], %[a2], %[a3]\n"
#define CCNN_MIN4 "v_min_f32_e32 %[a0], %[a0], %[a1]\n v_min3_f32 %[a0], %[a0], %[a2], %[a3]\n"
#define CCNN_ACT1                                                                                   \
    "v_add_f32_e32 %[a0], %[cb], %[a0]\n"                                                           \
    "v_max_f32_e32 %[t0], 0, %[a0]\n v_mul_f32_e32 %[a0], %[w1], %[a0]\n"                           \
    "v_mul_f32_e32 %[t0], %[w2], %[t0]\n v_add_f32_e32 %[t0], %[bb], %[t0]\n"                       \
    "v_add_f32_e32 %[a0], %[t0], %[a0]\n"
// the same with fused multiply-adds (the FP16 form): fma(w1, c, fma(w2, max(0, c), bn_b)).
// v_fmamk_f32 reads two registers and a literal and issues like a multiply; v_fma_f32 with
// three registers takes twice as long
#define CCNN_ACT4H                                                                                  \
    "v_add_f32_e32 %[a0], %[cb], %[a0]\n v_add_f32_e32 %[a1], %[cb], %[a1]\n"                       \
    "v_add_f32_e32 %[a2], %[cb], %[a2]\n v_add_f32_e32 %[a3], %[cb], %[a3]\n"                       \
    "v_mov_b32_e32 %[b], %[bb]\n"                                                                   \
    "v_max_f32_e32 %[t0], 0, %[a0]\n v_max_f32_e32 %[t1], 0, %[a1]\n"                               \
    "v_max_f32_e32 %[t2], 0, %[a2]\n v_max_f32_e32 %[t3], 0, %[a3]\n"                               \
    "v_fmamk_f32 %[t0], %[t0], %[w2], %[b]\n v_fmamk_f32 %[t1], %[t1], %[w2], %[b]\n"               \
    "v_fmamk_f32 %[t2], %[t2], %[w2], %[b]\n v_fmamk_f32 %[t3], %[t3], %[w2], %[b]\n"               \
    "v_fmamk_f32 %[a0], %[a0], %[w1], %[t0]\n v_fmamk_f32 %[a1], %[a1], %[w1], %[t1]\n"             \
    "v_fmamk_f32 %[a2], %[a2], %[w1], %[t2]\n v_fmamk_f32 %[a3], %[a3], %[w1], %[t3]\n"
#define CCNN_ACT1H                                                                                  \
    "v_add_f32_e32 %[a0], %[cb], %[a0]\n v_mov_b32_e32 %[b], %[bb]\n"                               \
    "v_max_f32_e32 %[t0], 0, %[a0]\n v_fmamk_f32 %[t0], %[t0], %[w2], %[b]\n"                       \
    "v_fmamk_f32 %[a0], %[a0], %[w1], %[t0]\n"
#define CCNN_ACC                                                                                    \
    [a0] "=&v"(a0), [a1] "=&v"(a1), [a2] "=&v"(a2), [a3] "=&v"(a3), [t0] "=&v"(t0), [t1] "=&v"(t1), \
        [t2] "=&v"(t2), [t3] "=&v"(t3)
#define CCNN_PAR                                                                                    \
    [cb] "n"(weight_bits<N, OB + M>), [w1] "n"(weight_bits<N, OB + MAPS + M>),                      \
        [w2] "n"(weight_bits<N, OB + 2 * MAPS + M>), [bb] "n"(weight_bits<N, OB + 3 * MAPS + M>)
#define CCNN_K(J) [k##J] "n"(weight_bits<N, OK + J>)
#define CCNN_W(R, C) [w##R##C] "v"(w[R][C])

// how the map's pool commutes with its activation: 1 rising, -1 falling, 0 not
template <class N, int OB, int MAPS, int M>
constexpr int act_order()
{
    constexpr float w1 = weight_v<N, OB + MAPS + M>, w2 = weight_v<N, OB + 2 * MAPS + M>;
    if (weight_v<N, OB + 3 * MAPS + M> == 0.f) return 0;
    return w1 > 0.f && w2 > 0.f ? 1 : w1 < 0.f && w2 < 0.f ? -1 : 0;
}

// 4x4 kernel at offset OK over a 5x5 window; activation parameters of map M (of MAPS) at OB
template <class N, int OK, int OB, int MAPS, int M>
__device__ __forceinline__ float conv4_act_pool(const float (&w)[5][5])
{
#define CCNN_CONV4                                                                                          \
    CCNN_TAP0(k0, w00, w01, w10, w11) CCNN_TAP(k1, w01, w02, w11, w12) CCNN_TAP(k2, w02, w03, w12, w13)     \
    CCNN_TAP(k3, w03, w04, w13, w14) CCNN_TAP(k4, w10, w11, w20, w21) CCNN_TAP(k5, w11, w12, w21, w22)      \
    CCNN_TAP(k6, w12, w13, w22, w23) CCNN_TAP(k7, w13, w14, w23, w24) CCNN_TAP(k8, w20, w21, w30, w31)      \
    CCNN_TAP(k9, w21, w22, w31, w32) CCNN_TAP(k10, w22, w23, w32, w33) CCNN_TAP(k11, w23, w24, w33, w34)    \
    CCNN_TAP(k12, w30, w31, w40, w41) CCNN_TAP(k13, w31, w32, w41, w42) CCNN_TAP(k14, w32, w33, w42, w43)   \
    CCNN_TAP(k15, w33, w34, w43, w44)
#define CCNN_IN4                                                                                            \
    CCNN_W(0, 0), CCNN_W(0, 1), CCNN_W(0, 2), CCNN_W(0, 3), CCNN_W(0, 4), CCNN_W(1, 0), CCNN_W(1, 1),       \
        CCNN_W(1, 2), CCNN_W(1, 3), CCNN_W(1, 4), CCNN_W(2, 0), CCNN_W(2, 1), CCNN_W(2, 2), CCNN_W(2, 3),   \
        CCNN_W(2, 4), CCNN_W(3, 0), CCNN_W(3, 1), CCNN_W(3, 2), CCNN_W(3, 3), CCNN_W(3, 4), CCNN_W(4, 0),   \
        CCNN_W(4, 1), CCNN_W(4, 2), CCNN_W(4, 3), CCNN_W(4, 4), CCNN_K(0), CCNN_K(1), CCNN_K(2), CCNN_K(3), \
        CCNN_K(4), CCNN_K(5), CCNN_K(6), CCNN_K(7), CCNN_K(8), CCNN_K(9), CCNN_K(10), CCNN_K(11),           \
        CCNN_K(12), CCNN_K(13), CCNN_K(14), CCNN_K(15), CCNN_PAR
    constexpr int order = act_order<N, OB, MAPS, M>();
    float a0, a1, a2, a3, t0, t1, t2, t3;
    if constexpr (order > 0)
        asm(CCNN_CONV4 CCNN_MAX4 CCNN_ACT1 : CCNN_ACC : CCNN_IN4);
    else if constexpr (order < 0)
        asm(CCNN_CONV4 CCNN_MIN4 CCNN_ACT1 : CCNN_ACC : CCNN_IN4);
    else
        asm(CCNN_CONV4 CCNN_ACT4 CCNN_MAX4 : CCNN_ACC : CCNN_IN4);
    return a0;
#undef CCNN_CONV4
#undef CCNN_IN4
}

// 3x3 kernel over a 4x4 window
template <class N, int OK, int OB, int MAPS, int M>
__device__ __forceinline__ float conv3_act_pool(const float (&w)[4][4])
{
#define CCNN_CONV3                                                                                          \
    CCNN_TAP0(k0, w00, w01, w10, w11) CCNN_TAP(k1, w01, w02, w11, w12) CCNN_TAP(k2, w02, w03, w12, w13)     \
    CCNN_TAP(k3, w10, w11, w20, w21) CCNN_TAP(k4, w11, w12, w21, w22) CCNN_TAP(k5, w12, w13, w22, w23)      \
    CCNN_TAP(k6, w20, w21, w30, w31) CCNN_TAP(k7, w21, w22, w31, w32) CCNN_TAP(k8, w22, w23, w32, w33)
#define CCNN_IN3                                                                                            \
    CCNN_W(0, 0), CCNN_W(0, 1), CCNN_W(0, 2), CCNN_W(0, 3), CCNN_W(1, 0), CCNN_W(1, 1), CCNN_W(1, 2),       \
        CCNN_W(1, 3), CCNN_W(2, 0), CCNN_W(2, 1), CCNN_W(2, 2), CCNN_W(2, 3), CCNN_W(3, 0), CCNN_W(3, 1),   \
        CCNN_W(3, 2), CCNN_W(3, 3), CCNN_K(0), CCNN_K(1), CCNN_K(2), CCNN_K(3), CCNN_K(4), CCNN_K(5),       \
        CCNN_K(6), CCNN_K(7), CCNN_K(8), CCNN_PAR
    constexpr int order = act_order<N, OB, MAPS, M>();
    float a0, a1, a2, a3, t0, t1, t2, t3;
    if constexpr (order > 0)
        asm(CCNN_CONV3 CCNN_MAX4 CCNN_ACT1 : CCNN_ACC : CCNN_IN3);
    else if constexpr (order < 0)
        asm(CCNN_CONV3 CCNN_MIN4 CCNN_ACT1 : CCNN_ACC : CCNN_IN3);
    else
        asm(CCNN_CONV3 CCNN_ACT4 CCNN_MAX4 : CCNN_ACC : CCNN_IN3);
    return a0;
#undef CCNN_CONV3
#undef CCNN_IN3
}

// The pool of lrelu_bn_fma over the four convolutions of map M, in the FP16 form. A dot
// product's result may be read by another kind of instruction after three wait states, which
// the compiler does not place before an assembly block: the blocks begin with four.
#define CCNN_AFTER_DOT "s_nop 3\n"
template <class N, int OB, int MAPS, int M>
__device__ __forceinline__ float act_pool_fma(float a0, float a1, float a2, float a3)
{
    constexpr int order = act_order<N, OB, MAPS, M>();
    float t0, t1, t2, t3, b;
#define CCNN_ACCH                                                                                           \
    [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3), [t0] "=&v"(t0), [t1] "=&v"(t1),             \
        [t2] "=&v"(t2), [t3] "=&v"(t3), [b] "=&v"(b)
    if constexpr (order > 0)
        asm(CCNN_AFTER_DOT CCNN_MAX4 CCNN_ACT1H : CCNN_ACCH : CCNN_PAR);
    else if constexpr (order < 0)
        asm(CCNN_AFTER_DOT CCNN_MIN4 CCNN_ACT1H : CCNN_ACCH : CCNN_PAR);
    else
        asm(CCNN_AFTER_DOT CCNN_ACT4H CCNN_MAX4 : CCNN_ACCH : CCNN_PAR);
    return a0;
#undef CCNN_ACCH
}
#undef CCNN_TAP0
#undef CCNN_TAP
#undef CCNN_ACT4
#undef CCNN_AFTER_DOT
#undef CCNN_ACT4H
#undef CCNN_ACT1H
#undef CCNN_ACT1
#undef CCNN_MAX4
#undef CCNN_MIN4
#undef CCNN_ACC
#undef CCNN_PAR
#undef CCNN_K
#undef CCNN_W

// x * k + y, fused, k a literal given by its bits
template <int BITS>
__device__ __forceinline__ float fma_k(float x, float y)
{
    float r;
    asm("v_fmamk_f32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "n"(BITS), "v"(y));
    return r;
}
// lrelu_bn_fma of map M
template <class N, int OB, int MAPS, int M>
__device__ __forceinline__ float lrelu_bn_fma_w(float conv)
{
    const float c = conv + weight_v<N, OB + M>;
    const float t = fma_k<weight_bits<N, OB + 2 * MAPS + M>>(fmaxf(0.f, c), weight_v<N, OB + 3 * MAPS + M>);
    return fma_k<weight_bits<N, OB + MAPS + M>>(c, t);
}
// two weights rounded to FP16 in one word, as Stage1H's tap pairs
template <class N, int A, int B>
constexpr uint32_t weight_half2 = (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)ConstNetOf<N>::net.w[A]) |
                                  (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)ConstNetOf<N>::net.w[B]) << 16;

// Activation and batch norm of map M of the layer whose parameters start at OB (MAPS maps),
// as lrelu_bn: constants that are used once, which the compiler makes literals by itself.
template <class N, int OB, int MAPS, int M>
__device__ __forceinline__ float lrelu_bn_w(float conv)
{
    const float c = conv + weight_v<N, OB + M>;
    return (weight_v<N, OB + 2 * MAPS + M> * fmaxf(0.f, c) + weight_v<N, OB + 3 * MAPS + M>)
         + weight_v<N, OB + MAPS + M> * c;
}

}  // namespace ccnn
