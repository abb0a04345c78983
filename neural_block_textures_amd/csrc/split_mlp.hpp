// The MLP of the fixed shapes on the 16-bit matrix instructions of gfx950 (v_mfma_f32_16x16x32_f16) with every operand
// in two 16-bit parts, as the ES population evaluates it (kern_pop.hpp, k_pop_split).
//
// A 32-bit value x is hi + lo with hi = x rounded to 11 significant bits and lo = x - hi rounded to 11: 22 bits and
// lo's sign, so what is left is at most one unit in the last place of x (nothing for three values of four). A product is
// w_hi x_hi + w_hi x_lo + w_lo x_hi (the fourth term is below 2^-22 of it, and is kept where a step has room for it),
// each exact in the instruction, which adds its 32 products to a 32-bit accumulator with fewer roundings than the
// 8 chained steps of the 32-bit instruction. Against 64-bit sums the results are as close as those of the 32-bit
// chains: over 72 ES steps of the shapes of this library the gradient's error is 0.98 times theirs (geometric mean). The instruction does 1024 multiply-adds and adds per cycle
// and SIMD against 64 of v_mfma_f32_16x16x4_f32, so three products cost a fifth of the 32-bit layer's time; what is
// left is VALU work: one instruction for the activation and two for the split of each hidden value. On gfx950 the time of a mix
// of matrix and VALU instructions is close to the sum of both (measured: a matrix instruction of 16 cycles hides about 5
// cycles of VALU instructions).
//
// Range. 16-bit parts span 2^-24 .. 65504, so the layers' weights are scaled by powers of two (SplitScale, split_pow2) to a
// typical size of 1 (hidden layers) or 2^9. Powers of two commute with every rounding and with the activation, so they change no
// result; the hidden values have room up to a few hundred, and keep both parts' bits down to 1/4. Features are not scaled, but
// their lo parts are (kSplitLo), against weights divided by as much: with the lo parts of small features subnormal, latents of 0.01
// gave gradients up to 1.7 and per-pixel latent differences up to 2.9 times as far from 64 bits as the 32-bit kernels. A value
// past the range becomes an infinity and its lo part the opposite one, so every unit it feeds is a NaN: the kernel sees the NaN and
// evaluates its slots again in 32 bits, from the 32-bit weights. So it does where a layer's weights are too far apart for the
// parts (split_pow2). Nothing is ever clipped.
//
// Operand layout (measured on gfx950): lane l, half j of A holds A[l % 16][8 (l / 16) + j], of B holds
// B[8 (l / 16) + j][l % 16]; C/D as the 32-bit instruction's. The 32 contraction slots are free to hold any input and
// part, as long as A and B agree: a layer's results are fed to the next as the lane holds them (mfma_mlp.hpp,
// hidden_input), hi parts in one operand, lo parts in another.
#pragma once
#include "mfma_mlp.hpp"

namespace ntc_hip {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

template <class S, bool = MfmaShape<S>::kOk>
struct SplitShape { static constexpr bool kOk = false; };
template <class S>
struct SplitShape<S, true> {
    using Q = MfmaShape<S>;
    static constexpr bool kOk = split_pays(Q::kIn, Q::kNL);
    static constexpr int kS1 = split_inputs(Q::kIn) / 8;   // first-layer steps
    // the kV hidden values of a lane in operands of eight slots: kFull operands of eight values per part (the last one
    // padded when it holds five or more), then kRem <= 4 values with both parts in one operand
    static constexpr int kV = Q::kKsH;
    static constexpr int kFull = kV / 8 + (kV % 8 > 4 ? 1 : 0);
    static constexpr int kRem = kV % 8 > 4 ? 0 : kV % 8;
    static constexpr int kA = 2 * kFull + (kRem == 0 ? 0 : (kRem <= 2 ? 1 : 2));   // weight operands per tile
    static constexpr int kB = 2 * kFull + (kRem == 0 ? 0 : 1);                     // value operands
    static constexpr int kOutVar = Q::kNout <= 4 ? 4 : 1;
};

// The value that slot j of weight operand a holds the weight of (-1: none), and whether it holds the lo part. An operand
// of kRem <= 2 values holds them as (w_hi, w_hi, w_lo, w_lo) against (x_hi, x_lo, x_hi, x_lo); kRem of 3 or 4 takes two
// weight operands, (w_hi, w_hi) then (w_lo, w_lo), against (x_hi, x_lo).
template <class S>
constexpr int split_value(int a, int j) {
    using P = SplitShape<S>;
    if (a < 2 * P::kFull) return 8 * (a / 2) + j < P::kV ? 8 * (a / 2) + j : -1;
    const int w = P::kRem <= 2 ? j & 1 : j & 3;
    return w < P::kRem ? 8 * P::kFull + w : -1;
}
template <class S>
constexpr bool split_low(int a, int j) {
    using P = SplitShape<S>;
    if (a < 2 * P::kFull) return a & 1;
    return P::kRem <= 2 ? j >= 4 : a - 2 * P::kFull == 1;
}

__device__ __forceinline__ f4v mfma_h(h8v a, h8v b, f4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// a value every lane holds, in a VGPR: a VALU instruction with an SGPR operand takes 4.5 cycles of a SIMD, with VGPRs or a
// constant only 2.5 (measured)
__device__ __forceinline__ float in_vgpr(float x) {
    asm("" : "+v"(x));
    return x;
}

// x and y in two parts: hi, then lo = x - hi (exact: v_fma_mix_f32 reads hi's halves as they are) rounded to 16 bits. neg is
// -1 in a VGPR (as a constant it turns the fused operation into a conversion and a subtraction). 18 cycles a pair; lo by
// v_fma_mixlo_f16 and v_fma_mixhi_f16 is an instruction less, but each of those takes 8.6 cycles: a 512-pair step of the
// 14-32-32-3 model on 65536 slots took 784 us with them and 766 us without.
__device__ __forceinline__ void split2(float x, float y, float neg, h2v& hi, h2v& lo) {
    hi = __builtin_convertvector((f2v){ x, y }, h2v);
    lo = __builtin_convertvector((f2v){ __builtin_fmaf((float)hi[0], neg, x), __builtin_fmaf((float)hi[1], neg, y) }, h2v);
}

// the power-of-two scales of one step's layers (scales[0 .. 2]: first, second hidden layer, output layer; [3]: what an
// output pre-activation is multiplied by), written by the minibatch launch
struct SplitScale { float s1, s2, s3, inv; };
__device__ __forceinline__ SplitScale split_scale(const float* __restrict__ p) {
    const CFloat* c = (const CFloat*)p;
    return { c[0], c[1], c[2], c[3] };
}

// A member's parameters in LDS, 4 bytes each: a weight's two parts (hi in the low half), a bias as it is. Weight rows are an
// odd number of words apart (the operand gather reads a column of 16 rows at a time). pos(k) = where flat parameter k is;
// layer(k) = 0, 1, 2 for the first hidden layer, the second, the output layer; bias(k).
template <class S>
struct SplitLds {
    using Q = MfmaShape<S>;
    static constexpr int NIN = Q::kIn, H = Q::kH, NO = Q::kNout;
    static constexpr int kRow1 = NIN | 1, kRowH = H | 1;
    // flat parameter offsets of each layer's weights
    static constexpr int kFlat2 = H * NIN + H, kFlat3 = kFlat2 + (Q::kNL - 1) * (H * H + H);
    static constexpr int kB1 = H * kRow1, kW2 = kB1 + H, kB2 = kW2 + H * kRowH;
    static constexpr int kW3 = Q::kNL > 1 ? kB2 + H : kW2, kB3 = kW3 + NO * kRowH, kWords = (kB3 + NO + 3) & ~3;
    __device__ __forceinline__ static int layer(int k) { return k >= kFlat3 ? 2 : (Q::kNL > 1 && k >= kFlat2 ? 1 : 0); }
    __device__ __forceinline__ static int local(int k) { return k - (k >= kFlat3 ? kFlat3 : (Q::kNL > 1 && k >= kFlat2 ? kFlat2 : 0)); }
    __device__ __forceinline__ static bool bias(int k) { return local(k) >= (k >= kFlat3 ? NO * H : (k >= kFlat2 ? H * H : H * NIN)); }
    __device__ __forceinline__ static int pos(int k) {
        const int q = local(k), l = layer(k);
        if (l == 0) return q < H * NIN ? (q / NIN) * kRow1 + q % NIN : kB1 + q - H * NIN;
        const int n = l == 2 ? NO : H;
        return (l == 2 ? kW3 : kW2) + (q < n * H ? (q / H) * kRowH + q % H : n * kRowH + q - n * H);
    }
};

// The factors of a member's parameters: hidden layers times b = 1 / (1 + c), so that the folded activation x' + c |x'| of
// x' = b x is x for x > 0 whatever c was rounded to; the output layer times out (-log2 e for the hardware sigmoid); the
// layers' powers of two, a bias with those of the layers before it.
struct SplitFactors { double w1, w2, w3, b1, b2, b3; };
__device__ __forceinline__ SplitFactors split_factors(const SplitScale& sc, float fold_c, double out) {
    const double b = 1.0 / (1.0 + (double)fold_c), t1 = sc.s1, t2 = t1 * sc.s2;
    return { b * sc.s1, b * sc.s2, out * sc.s3, b * t1, b * t2, out * t2 * sc.s3 };
}

// A weight (or bias) w0 + s eps times its factor as SplitLds holds it. The sum and the product are formed in 64 bits and
// rounded once, when lo is: with a member's weight rounded to 32 bits first and its factor's product rounded again, as the
// 32-bit kernels form it, the two parts' own rounding made the gradient's error 1.2 to 1.5 times theirs; a weight's error is
// the same in every slot, so unlike a sum's it does not average out over the minibatch.
__device__ __forceinline__ unsigned split_param(float w0, float s, float eps, double factor, bool bias) {
    const double v = __builtin_fma((double)s, (double)eps, (double)w0) * factor;
    const float f = (float)v;
    const _Float16 h = (_Float16)f;
    const _Float16 l = (_Float16)(float)(v - (double)(float)h);
    return bias ? __float_as_uint(f) : (unsigned)__builtin_bit_cast(unsigned short, h) | ((unsigned)__builtin_bit_cast(unsigned short, l) << 16);
}

// One member's parameters in operand layout.
template <class S>
struct SplitWeights {
    using Q = MfmaShape<S>;
    using P = SplitShape<S>;
    h8v a1[Q::kHt][P::kS1];
    f4v c1[Q::kHt];
    h8v ah[Q::kNL > 1 ? Q::kHt : 1][P::kA];
    f4v ch[Q::kNL > 1 ? Q::kHt : 1];
    // more than 4 outputs: the output tile's rows as out_at. At most 4: variant t holds output c in row 4 t + c, so four
    // tiles' outputs meet in one accumulator, tile t's in lane group t: each lane ends with the outputs of its own pixel.
    h8v ao[P::kOutVar][P::kA];
    f4v co;
};

// Gathers a member's parameters from LDS (SplitLds) into operand layout. Weights that a lane has no unit or input for are
// zero.
template <class S>
__device__ __forceinline__ void split_load(SplitWeights<S>& W, const unsigned* __restrict__ lds, int lane) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S>;
    using L = SplitLds<S>;
    constexpr int NIN = Q::kIn, H = Q::kH, NO = Q::kNout;
    constexpr unsigned kHi = 0x05040100u, kLo = 0x07060302u;   // the low, the high halves of two words
    const int i16 = lane & 15, g = lane >> 4;
    auto at = [&](bool ok, int k) { const unsigned v = lds[k]; return ok ? v : 0u; };
    auto bias = [&](bool ok, int k) { return __uint_as_float(at(ok, k)); };
    // the weights of features' lo parts: of a power of two, so exact down to a scaled weight of 2^-3, then within 2^-25
    const bool low = P::kS1 == 1 ? (g & 1) != 0 : g >= 2;
    auto for_features = [&](h8v& a) { a *= (_Float16)(low ? 1.0f / kSplitLo : 1.0f); };
    // slots 2 j and 2 j + 1 of an operand from two parameters
    auto put = [&](h8v& a, int j, unsigned x, unsigned y, unsigned half) {
        u4v v = __builtin_bit_cast(u4v, a);
        v[j] = __builtin_amdgcn_perm(y, x, half);
        a = __builtin_bit_cast(h8v, v);
    };
#pragma unroll
    for (int ot = 0; ot < Q::kHt; ot++) {
        const int u = unit_of<Q>(ot, i16), row = min(u, H - 1) * L::kRow1;
        unsigned w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int in = P::kS1 == 1 ? j : 8 * (g & 1) + j;
            w[j] = at(u < H && in < NIN, row + min(in, NIN - 1));
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if constexpr (P::kS1 == 1) {   // slots of groups 0 .. 3: (w_hi, w_hi, w_lo, w_lo) against (f_hi, f_lo, f_hi, f_lo)
                put(W.a1[ot][0], j, w[2 * j], w[2 * j + 1], g >= 2 ? kLo : kHi);
            } else {                       // step 0 w_hi, step 1 w_lo, against (f_hi 0-7, f_hi 8-15, f_lo 0-7, f_lo 8-15)
                put(W.a1[ot][0], j, w[2 * j], w[2 * j + 1], kHi);
                put(W.a1[ot][1], j, w[2 * j], w[2 * j + 1], kLo);
            }
        }
#pragma unroll
        for (int s = 0; s < P::kS1; s++) for_features(W.a1[ot][s]);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ur = unit_of<Q>(ot, 4 * g + r);
            W.c1[ot][r] = bias(ur < H, L::kB1 + min(ur, H - 1));
        }
    }
    // the weights of the row at `row` (valid if ok) for the values this lane group holds, into the operands of one tile
    auto gather = [&](h8v (&a)[P::kA], bool ok, int row) {
        unsigned w[P::kV + 1];
        w[P::kV] = 0u;
#pragma unroll
        for (int v = 0; v < P::kV; v++) {
            const int in = hidden_input<Q>(v, g);
            w[v] = at(ok && in < H, row + min(in, H - 1));
        }
#pragma unroll
        for (int q = 0; q < P::kA; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int x = split_value<S>(q, 2 * j), y = split_value<S>(q, 2 * j + 1);
                put(a[q], j, w[x < 0 ? P::kV : x], w[y < 0 ? P::kV : y], split_low<S>(q, 2 * j) ? kLo : kHi);
            }
    };
    if constexpr (Q::kNL > 1) {
#pragma unroll
        for (int ot = 0; ot < Q::kHt; ot++) {
            const int u = unit_of<Q>(ot, i16);
            gather(W.ah[ot], u < H, L::kW2 + min(u, H - 1) * L::kRowH);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int ur = unit_of<Q>(ot, 4 * g + r);
                W.ch[ot][r] = bias(ur < H, L::kB2 + min(ur, H - 1));
            }
        }
    }
    if constexpr (valu_out<S>()) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int c = i16 - 4 * t;
            gather(W.ao[t], c >= 0 && c < NO, L::kW3 + min(max(c, 0), NO - 1) * L::kRowH);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) W.co[r] = bias(r < NO, L::kB3 + min(r, NO - 1));
    } else {
        const int orow = out_at<S>(i16 >> 2, i16 & 3);
        gather(W.ao[0], orow >= 0, L::kW3 + max(orow, 0) * L::kRowH);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int oc = out_at<S>(g, r);
            W.co[r] = bias(oc >= 0, L::kB3 + max(oc, 0));
        }
    }
}

// a hidden layer's results of one tile through the activation, as the next layer's operands
template <class S>
__device__ __forceinline__ void split_act(const f4v (&acc)[MfmaShape<S>::kHt], float k, float neg, h8v (&b)[SplitShape<S>::kB]) {
    using P = SplitShape<S>;
    constexpr int V2 = P::kFull * 8 + (P::kRem ? (P::kRem <= 2 ? 2 : 4) : 0);
    h2v hi[V2 / 2], lo[V2 / 2];
#pragma unroll
    for (int q = 0; q < V2 / 2; q++) {
        const float x = 2 * q < P::kV ? act<kActFold>(acc[2 * q < P::kV ? q / 2 : 0][(2 * q) & 3], k) : 0.0f;
        const float y = 2 * q + 1 < P::kV ? act<kActFold>(acc[2 * q + 1 < P::kV ? q / 2 : 0][(2 * q + 1) & 3], k) : 0.0f;
        split2(x, y, neg, hi[q], lo[q]);
    }
    auto join = [](h2v a, h2v b, h2v c, h2v d) {
        return __builtin_shufflevector(__builtin_shufflevector(a, b, 0, 1, 2, 3), __builtin_shufflevector(c, d, 0, 1, 2, 3), 0, 1, 2, 3, 4, 5, 6, 7);
    };
#pragma unroll
    for (int f = 0; f < P::kFull; f++) {
        b[2 * f] = join(hi[4 * f], hi[4 * f + 1], hi[4 * f + 2], hi[4 * f + 3]);
        b[2 * f + 1] = join(lo[4 * f], lo[4 * f + 1], lo[4 * f + 2], lo[4 * f + 3]);
    }
    if constexpr (P::kRem > 2) b[2 * P::kFull] = join(hi[4 * P::kFull], hi[4 * P::kFull + 1], lo[4 * P::kFull], lo[4 * P::kFull + 1]);
    else if constexpr (P::kRem > 0) b[2 * P::kFull] = join(hi[4 * P::kFull], lo[4 * P::kFull], hi[4 * P::kFull], lo[4 * P::kFull]);
}

// c plus one tile row block's products with the values b (the small terms last); All: the products of two lo parts too
template <class S, bool All = false>
__device__ __forceinline__ f4v split_dot(const h8v (&a)[SplitShape<S>::kA], const h8v (&b)[SplitShape<S>::kB], f4v c) {
    using P = SplitShape<S>;
#pragma unroll
    for (int f = 0; f < P::kFull; f++) c = mfma_h(a[2 * f], b[2 * f], c);
#pragma unroll
    for (int q = 2 * P::kFull; q < P::kA; q++) c = mfma_h(a[q], b[2 * P::kFull], c);
#pragma unroll
    for (int f = 0; f < P::kFull; f++) {
        c = mfma_h(a[2 * f], b[2 * f + 1], c);
        c = mfma_h(a[2 * f + 1], b[2 * f], c);
        if constexpr (All) c = mfma_h(a[2 * f + 1], b[2 * f + 1], c);
    }
    return c;
}

// the hidden layers of one tile from its first-layer operand (the split features of a slot: split_features), the last
// one's values as operands
template <class S, bool All = false>
__device__ __forceinline__ void split_hidden(const SplitWeights<S>& W, h8v f, float k, float neg, h8v (&b)[SplitShape<S>::kB]) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S>;
    f4v acc[Q::kHt];
#pragma unroll
    for (int ot = 0; ot < Q::kHt; ot++) acc[ot] = mfma_h(W.a1[ot][0], f, W.c1[ot]);
    if constexpr (P::kS1 > 1)
#pragma unroll
        for (int ot = 0; ot < Q::kHt; ot++) acc[ot] = mfma_h(W.a1[ot][1], f, acc[ot]);
    split_act<S>(acc, k, neg, b);
    if constexpr (Q::kNL > 1) {
        f4v a2[Q::kHt];
#pragma unroll
        for (int ot = 0; ot < Q::kHt; ot++) a2[ot] = split_dot<S, All>(W.ah[ot], b, W.ch[ot]);
        split_act<S>(a2, k, neg, b);
    }
}

// split_hidden of N tiles, a layer of every tile at a time: their matrix and VALU instructions are independent
template <class S, int N>
__device__ __forceinline__ void split_hidden_n(const SplitWeights<S>& W, const h8v (&f)[N], float k, float neg, h8v (&b)[N][SplitShape<S>::kB]) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S>;
    f4v acc[N][Q::kHt];
#pragma unroll
    for (int s = 0; s < P::kS1; s++)
#pragma unroll
        for (int n = 0; n < N; n++)
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++) acc[n][ot] = mfma_h(W.a1[ot][s], f[n], s == 0 ? W.c1[ot] : acc[n][ot]);
#pragma unroll
    for (int n = 0; n < N; n++) split_act<S>(acc[n], k, neg, b[n]);
    if constexpr (Q::kNL > 1) {
        f4v a2[N][Q::kHt];
#pragma unroll
        for (int n = 0; n < N; n++)
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++) a2[n][ot] = split_dot<S>(W.ah[ot], b[n], W.ch[ot]);
#pragma unroll
        for (int n = 0; n < N; n++) split_act<S>(a2[n], k, neg, b[n]);
    }
}

}   // namespace ntc_hip
