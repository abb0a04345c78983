// The MLP of the fixed shapes on the 16-bit matrix instructions of gfx950 (v_mfma_f32_16x16x32_f16) with every operand
// in 16-bit parts, as the population, the latent pairs and the selector search evaluate it (kern_pop.hpp).
//
// A 32-bit value x is hi + lo with hi = x rounded to 11 significant bits and lo = x - hi rounded to 11: 22 bits and
// lo's sign, so what is left is at most one unit in the last place of x, and nothing for three values of four, where both parts
// are normal numbers (Range, below). Values have these two parts. So have weights where all evaluations share them (latent pairs,
// selector search: four products). A population's members differ in their weights, whose rounding is the same in every slot and
// does not average out over the minibatch: theirs have a third part, what hi and lo leave, and a product is w_hi x_hi + w_hi x_lo +
// w_lo x_hi + w_last x_hi (with two parts their gradients were up to 1.3 times as far from 64 bits as the 32-bit kernels'). The
// products are exact in the instruction, which adds its 32 to the accumulator with an error of 0.6 units of the sum (RMS,
// measured; a chain of 32 fused operations: 1.6). The small products come first, so that only the last steps round at the size
// of the sum: the other way round the errors were a third larger. Errors against 64 bits over those of the 32-bit kernels, on nine
// to eleven models each with ordinary, small and large weights and latents: ES members' loss differences 0.38 to 0.97 times, central
// differences' 0.81 to 1.02, per-pixel latent differences 0.68 to 0.98 (1.13 for a 16-wide model with its weights three times as
// large).
//
// The instruction does 1024 multiply-adds and adds per cycle and SIMD against 64 of v_mfma_f32_16x16x4_f32, so four products cost
// a quarter of the 32-bit layer's time; what is left is VALU work: one instruction for the activation and two for the split of each
// hidden value. On gfx950 the time of a mix of matrix and VALU instructions is close to the sum of both (measured: a matrix
// instruction of 16 cycles hides about 5 cycles of VALU instructions).
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

// Parts of a weight (a value has two): three in the population, two where all evaluations share the weights.
template <class S, int Parts = 2, bool = MfmaShape<S>::kOk>
struct SplitShape { static constexpr bool kOk = false; };
template <class S, int Parts>
struct SplitShape<S, Parts, true> {
    using Q = MfmaShape<S>;
    static constexpr bool kOk = split_pays(Q::kIn, Q::kNL);
    static constexpr int kS1 = split_inputs(Q::kIn) / 8;   // first-layer steps
    // the kV hidden values of a lane in operands of eight slots: kFull operands of eight values per part (the last one
    // padded when it holds five or more), then kRem <= 4 values with both parts in one operand
    static constexpr int kV = Q::kKsH;
    static constexpr int kFull = kV / 8 + (kV % 8 > 4 ? 1 : 0);
    static constexpr int kRem = kV % 8 > 4 ? 0 : kV % 8;
    static constexpr int kA = 2 * kFull + (kRem == 0 ? 0 : (kRem <= 2 ? 1 : 2));                 // weight operands per tile
    static constexpr int kB = 2 * kFull + (kRem == 0 ? 0 : (kRem > 2 && Parts == 3 ? 2 : 1));    // value operands
    static constexpr int kOutVar = Q::kNout <= 4 ? 4 : 1;
    // Three parts: the last parts of a layer's full operands follow its others, kFull of them. Operands of a member that stay in
    // LDS, 64 lanes of 16 bytes each, for registers: the hidden layer's last parts (kHidLds), the output layer's operands (kOutLds),
    // the first layer's second step (kW1Lds).
    static constexpr int kLast = Parts == 3 ? kFull : 0, kAll = kA + kLast;
    static constexpr bool kHidLds = Parts == 3 && kFull > 0 && Q::kNL > 1 && Q::kHt > 3;
    static constexpr bool kOutLds = Parts == 3 && kOutVar > 1 && Q::kHt > 2;
    static constexpr bool kW1Lds = Parts == 3 && kS1 > 1 && Q::kHt > 3;
    static constexpr int kAH = kHidLds ? kA : kAll, kAO = kOutLds ? 0 : kAll;           // the others, in registers
    static constexpr int kOut0 = kHidLds ? Q::kHt * kLast : 0, kW1 = kOut0 + (kOutLds ? kAll : 0);   // (where they begin)
    static constexpr int kLdsOps = kW1 + (kW1Lds ? Q::kHt : 0);
};

// The value that slot j of weight operand a holds the weight of (-1: none), and the part of it. An operand of kRem <= 2 values
// holds them as (w_hi, w_hi, w_lo, w_last) against (x_hi, x_lo, x_hi, x_hi); two parts: w_lo against (x_hi, x_lo). kRem of 3 or 4
// takes two weight operands, (w_hi, w_hi) against (x_hi, x_lo), then (w_lo, w_last) against (x_hi, x_hi); two parts: (w_lo, w_lo)
// against (x_hi, x_lo).
// (Full operands hold hi parts, then lo parts; their last parts are operands kA, kA + 1, ..)
template <class S, int Parts>
constexpr int split_value(int a, int j) {
    using P = SplitShape<S, Parts>;
    const int f = a >= P::kA ? a - P::kA : (a < 2 * P::kFull ? a / 2 : -1);
    if (f >= 0) return 8 * f + j < P::kV ? 8 * f + j : -1;
    const int w = P::kRem <= 2 ? j & 1 : j & 3;
    return w < P::kRem ? 8 * P::kFull + w : -1;
}
template <class S, int Parts>
constexpr int split_part(int a, int j) {
    using P = SplitShape<S, Parts>;
    if (a >= P::kA) return 2;
    if (a < 2 * P::kFull) return a % 2;
    const int quarter = P::kRem <= 2 ? j / 2 : 2 * (a - 2 * P::kFull) + j / 4;
    return quarter < 2 ? 0 : quarter - (Parts == 2 && quarter == 3 ? 2 : 1);
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

// A weight (or bias) w0 + s eps times its factor as SplitLds holds it, and a weight's last part. The sum and the product are
// formed in 64 bits and each part rounded once.
__device__ __forceinline__ unsigned split_param(float w0, float s, float eps, double factor, bool bias, unsigned short& last) {
    const double v = __builtin_fma((double)s, (double)eps, (double)w0) * factor;
    const float f = (float)v;
    const _Float16 h = (_Float16)f;
    const double r = v - (double)(float)h;
    const _Float16 l = (_Float16)(float)r;
    last = __builtin_bit_cast(unsigned short, (_Float16)(float)(r - (double)(float)l));
    return bias ? __float_as_uint(f) : (unsigned)__builtin_bit_cast(unsigned short, h) | ((unsigned)__builtin_bit_cast(unsigned short, l) << 16);
}

// One member's parameters in operand layout.
template <class S, int Parts>
struct SplitWeights {
    using Q = MfmaShape<S>;
    using P = SplitShape<S, Parts>;
    h8v a1[Q::kHt][P::kW1Lds ? 1 : P::kS1];
    f4v c1[Q::kHt];
    h8v ah[Q::kNL > 1 ? Q::kHt : 1][P::kAH];
    f4v ch[Q::kNL > 1 ? Q::kHt : 1];
    // more than 4 outputs: the output tile's rows as out_at. At most 4: variant t holds output c in row 4 t + c, so four
    // tiles' outputs meet in one accumulator, tile t's in lane group t: each lane ends with the outputs of its own pixel.
    h8v ao[P::kOutLds ? 1 : P::kOutVar][P::kOutLds ? 1 : P::kAO];   // (kOutLds: not held)
    f4v co;
    // the operands in LDS, and this lane's places: the hidden layer's last parts, the output layer's (variant t)
    const h8v* ops;
    int last, out[P::kOutVar];
    // Called in the loop over tiles: the places as new values, so that the loads from them stay in the loop (they do not change,
    // and out of the loop they would take the registers that they are in LDS to save).
    __device__ __forceinline__ void reload() {
        if constexpr (P::kHidLds || P::kW1Lds) asm volatile("" : "+v"(last));
        if constexpr (P::kOutLds)
#pragma unroll
            for (int t = 0; t < P::kOutVar; t++) asm volatile("" : "+v"(out[t]));
    }
};

// Gathers a member's parameters from LDS (SplitLds; last: the weights' last parts at the same places, three parts only) into
// operand layout, kept: those that split_keep puts back into LDS. Weights that a lane has no unit or input for are zero.
template <class S, int Parts>
__device__ __forceinline__ void split_load(SplitWeights<S, Parts>& W, const unsigned* __restrict__ lds, const unsigned short* __restrict__ last, int lane,
                                           h8v (&kept)[SplitShape<S, Parts>::kLdsOps + 1]) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S, Parts>;
    using L = SplitLds<S>;
    constexpr int NIN = Q::kIn, H = Q::kH, NO = Q::kNout;
    constexpr unsigned kHi = 0x05040100u, kLo = 0x07060302u;   // the low, the high halves of two words
    const int i16 = lane & 15, g = lane >> 4;
    auto at = [&](bool ok, int k) { const unsigned v = lds[k]; return ok ? v : 0u; };
    auto last_at = [&](bool ok, int k) {
        if constexpr (Parts == 2) return 0u;
        else { const unsigned v = last[k]; return ok ? v : 0u; }
    };
    auto bias = [&](bool ok, int k) { return __uint_as_float(at(ok, k)); };
    // slots 2 j and 2 j + 1 of an operand from two parameters
    auto put = [&](h8v& a, int j, unsigned x, unsigned y, unsigned half) {
        u4v v = __builtin_bit_cast(u4v, a);
        v[j] = __builtin_amdgcn_perm(y, x, half);
        a = __builtin_bit_cast(h8v, v);
    };
#pragma unroll
    for (int ot = 0; ot < Q::kHt; ot++) {
        const int u = unit_of<Q>(ot, i16), row = min(u, H - 1) * L::kRow1;
        constexpr int kIn = P::kS1 == 1 ? 8 : 4;   // inputs a lane holds weights of: all 8, or 4 g .. 4 g + 3
        unsigned w[kIn], t[kIn];
#pragma unroll
        for (int j = 0; j < kIn; j++) {
            const int in = P::kS1 == 1 ? j : 4 * g + j;
            w[j] = at(u < H && in < NIN, row + min(in, NIN - 1));
            t[j] = last_at(u < H && in < NIN, row + min(in, NIN - 1));
        }
        // weights that meet features' lo parts are divided by kSplitLo: exact down to a scaled weight of 2^-3, then within 2^-25
        const _Float16 lo = (_Float16)(1.0f / kSplitLo), one = (_Float16)1.0f;
        if constexpr (P::kS1 == 1) {   // lane groups 0 .. 3: (w_hi, w_hi, w_lo, w_last) against (f_hi, f_lo, f_hi, f_hi); two parts:
                                       // w_lo against f_lo in the last
            const bool l3 = Parts == 3 && g == 3;
#pragma unroll
            for (int j = 0; j < 4; j++) put(W.a1[ot][0], j, l3 ? t[2 * j] : w[2 * j], l3 ? t[2 * j + 1] : w[2 * j + 1], g >= 2 && !l3 ? kLo : kHi);
            W.a1[ot][0] *= g == 1 || (g == 3 && Parts == 2) ? lo : one;
        } else {                       // (w_hi, w_hi) against (f_hi, f_lo), then (w_lo, w_last) against (f_hi, f_hi); two parts: (w_lo,
                                       // w_lo) against (f_hi, f_lo)
            const h8v low = { one, one, one, one, lo, lo, lo, lo };
            h8v& second = P::kW1Lds ? kept[P::kW1Lds ? P::kW1 + ot : 0] : W.a1[ot][P::kW1Lds ? 0 : 1];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int q = 2 * (j & 1);
                put(W.a1[ot][0], j, w[q], w[q + 1], kHi);
                put(second, j, Parts == 3 && j >= 2 ? t[q] : w[q], Parts == 3 && j >= 2 ? t[q + 1] : w[q + 1], Parts == 3 && j >= 2 ? kHi : kLo);
            }
            W.a1[ot][0] *= low;
            if constexpr (Parts == 2) second *= low;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ur = unit_of<Q>(ot, 4 * g + r);
            W.c1[ot][r] = bias(ur < H, L::kB1 + min(ur, H - 1));
        }
    }
    // the weights of the row at `row` (valid if ok) for the values this lane group holds, into the operands of one tile
    // (operand q to to(q))
    auto gather = [&](auto to, bool ok, int row) {
        unsigned w[P::kV + 1], t[P::kV + 1];
        w[P::kV] = t[P::kV] = 0u;
#pragma unroll
        for (int v = 0; v < P::kV; v++) {
            const int in = hidden_input<Q>(v, g);
            w[v] = at(ok && in < H, row + min(in, H - 1));
            t[v] = last_at(ok && in < H, row + min(in, H - 1));
        }
#pragma unroll
        for (int q = 0; q < P::kAll; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int vx = split_value<S, Parts>(q, 2 * j), vy = split_value<S, Parts>(q, 2 * j + 1), part = split_part<S, Parts>(q, 2 * j);
                const int x = vx < 0 ? P::kV : vx, y = vy < 0 ? P::kV : vy;
                put(to(q), j, part == 2 ? t[x] : w[x], part == 2 ? t[y] : w[y], part == 1 ? kLo : kHi);
            }
    };
    if constexpr (Q::kNL > 1) {
#pragma unroll
        for (int ot = 0; ot < Q::kHt; ot++) {
            const int u = unit_of<Q>(ot, i16);
            gather([&](int q) -> h8v& { return q < P::kAH ? W.ah[ot][q < P::kAH ? q : 0] : kept[q < P::kAH ? 0 : ot * P::kLast + q - P::kA]; }, u < H,
                   L::kW2 + min(u, H - 1) * L::kRowH);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int ur = unit_of<Q>(ot, 4 * g + r);
                W.ch[ot][r] = bias(ur < H, L::kB2 + min(ur, H - 1));
            }
        }
    }
    auto out = [&](int t, int q) -> h8v& { return P::kOutLds ? kept[P::kOutLds ? P::kOut0 + q : 0] : W.ao[t][P::kOutLds ? 0 : q]; };
    if constexpr (valu_out<S>()) {
#pragma unroll
        for (int t = 0; t < (P::kOutLds ? 1 : 4); t++) {
            const int c = i16 - 4 * t;
            gather([&](int q) -> h8v& { return out(t, q); }, c >= 0 && c < NO, L::kW3 + min(max(c, 0), NO - 1) * L::kRowH);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) W.co[r] = bias(r < NO, L::kB3 + min(r, NO - 1));
    } else {
        const int orow = out_at<S>(i16 >> 2, i16 & 3);
        gather([&](int q) -> h8v& { return out(0, q); }, orow >= 0, L::kW3 + max(orow, 0) * L::kRowH);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int oc = out_at<S>(g, r);
            W.co[r] = bias(oc >= 0, L::kB3 + max(oc, 0));
        }
    }
}

// Puts the kept operands into the member's place in LDS (kLdsOps x 64; one of its waves writes) and finds this lane's. Variant
// t of the output layer's is variant 0 of the lane 4 t below, and where that has no output a lane of zeros (row 15).
template <class S, int Parts>
__device__ __forceinline__ void split_keep(SplitWeights<S, Parts>& W, const h8v (&kept)[SplitShape<S, Parts>::kLdsOps + 1], h8v* __restrict__ ops, bool write,
                                           int lane) {
    using P = SplitShape<S, Parts>;
    if (write)
#pragma unroll
        for (int q = 0; q < P::kLdsOps; q++) ops[64 * q + lane] = kept[q];
    W.ops = ops;
    W.last = lane;
    const int i16 = lane & 15;
#pragma unroll
    for (int t = 0; t < P::kOutVar; t++) {
        const int c = i16 - 4 * t, from = P::kOutVar == 1 || (c >= 0 && c < MfmaShape<S>::kNout) ? lane - 4 * t : lane | 15;
        W.out[t] = 64 * P::kOut0 + from;
    }
}

// a hidden layer's results of one tile through the activation, as the next layer's operands
template <class S, int Parts, int Act>
__device__ __forceinline__ void split_act(const f4v (&acc)[MfmaShape<S>::kHt], float k, float neg, h8v (&b)[SplitShape<S, Parts>::kB]) {
    using P = SplitShape<S, Parts>;
    constexpr int V2 = P::kFull * 8 + (P::kRem ? (P::kRem <= 2 ? 2 : 4) : 0);
    h2v hi[V2 / 2], lo[V2 / 2];
#pragma unroll
    for (int q = 0; q < V2 / 2; q++) {
        const float x = 2 * q < P::kV ? act<Act>(acc[2 * q < P::kV ? q / 2 : 0][(2 * q) & 3], k) : 0.0f;
        const float y = 2 * q + 1 < P::kV ? act<Act>(acc[2 * q + 1 < P::kV ? q / 2 : 0][(2 * q + 1) & 3], k) : 0.0f;
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
    constexpr int R = 4 * P::kFull, F = 2 * P::kFull;
    if constexpr (P::kRem > 2) {
        b[F] = join(hi[R], hi[R + 1], lo[R], lo[R + 1]);
        if constexpr (Parts == 3) b[F + 1] = join(hi[R], hi[R + 1], hi[R], hi[R + 1]);
    } else if constexpr (P::kRem > 0) {
        b[F] = join(hi[R], lo[R], hi[R], Parts == 3 ? hi[R] : lo[R]);
    }
}

// c plus one tile row block's products with the values b, the small terms first: they are added to the bias, and only the last
// steps round at the size of the whole sum. a(q): its weight operand q (of kA, then the full operands' last parts)
template <class S, int Parts, class A>
__device__ __forceinline__ f4v split_dot(A a, const h8v (&b)[SplitShape<S, Parts>::kB], f4v c) {
    using P = SplitShape<S, Parts>;
    constexpr int F = 2 * P::kFull;
#pragma unroll
    for (int f = 0; f < P::kFull; f++) {
        if constexpr (Parts == 2) c = mfma_h(a(2 * f + 1), b[2 * f + 1], c);
        c = mfma_h(a(2 * f), b[2 * f + 1], c);
        c = mfma_h(a(2 * f + 1), b[2 * f], c);
        if constexpr (Parts == 3) c = mfma_h(a(P::kA + f), b[2 * f], c);
    }
    if constexpr (P::kRem > 2) c = mfma_h(a(F + 1), b[F + (Parts == 3 ? 1 : 0)], c);
    if constexpr (P::kRem > 0) c = mfma_h(a(F), b[F], c);
#pragma unroll
    for (int f = 0; f < P::kFull; f++) c = mfma_h(a(2 * f), b[2 * f], c);
    return c;
}
// of hidden tile ot, and of the output layer (variant t)
template <class S, int Parts>
__device__ __forceinline__ f4v split_dot_hidden(const SplitWeights<S, Parts>& W, int ot, const h8v (&b)[SplitShape<S, Parts>::kB]) {
    using P = SplitShape<S, Parts>;
    return split_dot<S, Parts>([&](int q) { return q < P::kAH ? W.ah[ot][q < P::kAH ? q : 0] : W.ops[W.last + 64 * (ot * P::kLast + q - P::kA)]; }, b, W.ch[ot]);
}
template <class S, int Parts>
__device__ __forceinline__ f4v split_dot_out(const SplitWeights<S, Parts>& W, int t, const h8v (&b)[SplitShape<S, Parts>::kB], f4v c) {
    using P = SplitShape<S, Parts>;
    return split_dot<S, Parts>([&](int q) { return P::kOutLds ? W.ops[W.out[t] + 64 * q] : W.ao[P::kOutLds ? 0 : t][P::kOutLds ? 0 : q]; }, b, c);
}

// The hidden layers of N tiles from their first-layer operands (the split features of a slot each), the last one's values as
// operands: a layer of every tile at a time, so that their matrix and VALU instructions are independent.
template <class S, int Parts, int Act, int N>
__device__ __forceinline__ void split_hidden_n(const SplitWeights<S, Parts>& W, const h8v (&f)[N], float k, float neg, h8v (&b)[N][SplitShape<S, Parts>::kB]) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S, Parts>;
    f4v acc[N][Q::kHt];
#pragma unroll
    for (int s = P::kS1 - 1; s >= 0; s--)
#pragma unroll
        for (int n = 0; n < N; n++) {
            const h8v x = s == 1 && Parts == 3 ? __builtin_shufflevector(f[n], f[n], 0, 1, 2, 3, 0, 1, 2, 3) : f[n];
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++)
                acc[n][ot] = mfma_h(s == 1 && P::kW1Lds ? W.ops[W.last + 64 * (P::kW1 + ot)] : W.a1[ot][P::kW1Lds ? 0 : s], x,
                                    s == P::kS1 - 1 ? W.c1[ot] : acc[n][ot]);
        }
#pragma unroll
    for (int n = 0; n < N; n++) split_act<S, Parts, Act>(acc[n], k, neg, b[n]);
    if constexpr (Q::kNL > 1) {
        f4v a2[N][Q::kHt];
#pragma unroll
        for (int n = 0; n < N; n++)
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++) a2[n][ot] = split_dot_hidden<S, Parts>(W, ot, b[n]);
#pragma unroll
        for (int n = 0; n < N; n++) split_act<S, Parts, Act>(a2[n], k, neg, b[n]);
    }
}

// split_hidden_n of one tile
template <class S, int Parts, int Act>
__device__ __forceinline__ void split_hidden(const SplitWeights<S, Parts>& W, h8v f, float k, float neg, h8v (&b)[SplitShape<S, Parts>::kB]) {
    h8v fs[1] = { f }, bs[1][SplitShape<S, Parts>::kB];
    split_hidden_n<S, Parts, Act, 1>(W, fs, k, neg, bs);
#pragma unroll
    for (int q = 0; q < SplitShape<S, Parts>::kB; q++) b[q] = bs[0][q];
}

}   // namespace ntc_hip
