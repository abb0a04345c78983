// Device code only (compiled into libntc_hip.so for the fixed shapes of shapes.hpp, and by hipRTC at
// init for the shape of a model that is none of them, jit.cpp); the launchers are in kernels_pop.hip.
//
// The population evaluation (MlpTrainer::step's member losses, main.cpp:1848-1861) on the
// matrix cores of gfx950, for the fixed shapes the matrix cores pay off for (MfmaShape::kOk) and
// 0 <= leak <= 1; other models use the VALU kernel of kernels_mlp.hip. In an ES step the kernel
// stages the pair's perturbed weights itself (no member weight sets in memory). The shapes split_pays takes run on k_pop_split
// (16-bit instructions, operands in parts), ES steps and central differences; the other shapes on k_pop_mfma (32-bit
// instructions), which the following is about.
//
// On this chip an FP32 matrix instruction and a VALU instruction do not run concurrently on a
// SIMD (a 16x16x4 f32 step costs 32 cycles, a VALU instruction 4, and their mixes take the sum),
// so everything around the matrix operations is counted in instructions: the activation is one
// instruction (kActFold's fused multiply-add on hidden layers whose weights were scaled by
// (1 + leak) / 2 when the member's weights were staged, which propagates a NaN as the reference's
// activation does); a hidden layer's outputs feed the next layer in the order
// the matrix instruction leaves them (no transpose; each unit's sum takes its inputs in another
// order than the reference's ascending one); the sigmoid is the hardware exp2 and reciprocal, its
// -log2(e) folded into the output layer; a lane's channel terms cw d d are fused multiply-adds in float
// over the tiles a wave evaluates at once, then added into a double; tile
// inputs are buffer loads with a loop-invariant lane offset and the tile's offset in an SGPR. Member
// losses stay within 1e-5 relative of the reference's (they are not bit-identical here anyway:
// the sigmoid differs in the last bits).
//
// Block (pair, chunk) has four waves: wave w evaluates member 2 pair + (w & 1) on the 16-slot
// tiles 2 j + (w >> 1) of the chunk, two tiles at a time, the next two tiles' inputs loading
// while the current ones compute. Each lane adds the float terms cw (d d) (main.cpp:1747) of its
// output channels into a double; the two waves of a member are added in a fixed order.
#pragma once
#include "split_mlp.hpp"

namespace ntc_hip {

constexpr int kPopWaves = 4;
// Models with at most 4 outputs and one 16-unit hidden tile take the pixel-per-lane output layer
// (mfma_out_own): four tiles per pass, exchanged through the wave's LDS so that every lane holds all hidden
// units of one pixel, then v_mfma_f32_4x4x1_16b_f32 steps leave that pixel's outputs in its own registers.
template <class S>
constexpr bool pop_own() { return valu_out<S>() && MfmaShape<S>::kHt == 1; }
// 16-slot tiles a wave evaluates at once (independent chains of matrix instructions; two for the other
// shapes: the 64-wide models then hold 236 VGPRs at two waves per SIMD)
template <class S>
constexpr int pop_u() { return pop_own<S>() ? 4 : 2; }

// The minibatch arrays are read through raw buffers (buffer_of): loads take a loop-invariant 32-bit lane
// offset (VGPR) and the tile's byte offset (SGPR), so no address arithmetic per load. num_records = the
// allocation (every read stays inside it: minibatch_rows(nin) feature rows, those past nin zero, and
// kMinibatchSlack floats past the last row of each array).

// The targets a lane needs per tile: the pixel-per-lane output layer leaves every output of the lane's
// own pixel in the lane (its nout targets, once per pass); models with at most 4 outputs otherwise take
// their output layer on the VALU (valu_out_g), which leaves output g of pixel j in lane (g, j): one
// target per tile; otherwise the D layout's out_regs per tile (outputs out_at(g, r)).
template <class S>
constexpr int pop_nt() { return pop_own<S>() ? MfmaShape<S>::kNout : (valu_out<S>() ? 1 : out_regs<S>()); }
template <class S>
constexpr int pop_tt() { return pop_own<S>() ? 1 : pop_u<S>(); }

// Whether the loop runs two whole passes as one straight-line block (so that one pass's output stage can
// overlap the next pass's hidden layers), masking only the passes at the chunk's end: measured on the
// MI355X, 3.5% faster for the 3-output 32-wide shapes (dct512: 0.425 -> 0.410 ms), 0.5-2% slower for the
// 12-output and the pixel-per-lane shapes (one more occupancy step of registers, or nothing to overlap).
template <class S>
constexpr bool pop_pairs_whole() { return valu_out<S>() && !pop_own<S>(); }

// a compile-time flag handed to a generic lambda
template <bool B>
struct WholeTag { static constexpr bool value = B; };

template <class S>
struct PopTileIn {
    float b1[pop_u<S>()][MfmaShape<S>::kKs1];
    float t[pop_tt<S>()][pop_nt<S>()];
};

// Inputs of tiles j .. j + U - 1 of this wave: soff = byte offset of tile j's first slot (uniform);
// tile u sits 32 slots further per u. With the pixel-per-lane output layer, lane (g, i) loads the
// targets of pixel i of tile g (its lane offsets include the 32 g slots).
template <class S>
__device__ __forceinline__ void pop_load(PopTileIn<S>& in, __amdgpu_buffer_rsrc_t rf, __amdgpu_buffer_rsrc_t rt, uint32_t soff,
                                         const uint32_t (&fo)[MfmaShape<S>::kKs1], const uint32_t (&to)[pop_nt<S>()]) {
    using Q = MfmaShape<S>;
#pragma unroll
    for (int u = 0; u < pop_u<S>(); u++) {
        const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane((int)(soff + 128u * u));   // uniform: an SGPR
#pragma unroll
        for (int ks = 0; ks < Q::kKs1; ks++) in.b1[u][ks] = buffer_f32(rf, fo[ks], so);
        if constexpr (!pop_own<S>()) {
#pragma unroll
            for (int r = 0; r < pop_nt<S>(); r++) in.t[u][r] = buffer_f32(rt, to[r], so);
        }
    }
    if constexpr (pop_own<S>()) {
        const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
#pragma unroll
        for (int c = 0; c < pop_nt<S>(); c++) in.t[0][c] = buffer_f32(rt, to[c], so);
    }
}

// 1 / (1 + e^-s) from the hardware exp2 and reciprocal (each within about 1 ulp), given
// s2 = -log2(e) s: the kernels scale the output layer by kNegLog2e (scale_output), so the matrix
// instruction delivers s2 directly
constexpr float kNegLog2e = -1.44269504088896341f;
constexpr double kNegLog2eD = -1.44269504088896340736;
__device__ __forceinline__ float sigmoid_hw2(float s2) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(s2)); }

// the output of a pre-activation: clamp(s + 0.5) with --clamp, else the sigmoid of a pre-activation
// delivered as -log2(e) s (the output layer is scaled when !clamp)
template <class S>
__device__ __forceinline__ float out_of(float s, bool clamp) {
    return clamp ? __builtin_amdgcn_fmed3f(s + 0.5f, 0.0f, 1.0f) : sigmoid_hw2(s);
}

// Where a member's parameters come from: the weight sets of a central-difference step (kSets), or -
// in an ES step - both members' weights w0 +- sigma eps (one fused operation each, main.cpp:1852-1856)
// staged in LDS, from the block's own draw of the pair's Gaussians (NS_MLP, step, pair, k; the chunk-0
// block writes them to eps for the update: kDraw, for populations with one or two chunks per pair) or
// from the Gaussians a separate kernel drew once for all chunks (kReadEps).
enum PopFrom : int { kSets = 0, kDraw = 1, kReadEps = 2 };
struct PopSource {
    const float* wsets;                    // central differences: 2 pairs x P
    NoiseFix nt; uint64_t seed; uint32_t step; float sigma;
    const float* w0; float* eps;           // ES: the current weights and the step's Gaussians [pair][P]
};

// waves per SIMD the register allocation aims at (more would spill)
template <class S>
constexpr int pop_occupancy() { return MfmaShape<S>::kH > 32 ? 2 : (MfmaShape<S>::kIn <= 8 ? 4 : 3); }

template <class S, int Act, bool Clamp, int From>
__global__ void __launch_bounds__(64 * kPopWaves) __attribute__((amdgpu_waves_per_eu(pop_occupancy<S>()))) k_pop_mfma(DevModel m, PopSource src, int M, int Mcap,
                                                           int chunk, int chunks, const float* __restrict__ feat,
                                                           const float* __restrict__ btgt, double* __restrict__ part) {
    using Q = MfmaShape<S>;
    constexpr bool Es = From != kSets;
    __shared__ double red[kPopWaves];
    __shared__ float wpm_s[Es ? 2 * Q::kP : 1];   // ES: the + member's weights, then the - member's
    // the pixel-per-lane output layer's transposes: kOwnWave floats per wave
    __shared__ __attribute__((aligned(16))) float own_s[pop_own<S>() ? kPopWaves * kOwnWave : 4];
    // the VALU output layer's reduce-scatters: kVoTile floats per tile of a pass, per wave
    constexpr int kVoWave = kVoTile * pop_u<S>();
    __shared__ __attribute__((aligned(16))) float vo_s[valu_out<S>() && !pop_own<S>() ? kPopWaves * kVoWave : 4];
    const int lane = tid_x() & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6);
    const int pair = bid_x(), ch = bid_y(), sgn = wave & 1, half = wave >> 1;
    const int i16 = lane & 15, g = lane >> 4;
    constexpr int NT = pop_nt<S>();
    constexpr bool kOwn = pop_own<S>();
    constexpr bool kVOut = valu_out<S>();
    // lane byte offsets of the feature rows 4 ks + g (rows past nin are the array's zero rows) and target
    // rows out_at(g, r), or g (padding and rows past the last one read a valid row: their channel weights cw
    // are zero); the pixel-per-lane layer: target row r of pixel i16 of tile g
    uint32_t fo[Q::kKs1], to[NT];
#pragma unroll
    for (int ks = 0; ks < Q::kKs1; ks++) fo[ks] = 4u * ((uint32_t)(4 * ks + g) * (uint32_t)Mcap + (uint32_t)i16);
#pragma unroll
    for (int r = 0; r < NT; r++)
        to[r] = kOwn ? 4u * ((uint32_t)r * (uint32_t)Mcap + 32u * (uint32_t)g + (uint32_t)i16)
                     : 4u * ((uint32_t)(kVOut ? min(g, Q::kNout - 1) : max(out_at<S>(g, r), 0)) * (uint32_t)Mcap + (uint32_t)i16);
    const int s0 = ch * chunk, s1 = min(M, s0 + chunk);
    const int tiles = (s1 - s0 + 15) >> 4;
    const int mine = (tiles - half + 1) >> 1;   // this wave's tiles: 2 j + half, j < mine
    static_assert(minibatch_rows(Q::kIn) == 4 * Q::kKs1, "the feature rows the first layer's k-steps read");
    const __amdgpu_buffer_rsrc_t rf = buffer_of(feat, 4u * ((uint32_t)minibatch_rows(Q::kIn) * (uint32_t)Mcap + (uint32_t)kMinibatchSlack));
    const __amdgpu_buffer_rsrc_t rt = buffer_of(btgt, 4u * ((uint32_t)Q::kNout * (uint32_t)Mcap + (uint32_t)kMinibatchSlack));
    constexpr int U = pop_u<S>();
    // the first tiles' inputs load while the member's weights are staged
    PopTileIn<S> in0, in1;
    pop_load<S>(in0, rf, rt, 4u * (uint32_t)(s0 + 16 * half), fo, to);
    MfmaWeights<S> W;
    if constexpr (Es) {
        const uint64_t head = noise_head(src.seed, NS_MLP, src.step, (uint32_t)pair);
        float* eg = src.eps + (size_t)pair * Q::kP;
        for (int k = tid_x(); k < Q::kP; k += 64 * kPopWaves) {
            float e;
            if constexpr (From == kDraw) {
                e = gauss_at(src.nt, head, (uint64_t)k);
                if (ch == 0) eg[k] = e;
            } else {
                e = eg[k];
            }
            const float w0 = src.w0[k];
            wpm_s[k] = __builtin_fmaf(src.sigma, e, w0);
            wpm_s[Q::kP + k] = __builtin_fmaf(-src.sigma, e, w0);
        }
        __syncthreads();
        mfma_load<S>(W, wpm_s + sgn * Q::kP, lane);
    } else {
        mfma_load<S>(W, src.wsets + (size_t)(2 * pair + sgn) * Q::kP, lane);
    }
    if constexpr (!Clamp) scale_output<S>(W, kNegLog2e);
    if constexpr (Act == kActFold) scale_hidden<S>(W, fold_scale(m.leak));
    const float ak = act_k_of<Act>(m);
    // the channel weight of each of this lane's outputs (pixel-per-lane layer: output r; D layout: rows
    // 4 g + r; VALU output layer: output g), zero past the last output
    float cw[NT];
#pragma unroll
    for (int r = 0; r < NT; r++) {
        cw[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < Q::kNout; c++)
            if ((kOwn ? r : (kVOut ? g : out_at<S>(g, r))) == c) cw[r] = m.cw[c];
    }
    double e = 0.0;
    // One pass: tiles j .. j + U - 1 from c, while tiles j + U .. load into n. The loop alternates
    // two input sets, so no registers are copied between passes. The loads are issued on every pass
    // (the last one reloads its own tiles) so that the wait for them falls in the next pass.
    // whole: every tile of the pass lies inside the chunk (known at compile time: no per-lane checks)
    auto pass = [&](PopTileIn<S>& c, PopTileIn<S>& n, int j, auto whole) {
        constexpr bool kWhole = decltype(whole)::value;
        j = __builtin_amdgcn_readfirstlane(j);   // uniform: the tile arithmetic stays in SGPRs
        pop_load<S>(n, rf, rt, 4u * (uint32_t)(s0 + 16 * (2 * (j + U < mine ? j + U : j) + half)), fo, to);
        if constexpr (kOwn) {
            // the lane's own pixel (pixel i16 of tile j + g): its channel terms cw (d d), one multiply and one
            // fused multiply-add each, summed in float, then into the double
            float x[U][Q::kKsH];
            mfma_hidden<S, U, Act>(W, c.b1, ak, x);
            const f4v o = mfma_out_own<S>(W, x, own_s + wave * kOwnWave, g, i16);
            float tsum = 0.0f;
#pragma unroll
            for (int r = 0; r < NT; r++) {
                const float d = out_of<S>(o[r], Clamp) - c.t[0][r];
                tsum = __builtin_fmaf(__fmul_rn(cw[r], d), d, tsum);
            }
            if (kWhole || (j + g < mine && s0 + 16 * (2 * (j + g) + half) + i16 < s1)) e += (double)tsum;
        } else {
            // this lane's outputs' channel terms cw (d d): one multiply and one fused multiply-add each,
            // summed in float over the pass's tiles, then into the double
            float dq[pop_tt<S>()][NT], dd[pop_tt<S>()][NT];
            if constexpr (kVOut) {
                float x[U][Q::kKsH];
                mfma_hidden<S, U, Act>(W, c.b1, ak, x);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    dd[u][0] = out_of<S>(valu_out_g<S>(W, x[u], vo_s + wave * kVoWave + u * kVoTile, g, i16), Clamp) - c.t[u][0];
                    dq[u][0] = __fmul_rn(cw[0], dd[u][0]);
                }
            } else {
                f4v o[U];
                mfma_forward<S, U, Act>(W, c.b1, ak, o);
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int r = 0; r < NT; r++) {
                        dd[u][r] = out_of<S>(o[u][r], Clamp) - c.t[u][r];
                        dq[u][r] = __fmul_rn(cw[r], dd[u][r]);
                    }
            }
            {
                if (kWhole || (j + U <= mine && s0 + 16 * (2 * (j + U - 1) + half) + 16 <= s1)) {   // all U tiles whole (uniform)
                    float tsum = 0.0f;
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int r = 0; r < NT; r++) tsum = __builtin_fmaf(dq[u][r], dd[u][r], tsum);
                    e += (double)tsum;
                } else {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int st = s0 + 16 * (2 * (j + u) + half);   // first slot of the tile (uniform)
                        float tsum = 0.0f;
#pragma unroll
                        for (int r = 0; r < NT; r++) tsum = __builtin_fmaf(dq[u][r], dd[u][r], tsum);
                        if (j + u < mine && st + i16 < s1) e += (double)tsum;
                    }
                }
            }
        }
    };
    // this wave's tiles that lie wholly inside the chunk (tile t: slots s0 + 16 (2 t + half) + 0 .. 15)
    const int nwhole = min(mine, max(0, (s1 - s0 - 16 * half + 16) >> 5));
    int j = 0;
    for (; pop_pairs_whole<S>() && j + 2 * U <= nwhole; j += 2 * U) {   // two whole passes: one straight-line block
        pass(in0, in1, j, WholeTag<true>{});
        pass(in1, in0, j + U, WholeTag<true>{});
    }
    for (; j < mine; j += 2 * U) {
        pass(in0, in1, j, WholeTag<false>{});
        if (j + U >= mine) break;
        pass(in1, in0, j + U, WholeTag<false>{});
    }
    e = wave_sum(e);
    if (lane == 0) red[wave] = e;
    __syncthreads();
    if (tid_x() == 0) {
        part[(size_t)(2 * pair) * chunks + ch] = red[0] + red[2];
        part[(size_t)(2 * pair + 1) * chunks + ch] = red[1] + red[3];
    }
}

// Waves per SIMD that the split kernels' register allocation aims at. k_lat_split and k_qat_split: split_waves, at which several
// shapes keep values in scratch. k_pop_split holds three parts of the weights: at three waves its loop over tiles reloads up to
// 28 values a pass from scratch for the 36-wide models of more than 8 inputs and the 48-wide ones, at two none (512 pairs on 4096
// slots, MI355X: 10-36-36-12 299 -> 118 us, 14-48-48-12 771 -> 147 us).
constexpr int split_waves(int nin, int H, int nout) { return H > 48 ? 2 : ((nin <= 8 && H <= 32 && (nout > 4 || H <= 16)) ? 4 : 3); }
constexpr int pop_split_waves(int nin, int H, int nout) { return H > 40 || (H > 32 && nin > 8) ? 2 : split_waves(nin, H, nout); }
template <class S>
constexpr int split_occupancy() { return split_waves(MfmaShape<S>::kIn, MfmaShape<S>::kH, MfmaShape<S>::kNout); }
template <class S>
constexpr int pop_split_occupancy() { return pop_split_waves(MfmaShape<S>::kIn, MfmaShape<S>::kH, MfmaShape<S>::kNout); }
// the minibatch slot by slot (device_common.hpp, split_inputs) and the step's layer scales (split_mlp.hpp)
struct SplitIn {
    const u4v* feat;
    const float* tgt;
    const float* scales;
};

// Stages both members of an ES pair in LDS (SplitLds): w0 + sigma eps, then w0 - sigma eps (main.cpp:1852-1856), in three
// parts with their factors. The Gaussians are drawn here (kDraw: the chunk-0 block writes them for the update) or read
// (kReadEps). Central differences (kSets): pair j < P is w0 with weight j at w + h and w - h (h = sigma; the 32-bit sums,
// main.cpp:1905), pair P two copies of w0.
template <class S, int From>
__device__ __forceinline__ void split_stage(const PopSource& src, const SplitFactors f, int pair, int ch, unsigned* __restrict__ lds,
                                            unsigned short* __restrict__ last) {
    using L = SplitLds<S>;
    constexpr int kP = MfmaShape<S>::kP;
    const uint64_t head = noise_head(src.seed, NS_MLP, src.step, (uint32_t)pair);
    float* eg = src.eps + (size_t)pair * kP;
    for (int k = tid_x(); k < kP; k += 64 * kPopWaves) {
        const float w0 = src.w0[k];
        float wp = w0, wm = w0, s = src.sigma, e = 0.0f;
        if constexpr (From == kSets) {
            if (k == pair) { wp = w0 + s; wm = w0 - s; }
            s = 0.0f;
        } else if constexpr (From == kDraw) {
            e = gauss_at(src.nt, head, (uint64_t)k);
            if (ch == 0) eg[k] = e;
        } else {
            e = eg[k];
        }
        const int l = L::layer(k), at = L::pos(k);
        const bool b = L::bias(k);
        const double fw = l == 0 ? f.w1 : (l == 1 ? f.w2 : f.w3), fb = l == 0 ? f.b1 : (l == 1 ? f.b2 : f.b3), ff = b ? fb : fw;
        lds[at] = split_param(wp, s, e, ff, b, last[at]);
        lds[L::kWords + at] = split_param(wm, -s, e, ff, b, last[L::kWords + at]);
    }
}

// Parameter k of a member in 32 bits: w0 + s eps, one fused operation (main.cpp:1852-1856); central differences: w0 with weight
// `hit` at w + s (main.cpp:1905).
template <int From>
struct MemberAt {
    const float *w0, *eps;
    float s;
    int hit;
    __device__ __forceinline__ float operator()(int k) const {
        if constexpr (From == kSets) return k == hit ? w0[k] + s : w0[k];
        else return __builtin_fmaf(s, eps[k], w0[k]);
    }
};

// ---- The population on the 16-bit matrix instructions with 32-bit operands in parts (split_mlp.hpp: weights in three, values in
// two), for the shapes of at most 16 inputs and two hidden layers: ES steps, and central differences (kSets), whose members it
// forms from the weights themselves (no weight sets in memory).
//
// Block (pair, chunk) has four waves: wave w evaluates member 2 pair + (w & 1) on the passes 2 q + (w >> 1) of the chunk's
// slots, 32 slots a pass (two 16-slot tiles) for the models with more than 4 outputs, 64 (four tiles) for the others, whose
// four output tiles meet in one accumulator so that every lane ends with the outputs of its own slot. A member's operands and
// biases stay in VGPRs for the whole chunk, but for those of the widest models that SplitShape keeps in LDS, so a pass reads only
// its inputs, the next pass's while it computes: 16 bytes of features per lane and tile and the lane's targets, both laid out slot
// by slot by the minibatch launch.
// What bounds it is the issue of matrix and VALU instructions, which hardly overlap: a 32-wide, 12-output tile takes 14
// matrix instructions of 16 cycles and about 66 VALU ones (2.5 cycles each, conversions 4.5, exp2 and the reciprocal 8.6), where
// the 32-bit instructions of k_pop_mfma take 28 of 32 cycles beside their VALU work. Whole launches, k_pop_mfma and
// k_pop_split with weights in two parts and in three (MI355X, ms): material512 0.97 (its former pair-sharing kernel), 0.48, 0.51;
// two levels with 512 pairs on 65536 slots 1.58, 0.72, 0.82; 36-wide with 777 pairs on 5001 slots 0.37, 0.145, 0.16; 64-wide with
// 8192 pairs on 262144 slots 386, 119, 143.
// A lane adds its channel terms cw (d d) in float over a pass's slots, then into a double, as the other population kernels;
// central differences in double throughout (in float, their loss differences were 1.02 to 1.13 times as far from 64 bits as
// k_pop_mfma's).
// Values past the 16-bit range make NaN outputs (split_mlp.hpp), so a wave whose sum is a NaN evaluates its slots again in
// 32 bits, from the 32-bit weights, as k_pop_mfma does; with --clamp, where a NaN output becomes 0, the output pre-activations
// are tested. A model of such values pays for both evaluations in every step: its hidden values, scaled as the weights are
// (split_pow2), pass 65504.
template <class S>
constexpr int split_u() { return valu_out<S>() ? 4 : 2; }
// Tiles whose layers are evaluated together, so that one tile's activations stand between another's matrix instructions: all
// of a pass with one hidden tile, two with two, one with more (registers). Against one at a time (MI355X): ten iterations of
// the 16-wide 256 x 256 run 577 -> 572 us, a step of two levels 748 -> 729, of the 32-wide plane 236 -> 227.
template <class S>
constexpr int split_together() { return MfmaShape<S>::kHt == 1 ? split_u<S>() : (MfmaShape<S>::kHt == 2 ? 2 : 1); }

template <int From>
struct SlotSum { using T = float; };
template <>
struct SlotSum<kSets> { using T = double; };

template <class S, bool Clamp, int From, bool UnitCw>
__global__ void __launch_bounds__(64 * kPopWaves) __attribute__((amdgpu_waves_per_eu(pop_split_occupancy<S>()))) k_pop_split(DevModel m, PopSource src, int M, int Mcap,
                                                            int chunk, int chunks, SplitIn in, const float* __restrict__ feat,
                                                            double* __restrict__ part) {
    using Q = MfmaShape<S>;
    // central differences: members one weight apart, so the reference's activation (see launch_pop_matrix)
    constexpr int Act = From == kSets ? kActMax : kActFold;
    using P = SplitShape<S, 3>;
    static_assert(P::kOk, "a shape the split kernel takes");
    constexpr int NIN = Q::kIn, NO = Q::kNout, RO = out_regs<S>(), U = split_u<S>();
    constexpr bool kVOut = valu_out<S>();
    constexpr int TS = split_targets(NO), FB = 4 * split_inputs(NIN);   // floats of targets and bytes of features per slot
    constexpr int NT = kVOut ? NO : RO;                                  // target values a lane takes per read
    constexpr int TT = kVOut ? 1 : U;                                    // reads per pass
    __shared__ double red[kPopWaves];
    // the + member's parameters, then the - member's, and their weights' last parts; then their operands that stay in LDS
    constexpr int kWords = SplitLds<S>::kWords, kMem = 3 * kWords > 512 * P::kLdsOps ? 3 * kWords : 512 * P::kLdsOps;
    __shared__ __attribute__((aligned(16))) unsigned par_s[kMem];
    unsigned short* const last_s = (unsigned short*)(par_s + 2 * kWords);
    __shared__ __attribute__((aligned(16))) float vo_s[kVOut ? kPopWaves * kVoTile : 4];   // the 32-bit evaluation's output sums
    const int lane = tid_x() & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6);
    const int pair = bid_x(), ch = bid_y(), sgn = wave & 1, half = wave >> 1;
    const int i16 = lane & 15, g = lane >> 4;
    const int s0 = ch * chunk, s1 = min(M, s0 + chunk);
    constexpr int PS = 16 * U;                                           // slots per pass
    const int mine = ((s1 - s0 + PS - 1) / PS - half + 1) >> 1;          // this wave's passes: 2 q + half, q < mine
    const uint32_t slots = (uint32_t)Mcap + (uint32_t)kSplitSlack;
    const __amdgpu_buffer_rsrc_t rf = buffer_of((const float*)in.feat, slots * (uint32_t)FB), rt = buffer_of(in.tgt, slots * 4u * TS);
    const uint32_t fo = (uint32_t)(FB * i16 + 16 * (P::kS1 == 1 ? (g == 1 ? 1 : 0) : g));
    const uint32_t to = kVOut ? 4u * (uint32_t)(TS * lane) : 4u * (uint32_t)(TS * i16 + RO * g);
    struct In { h8v f[U]; float t[TT][NT]; };
    auto load = [&](In& n, int q) {
        const uint32_t s = (uint32_t)__builtin_amdgcn_readfirstlane(s0 + PS * (2 * q + half));
#pragma unroll
        for (int u = 0; u < U; u++) n.f[u] = __builtin_bit_cast(h8v, __builtin_amdgcn_raw_buffer_load_b128(rf, (int)fo, (int)((s + 16u * u) * FB), 0));
#pragma unroll
        for (int u = 0; u < TT; u++)
#pragma unroll
            for (int r = 0; r < NT; r++) n.t[u][r] = buffer_f32(rt, to + 4u * r, (s + 16u * u) * (4u * TS));
    };
    In in0, in1;
    load(in0, 0);
    const SplitScale sc = split_scale(in.scales);
    split_stage<S, From>(src, split_factors(sc, Act == kActMax ? 0.0f : m.fold_c, Clamp ? 1.0 : kNegLog2eD), pair, ch, par_s, last_s);
    __syncthreads();
    SplitWeights<S, 3> W;
    {
        h8v kept[P::kLdsOps + 1];
        split_load<S, 3>(W, par_s + sgn * kWords, last_s + sgn * kWords, lane, kept);
        if constexpr (P::kLdsOps > 0) {
            __syncthreads();
            split_keep<S, 3>(W, kept, (h8v*)par_s + sgn * 64 * P::kLdsOps, half == 0, lane);
            __syncthreads();
        }
    }
    const float ak = in_vgpr(act_k_of<Act>(m)), neg = in_vgpr(-1.0f), inv = in_vgpr(sc.inv);
    // the channel weight of each of this lane's output registers (0 past the last output)
    float cw[NT];
#pragma unroll
    for (int r = 0; r < NT; r++) {
        cw[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < NO; c++)
            if ((kVOut ? r : out_at<S>(g, r)) == c) cw[r] = m.cw[c];
    }
    constexpr bool kUnit = UnitCw && (kVOut || NO == 4 * RO);   // (padding outputs need their zero weight)
    double e = 0.0;
    bool bad = false;   // --clamp: an output pre-activation was a NaN
    // sum plus this lane's channel terms, in 32 bits; central differences, whose loss differences are small against the
    // losses: in 64
    using Sum = typename SlotSum<From>::T;
    auto terms = [&](const f4v& o, const float (&t)[NT], Sum sum) {
#pragma unroll
        for (int r = 0; r < NT; r++) {
            const float s = o[r] * inv;
            if constexpr (Clamp) bad |= !not_nan_bits(s);
            const float d = out_of<S>(s, Clamp) - t[r];
            if constexpr (From == kSets) sum = __builtin_fma(kUnit ? (double)d : (double)cw[r] * (double)d, (double)d, sum);
            else sum = __builtin_fmaf(kUnit ? d : __fmul_rn(cw[r], d), d, sum);
        }
        return sum;
    };
    auto pass = [&](In& c, In& n, int q) {
        q = __builtin_amdgcn_readfirstlane(q);
        load(n, q + 1 < mine ? q + 1 : q);
        W.reload();
        const int s = s0 + PS * (2 * q + half);   // the pass's first slot
        if constexpr (kVOut) {
            f4v o = W.co;
            constexpr int N = split_together<S>();
#pragma unroll
            for (int u = 0; u < U; u += N) {
                h8v b[N][P::kB], fs[N];
#pragma unroll
                for (int n = 0; n < N; n++) fs[n] = c.f[u + n];
                split_hidden_n<S, 3, Act, N>(W, fs, ak, neg, b);
#pragma unroll
                for (int n = 0; n < N; n++) o = split_dot_out<S, 3>(W, u + n, b[n], o);
            }
            const Sum ts = terms(o, c.t[0], 0);
            if (s + lane < s1) e += (double)ts;
        } else {
            f4v o[U];
            constexpr int N = split_together<S>();
#pragma unroll
            for (int u = 0; u < U; u += N) {
                h8v b[N][P::kB], fs[N];
#pragma unroll
                for (int n = 0; n < N; n++) fs[n] = c.f[u + n];
                split_hidden_n<S, 3, Act, N>(W, fs, ak, neg, b);
#pragma unroll
                for (int n = 0; n < N; n++) o[u + n] = split_dot_out<S, 3>(W, 0, b[n], W.co);
            }
            if (s + PS <= s1) {   // every slot inside the chunk (uniform)
                Sum ts = 0;
#pragma unroll
                for (int u = 0; u < U; u++) ts = terms(o[u], c.t[u], ts);
                e += (double)ts;
            } else {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const Sum ts = terms(o[u], c.t[u], 0);
                    if (s + 16 * u + i16 < s1) e += (double)ts;
                }
            }
        }
    };
    for (int q = 0; q < mine; q += 2) {
        pass(in0, in1, q);
        if (q + 1 < mine) pass(in1, in0, q + 1);
    }
    if (__builtin_amdgcn_ballot_w64(bad || !not_nan_bits_d(e)) != 0) {
        // 32 bits: the wave's slots again, a 16-slot tile at a time, from the minibatch's 32-bit feature rows and the member's
        // 32-bit weights, as k_pop_mfma evaluates them
        e = 0.0;
        float* const eg = src.eps + (size_t)pair * Q::kP;
        if constexpr (From == kDraw) {
            if (ch != 0) {   // (the chunk-0 block, which may not have run, writes the same values)
                const uint64_t head = noise_head(src.seed, NS_MLP, src.step, (uint32_t)pair);
                for (int k = lane; k < Q::kP; k += 64) eg[k] = gauss_at(src.nt, head, (uint64_t)k);
                __threadfence_block();
            }
        }
        MfmaWeights<S> W32;
        mfma_load_from<S>(W32, MemberAt<From>{ src.w0, eg, sgn ? -src.sigma : src.sigma, pair }, lane);
        if constexpr (!Clamp) scale_output<S>(W32, kNegLog2e);
        if constexpr (Act == kActFold) scale_hidden<S>(W32, fold_scale(m.leak));
        const __amdgpu_buffer_rsrc_t r32 = buffer_of(feat, 4u * ((uint32_t)minibatch_rows(NIN) * (uint32_t)Mcap + (uint32_t)kMinibatchSlack));
        for (int q = 0; q < mine; q++)
            for (int u = 0; u < U; u++) {
                const int st = s0 + PS * (2 * q + half) + 16 * u;
                if (st >= s1) break;
                float b1[1][Q::kKs1], x[1][Q::kKsH];
#pragma unroll
                for (int ks = 0; ks < Q::kKs1; ks++)
                    b1[0][ks] = buffer_f32(r32, 4u * ((uint32_t)(4 * ks + g) * (uint32_t)Mcap + (uint32_t)i16), 4u * (uint32_t)st);
                mfma_hidden<S, 1, Act>(W32, b1, ak, x);
                float ts = 0.0f;
                if constexpr (kVOut) {
                    const float d = out_of<S>(valu_out_g<S>(W32, x[0], vo_s + wave * kVoTile, g, i16), Clamp) -
                                    buffer_f32(rt, 4u * (uint32_t)(TS * i16 + min(g, NO - 1)), (uint32_t)st * (4u * TS));
                    ts = g < NO ? __fmul_rn(__fmul_rn(m.cw[min(g, NO - 1)], d), d) : 0.0f;
                } else {
                    f4v o[1];
                    mfma_output<S, 1>(W32, x, o);
#pragma unroll
                    for (int r = 0; r < RO; r++) {
                        const float d = out_of<S>(o[0][r], Clamp) - buffer_f32(rt, to + 4u * r, (uint32_t)st * (4u * TS));
                        ts = __builtin_fmaf(__fmul_rn(cw[r], d), d, ts);
                    }
                }
                if (st + i16 < s1) e += (double)ts;
            }
    }
    e = wave_sum(e);
    if (lane == 0) red[wave] = e;
    __syncthreads();
    if (tid_x() == 0) {
        part[(size_t)(2 * pair) * chunks + ch] = red[0] + red[2];
        part[(size_t)(2 * pair + 1) * chunks + ch] = red[1] + red[3];
    }
}

// The latent pair evaluation (LatentTrainer::step_impl, main.cpp:1990-2007) on the matrix cores:
// block (512 or 256 pixels, pair k), each wave a quarter of them in rounds of 64. In a round every
// lane builds the features of its own pixel with the pair's texels perturbed by +sg eps and by
// -sg eps (features_pm: both members from one set of taps and texel loads), and an exchange through
// the wave's own LDS rows (tiles_of) turns the 64 pixels into the B operands of four 16-pixel tiles:
// no barrier, so a wave's feature loads overlap other waves' matrix work. Each
// tile's + and - members are evaluated together; a pixel's error is decode_err's float sum of
// cw (d d) over its channels (a lane's out_regs in ascending order, then the lane groups pairwise: within
// a few ulp of the reference's ascending chain), and dpix = (e+ - e-) * inv_px.
// rounds of 64 pixels per wave, at most: 2 (512 pixels per block), or 1 for wide inputs; the launch may
// take fewer (`rounds`) to spread a small image over more blocks. One rule for the kernel and its
// launchers (the host checks a launch's rounds against it: the kernel stops at this count).
__host__ __device__ constexpr int lat_rounds_of(int nin) { return nin <= 8 ? 2 : 1; }
template <class S>
constexpr int lat_rounds() { return lat_rounds_of(MfmaShape<S>::kIn); }

// The features of one pixel for both members of a latent pair at once (fixed shapes): every tap and texel
// load is shared, each member's texel value is its own fused zb +- sg eps (a level outside `mask` is
// unperturbed), and each member's blend is the single-member blend - so fp and fm equal features<S> with
// PerturbedLatent{ z, eps, sg, mask } and { z, eps, -sg, mask }. Texels are read through raw buffers with
// 32-bit byte offsets (a latent holds fewer than 2^30 floats). The code has no branch per texel: a level
// outside `mask` reads its Gaussians through an empty buffer (rn: every load returns 0 without touching
// memory), so fma(+-sg, 0, zb) = zb, up to the sign of a zero texel, which no output can see (the layers'
// sums and the activation treat +0 and -0 alike). A branch per texel (or stores under a branch) makes the
// compiler keep the features in scratch.
template <int C>
__device__ __forceinline__ void sample_level_pm(const DevLevel& L, __amdgpu_buffer_rsrc_t rz, __amdgpu_buffer_rsrc_t re,
                                                float sg, const Tap& t, float* fp, float* fm) {
    const uint32_t off = (uint32_t)L.off, LW = (uint32_t)L.W, LC = (uint32_t)L.C;
    const uint32_t a = 4u * (off + ((uint32_t)t.y0 * LW + (uint32_t)t.x0) * LC);
    if (L.nearest) {
#pragma unroll
        for (int c = 0; c < C; c++) {
            const float zb = buffer_f32(rz, a + 4u * c, 0u), ee = buffer_f32(re, a + 4u * c, 0u);
            fp[c] = __builtin_fmaf(sg, ee, zb);
            fm[c] = __builtin_fmaf(-sg, ee, zb);
        }
        return;
    }
    const uint32_t tap[4] = { a, 4u * (off + ((uint32_t)t.y0 * LW + (uint32_t)t.x1) * LC),
                              4u * (off + ((uint32_t)t.y1 * LW + (uint32_t)t.x0) * LC),
                              4u * (off + ((uint32_t)t.y1 * LW + (uint32_t)t.x1) * LC) };
    const Blend w = blend_of(t);
#pragma unroll
    for (int c = 0; c < C; c++) {
        float vp[4], vm[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float zb = buffer_f32(rz, tap[q] + 4u * c, 0u), ee = buffer_f32(re, tap[q] + 4u * c, 0u);
            vp[q] = __builtin_fmaf(sg, ee, zb);
            vm[q] = __builtin_fmaf(-sg, ee, zb);
        }
        fp[c] = blend(w, vp[0], vp[1], vp[2], vp[3]);
        fm[c] = blend(w, vm[0], vm[1], vm[2], vm[3]);
    }
}

template <class S>
__device__ __forceinline__ void features_pm(const DevModel& m, __amdgpu_buffer_rsrc_t rz, __amdgpu_buffer_rsrc_t re, __amdgpu_buffer_rsrc_t rn,
                                            float sg, unsigned mask,
                                            int px, int py, float (&fp)[S::kMaxIn], float (&fm)[S::kMaxIn]) {
    static_assert(S::kFixed, "fixed shapes only");
    const float u = pixel_u(px, m.W), v = pixel_u(py, m.H);
    const Tap t0 = tap_of(m.lv[0].W, m.lv[0].H, m.lv[0].nearest != 0, u, v);
    Tap t1 = t0;
    sample_level_pm<S::kC0>(m.lv[0], rz, (mask & 1u) ? re : rn, sg, t0, fp, fm);
    if constexpr (S::kC1 > 0) {
        t1 = tap_of(m.lv[1].W, m.lv[1].H, m.lv[1].nearest != 0, u, v);
        sample_level_pm<S::kC1>(m.lv[1], rz, ((mask >> 1) & 1u) ? re : rn, sg, t1, fp + S::kC0, fm + S::kC0);
    }
    if constexpr (S::kC2 > 0) {
        const Tap t2 = tap_of(m.lv[2].W, m.lv[2].H, m.lv[2].nearest != 0, u, v);
        sample_level_pm<S::kC2>(m.lv[2], rz, ((mask >> 2) & 1u) ? re : rn, sg, t2, fp + S::kC0 + S::kC1, fm + S::kC0 + S::kC1);
    }
    constexpr int k0 = S::kC0 + S::kC1 + S::kC2;
#pragma unroll
    for (int q = 0; q < S::kNpos; q++) {
        const bool uv = m.pos[q] == 0;
        fp[k0 + 2 * q] = fm[k0 + 2 * q] = __builtin_fmaf(uv ? u : t1.fx, 2.0f, -1.0f);
        fp[k0 + 2 * q + 1] = fm[k0 + 2 * q + 1] = __builtin_fmaf(uv ? v : t1.fy, 2.0f, -1.0f);
    }
}

// The column and row of pixel base + lane for a wave's 64 pixels from base (a multiple of 64): when the
// image's width is a multiple of 64 they share one row (a scalar division), else each lane divides (pixels
// past the last clamped to it).
__device__ __forceinline__ void round_pixel(const DevModel& m, int base, int lane, int& px, int& py) {
    if (m.W % 64 == 0 && base < m.npix) {
        const int row = base / m.W;
        px = base - row * m.W + lane;
        py = row;
    } else {
        const int pr = min(base + lane, m.npix - 1);
        px = pr % m.W;
        py = pr / m.W;
    }
}


// One 16-pixel tile of a latent pair: both members' MLPs on the tile's first-layer operands bp / bm, each lane's
// channel terms cw (d d) (its out_regs in ascending order, or its one on the VALU output layer), the pixel's four
// lane groups added pairwise for each member (group_sums), and (e+ - e-) inv_px written to out[p] by lane group 0.
template <class S, int Act, bool Clamp>
__device__ __forceinline__ void lat_pair_tile(const DevModel& m, const MfmaWeights<S>& W, float ak, const float (&cw)[4],
                                              const float (&bp)[MfmaShape<S>::kKs1], const float (&bm)[MfmaShape<S>::kKs1],
                                              const float (&tt)[4], float* vo, float* sums, int g, int i16, int p,
                                              float* __restrict__ out) {
    using Q = MfmaShape<S>;
    constexpr bool kVOut = valu_out<S>();
    // the first layer's pre-activations of both members (D layout)
    f4v a1[2][Q::kHt];
    {
        float b1[2][Q::kKs1];
#pragma unroll
        for (int ks = 0; ks < Q::kKs1; ks++) { b1[0][ks] = bp[ks]; b1[1][ks] = bm[ks]; }
        mfma_layer1<S, 2>(W, b1, a1);
    }
    float ep = 0.0f, em = 0.0f;
    if constexpr (kVOut) {
        float x[2][Q::kKsH];
        mfma_hidden_from1<S, 2, Act>(W, a1, ak, x);
        const float dp = out_of<S>(valu_out_g<S>(W, x[0], vo, g, i16), Clamp) - tt[0],
                    dm = out_of<S>(valu_out_g<S>(W, x[1], vo + kVoTile, g, i16), Clamp) - tt[0];
        ep = __fmul_rn(cw[0], __fmul_rn(dp, dp));
        em = __fmul_rn(cw[0], __fmul_rn(dm, dm));
    } else {
        float x[2][Q::kKsH];
        mfma_hidden_from1<S, 2, Act>(W, a1, ak, x);
        f4v o[2];
        mfma_output<S, 2>(W, x, o);
#pragma unroll
        for (int r = 0; r < out_regs<S>(); r++) {
            const float dp = out_of<S>(o[0][r], Clamp) - tt[r], dm = out_of<S>(o[1][r], Clamp) - tt[r];
            ep = __builtin_fmaf(cw[r], __fmul_rn(dp, dp), ep);
            em = __builtin_fmaf(cw[r], __fmul_rn(dm, dm), em);
        }
    }
    float sp, sm;
    group_sums(ep, em, sums, g, i16, sp, sm);
    if (g == 0 && p < m.npix) out[p] = __fmul_rn(sp - sm, m.inv_px);
}

template <class S, int Act, bool Clamp>
__global__ void __launch_bounds__(256) k_lat_pair_mfma(DevModel m, const float* __restrict__ w, const float* __restrict__ zdec,
                                                      const float* __restrict__ eps, const float* __restrict__ tgt, float sg,
                                                      unsigned mask, float* __restrict__ dpix, int rounds) {
    using Q = MfmaShape<S>;
    constexpr int NO = Q::kNout, kRounds = lat_rounds<S>();
    // at most 4 outputs: the output layer on the VALU leaves output g of pixel j in lane (g, j)
    constexpr bool kVOut = valu_out<S>();
    const int k = bid_y();
    const int lane = tid_x() & 63, wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6), i16 = lane & 15, g = lane >> 4;
    // each wave's LDS exchanges (in place of lane swaps): both members' tile operands, the VALU output layer's
    // reduce-scatters of both members, the pixel sums of both members' errors
    constexpr int kTileLds = 2 * kTilesLds<S>;
    constexpr int kWaveLds = kTileLds + (kVOut ? 2 * kVoTile : 0) + kSumsLds;
    __shared__ __attribute__((aligned(16))) float lds[4 * kWaveLds];
    float* const tl = lds + wave * kWaveLds;
    float* const vo = tl + kTileLds;
    float* const sums = vo + (kVOut ? 2 * kVoTile : 0);
    const __amdgpu_buffer_rsrc_t rz = buffer_of(zdec, 4u * (uint32_t)m.nz), re = buffer_of(eps + (size_t)k * m.nz, 4u * (uint32_t)m.nz),
                                 rn = buffer_of(eps, 0u);   // a level outside the mask: no Gaussians (every load 0)
    float* out = dpix + (size_t)k * m.npix;
    MfmaWeights<S> W;
    mfma_load<S>(W, w, lane);
    if constexpr (!Clamp) scale_output<S>(W, kNegLog2e);
    if constexpr (Act == kActFold) scale_hidden<S>(W, fold_scale(m.leak));
    const float ak = act_k_of<Act>(m);
    float cw[4];
    if constexpr (kVOut) {
#pragma unroll
        for (int r = 0; r < 4; r++) cw[r] = (r == 0 && g < NO) ? m.cw[g] : 0.0f;
    } else {
        lane_cw<S>(m.cw, g, cw);
    }
    // the targets of the tile at pixel t0: lane (g, j) reads channels out_at(g, r) of pixel t0 + j (padding
    // reads a valid channel; rows past the last pixel are clamped); VALU output layer: channel g
    auto load_t = [&](int t0, float (&t)[4]) {
        const int pr = min(t0 + i16, m.npix - 1);
        if constexpr (kVOut) {
            t[0] = tgt[(size_t)pr * NO + min(g, NO - 1)];
#pragma unroll
            for (int r = 1; r < 4; r++) t[r] = 0.0f;
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) t[r] = r < out_regs<S>() ? tgt[(size_t)pr * NO + max(out_at<S>(g, r), 0)] : 0.0f;
        }
    };
    for (int rd = 0; rd < kRounds; rd++) {
        if (rd >= rounds) break;
        const int base = bid_x() * 256 * rounds + 64 * rounds * wave + 64 * rd;   // tile t: pixels base + 16 t + j
        float tn[4];
        load_t(base, tn);
        // both members' first-layer operands
        float bp[4][Q::kKs1], bm[4][Q::kKs1];
        {
            int px, py;
            round_pixel(m, base, lane, px, py);
            float fp[S::kMaxIn], fm[S::kMaxIn];
            features_pm<S>(m, rz, re, rn, sg, mask, px, py, fp, fm);
            tiles_of<S>(fp, bp, tl, g, i16);
            tiles_of<S>(fm, bm, tl + kTilesLds<S>, g, i16);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float tt[4];
#pragma unroll
            for (int r = 0; r < 4; r++) tt[r] = tn[r];
            if (t + 1 < 4) load_t(base + 16 * (t + 1), tn);
            const int p = base + 16 * t + i16;
            lat_pair_tile<S, Act, Clamp>(m, W, ak, cw, bp[t], bm[t], tt, vo, sums, g, i16, p, out);
        }
    }
}

// ---- The latent pair evaluation on the 16-bit matrix instructions with operands in two parts (split_mlp.hpp), for the shapes
// k_pop_split takes: as many blocks as fit the chip, each of which stages the current weights once (split_stage_plain); a
// wave takes 64 pixels of a pair at a time, every wave's next one a whole grid further, over all pairs. Each lane builds its
// pixel's features for both members (features_pm) and writes them split to the wave's LDS; lane group g of a 16-pixel tile
// reads back the 16 bytes of parts that its slots of the first layer take. A lane's channel terms of the + member less those of the - member
// are added over a pixel's four lane groups (more than 4 outputs; through LDS, so that each lane ends with one of the 64
// pixels), or are the pixel's own (at most 4: split_mlp.hpp, ao). A wave that met a NaN evaluates its rounds again in 32 bits
// (lat_pair_tile), as k_pop_split does.
// What bounds it is instruction issue, as in k_pop_split, with the feature loads (two floats a tap and channel) beside it.
// Against k_lat_pair_mfma (MI355X): 512 x 512, four maps, a searched and a 4-channel level, 4 pairs: 71 -> 40 us; RGB, levels of 8 and 4 channels,
// 16 pairs: 292 -> 165 us. All four products of the two parts are taken (1% of the step): over seven models of three seeds the
// gradient's error against 64 bits was 1.002 times the 32-bit kernel's, 1.004 without the product of the lo parts; with the small
// products first, the per-pixel differences' is 0.68 to 0.98 times it (split_mlp.hpp).
template <class S>
__device__ __forceinline__ SplitScale split_stage_plain(const DevModel& m, const float* __restrict__ w, double out, unsigned* __restrict__ lds) {
    using L = SplitLds<S>;
    constexpr int kP = MfmaShape<S>::kP, kN = (kP + 255) / 256;
    __shared__ SplitRange top[4][3];
    float v[kN];
    SplitRange r[3] = { { 0, 0, 0 }, { 0, 0, 0 }, { 0, 0, 0 } };
#pragma unroll
    for (int q = 0; q < kN; q++) v[q] = w[min(tid_x() + 256 * q, kP - 1)];
    const float fold = fold_scale(m.leak);
#pragma unroll
    for (int q = 0; q < kN; q++) {
        const int k = tid_x() + 256 * q;
        const bool b = k >= kP || L::bias(k);
#pragma unroll
        for (int l = 0; l < 3; l++) r[l].add(!b && L::layer(k) == l ? v[q] : 0.0f, 0.0f, l == 2 ? (float)fabs(out) : fold);
    }
#pragma unroll
    for (int l = 0; l < 3; l++) {
        r[l].add_wave();
        if ((tid_x() & 63) == 0) top[tid_x() >> 6][l] = r[l];
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 3; l++) {
        r[l] = top[0][l];
        for (int q = 1; q < 4; q++) r[l].add(top[q][l]);
    }
    SplitScale sc{ split_pow2(r[0], kSplitExp[0]), split_pow2(r[1], kSplitExp[1]), split_pow2(r[2], kSplitExp[2]), 0.0f };
    sc.inv = 1.0f / (sc.s1 * sc.s2 * sc.s3);
    const SplitFactors f = split_factors(sc, m.fold_c, out);
#pragma unroll
    for (int q = 0; q < kN; q++) {
        const int k = tid_x() + 256 * q;
        if (k < kP) {
            const int l = L::layer(k);
            const bool b = L::bias(k);
            const double fw = l == 0 ? f.w1 : (l == 1 ? f.w2 : f.w3), fb = l == 0 ? f.b1 : (l == 1 ? f.b2 : f.b3);
            unsigned short last;
            lds[L::pos(k)] = split_param(v[q], 0.0f, 0.0f, b ? fb : fw, b, last);
        }
    }
    __syncthreads();
    return sc;
}

// A wave's 64 pixels' features f (lane: one pixel) split to t, as split_piece orders them
template <class S>
__device__ __forceinline__ void split_write(const float (&f)[S::kMaxIn], float neg, u4v* __restrict__ t, int lane) {
    constexpr int N = split_inputs(S::kNin), C = N / 8;   // 16-byte pieces per part
    const float neg_lo = neg * kSplitLo;
    h2v hi[N / 2], lo[N / 2];
#pragma unroll
    for (int j = 0; j < N / 2; j++) {
        const int i = 2 * j;
        const float x = i < S::kNin ? f[i < S::kNin ? i : 0] : 0.0f, y = i + 1 < S::kNin ? f[i + 1 < S::kNin ? i + 1 : 0] : 0.0f;
        hi[j] = __builtin_convertvector((f2v){ x, y }, h2v);
        lo[j] = __builtin_convertvector((f2v){ __builtin_fmaf((float)hi[j][0], neg_lo, x * kSplitLo),
                                               __builtin_fmaf((float)hi[j][1], neg_lo, y * kSplitLo) }, h2v);
    }
#pragma unroll
    for (int q = 0; q < 2 * C; q++) {
        u4v a;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int p = split_piece(N, 8 * q + 2 * j);   // (an even half and the next one are parts of neighbouring inputs)
            a[j] = __builtin_bit_cast(unsigned, p < N ? hi[p / 2 % (N / 2)] : lo[p / 2 % (N / 2)]);
        }
        t[lane * 2 * C + q] = a;
    }
}
// the first-layer operand of pixel `px` (of the wave's 64) for lane group g
template <class S>
__device__ __forceinline__ h8v split_read(const u4v* __restrict__ t, int px, int g) {
    constexpr int C = split_inputs(S::kNin) / 8;
    return __builtin_bit_cast(h8v, t[px * 2 * C + (C == 1 ? (g & 1) : g)]);
}

template <class S, bool Clamp, bool UnitCw>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(split_occupancy<S>()))) k_lat_split(DevModel m, const float* __restrict__ w, const float* __restrict__ zdec,
                                                      const float* __restrict__ eps, const float* __restrict__ tgt, float sg,
                                                      unsigned mask, float* __restrict__ dpix, int K, int blocks) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S, 2>;
    constexpr int NO = Q::kNout, RO = out_regs<S>(), kEx = 64 * split_inputs(Q::kIn);   // floats of one member's exchange
    constexpr bool kVOut = valu_out<S>();
    constexpr int NT = kVOut ? NO : RO;
    static_assert(2 * kTilesLds<S> <= 2 * kEx && 2 * kVoTile + kSumsLds <= 2 * kEx, "the 32-bit evaluation's exchanges fit");
    __shared__ unsigned par_s[SplitLds<S>::kWords];
    __shared__ __attribute__((aligned(16))) float ex_s[4][2 * kEx];
    __shared__ __attribute__((aligned(16))) float sum_s[kVOut ? 1 : 4][kVOut ? 4 : 256];
    const int lane = tid_x() & 63, wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6), i16 = lane & 15, g = lane >> 4;
    const SplitScale sc = split_stage_plain<S>(m, w, Clamp ? 1.0 : kNegLog2eD, par_s);
    SplitWeights<S, 2> W;
    {
        h8v kept[1];
        split_load<S, 2>(W, par_s, nullptr, lane, kept);
    }
    const float ak = in_vgpr(act_k_of<kActFold>(m)), neg = in_vgpr(-1.0f), inv = in_vgpr(sc.inv);
    float cw[NT];
#pragma unroll
    for (int r = 0; r < NT; r++) {
        cw[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < NO; c++)
            if ((kVOut ? r : out_at<S>(g, r)) == c) cw[r] = m.cw[c];
    }
    constexpr bool kUnit = UnitCw && (kVOut || NO == 4 * RO);
    const __amdgpu_buffer_rsrc_t rz = buffer_of(zdec, 4u * (uint32_t)m.nz), rn = buffer_of(eps, 0u);
    float* const ex = ex_s[wave];
    const int R = (m.npix + 63) >> 6;                       // 64-pixel rounds of an image
    const int stride = 4 * blocks;
    // this wave's rounds: f(pair, first pixel)
    auto rounds = [&](auto f) {
        int k = 0;
        for (int rd = bid_x() * 4 + wave;; rd += stride) {
            while (rd >= R && k < K) { rd -= R; k++; }
            if (k >= K) break;
            f(k, 64 * rd);
        }
    };
    bool again = false;   // a round had a NaN
    rounds([&](int k, int base) {
        const __amdgpu_buffer_rsrc_t re = buffer_of(eps + (size_t)k * m.nz, 4u * (uint32_t)m.nz);
        float* const out = dpix + (size_t)k * m.npix;
        {
            int px, py;
            round_pixel(m, base, lane, px, py);
            float fp[S::kMaxIn], fm[S::kMaxIn];
            features_pm<S>(m, rz, re, rn, sg, mask, px, py, fp, fm);
            split_write<S>(fp, neg, (u4v*)ex, lane);
            split_write<S>(fm, neg, (u4v*)(ex + kEx), lane);
        }
        wave_lds_fence();
        bool bad = false;
        // this lane's channel terms of the + member less the - member's: cw (d+ d+ - d- d-) as cw (d+ - d-) (d+ + d-), which
        // rounds relative to the difference and not to each square (the two members' errors are close)
        auto terms = [&](const f4v& op, const f4v& om, const float (&t)[NT]) {
            float e = 0.0f;
#pragma unroll
            for (int r = 0; r < NT; r++) {
                const float sp = op[r] * inv, sm = om[r] * inv;
                if constexpr (Clamp) bad |= !not_nan_bits(sp) || !not_nan_bits(sm);
                const float vp = out_of<S>(sp, Clamp), vm = out_of<S>(sm, Clamp);
                const float d = vp - vm, c = (vp - t[r]) + (vm - t[r]);
                e = __builtin_fmaf(kUnit ? d : __fmul_rn(cw[r], d), c, e);
            }
            return e;
        };
        float diff;
        if constexpr (kVOut) {
            float t[NT];
            const int pr = min(base + lane, m.npix - 1);
#pragma unroll
            for (int r = 0; r < NT; r++) t[r] = tgt[(size_t)pr * NO + r];
            f4v o[2] = { W.co, W.co };
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int v = 0; v < 2; v++) {
                    h8v b[P::kB];
                    split_hidden<S, 2, kActFold>(W, split_read<S>((const u4v*)(ex + v * kEx), 16 * u + i16, g), ak, neg, b);
                    o[v] = split_dot_out<S, 2>(W, u, b, o[v]);
                }
            diff = terms(o[0], o[1], t);
        } else {
            float* const sums = sum_s[wave];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                float t[NT];
                const int pr = min(base + 16 * u + i16, m.npix - 1);
#pragma unroll
                for (int r = 0; r < NT; r++) t[r] = tgt[(size_t)pr * NO + max(out_at<S>(g, r), 0)];
                f4v o[2];
#pragma unroll
                for (int v = 0; v < 2; v++) {
                    h8v b[P::kB];
                    split_hidden<S, 2, kActFold>(W, split_read<S>((const u4v*)(ex + v * kEx), 16 * u + i16, g), ak, neg, b);
                    o[v] = split_dot_out<S, 2>(W, 0, b, W.co);
                }
                sums[(16 * u + i16) * 4 + g] = terms(o[0], o[1], t);
            }
            wave_lds_fence();
            const f4v v = *reinterpret_cast<const f4v*>(sums + 4 * lane);
            diff = (v[0] + v[2]) + (v[1] + v[3]);
        }
        wave_lds_fence();
        again |= __builtin_amdgcn_ballot_w64(bad || !not_nan_bits(diff)) != 0;
        if (base + lane < m.npix) out[base + lane] = __fmul_rn(diff, m.inv_px);
    });
    if (!again) return;
    // 32 bits, all of the wave's rounds
    MfmaWeights<S> F;
    mfma_load<S>(F, w, lane);
    if constexpr (!Clamp) scale_output<S>(F, kNegLog2e);
    scale_hidden<S>(F, fold_scale(m.leak));
    rounds([&](int k, int base) {
        const __amdgpu_buffer_rsrc_t re = buffer_of(eps + (size_t)k * m.nz, 4u * (uint32_t)m.nz);
        float* const out = dpix + (size_t)k * m.npix;
        float bp[4][Q::kKs1], bm[4][Q::kKs1], cw4[4];
        {
            int px, py;
            round_pixel(m, base, lane, px, py);
            float fp[S::kMaxIn], fm[S::kMaxIn];
            features_pm<S>(m, rz, re, rn, sg, mask, px, py, fp, fm);
            tiles_of<S>(fp, bp, ex, g, i16);
            tiles_of<S>(fm, bm, ex + kTilesLds<S>, g, i16);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) cw4[r] = kVOut ? ((r == 0 && g < NO) ? m.cw[min(g, NO - 1)] : 0.0f) : (r < NT ? cw[r < NT ? r : 0] : 0.0f);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            float t[4];
            const int pr = min(base + 16 * u + i16, m.npix - 1);
#pragma unroll
            for (int r = 0; r < 4; r++) t[r] = tgt[(size_t)pr * NO + (kVOut ? min(g, NO - 1) : max(out_at<S>(g, r), 0))];
            lat_pair_tile<S, kActFold, Clamp>(m, F, ak, cw4, bp[u], bm[u], t, ex, ex + 2 * kVoTile, g, i16, base + 16 * u + i16, out);
        }
    });
}

// The selector search's occupancy target: four waves per SIMD for the 8-input, 32-wide models with more than 4
// outputs and the folded activation, which fit in 128 VGPRs without scratch (the compiler alone gives them 130 and
// three waves); the compiler's choice for the other shapes, several of which spill at four.
template <class S, int Act>
constexpr int qat_occupancy() {
    return (MfmaShape<S>::kIn <= 8 && MfmaShape<S>::kH == 32 && !valu_out<S>() && Act == kActFold) ? 4 : 1;
}

// The selector search (qat_search, main.cpp:2088-2139) on the matrix cores, for a nearest level 0
// of the image's size (each texel's cell is its own pixel): wave = 64 pixels in four 16-pixel tiles.
// Every lane builds the features of its own pixel (features<S>) and tiles_of turns them into the four
// tiles' B operands. Per tile and channel, every candidate value is one MLP evaluation of the tile with
// that feature replaced (two candidates at a time); the first layer's sums over the other inputs are formed
// once per tile and channel and the candidate's term is added to them last (the reference adds it in input
// order, main.cpp:603-627: the same products, one rounding order apart). The choice is the reference's: the current grid
// value first, then every other value with strict <, so the first strictly smaller loss wins
// (main.cpp:2101-2132). The winner enters the features of the next channel and is written to the
// decode buffer. A candidate's loss is the pixel's float sum of cw (d d) over its channels (a lane's
// out_regs, then the pixel's four lanes pairwise, the same value in each of them) with the hidden
// activation of act<Act>: the reference adds the float terms in double with its own activation, so a
// choice can differ from the reference's only between candidates whose losses agree to a few float
// roundings (the reference's own check accepts such rounding ties, main.cpp:3143-3144).
// The search on the 64 pixels from base (tile t: pixels base + 16 t + j) of one wave, on the 32-bit instructions.
// UnitCw: every channel weight is 1, so a candidate's error terms are d d (fused into the sum where a lane holds several)
template <class S, int Act, bool Clamp, bool UnitCw>
__device__ __forceinline__ void qat_round(const DevModel& m, const MfmaWeights<S>& W, float ak, const float (&cw)[4], float* __restrict__ zdec,
                                          const float* __restrict__ tgt, const int* __restrict__ qat_bits, const float* __restrict__ grid,
                                          int base, int lane, float* tl, float* vo, float* sums) {
    using Q = MfmaShape<S>;
    constexpr int NO = Q::kNout, C0 = S::kC0;
    constexpr bool kVOut = valu_out<S>();
    const int i16 = lane & 15, g = lane >> 4;
    float f[S::kMaxIn];
    {
        const int pr = min(base + lane, m.npix - 1);
        features<S>(m, PlainLatent{ zdec }, pr % m.W, pr / m.W, f);
    }
    float b[4][Q::kKs1];
    tiles_of<S>(f, b, tl, g, i16);
    // the targets of tile t: lane (g, j) holds channels out_at(g, r) (VALU output layer: g) of pixel j; loaded one
    // tile ahead, so only the first tile's loads are waited for before the search starts
    auto load_t = [&](int t, float (&tv)[4]) {
        const int pr = min(base + 16 * t + i16, m.npix - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) tv[r] = tgt[(size_t)pr * NO + (kVOut ? min(g, NO - 1) : max(out_at<S>(g, r), 0))];
    };
    // per channel: its bit depth, its grid, and the current grid index of the lane's own pixel
    int bits[C0], cur_own[C0];
    const float* gvs[C0];
#pragma unroll
    for (int c = 0; c < C0; c++) {
        bits[c] = qat_bits[c];
        gvs[c] = grid + bits[c] * 257;
        cur_own[c] = qat_index(f[c], bits[c]);
    }
    float tn[4];
    load_t(0, tn);
    // Tile by tile (a tile's pixels are independent of the other tiles'), each tile's channels in order: the winner of
    // channel c enters the features of channel c + 1, as in the reference's per-texel loop.
#pragma unroll
    for (int t = 0; t < 4; t++) {
        float tt[4];
#pragma unroll
        for (int r = 0; r < 4; r++) tt[r] = tn[r];
        if (t + 1 < 4) load_t(t + 1, tn);
#pragma unroll
        for (int c = 0; c < C0; c++) {
            const int levels = (1 << bits[c]) - 1;
            const float* gv = gvs[c];
            // the channel's current index of pixel j of tile t, from the lane that built the pixel's features
            const int cur = __builtin_amdgcn_ds_bpermute((16 * t + i16) << 2, cur_own[c]);
            // the losses and grid values of the current candidate and of the best other one so far: the winner's
            // value comes from these registers, not from a load of the grid after the search
            // best over the other candidates in ascending k, from +inf with a strict <; a NaN loss never wins and a NaN
            // current loss keeps the current value, as the reference's running minimum from the current loss gives
            // (main.cpp:2122-2127). The NaN tests are on the bits: this file is compiled assuming no NaNs.
            // (selects, not branches: the choice is per lane. A best_l still at +inf means no other candidate won.)
            float cur_l = 0.0f, best_l = __builtin_inff(), cur_v = 0.0f, best_v = 0.0f;
            // The first layer's sums of the tile without input c (a zero in its place: fma(w, 0, s) = s) and, in D
            // layout, the weight of input c into each of this lane's units (read from the lane of W.a1 that holds
            // it): a candidate's first-layer pre-activations are then one fused multiply-add, w_c gc + base, and
            // the matrix cores take only the layers after the first for each candidate.
            f4v s1[1][Q::kHt];
            {
                float b0[1][Q::kKs1];
#pragma unroll
                for (int ks = 0; ks < Q::kKs1; ks++) b0[0][ks] = (ks == c / 4 && g == c % 4) ? 0.0f : b[t][ks];
                mfma_layer1<S, 1>(W, b0, s1);
            }
            float w1c[Q::kHt][4];
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    w1c[ot][r] = __int_as_float(__builtin_amdgcn_ds_bpermute(((c % 4) * 16 + 4 * g + r) << 2, __float_as_int(W.a1[ot][c / 4])));
            for (int kc = 0; kc <= levels; kc += 2) {   // 2^bits candidates: two tiles at a time
                const float gc[2] = { gv[kc], gv[kc + 1] };
                f4v a1[2][Q::kHt];
#pragma unroll
                for (int v = 0; v < 2; v++)
#pragma unroll
                    for (int ot = 0; ot < Q::kHt; ot++)
#pragma unroll
                        for (int r = 0; r < 4; r++) a1[v][ot][r] = __builtin_fmaf(w1c[ot][r], gc[v], s1[0][ot][r]);
                float lv[2];   // this lane's channels, then the pixel's lanes
                float x[2][Q::kKsH];
                mfma_hidden_from1<S, 2, Act>(W, a1, ak, x);
                if constexpr (kVOut) {
#pragma unroll
                    for (int v = 0; v < 2; v++) {
                        const float d = out_of<S>(valu_out_g<S>(W, x[v], vo + v * kVoTile, g, i16), Clamp) - tt[0];
                        constexpr bool kUnit = UnitCw && NO == 4;
                        lv[v] = kUnit ? __fmul_rn(d, d) : __fmul_rn(cw[0], __fmul_rn(d, d));   // cw (d d), main.cpp:2119
                    }
                } else {
                    f4v o[2];
                    mfma_output<S, 2>(W, x, o);
#pragma unroll
                    for (int v = 0; v < 2; v++) {
                        lv[v] = 0.0f;
#pragma unroll
                        for (int r = 0; r < out_regs<S>(); r++) {
                            const float d = out_of<S>(o[v][r], Clamp) - tt[r];
                            constexpr bool kUnit = UnitCw && NO == 4 * out_regs<S>();
                            lv[v] = kUnit ? __builtin_fmaf(d, d, lv[v]) : __builtin_fmaf(cw[r], __fmul_rn(d, d), lv[v]);
                        }
                    }
                }
                float ls[2];
                group_sums(lv[0], lv[1], sums, g, i16, ls[0], ls[1]);
#pragma unroll
                for (int v = 0; v < 2; v++) {
                    const float l = ls[v];
                    const bool is_cur = kc + v == cur;
                    const bool better = !is_cur && not_nan_bits(l) && l < best_l;
                    cur_l = is_cur ? l : cur_l;
                    cur_v = is_cur ? gc[v] : cur_v;
                    best_l = better ? l : best_l;
                    best_v = better ? gc[v] : best_v;
                }
            }
            // cur is in 0 .. levels (qat_index clamps), so cur_v is its grid value
            const float win_v = (not_nan_bits(cur_l) && best_l < cur_l) ? best_v : cur_v;
            if (g == c % 4) b[t][c / 4] = win_v;
            const int p = base + 16 * t + i16;
            if (g == 0 && p < m.npix) zdec[m.lv[0].off + (size_t)p * m.lv[0].C + c] = win_v;
        }
    }
}

template <class S, int Act, bool Clamp, bool UnitCw = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qat_occupancy<S, Act>()))) k_qat_mfma(DevModel m, const float* __restrict__ w, float* __restrict__ zdec,
                                                 const float* __restrict__ tgt, const int* __restrict__ qat_bits,
                                                 const float* __restrict__ grid) {
    using Q = MfmaShape<S>;
    constexpr int NO = Q::kNout;
    const int lane = tid_x() & 63, wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6), g = lane >> 4;
    constexpr bool kVOut = valu_out<S>();   // the output layer on the VALU: output g of pixel j in lane (g, j)
    // each wave's LDS exchanges (in place of lane swaps): the tile operands, the VALU output layer's
    // reduce-scatters of both candidates, the candidates' pixel sums
    constexpr int kWaveLds = kTilesLds<S> + (kVOut ? 2 * kVoTile : 0) + kSumsLds;
    __shared__ __attribute__((aligned(16))) float lds[4 * kWaveLds];
    float* const tl = lds + wave * kWaveLds;
    float* const vo = tl + kTilesLds<S>;
    float* const sums = vo + (kVOut ? 2 * kVoTile : 0);
    MfmaWeights<S> W;
    mfma_load<S>(W, w, lane);
    if constexpr (!Clamp) scale_output<S>(W, kNegLog2e);
    if constexpr (Act == kActFold) scale_hidden<S>(W, fold_scale(m.leak));
    const float ak = act_k_of<Act>(m);
    float cw[4];
    if constexpr (kVOut) {
#pragma unroll
        for (int r = 0; r < 4; r++) cw[r] = (r == 0 && g < NO) ? m.cw[g] : 0.0f;
    } else {
        lane_cw<S>(m.cw, g, cw);
    }
    qat_round<S, Act, Clamp, UnitCw>(m, W, ak, cw, zdec, tgt, qat_bits, grid, bid_x() * 256 + wave * 64, lane, tl, vo, sums);
}

// ---- The selector search on the 16-bit matrix instructions with operands in two parts, for the shapes k_pop_split takes and
// 0 <= leak <= 1. As k_qat_mfma, with blocks that stay on the chip as k_lat_split's: a wave takes 64 pixels at a time. The
// searched inputs are left out of the first layer's operands (zeros in their places); each tile's first layer is formed once,
// the other searched channels' terms and a candidate's are added to it in 32 bits, one fused multiply-add each. A candidate
// then takes the layers after the first: 9 matrix instructions of 16 cycles for the 32-wide, 12-output models where the
// 32-bit ones are 24 of 32. The winners are written when all of a round's losses are numbers; a round with a NaN is left as
// it was and searched in 32 bits at the end (qat_round), the launch giving a wave at most 64 rounds.
// material512, two channels of four values (MI355X): 73 -> 38 us.
// With one hidden layer a candidate is the output layer alone, of which at most 4 outputs are a small part of a matrix tile: those
// models stay on k_qat_mfma, whose output layer is on the VALU (7-32-3, one channel, 512 x 512: 26 us against 31).
// (a wave per SIMD fewer than k_lat_split with more than one searched channel, whose first-layer weights are in registers too)
constexpr int qat_waves(int nin, int H, int nout, int c0) { return split_waves(nin, H, nout) - (c0 > 1 && H <= 48 ? 1 : 0); }
template <class S, bool Clamp, bool UnitCw>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qat_waves(S::kNin, S::kH, S::kNout, S::kC0)))) k_qat_split(DevModel m, const float* __restrict__ w, float* __restrict__ zdec,
                                                 const float* __restrict__ tgt, const int* __restrict__ qat_bits,
                                                 const float* __restrict__ grid, int blocks) {
    using Q = MfmaShape<S>;
    using P = SplitShape<S, 2>;
    constexpr int NO = Q::kNout, RO = out_regs<S>(), C0 = S::kC0, kEx = 64 * split_inputs(Q::kIn);
    constexpr bool kVOut = valu_out<S>();
    constexpr int NT = kVOut ? NO : RO;
    static_assert(kTilesLds<S> <= kEx, "the 32-bit search's tile operands fit");
    __shared__ unsigned par_s[SplitLds<S>::kWords];
    __shared__ __attribute__((aligned(16))) float lds[4][kEx + (kVOut ? 2 * kVoTile : 0) + kSumsLds];
    const int lane = tid_x() & 63, wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6), i16 = lane & 15, g = lane >> 4;
    float* const ex = lds[wave];
    float* const vo = ex + kEx;
    float* const sums = vo + (kVOut ? 2 * kVoTile : 0);
    const SplitScale sc = split_stage_plain<S>(m, w, Clamp ? 1.0 : kNegLog2eD, par_s);
    SplitWeights<S, 2> W;
    {
        h8v kept[1];
        split_load<S, 2>(W, par_s, nullptr, lane, kept);
    }
    const float ak = in_vgpr(act_k_of<kActFold>(m)), neg = in_vgpr(-1.0f), inv = in_vgpr(sc.inv);
    // the first layer's weights of the searched inputs for this lane's units, with the layer's factors
    float w1[C0][Q::kHt][4];
    {
        const double b = split_factors(sc, m.fold_c, 1.0).w1;
#pragma unroll
        for (int c = 0; c < C0; c++)
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int u = unit_of<Q>(ot, 4 * g + r);
                    const float v = (float)((double)w[min(u, Q::kH - 1) * Q::kIn + c] * b);
                    w1[c][ot][r] = u < Q::kH ? v : 0.0f;
                }
    }
    float cw[NT];
#pragma unroll
    for (int r = 0; r < NT; r++) {
        cw[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < NO; c++)
            if ((kVOut ? r : out_at<S>(g, r)) == c) cw[r] = m.cw[c];
    }
    constexpr bool kUnit = UnitCw && (kVOut || NO == 4 * RO);
    const int R = (m.npix + 63) >> 6;
    unsigned long long again = 0;   // rounds that had a NaN
    int n = 0;
    for (int rd = bid_x() * 4 + wave; rd < R; rd += 4 * blocks, n++) {
        const int base = 64 * rd;
        float f[S::kMaxIn];
        {
            const int pr = min(base + lane, m.npix - 1);
            features<S>(m, PlainLatent{ zdec }, pr % m.W, pr / m.W, f);
        }
        float own[C0];      // the lane's own pixel's channels and their grid indices
        int cur_own[C0];
#pragma unroll
        for (int c = 0; c < C0; c++) {
            own[c] = f[c]; cur_own[c] = qat_index(f[c], qat_bits[c]);
            f[c] = 0.0f;
        }
        split_write<S>(f, neg, (u4v*)ex, lane);
        wave_lds_fence();
        float win[4][C0];
        bool bad = false;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float tt[NT];
            const int pr = min(base + 16 * t + i16, m.npix - 1);
#pragma unroll
            for (int r = 0; r < NT; r++) tt[r] = tgt[(size_t)pr * NO + (kVOut ? r : max(out_at<S>(g, r), 0))];
            const h8v b1 = split_read<S>((const u4v*)ex, 16 * t + i16, g);
            f4v s0[Q::kHt];
#pragma unroll
            for (int ot = 0; ot < Q::kHt; ot++) {
                s0[ot] = W.c1[ot];
#pragma unroll
                for (int s = P::kS1 - 1; s >= 0; s--) s0[ot] = mfma_h(W.a1[ot][s], b1, s0[ot]);
            }
#pragma unroll
            for (int c = 0; c < C0; c++) win[t][c] = __int_as_float(__builtin_amdgcn_ds_bpermute((16 * t + i16) << 2, __float_as_int(own[c])));
#pragma unroll
            for (int c = 0; c < C0; c++) {
                const int levels = (1 << qat_bits[c]) - 1;
                const float* gv = grid + qat_bits[c] * 257;
                const int cur = __builtin_amdgcn_ds_bpermute((16 * t + i16) << 2, cur_own[c]);
                f4v sb[Q::kHt];   // without channel c
#pragma unroll
                for (int ot = 0; ot < Q::kHt; ot++) {
                    sb[ot] = s0[ot];
#pragma unroll
                    for (int q = 0; q < C0; q++)
                        if (q != c)
#pragma unroll
                            for (int r = 0; r < 4; r++) sb[ot][r] = __builtin_fmaf(w1[q][ot][r], win[t][q], sb[ot][r]);
                }
                // the running minimum as in qat_round: the current value first, then the others in ascending order, strict <
                float cur_l = 0.0f, best_l = __builtin_inff(), cur_v = 0.0f, best_v = 0.0f;
                for (int kc = 0; kc <= levels; kc += 2) {
                    const float gc[2] = { gv[kc], gv[kc + 1] };
                    float lv[2];
#pragma unroll
                    for (int v = 0; v < 2; v++) {
                        f4v a1[Q::kHt];
#pragma unroll
                        for (int ot = 0; ot < Q::kHt; ot++)
#pragma unroll
                            for (int r = 0; r < 4; r++) a1[ot][r] = __builtin_fmaf(w1[c][ot][r], gc[v], sb[ot][r]);
                        h8v b[P::kB];
                        split_act<S, 2, kActFold>(a1, ak, neg, b);
                        if constexpr (Q::kNL > 1) {
                            f4v a2[Q::kHt];
#pragma unroll
                            for (int ot = 0; ot < Q::kHt; ot++) a2[ot] = split_dot_hidden<S, 2>(W, ot, b);
                            split_act<S, 2, kActFold>(a2, ak, neg, b);
                        }
                        const f4v o = split_dot_out<S, 2>(W, 0, b, W.co);   // (at most 4 outputs: lane group 0 holds them)
                        lv[v] = 0.0f;
#pragma unroll
                        for (int r = 0; r < NT; r++) {
                            const float s = o[r] * inv;
                            if constexpr (Clamp) bad |= !not_nan_bits(s);
                            const float d = out_of<S>(s, Clamp) - tt[r];
                            lv[v] = kUnit ? __builtin_fmaf(d, d, lv[v]) : __builtin_fmaf(cw[r], __fmul_rn(d, d), lv[v]);
                        }
                    }
                    float ls[2];
                    if constexpr (kVOut) {
#pragma unroll
                        for (int v = 0; v < 2; v++) ls[v] = __int_as_float(__builtin_amdgcn_ds_bpermute(i16 << 2, __float_as_int(lv[v])));
                    } else {
                        group_sums(lv[0], lv[1], sums, g, i16, ls[0], ls[1]);
                    }
#pragma unroll
                    for (int v = 0; v < 2; v++) {
                        const float l = ls[v];
                        const bool is_cur = kc + v == cur, better = !is_cur && l < best_l;
                        bad |= !not_nan_bits(l);
                        cur_l = is_cur ? l : cur_l;
                        cur_v = is_cur ? gc[v] : cur_v;
                        best_l = better ? l : best_l;
                        best_v = better ? gc[v] : best_v;
                    }
                }
                win[t][c] = best_l < cur_l ? best_v : cur_v;
            }
        }
        wave_lds_fence();
        if (__builtin_amdgcn_ballot_w64(bad) != 0) {
            again |= 1ull << n;
            continue;
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int p = base + 16 * t + i16;
            if (g == 0 && p < m.npix)
#pragma unroll
                for (int c = 0; c < C0; c++) zdec[m.lv[0].off + (size_t)p * m.lv[0].C + c] = win[t][c];
        }
    }
    if (again == 0) return;
    MfmaWeights<S> F;
    mfma_load<S>(F, w, lane);
    if constexpr (!Clamp) scale_output<S>(F, kNegLog2e);
    scale_hidden<S>(F, fold_scale(m.leak));
    float cw4[4];
#pragma unroll
    for (int r = 0; r < 4; r++) cw4[r] = kVOut ? ((r == 0 && g < NO) ? m.cw[min(g, NO - 1)] : 0.0f) : (r < NT ? cw[r < NT ? r : 0] : 0.0f);
    n = 0;
    for (int rd = bid_x() * 4 + wave; rd < R; rd += 4 * blocks, n++)
        if ((again >> n) & 1ull) qat_round<S, kActFold, Clamp, false>(m, F, ak, cw4, zdec, tgt, qat_bits, grid, 64 * rd, lane, ex, vo, sums);
}

}   // namespace ntc_hip
