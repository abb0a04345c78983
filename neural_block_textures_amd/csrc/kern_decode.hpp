// The full decode (Decoder::decode_full, main.cpp:1712-1718) on the FP32 matrix cores of gfx950, bit for bit the VALU
// kernel's (k_decode): device code only, compiled into libntc_hip.so for the fixed shapes and by hipRTC for others.
//
// v_mfma_f32_16x16x4_f32 adds its four products in order, each step a rounded fused multiply-add (mfma_mlp.hpp), so a chain
// of them is the reference's s = b[j]; s = fma(w[j][i], a[i], s) if its k-steps take the inputs in ascending order. The row
// of a hidden tile that lane group g holds in register r is therefore unit 4 r + g of the tile (dec_unit): k-step 4 t + r of
// the next layer takes register r of tile t, and lane group g's value is input 4 (4 t + r) + g. The activation and the output
// are the VALU kernel's functions.
//
// What bounds it: the matrix instructions (a SIMD does 32 multiply-adds a cycle on them; with a weight in an SGPR, as the
// VALU kernel holds them, a fused multiply-add takes 4.5 cycles for 64) and, where the error is asked for, nothing is
// written: the squared 8-bit differences are summed in the same kernel. A wave loads the weights once and takes rounds of 64
// pixels until the image ends: each lane builds one pixel's features, an exchange through the wave's LDS turns them into four
// 16-pixel tiles.
// The error of four 2048 x 2048 maps (14-64-64-12): decode and error kernels of 925 + 107 us, now one of 573 us (the 96 matrix
// instructions of a tile alone: 375 us; the activations, sigmoids and features of a tile, which do not overlap them, the rest).
#pragma once
#include "kern_valu.hpp"
#include "mfma_mlp.hpp"

namespace ntc_hip {

// Matrix instructions of a 16-pixel tile, every output a row of one output tile.
__host__ __device__ constexpr int decode_mfmas(int nin, int H, int NL) {
    const int ht = (H + 15) / 16, ks = 4 * (ht - 1) + (H - 16 * (ht - 1) + 3) / 4;
    return ht * ((nin + 3) / 4) + (NL - 1) * ht * ks + ks;
}
// The registers it takes (within 4 of the compiler's count for 6 and 14 inputs, 16 to 64 wide, one to six layers): weights and
// biases of every layer, which stay in them, the tiles in flight and the first layer's operands. And the waves per SIMD that
// they leave room for, at most 4.
__host__ __device__ constexpr int decode_regs(int nin, int H, int NL) {
    const int ht = (H + 15) / 16, ks = 4 * (ht - 1) + (H - 16 * (ht - 1) + 3) / 4, ks1 = (nin + 3) / 4;
    return ht * ks1 + 4 * ht + ks + 4 + (NL - 1) * ht * (ks + 4) + 42 + 8 * ks1;
}
__host__ __device__ constexpr int decode_waves(int nin, int H, int NL) {
    const int r = decode_regs(nin, H, NL), w = H > 48 ? 2 : (H > 32 ? 3 : 4);
    return r <= 128 && w > 3 ? 4 : (r <= 168 && w > 2 ? 3 : (r <= 256 ? 2 : 1));
}
// Whether it pays: a matrix instruction takes 32 cycles against about 1.1 of a multiply-add on the VALU (4.5 cycles for 64
// pixels). 16-wide decoders and wider ones do (16: 320 cycles against 450), 17-wide ones do not (their second tile holds one
// unit: 608 against 516). And its registers must fit with two waves or more.
__host__ __device__ constexpr bool decode_pays(int nin, int H, int NL, int nout) {
    return nout <= 16 && NL >= 1 && 32 * decode_mfmas(nin, H, NL) < nin * H + (NL - 1) * H * H + H * nout && decode_waves(nin, H, NL) >= 2;
}
// Whether it also pays for at most 4 outputs as floats on `groups` 256-pixel groups, `fill` of them a full chip: their stores are
// a float a lane, and a full chip hides the VALU kernel's latencies. Below a full chip it does (MI355X, us, VALU -> here: 16-wide
// 256 x 256 9.5 -> 7.8, 24-wide 11.9 -> 9.7); above, where the matrix instructions are a quarter ahead (32-wide 1024 x 1024 60.6 ->
// 55.2, 2048 x 2048 218 -> 188) and not where less (16-wide 27.5 -> 29.3 and 87.8 -> 97.1, 24-wide 41.0 -> 43.5 and 141 -> 149), nor
// on just a full chip (32-wide 512 x 512 21.7 -> 22.9).
__host__ __device__ constexpr bool decode_float_pays(int nin, int H, int NL, int nout, size_t groups, size_t fill) {
    return nout > 4 || groups < fill ||
           (groups >= 2 * fill && 4 * 32 * decode_mfmas(nin, H, NL) <= 3 * (nin * H + (NL - 1) * H * H + H * nout));
}
template <class S, bool = S::kFixed && S::kUniform>
struct DecodeOk { static constexpr bool value = false; };
template <class S>
struct DecodeOk<S, true> { static constexpr bool value = decode_pays(S::kNin, S::kH, S::kNL, S::kNout); };

enum DecodeTo : int { kToFloat = 0, kToBytes = 1, kToError = 2 };

__host__ __device__ constexpr int dec_unit(int ot, int row) { return 16 * ot + 4 * (row & 3) + (row >> 2); }
// 16-pixel tiles evaluated at once, so that enough chains of matrix instructions are independent
constexpr int dec_tiles(int ht) { return ht == 1 ? 4 : (ht == 2 ? 2 : 1); }

template <class S>
struct DecWeights {
    static constexpr int kHt = (S::kH + 15) / 16, kKs1 = (S::kNin + 3) / 4, kLast = (S::kH - 16 * (kHt - 1) + 3) / 4,
                         kKsH = 4 * (kHt - 1) + kLast, kDeep = S::kNL > 1 ? S::kNL - 1 : 1, kOut = (S::kNout + 3) / 4;
    static constexpr int regs(int ot) { return ot == kHt - 1 ? kLast : 4; }
    float a1[kHt][kKs1];
    f4v c1[kHt];
    float ah[kDeep][kHt][kKsH];
    f4v ch[kDeep][kHt];
    float ao[kKsH];   // row 4 g + r of the output tile: output kOut g + r, r < kOut
    f4v co;

    __device__ __forceinline__ void load(const float* __restrict__ w, int i16, int g) {
        constexpr int NIN = S::kNin, H = S::kH, NO = S::kNout;
        auto at = [&](bool ok, int k) { const float v = w[k]; return ok ? v : 0.0f; };
#pragma unroll
        for (int ot = 0; ot < kHt; ot++) {
            const int u = dec_unit(ot, i16), uc = min(u, H - 1);
#pragma unroll
            for (int ks = 0; ks < kKs1; ks++) a1[ot][ks] = at(u < H && 4 * ks + g < NIN, uc * NIN + min(4 * ks + g, NIN - 1));
#pragma unroll
            for (int r = 0; r < 4; r++) c1[ot][r] = at(dec_unit(ot, 4 * g + r) < H, H * NIN + min(dec_unit(ot, 4 * g + r), H - 1));
        }
        int p = H * NIN + H;
#pragma unroll
        for (int l = 0; l < S::kNL - 1; l++) {
#pragma unroll
            for (int ot = 0; ot < kHt; ot++) {
                const int u = dec_unit(ot, i16), uc = min(u, H - 1);
#pragma unroll
                for (int ks = 0; ks < kKsH; ks++) ah[l][ot][ks] = at(u < H && 4 * ks + g < H, p + uc * H + min(4 * ks + g, H - 1));
#pragma unroll
                for (int r = 0; r < 4; r++)
                    ch[l][ot][r] = at(dec_unit(ot, 4 * g + r) < H, p + H * H + min(dec_unit(ot, 4 * g + r), H - 1));
            }
            p += H * H + H;
        }
        const int row = kOut * (i16 >> 2) + (i16 & 3), rc = min(row, NO - 1);
        const bool live = (i16 & 3) < kOut && row < NO;
#pragma unroll
        for (int ks = 0; ks < kKsH; ks++) ao[ks] = at(live && 4 * ks + g < H, p + rc * H + min(4 * ks + g, H - 1));
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int c = kOut * g + r;
            co[r] = at(r < kOut && c < NO, p + NO * H + min(c, NO - 1));
        }
    }

    // the output pre-activations of U tiles from their first-layer operands
    template <int U>
    __device__ __forceinline__ void forward(const float (&b)[U][kKs1], float leak, f4v (&o)[U]) const {
        float x[U][kKsH];
        f4v acc[U][kHt];
        auto next = [&] {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int ot = 0; ot < kHt; ot++)
#pragma unroll
                    for (int r = 0; r < regs(ot); r++) x[u][4 * ot + r] = activate(acc[u][ot][r], leak);
        };
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int ot = 0; ot < kHt; ot++) acc[u][ot] = c1[ot];
#pragma unroll
        for (int ks = 0; ks < kKs1; ks++)
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int ot = 0; ot < kHt; ot++) acc[u][ot] = mfma4(a1[ot][ks], b[u][ks], acc[u][ot]);
        next();
#pragma unroll
        for (int l = 0; l < S::kNL - 1; l++) {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int ot = 0; ot < kHt; ot++) acc[u][ot] = ch[l][ot];
#pragma unroll
            for (int ks = 0; ks < kKsH; ks++)
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int ot = 0; ot < kHt; ot++) acc[u][ot] = mfma4(ah[l][ot][ks], x[u][ks], acc[u][ot]);
            next();
        }
#pragma unroll
        for (int u = 0; u < U; u++) o[u] = co;
#pragma unroll
        for (int ks = 0; ks < kKsH; ks++)
#pragma unroll
            for (int u = 0; u < U; u++) o[u] = mfma4(ao[ks], x[u][ks], o[u]);
    }
};

// save_png's rounding: lround of the [0, 1]-clamped value times 255
__device__ __forceinline__ int to_byte(float v) { return (int)roundf(__fmul_rn(fminf(1.0f, fmaxf(0.0f, v)), 255.0f)); }

// Pixels 0 .. ew eh - 1 of the extent (raster order within it) to out: W H nout floats (kToFloat) or bytes (kToBytes), the
// extent then being the image; or four sums of squared 8-bit differences from tgt per block (kToError).
template <class S, int To>
__global__ void __launch_bounds__(kTPB) __attribute__((amdgpu_waves_per_eu(decode_waves(S::kNin, S::kH, S::kNL)))) k_decode_mfma(DevModel m, const float* __restrict__ w, const float* __restrict__ z,
                                                                      const float* __restrict__ tgt, int ew, int eh, void* __restrict__ out) {
    using D = DecWeights<S>;
    constexpr int NO = S::kNout, U = dec_tiles(D::kHt);
    __shared__ __attribute__((aligned(16))) float lds[kTPB / 64][4 * D::kKs1 * 64];
    __shared__ unsigned long long red[kTPB / 64][4];
    const int lane = tid_x() & 63, wave = __builtin_amdgcn_readfirstlane(tid_x() >> 6), i16 = lane & 15, g = lane >> 4;
    float* const tl = lds[wave];
    const int n = ew * eh;
    D W;
    W.load(w, i16, g);
    unsigned sq[D::kOut];   // squared differences of this lane's output registers
#pragma unroll
    for (int r = 0; r < D::kOut; r++) sq[r] = 0u;
    for (int base = (bid_x() * (kTPB / 64) + wave) * 64; base < n; base += (int)gridDim.x * kTPB) {
        float b[4][D::kKs1];
        {
            const int i = min(base + lane, n - 1);
            float f[S::kMaxIn];
            features<S>(m, PlainLatent{ z }, i % ew, i / ew, f);
            tiles_of_n<D::kKs1>(f, b, tl, g, i16);
        }
#pragma unroll
        for (int t0 = 0; t0 < 4; t0 += U) {
            float bu[U][D::kKs1];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int ks = 0; ks < D::kKs1; ks++) bu[u][ks] = b[t0 + u][ks];
            f4v o[U];
            W.template forward<U>(bu, m.leak, o);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = base + 16 * (t0 + u) + i16;
                if (i >= n) continue;
                const size_t p = ew == m.W ? (size_t)i : (size_t)(i / ew) * m.W + i % ew;
#pragma unroll
                for (int r = 0; r < D::kOut; r++) {
                    const int c = D::kOut * g + r;
                    if (c >= NO) continue;
                    const float v = output_of(o[u][r], m.clamp_out);
                    if constexpr (To == kToFloat) ((float*)out)[p * NO + c] = v;
                    else if constexpr (To == kToBytes) ((uint8_t*)out)[p * NO + c] = (uint8_t)to_byte(v);
                    else {
                        const int d = to_byte(v) - to_byte(tgt[p * NO + c]);
                        sq[r] += (unsigned)(d * d);
                    }
                }
            }
        }
    }
    if constexpr (To == kToError) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            unsigned long long v = 0;
#pragma unroll
            for (int r = 0; r < D::kOut; r++)
                if ((D::kOut * g + r) / 3 == t) v += sq[r];
            for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s, 64);
            if (lane == 0) red[wave][t] = v;
        }
        __syncthreads();
        if (tid_x() < 4) {
            unsigned long long v = 0;
            for (int q = 0; q < kTPB / 64; q++) v += red[q][tid_x()];
            ((unsigned long long*)out)[(size_t)bid_x() * 4 + tid_x()] = v;
        }
    }
}

}   // namespace ntc_hip
