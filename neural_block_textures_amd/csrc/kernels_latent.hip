// Latent-side kernels of the gfx950 ES backend: the latent Gaussians of one step, the antithetic
// pair evaluation over the full image, the footprint gather that turns per-pixel loss differences
// into the latent gradient, and the exhaustive --qat selector search.
//
// Reference semantics (main.cpp): LatentTrainer::step_impl 1974-2044 (perturb texels, decode_err
// twice, raster-order scatter into the distinct taps, grad += w * eps), dct_rate_pass 1935-1952,
// qat_search 2088-2139.
#include "kern_valu.hpp"
#include "mfma_mlp.hpp"
#include "jit.hpp"
#include "shapes.hpp"
#include "trainer_impl.hpp"

namespace ntc_hip {


__device__ __forceinline__ int level_of(const DevModel& m, long long i) {
    int l = 0;
    for (int q = 1; q < m.nlev; q++) if (i >= m.lv[q].off) l = q;
    return l;
}

// eps[k][i] = gauss(seed, NS_LAT, step, k0 + k, i) for the ES-perturbed levels (the other levels' entries are
// never read and are left as they are): the group of pairs k0 .. k0 + gridDim.y - 1 of a latent step; the
// first group's pair-0 threads also clear the latent gradient. Grid: latent entries x pairs (blockIdx.y = k).
__global__ void __launch_bounds__(kTPB) k_lat_eps(NoiseFix nt, DevModel m, uint64_t seed, uint32_t step, unsigned mask, int k0,
                                                 float* __restrict__ eps, float* __restrict__ zgrad) {
    const long long i = (long long)blockIdx.x * kTPB + threadIdx.x;
    if (i >= m.nz) return;
    const int k = blockIdx.y;
    if (k0 + k == 0) zgrad[i] = 0.0f;
    const int l = level_of(m, i);
    if ((mask >> l) & 1u) eps[(size_t)k * m.nz + i] = gauss_at(nt, noise_head(seed, NS_LAT, step, (uint32_t)(k0 + k)), (uint64_t)i);
}

// Footprint gather per level (the gather form of the reference's raster-order scatter,
// main.cpp:2011-2037): the loss difference a texel's taps collect from pair k is the sum of dpix[k]
// over the pixel rectangle that reads the texel, in raster order (the rectangle comes from the host's
// range table, built with the same tap arithmetic); then grad += (d * scale) * eps per channel, pair
// after pair. With the --dct-lambda rate term, level 0 also receives (rate_scale * dbits) * scale * eps
// right after each pair's mse term. A texel's gradient is final when its block has added its pairs (one block owns
// it), so with `adam` the block also takes the texel's Adam step (the latent ES step's
// update, main.cpp:2036-2037), and with zq_copy writes the new value to the decode copy too (a level that is neither
// --qes nor DCT coded, where the snap would copy it). With `first` the gradient starts from zero rather than from grad
// (the step's first group of pairs).
//
// A block has one to four waves (four pairs a wave: as many as the step's pairs fill) and takes 16 neighbouring texels of a
// row: lane group q of a wave sums pair q of the wave's four, lane j of it texel j. The sum is one chain of rounded adds, so
// its length is fixed; what can be fast is what feeds it.
// kNarrow (rectangles of at most 16 columns): each lane reads its run from memory, the 16 lanes of a pair a few lines.
// Wider ones, kRows: texels lie further apart than a line, so a wave copies its pairs' rows to LDS, whole lines at a time and the
// next row in flight while one is added, and every lane reads its texel's run from there; with four waves all 16 pairs' chains
// run at once. Levels of 128 x 128 x 8 and 32 x 32 x 4 under 512 x 512 pixels, 16 pairs (MI355X): 190 -> 78 us (104 with the four rows a multiple of 64
// floats apart: sixteen lanes on a bank).
// Wider ones with at most four pairs, kRuns: one wave's rows to LDS take longer than each lane's own runs of 16 from memory, the
// next run in flight while one is added. The same levels, 1, 2, 4 and 8 pairs: 43, 46, 53 and 99 us against 57, 57, 58 and 63.
// kUnit (a level 0 of one pixel per texel): a thread per texel, its pairs in order; a 512 x 512 x 1 plane and a 128 x 128 x 4
// level, 4 pairs: 31 -> 23 us.
//
// Blocks past the gather's own (blockIdx.x >= start[n]) draw the next latent step's Gaussians for the perturbed
// levels (the entries lo .. hi - 1 whose level is in `mask`; block d = pair d / eb, entries lo + 2 blockDim (d % eb) ..):
// the values k_lat_eps would draw for step next_step, written to eps_next. They run beside the gather's blocks,
// so the next step needs no draw launch of its own.
//
// One launch gathers every perturbed level of the step (GatherLevels: blocks start[i] .. start[i + 1] - 1 take level
// lv[i]); the rate term goes to level 0, and zq_copy[i] (or null) is level lv[i]'s decode copy.
constexpr int kGatherTex = 16, kGatherPairs = 4, kGatherWaves = 4, kGatherRun = 32, kWideCols = 320,
              kWideRow = kWideCols + 4;   // (the four pairs' rows in LDS: texels 16 columns apart then share a bank four at a time, not sixteen)
enum GatherMode : int { kNarrow = 0, kUnit = 1, kRows = 2, kRuns = 3 };
struct LatAhead {
    NoiseFix nt; uint64_t seed; uint32_t next_step; unsigned mask;
    float* eps_next; int eb; long long lo, hi;
};
struct GatherLevels {
    int n;
    int lv[kMaxLevels];
    int start[kMaxLevels + 1];
    int mode[kMaxLevels];
    float* zq_copy[kMaxLevels];
};
// Wide: kRows or kRuns if a level of the launch is, else kNarrow. Waves: a block's most. Steps of at most four pairs, which need
// one, are compiled for one (barriers and the wave's index go: levels of 128 x 128 x 8 and 32 x 32 x 4 under 512 x 512 pixels, 4
// pairs, 56.2 -> 54.7 us). The loop over pairs in `channel` is not unrolled: by four it took 104 scalar registers, which leave 7
// waves a SIMD for 8 (1024 x 1024 x 4 and 256 x 256 x 8 under 2048 x 2048 pixels, 4 pairs, 381 -> 376 us).
template <int Wide, int Waves>
__global__ void __launch_bounds__(64 * Waves) k_lat_gather(DevModel m, GatherLevels G, int K, float scale,
                                                                  const float* __restrict__ dpix,
                                                                  const float* __restrict__ eps, const int* __restrict__ ranges,
                                                                  int rate0, float rate_scale, int dct_bw, int dct_n,
                                                                  const int32_t* __restrict__ dbits, float* __restrict__ grad,
                                                                  int first, int adam, float* __restrict__ z, float* __restrict__ zm,
                                                                  float* __restrict__ zv, float lr, float c1, float c2, LatAhead ah) {
    const int threads = Waves == 1 ? 64 : (int)blockDim.x;
    if ((int)blockIdx.x >= G.start[G.n]) {   // a draw-ahead block (uniform: the whole block returns here)
        const int d = (int)blockIdx.x - G.start[G.n], k = d / ah.eb;
        const uint64_t head = noise_head(ah.seed, NS_LAT, ah.next_step, (uint32_t)k);
        const long long i0 = ah.lo + (long long)(d - k * ah.eb) * 2 * threads, i1 = min(ah.hi, i0 + 2 * threads);
        for (long long i = i0 + threadIdx.x; i < i1; i += threads)
            if ((ah.mask >> level_of(m, i)) & 1u) ah.eps_next[(size_t)k * m.nz + i] = gauss_at(ah.nt, head, (uint64_t)i);
        return;
    }
    __shared__ float dsum[Waves * kGatherPairs][kGatherTex];
    extern __shared__ float stage_s[];   // with a level of kRows: kGatherPairs x kWideRow floats per wave
    int li = 0;   // this block's level (uniform)
    while (li + 1 < G.n && (int)blockIdx.x >= G.start[li + 1]) li++;
    const int level = G.lv[li], blk0 = (int)blockIdx.x - G.start[li];
    const DevLevel& L = m.lv[level];
    const int rate = rate0 && level == 0;
    float* const zq_copy = G.zq_copy[li];
    // the pairs k0 .. k0 + kn - 1 (their sums d(k)) on channel c of texel (tx, ty), after the gradient so far; after the last
    // pair the channel's Adam step
    auto channel = [&](int tx, int ty, int c, int k0, int kn, auto d) {
        const size_t i = (size_t)(L.off + ((long long)ty * L.W + tx) * L.C + c);
        const int blk = (ty / 8) * dct_bw + tx / 8;
        float gc = (first && k0 == 0) ? 0.0f : grad[i];
        for (int kk = 0; kk < kn; kk++) {
            const float ei = eps[(size_t)(k0 + kk) * m.nz + i];
            gc = __builtin_fmaf(d(kk) * scale, ei, gc);
            if (rate) {
                const int32_t db = dbits[(size_t)(k0 + kk) * dct_n + (size_t)blk * L.C + c];
                gc = __builtin_fmaf(__fmul_rn(__fmul_rn(rate_scale, (float)db), scale), ei, gc);
            }
        }
        grad[i] = gc;
        if (adam && k0 + kn >= K) {
            adam_at(z, zm, zv, i, gc, lr, c1, c2);
            if (zq_copy) zq_copy[i] = z[i];   // a level the decode copy takes as it is
        }
    };
    if (G.mode[li] == kUnit) {   // a thread per texel; a sum of one value (from +0, as the longer ones)
        const int t = blk0 * threads + (int)threadIdx.x;
        if (t >= L.W * L.H) return;
        for (int c = 0; c < L.C; c++)
            channel(t % L.W, t / L.W, c, 0, K, [&](int kk) { return 0.0f + dpix[(size_t)kk * m.npix + t]; });
        return;
    }
    const int lane = threadIdx.x & 63, wave = Waves == 1 ? 0 : threadIdx.x >> 6, j = lane % kGatherTex, q = lane / kGatherTex;
    const int tiles = (L.W + kGatherTex - 1) / kGatherTex, ty = blk0 / tiles, tx = (blk0 - ty * tiles) * kGatherTex + j;
    const bool live = tx < L.W;
    const int* R = ranges + L.rng;
    const int y0 = R[2 * L.W + ty], y1 = R[2 * L.W + L.H + ty];
    const int x0 = live ? R[tx] : m.W, x1 = live ? R[L.W + tx] : 0;   // (a texel that no pixel reads has x0 >= x1)
    const int round = kGatherPairs * (threads >> 6);
    for (int k0 = 0; k0 < K; k0 += round) {
        const int kw = k0 + kGatherPairs * wave, k = kw + q;   // this wave's first pair, this lane's
        float d = 0.0f;
        if (Wide == kNarrow || G.mode[li] == kNarrow) {
            if (k < K && x0 < x1 && y0 < y1) {
                // the rectangle's values in raster order, loaded in groups of kGatherRun across row ends and then added in
                // order (the loads of a group overlap; the sum stays one chain). A slot past the rectangle's end adds +0, which
                // leaves the sum as it is: the sum starts at +0 and a rounded sum is -0 only when both operands
                // are, so it is never -0.
                const float* dp = dpix + (size_t)k * m.npix;
                const int fw = x1 - x0, n = fw * (y1 - y0);
                if (n == 1) {
                    d += dp[(size_t)y0 * m.W + x0];
                } else {
                    int row = y0, col = 0;   // position of the group's first slot
                    for (int s = 0; s < n; s += kGatherRun) {
                        float v[kGatherRun];
                        int r = row, cc = col;
#pragma unroll
                        for (int i = 0; i < kGatherRun; i++) {
                            v[i] = s + i < n ? dp[(size_t)r * m.W + x0 + cc] : 0.0f;
                            if (++cc == fw) { cc = 0; r++; }
                        }
                        row = r; col = cc;
#pragma unroll
                        for (int i = 0; i < kGatherRun; i++) d += v[i];
                    }
                }
            }
        } else if constexpr (Wide == kRuns) {
            if (k < K && x0 < x1 && y0 < y1) {
                // runs of 16 in raster order (a row's last run padded with +0), two buffers
                const float* dp = dpix + (size_t)k * m.npix;
                float va[16], vb[16];
                auto load_run = [&](float (&v)[16], int py, int px) {
                    const float* rw = dp + (size_t)py * m.W;
#pragma unroll
                    for (int i = 0; i < 16; i++) v[i] = px + i < x1 ? rw[px + i] : 0.0f;
                };
                auto step = [&](int& py, int& px) { px += 16; if (px >= x1) { px = x0; py++; } };
                int py = y0, px = x0;
                load_run(va, py, px);
                while (true) {
                    step(py, px);
                    if (py < y1) load_run(vb, py, px);
#pragma unroll
                    for (int i = 0; i < 16; i++) d += va[i];
                    if (py >= y1) break;
                    step(py, px);
                    if (py < y1) load_run(va, py, px);
#pragma unroll
                    for (int i = 0; i < 16; i++) d += vb[i];
                    if (py >= y1) break;
                }
            }
        } else if (kw < K) {
            // the columns under the tile's texels
            int xa = x0 < x1 ? x0 : m.W, xb = x0 < x1 ? x1 : 0;
            for (int o = 8; o > 0; o >>= 1) { xa = min(xa, __shfl_xor(xa, o, 64)); xb = max(xb, __shfl_xor(xb, o, 64)); }
            xa = __builtin_amdgcn_readfirstlane(xa); xb = __builtin_amdgcn_readfirstlane(xb);
            // kWideCols columns of a row of the wave's pairs at a time (a step), in raster order, kAhead steps in flight; what
            // lies past the columns asked for is copied too (buffer loads: past the image's end they read 0), never added
            constexpr int kAhead = 3, kPer = kWideCols / 64;
            float* const st = stage_s + wave * kGatherPairs * kWideRow;
            const int wide = max(0, xb - xa), per_row = (wide + kWideCols - 1) / kWideCols, steps = per_row * max(0, y1 - y0);
            float v[kAhead][kGatherPairs][kPer];
            int lc = xa, ly = y0;   // the next step to load
            auto load = [&](float (&b)[kGatherPairs][kPer]) {
                const uint32_t at = 4u * ((uint32_t)ly * (uint32_t)m.W + (uint32_t)lc);
#pragma unroll
                for (int p = 0; p < kGatherPairs; p++) {
                    const __amdgpu_buffer_rsrc_t rd = buffer_of(dpix + (size_t)min(kw + p, K - 1) * m.npix, 4u * (uint32_t)m.npix);
#pragma unroll
                    for (int s = 0; s < kPer; s++) b[p][s] = buffer_f32(rd, 4u * (uint32_t)(lane + 64 * s), at);
                }
                lc += kWideCols;
                if (lc >= xb) { lc = xa; ly++; }
            };
#pragma unroll
            for (int b = 0; b < kAhead; b++) if (b < steps) load(v[b]);
            int cs = xa;
            for (int n = 0; n < steps; n += kAhead)
#pragma unroll
                for (int b = 0; b < kAhead; b++) {
                    if (n + b >= steps) break;
#pragma unroll
                    for (int p = 0; p < kGatherPairs; p++)
#pragma unroll
                        for (int s = 0; s < kPer; s++) st[p * kWideRow + lane + 64 * s] = v[b][p][s];
                    wave_lds_fence();
                    if (n + b + kAhead < steps) load(v[b]);
                    const int c0 = max(x0, cs), cnt = min(x1, cs + kWideCols) - c0;
                    const float* run = st + q * kWideRow + (c0 - cs);
                    int s = 0;
                    for (; s + 16 <= cnt; s += 16) {
                        float a[16];
#pragma unroll
                        for (int i = 0; i < 16; i++) a[i] = run[s + i];
#pragma unroll
                        for (int i = 0; i < 16; i++) d += a[i];
                    }
                    for (; s < cnt; s++) d += run[s];
                    wave_lds_fence();
                    cs += kWideCols;
                    if (cs >= xb) cs = xa;
                }
        }
        dsum[kGatherPairs * wave + q][j] = d;
        __syncthreads();
        // the round's pairs in order on every channel of the texel (thread (wave, q) takes channels 4 wave + q, + round, ...)
        if (live)
            for (int c = kGatherPairs * wave + q; c < L.C; c += round)
                channel(tx, ty, c, k0, min(K - k0, round), [&](int kk) { return dsum[kk][j]; });
        __syncthreads();
    }
}

// ---------------------------------------------------------------- launchers
void launch_lat_eps(Impl& I, int k0, int K, unsigned mask) {
    ProfScope ps(I, "lat_eps");
    hipLaunchKernelGGL(k_lat_eps, dim3(blocks_for(I.nz, kTPB), K), dim3(kTPB), 0, I.stream, I.noise, I.dm, I.d.seed,
                       (uint32_t)I.lat_step_no, mask, k0, I.eps_lat, I.zgrad);
    NTC_CHECK(hipGetLastError());
}

void launch_lat_pair_valu(Impl& I, int K, float sigma, unsigned mask) {
    if (I.jit) {
        jit_launch(k_lat_pair<ShapeDefault>, I, "k_lat_pair", "", dim3(blocks_for(I.npix, kTPB), K), dim3(kTPB), 0, I.dm, I.w, I.zdec,
                   I.eps_lat, I.tgt, sigma, mask, I.dpix);
    } else dispatch_shape(I.dm, [&](auto s) {
        using S = decltype(s);
        hipLaunchKernelGGL(k_lat_pair<S>, dim3(blocks_for(I.npix, kTPB), K), dim3(kTPB), 0, I.stream, I.dm, I.w, I.zdec, I.eps_lat,
                           I.tgt, sigma, mask, I.dpix);
    });
    NTC_CHECK(hipGetLastError());
}

void launch_lat_gather(Impl& I, unsigned mask, int k0, int K, float scale, bool rate, float lr, int t, int ahead_K, float* zq_rest) {
    const float c1 = t > 0 ? 1.0f - powf(0.9f, (float)t) : 1.0f, c2 = t > 0 ? 1.0f - powf(0.999f, (float)t) : 1.0f;
    GatherLevels G{};
    size_t grid = 0;
    int wide = kNarrow;
    const int threads = 64 * std::min(kGatherWaves, (K + kGatherPairs - 1) / kGatherPairs);
    auto mode = [&](int l) { return l == 0 && I.lv0_unit_cells ? kUnit : (I.lv_cols[l] > 16 ? (K > kGatherPairs ? kRows : kRuns) : kNarrow); };
    for (int pass = 0; pass < 2; pass++)   // the wide levels' blocks first: they take longest
        for (int l = 0; l < I.d.nlev; l++)
            if (((mask >> l) & 1u) && (mode(l) >= kRows) == (pass == 0)) {
                G.lv[G.n] = l;
                G.start[G.n] = (int)grid;
                G.mode[G.n] = mode(l);
                if (pass == 0) wide = mode(l);
                G.zq_copy[G.n] = l > 0 ? zq_rest : nullptr;
                grid += mode(l) == kUnit ? (size_t)blocks_for((size_t)I.d.lv[l].W * I.d.lv[l].H, threads)
                                         : (size_t)blocks_for((size_t)I.d.lv[l].W, kGatherTex) * (size_t)I.d.lv[l].H;
                G.n++;
            }
    G.start[G.n] = (int)grid;
    LatAhead ah{};
    ah.eb = 1;
    if (ahead_K > 0) {   // the next step's Gaussians: the range of entries the perturbed levels span
        ah.nt = I.noise; ah.seed = I.d.seed; ah.next_step = (uint32_t)(I.lat_step_no + 1); ah.mask = mask; ah.eps_next = I.eps_ahead;
        ah.lo = (long long)I.nz; ah.hi = 0;
        for (int l = 0; l < I.d.nlev; l++)
            if ((mask >> l) & 1u) {
                ah.lo = std::min<long long>(ah.lo, I.dm.lv[l].off);
                ah.hi = std::max<long long>(ah.hi, I.dm.lv[l].off + (long long)I.d.lv[l].W * I.d.lv[l].H * I.d.lv[l].C);
            }
        ah.eb = blocks_for((size_t)(ah.hi - ah.lo), 2 * threads);
        grid += (size_t)ah.eb * (size_t)ahead_K;
    }
    if (grid > 0x7fffffff) {
        fprintf(stderr, "ntc_hip backend: latent gather launch of %zu blocks\n", grid);
        exit(1);
    }
    ProfScope ps(I, "lat_gather");
    auto* const kern = wide == kRows   ? k_lat_gather<kRows, kGatherWaves>
                       : wide == kRuns ? k_lat_gather<kRuns, 1>
                       : threads == 64 ? k_lat_gather<kNarrow, 1>
                                       : k_lat_gather<kNarrow, kGatherWaves>;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads),
                       wide == kRows ? (size_t)threads / 64 * kGatherPairs * kWideRow * sizeof(float) : 0, I.stream, I.dm, G, K,
                       scale, I.dpix, I.eps_lat,
                       I.ranges, rate ? 1 : 0, I.ddct.rate_scale, I.ddct.BW, I.ddct.n, rate ? I.dct_dbits + (size_t)k0 * I.ddct.n : nullptr,
                       I.zgrad, k0 == 0 ? 1 : 0, t > 0 ? 1 : 0, I.z, I.zm,
                       I.zv, lr, c1, c2, ah);
    NTC_CHECK(hipGetLastError());
}

void launch_qat_search(Impl& I) {
    const size_t ntx = (size_t)I.d.lv[0].W * I.d.lv[0].H;
    ProfScope ps(I, "qat_search");
    if (qat_on_matrix_cores(I)) {
        launch_qat_mfma(I);
        return;
    }
    if (I.jit) {
        jit_launch(k_qat_search<ShapeDefault>, I, "k_qat_search", "", dim3(blocks_for(ntx, kTPB)), dim3(kTPB), 0, I.dm, I.w, I.zdec,
                   I.tgt, I.ranges, I.qat_bits, I.qat_grid);
    } else dispatch_shape(I.dm, [&](auto s) {
        using S = decltype(s);
        hipLaunchKernelGGL(k_qat_search<S>, dim3(blocks_for(ntx, kTPB)), dim3(kTPB), 0, I.stream, I.dm, I.w, I.zdec, I.tgt, I.ranges,
                           I.qat_bits, I.qat_grid);
    });
    NTC_CHECK(hipGetLastError());
}

}   // namespace ntc_hip
