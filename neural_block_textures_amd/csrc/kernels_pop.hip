// Launchers of the matrix-core kernels of kern_pop.hpp.
#include "jit.hpp"
#include "kern_pop.hpp"
#include "shapes.hpp"
#include "trainer_impl.hpp"

namespace ntc_hip {

// every channel weight of the model is 1
static bool unit_cw(const Impl& I) {
    bool unit = true;
    for (int c = 0; c < I.dm.nout; c++) unit = unit && I.dm.cw[c] == 1.0f;
    return unit;
}

bool qat_on_matrix_cores(const Impl& I) {
    if (!I.lv0_unit_cells || I.valu_only) return false;
    if (I.jit) return jit_mfma(I);
    bool ok = false;
    dispatch_shape(I.dm, [&](auto s) { ok = MfmaShape<decltype(s)>::kOk; });
    return ok;
}

// the population and latent-pair evaluations on the matrix cores take 0 <= leak <= 1 (kActFold, kActMax)
bool pop_on_matrix_cores(const Impl& I) {
    if (I.valu_only || !(I.dm.leak >= 0.0f && I.dm.leak <= 1.0f)) return false;
    if (I.jit) return jit_mfma(I);
    bool ok = false;
    dispatch_shape(I.dm, [&](auto s) { ok = MfmaShape<decltype(s)>::kOk; });
    return ok;
}

#ifndef NTC_POP_MIN_BLOCKS
#define NTC_POP_MIN_BLOCKS 2048
#endif
int pop_chunk(const Impl& I, int pairs, int M) {
    if (pop_on_matrix_cores(I)) {
        // at least NTC_POP_MIN_BLOCKS blocks where the population allows, at least 256 slots per chunk
        const int want = std::max(1, std::min((NTC_POP_MIN_BLOCKS + pairs - 1) / pairs, M / 256));
        const int chunk = ((M + want - 1) / want + 15) & ~15;
        return std::max(chunk, 16);
    }
    return std::min(M, 1024);
}

template <class S, int Act, int From>
static void launch_pop_mfma(Impl& I, const PopSource& src, int pairs, int M, int chunk, int chunks) {
    auto kern = I.dm.clamp_out ? k_pop_mfma<S, Act, true, From> : k_pop_mfma<S, Act, false, From>;
    launch_timed(kern, I, dim3(pairs, chunks), dim3(64 * kPopWaves), 0, I.dm, src, M, I.Mcap, chunk, chunks, I.feat, I.btgt, I.part);
}

static void check_pop_launch(const Impl& I, int pairs, int chunk, int chunks) {
    if ((size_t)2 * pairs * chunks > I.part_cap) {
        fprintf(stderr, "ntc_hip backend: population evaluation needs %d partial sums, buffer holds %zu\n", 2 * pairs * chunks,
                I.part_cap);
        exit(1);
    }
    if (chunk % 16 != 0) {
        fprintf(stderr, "ntc_hip backend: matrix-core population evaluation needs 16-slot chunks (got %d)\n", chunk);
        exit(1);
    }
}

template <int From>
static void launch_pop_matrix(Impl& I, const PopSource& src, int pairs, int M, int chunk, int chunks) {
    if (I.jit) {   // the same choice of activation as below
        const int act = From == kSets ? kActMax : kActFold;
        jit_launch(k_pop_mfma<ShapeMaterial, kActFold, false, From>, I, "k_pop_mfma",
                   std::to_string(act) + (I.dm.clamp_out ? ", true, " : ", false, ") + std::to_string(From), dim3(pairs, chunks),
                   dim3(64 * kPopWaves), 0, I.dm, src, M, I.Mcap, chunk, chunks, I.feat, I.btgt, I.part);
        NTC_CHECK(hipGetLastError());
        return;
    }
    dispatch_shape(I.dm, [&](auto s) {
        using S = decltype(s);
        if constexpr (MfmaShape<S>::kOk) {
            // central differences compare members one weight apart (w_j +- h): their activations are the
            // reference's bit for bit; the ES members (w +- sigma eps) take the one-instruction folded form
            if constexpr (From == kSets) launch_pop_mfma<S, kActMax, From>(I, src, pairs, M, chunk, chunks);
            else launch_pop_mfma<S, kActFold, From>(I, src, pairs, M, chunk, chunks);
        }
    });
    NTC_CHECK(hipGetLastError());
}

template <int From>
static void launch_pop_split(Impl& I, const PopSource& src, int N, int M, int chunk, int chunks);

void launch_pop_eval(Impl& I, int pairs, int M, int chunk, int chunks) {
    ProfScope ps(I, "pop_eval", pop_on_matrix_cores(I));   // the matrix path is one launch
    if (!pop_on_matrix_cores(I)) {
        if ((size_t)2 * pairs * chunks > I.part_cap) {
            fprintf(stderr, "ntc_hip backend: population evaluation needs %d partial sums, buffer holds %zu\n", 2 * pairs * chunks,
                    I.part_cap);
            exit(1);
        }
        launch_pop_eval_valu(I, pairs, M, chunk, chunks);
        return;
    }
    check_pop_launch(I, pairs, chunk, chunks);
    PopSource src{};
    src.wsets = I.wsets;
    launch_pop_matrix<kSets>(I, src, pairs, M, chunk, chunks);
}

// the central-difference population (P + 1 pairs) of a model on the split kernel, from the weights and h
void launch_pop_eval_fd(Impl& I, float h, int M, int chunk, int chunks) {
    check_pop_launch(I, I.P + 1, chunk, chunks);
    PopSource src{};
    src.w0 = I.w; src.sigma = h;
    ProfScope ps(I, "pop_eval", true);
    launch_pop_split<kSets>(I, src, I.P + 1, M, chunk, chunks);
}

// The split population kernel takes every step that the matrix cores take, of the shapes it has an operand layout for
// (split_pays) and minibatches its offsets hold. Against the 32-bit kernel on the MI355X: see k_pop_split. NTC_HIP_POP_PAIR=0
// (read at init) keeps k_pop_mfma for the population, and k_lat_pair_mfma for the latent pairs of the listed shapes: the 32-bit
// kernels that the tests compare the split ones with.
bool pop_split_fits(const Impl& I) {
    const char* env = getenv("NTC_HIP_POP_PAIR");
    // (its arrays are read through 32-bit offsets: for 9 to 12 inputs 67 million slots, where k_pop_mfma's hold 89 million)
    const uint64_t slots = (uint64_t)I.Mcap + kSplitSlack, most = (uint64_t)1 << 32;
    const bool fits = slots * 4u * split_inputs(I.dm.nin) < most && slots * 4u * split_targets(I.dm.nout) < most;
    return !(env && env[0] == '0') && split_pays(I.dm.nin, I.dm.nl) && fits;
}
bool pop_split_possible(const Impl& I) { return pop_on_matrix_cores(I) && pop_split_fits(I); }
bool pop_split_step(const Impl& I) { return I.pop_split && pop_on_matrix_cores(I); }

template <int From>
static void launch_pop_split(Impl& I, const PopSource& src, int N, int M, int chunk, int chunks) {
    const bool unit = unit_cw(I);
    const SplitIn in{ (const u4v*)I.sfeat, I.stgt, I.sscale };
    if (I.jit) {
        jit_launch(k_pop_split<ShapeMaterial, false, From, false>, I, "k_pop_split",
                   std::string(I.dm.clamp_out ? "true, " : "false, ") + std::to_string(From) + ", false", dim3(N, chunks), dim3(64 * kPopWaves), 0,
                   I.dm, src, M, I.Mcap, chunk, chunks, in, (const float*)I.feat, I.part);
        NTC_CHECK(hipGetLastError());
        return;
    }
    dispatch_shape(I.dm, [&](auto s) {
        using S = decltype(s);
        if constexpr (SplitShape<S>::kOk) {
            auto kern = I.dm.clamp_out ? k_pop_split<S, true, From, false>
                                       : (unit ? k_pop_split<S, false, From, true> : k_pop_split<S, false, From, false>);
            launch_timed(kern, I, dim3(N, chunks), dim3(64 * kPopWaves), 0, I.dm, src, M, I.Mcap, chunk, chunks, in, (const float*)I.feat,
                         I.part);
        }
    });
    NTC_CHECK(hipGetLastError());
}

void launch_pop_eval_es(Impl& I, int it, float sigma, int N, int M, int chunk, int chunks) {
    check_pop_launch(I, N, chunk, chunks);
    PopSource src{};
    src.nt = I.noise; src.seed = I.d.seed; src.step = (uint32_t)it; src.sigma = sigma;
    src.w0 = I.w; src.eps = I.eps_mlp;
    ProfScope ps(I, "pop_eval", true);
    if (pop_split_step(I)) {
        if (pop_reads_eps(chunks)) launch_pop_split<kReadEps>(I, src, N, M, chunk, chunks);
        else launch_pop_split<kDraw>(I, src, N, M, chunk, chunks);
        return;
    }
    if (pop_reads_eps(chunks)) launch_pop_matrix<kReadEps>(I, src, N, M, chunk, chunks);   // drawn by the minibatch launch
    else launch_pop_matrix<kDraw>(I, src, N, M, chunk, chunks);
}

// rounds per wave of the latent pair kernel: lat_rounds_of(nin) (the shape's most; the compiled shape has
// nin inputs), one where two would leave the launch under 2048 blocks. A count above the compiled kernel's
// would leave pixels of every block unevaluated: refused.
static int lat_rounds_for(const Impl& I, int most, int K) {
    if (most < 1 || most > lat_rounds_of(I.dm.nin)) {
        fprintf(stderr, "ntc_hip backend: latent pair launch with %d rounds for a %d-input model (at most %d)\n", most, I.dm.nin,
                lat_rounds_of(I.dm.nin));
        exit(1);
    }
    if (most > 1 && (size_t)((I.npix + 511) / 512) * (size_t)K < 2048) return 1;
    return most;
}

bool lat_pair_on_matrix_cores(const Impl& I) { return pop_on_matrix_cores(I); }

// k_lat_split for the models whose population is split, and for every shape compiled at init that it takes (no other
// latent pair kernel is compiled for those); k_lat_pair_mfma for the rest, which in a default run are shapes compiled at
// init, and with NTC_HIP_POP_PAIR=0 the listed ones.
bool lat_split_step(const Impl& I) { return lat_pair_on_matrix_cores(I) && split_pays(I.dm.nin, I.dm.nl) && (I.jit || I.pop_split); }
// k_qat_split for the shapes it pays for and 0 <= leak <= 1, whatever NTC_HIP_POP_PAIR is; k_qat_mfma for the rest
bool qat_split_step(const Impl& I) {
    return qat_on_matrix_cores(I) && split_qat_pays(I.dm.nin, I.dm.nl, I.dm.nout) && I.dm.leak >= 0.0f && I.dm.leak <= 1.0f;
}

void launch_lat_pair(Impl& I, int K, float sigma, unsigned mask) {
    ProfScope ps(I, "lat_pair");
    if (!lat_pair_on_matrix_cores(I)) {
        launch_lat_pair_valu(I, K, sigma, mask);
        return;
    }
    if (lat_split_step(I)) {
        // as many blocks as fit the chip, or as 64-pixel rounds fill
        const size_t rounds = (I.npix + 63) / 64 * (size_t)K;
        const unsigned blocks = (unsigned)std::min<size_t>((size_t)I.cus * split_waves(I.dm.nin, I.dm.hidden[0], I.dm.nout), (rounds + 3) / 4);
        if (I.jit) {
            jit_launch(k_lat_split<ShapeMaterial, false, false>, I, "k_lat_split", I.dm.clamp_out ? "true, false" : "false, false", dim3(blocks),
                       dim3(256), 0, I.dm, I.w, I.zdec, I.eps_lat, I.tgt, sigma, mask, I.dpix, K, (int)blocks);
        } else dispatch_shape(I.dm, [&](auto s) {
            using S = decltype(s);
            if constexpr (SplitShape<S>::kOk) {
                auto kern = I.dm.clamp_out ? k_lat_split<S, true, false> : (unit_cw(I) ? k_lat_split<S, false, true> : k_lat_split<S, false, false>);
                hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, I.stream, I.dm, I.w, I.zdec, I.eps_lat, I.tgt, sigma, mask, I.dpix, K,
                                   (int)blocks);
            }
        });
        NTC_CHECK(hipGetLastError());
        return;
    }
    if (I.jit) {
        const int rounds = lat_rounds_for(I, lat_rounds_of(I.dm.nin), K), pix = 256 * rounds;
        jit_launch(k_lat_pair_mfma<ShapeMaterial, kActFold, false>, I, "k_lat_pair_mfma",
                   std::to_string((int)kActFold) + (I.dm.clamp_out ? ", true" : ", false"), dim3((unsigned)((I.npix + pix - 1) / pix), K), dim3(256), 0,
                   I.dm, I.w, I.zdec, I.eps_lat, I.tgt, sigma, mask, I.dpix, rounds);
    } else dispatch_shape(I.dm, [&](auto s) {
        using S = decltype(s);
        if constexpr (MfmaShape<S>::kOk) {
            const int rounds = lat_rounds_for(I, lat_rounds<S>(), K), pix = 256 * rounds;
            auto kern = I.dm.clamp_out ? k_lat_pair_mfma<S, kActFold, true> : k_lat_pair_mfma<S, kActFold, false>;
            hipLaunchKernelGGL(kern, dim3((unsigned)((I.npix + pix - 1) / pix), K), dim3(256), 0, I.stream, I.dm, I.w, I.zdec, I.eps_lat, I.tgt,
                               sigma, mask, I.dpix, rounds);
        }
    });
    NTC_CHECK(hipGetLastError());
}

void launch_qat_mfma(Impl& I) {
    if (qat_split_step(I)) {
        // as many blocks as fit the chip; more where a wave would have over 64 rounds (its mask of rounds to search again)
        const size_t rounds = (I.npix + 63) / 64;
        const size_t fill = std::max((size_t)I.cus * qat_waves(I.dm.nin, I.dm.hidden[0], I.dm.nout, I.dm.lv[0].C), (rounds + 255) / 256);
        const unsigned blocks = (unsigned)std::min(fill, (rounds + 3) / 4);
        if (I.jit) {
            jit_launch(k_qat_split<ShapeMaterial, false, false>, I, "k_qat_split", I.dm.clamp_out ? "true, false" : "false, false", dim3(blocks),
                       dim3(256), 0, I.dm, I.w, I.zdec, I.tgt, I.qat_bits, I.qat_grid, (int)blocks);
        } else dispatch_shape(I.dm, [&](auto s) {
            using S = decltype(s);
            if constexpr (SplitShape<S>::kOk) {
                auto kern = I.dm.clamp_out ? k_qat_split<S, true, false> : (unit_cw(I) ? k_qat_split<S, false, true> : k_qat_split<S, false, false>);
                hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, I.stream, I.dm, I.w, I.zdec, I.tgt, I.qat_bits, I.qat_grid, (int)blocks);
            }
        });
        NTC_CHECK(hipGetLastError());
        return;
    }
    if (I.jit) {
        const float leak = I.dm.leak;
        const int act = leak >= 0.0f && leak <= 1.0f ? kActFold : kActAny;
        jit_launch(k_qat_mfma<ShapeMaterial, kActFold, false>, I, "k_qat_mfma", std::to_string(act) + (I.dm.clamp_out ? ", true" : ", false"),
                   dim3((unsigned)((I.npix + 255) / 256)),
                   dim3(256), 0, I.dm, I.w, I.zdec, I.tgt, I.qat_bits, I.qat_grid);
        NTC_CHECK(hipGetLastError());
        return;
    }
    dispatch_shape(I.dm, [&](auto s) {
        using S = decltype(s);
        if constexpr (MfmaShape<S>::kOk)
        {
            // (every listed shape with 0 <= leak <= 1 is the split kernel's)
            auto kern = I.dm.clamp_out ? k_qat_mfma<S, kActAny, true> : k_qat_mfma<S, kActAny, false>;
            hipLaunchKernelGGL(kern, dim3((unsigned)((I.npix + 255) / 256)), dim3(256), 0, I.stream, I.dm, I.w, I.zdec, I.tgt,
                               I.qat_bits, I.qat_grid);
        }
    });
    NTC_CHECK(hipGetLastError());
}

}   // namespace ntc_hip
