// Enqueues every launch of one chunk of a Muon step (momentum -> norm -> normalise -> Newton-Schulz
// products, the last of which takes the parameter step) from one call.  What bounds a step over small
// matrices is the host: issued one by one from Python the 18 launches of a 64 x 576 matrix took
// 137 us of which the GPU worked 70.
#include "common.h"

namespace muon_amd {

// Launches in order, each bracketed by the next two of the caller's events when there are some.
struct Enqueue {
    hipStream_t stream;
    void* const* events;
    int rc = MUON_AMD_OK;

    template <typename F>
    void operator()(F&& launch) {
        if (rc != MUON_AMD_OK) return;
        if (events) record();
        rc = launch();
        if (rc == MUON_AMD_OK && events) record();
    }
    void record() {
        if (hipEventRecord(static_cast<hipEvent_t>(*events++), stream) != hipSuccess) rc = check_launch("event record");
    }
};

}  // namespace muon_amd

using namespace muon_amd;

extern "C" {

size_t muon_amd_sizeof_chunk_run(void) { return sizeof(MuonChunkRun); }

int muon_amd_run_chunk(const MuonChunkRun* run, float one_minus_beta, float beta, int nesterov, int mutate_grad,
                       float eps, float lr, float wd_factor, const float* scalars_dev, int skip_momentum,
                       void* const* events, void* stream) {
    MUON_REQUIRE(run, "run_chunk: null plan");
    const MuonChunkRun& c = *run;
    MUON_REQUIRE(c.steps >= 0 && (c.steps == 0 || c.scalars), "run_chunk: steps=%d", c.steps);
    const float* const sc_apply = scalars_dev ? scalars_dev + 2 : nullptr;
    Enqueue go{static_cast<hipStream_t>(stream), events};
    if (!skip_momentum)
        go([&] {
            return muon_amd_momentum(c.mats, c.block_prefix, c.nmat, c.nblocks, one_minus_beta, beta, nesterov,
                                     mutate_grad, scalars_dev, stream);
        });
    const int norm_flags = c.flags | (c.aol ? MUON_AMD_NORM_UNIT : 0);
    if (c.norm_in_normalize) {
        go([&] {
            return launch_norm_normalize(c.mats, c.tile_prefix, c.nmat, c.ntiles, eps, norm_flags, c.split_counters,
                                         c.split_slots, go.stream);
        });
    } else {
        go([&] { return launch_norm_finalize(c.mats, c.nmat, eps, norm_flags, c.split_counters, c.split_slots, go.stream); });
        go([&] { return muon_amd_normalize(c.mats, c.tile_prefix, c.nmat, c.ntiles, stream); });
    }
    const auto gemm = [&](int desc, int kind, const float* abg, int extra) {
        const MuonChunkLaunch& ln = c.launches[kind];
        float* const partials = ln.split_slots ? c.split_partials : nullptr;
        int32_t* const counters = ln.split_slots ? c.split_counters : nullptr;
        go([&] {
            return muon_amd_ns_gemm(c.gemm[desc], ln.jobs, ln.njobs, ln.tile_class, abg[0], abg[1], abg[2],
                                    c.flags | extra, partials, counters, stream);
        });
    };
    for (int it = 0; it < c.steps; ++it) {
        const float* const abg = c.scalars + 9 * it;          // {alpha, beta, gamma} of the three products
        const bool first_aol = c.aol && it == 0;
        gemm(it % 2 ? MUON_AMD_GRAM_ODD : MUON_AMD_GRAM_EVEN, first_aol ? MUON_AMD_LAUNCH_GRAM_ROWSUM : MUON_AMD_LAUNCH_GRAM,
             abg, first_aol ? MUON_AMD_GEMM_ROWSUM : 0);
        if (first_aol) {
            // muon.py:776-785: the row sums of |A| come out of the product's epilogue as partial sums (one
            // small launch adds them up), then X and A are rescaled in place (A becomes the Gram matrix
            // of the rescaled X, so this iteration needs no second X X^T)
            go([&] { return muon_amd_aol_rowsum_finalize(c.aol, c.aol_row_prefix, c.nmat, c.aol_row_blocks, eps, stream); });
            go([&] { return muon_amd_aol_rescale(c.aol, c.aol_seg_prefix, c.nmat, c.aol_seg_blocks, c.aol_mode, stream); });
        }
        // (A / s, rows only, is not symmetric: the polynomial over every tile, no mirrored store)
        if (first_aol && c.aol_mode == MUON_AMD_AOL_ROWS_ONLY)
            gemm(MUON_AMD_POLY_FULL, MUON_AMD_LAUNCH_POLY_FULL, abg + 3, 0);
        else
            gemm(MUON_AMD_POLY, MUON_AMD_LAUNCH_POLY, abg + 3, 0);
        if (it + 1 < c.steps) {
            gemm(it % 2 ? MUON_AMD_UPDATE_ODD : MUON_AMD_UPDATE_EVEN, MUON_AMD_LAUNCH_UPDATE, abg + 6, MUON_AMD_GEMM_Q_KMAJOR);
        } else {
            // the last update product takes the parameter step in its epilogue (muon.py:14, 98-99)
            const MuonChunkLaunch& ln = c.launches[MUON_AMD_LAUNCH_UPDATE];
            go([&] {
                return muon_amd_ns_gemm_apply(c.gemm[MUON_AMD_UPDATE_LAST], ln.jobs, ln.njobs, ln.tile_class, abg[6], abg[7],
                                              c.flags, c.mats, lr, wd_factor, sc_apply, stream);
            });
        }
    }
    if (c.steps == 0)          // no iteration: the parameter step is a launch of its own
        go([&] { return muon_amd_apply(c.mats, c.block_prefix, c.nmat, c.nblocks, lr, wd_factor, sc_apply, stream); });
    return go.rc;
}

}  // extern "C"
