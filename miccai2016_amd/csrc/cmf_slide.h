// Max-flow passes of many iterations over volumes larger than the chip
// (cmf_slide.hip).
#pragma once

#include "mh_common.h"

namespace mh {

// How the (axis 1, axis 2) plane is cut: nt1 x nt2 tiles of b1 x b2 voxels, and
// for each tile `slots` work-groups of 8 planes, so that a window of 8 slots
// planes is resident and a pass advances up to `levels` iterations. levels = 0:
// not worth it, or does not fit.
struct SlidePlan {
    int b1 = 0, b2 = 0, nt1 = 0, nt2 = 0, slots = 0, levels = 0;
    int blocks() const { return nt1 * nt2 * slots; }
};

// The plan for solves of these dims (with seeds: `sup`) whose criterion comes
// every `update` iterations, on this context's device or one of so many compute
// units; the bytes of LDS a work-group of it takes.
SlidePlan slide_plan(mh_ctx *ctx, const int dims[3], const mh_cmf_params *prm, bool sup);
SlidePlan slide_plan(int compute_units, const int dims[3], const mh_cmf_params *prm, bool sup);
int slide_lds_bytes(const SlidePlan &plan);

// Device bytes of the words its work-groups exchange.
int64_t slide_inbox_bytes(const SlidePlan &plan);

// One solve's fields: the state of iteration t, and where that of t + levels goes.
struct SlideFields {
    const float *hp, *tmp, *pt, *u;
    float *hpo, *tmpo, *pto, *uo;
    const float4 *q4;
    const float *alpha, *cs, *ct;
    const uint8_t *labels;
};

// The solve's control words the pass reads and writes: stop (a stopped solve
// is not advanced; kSlideAborted when the pass could not be completed, its
// input untouched), parity (the buffer set holding the state), the abort word,
// and the iteration and buffer set of an aborted pass.
struct SlideControl {
    int *stop, *parity, *abort, *abort_it, *abort_cur;
};
constexpr int kSlideAborted = 3;

// Enqueue one pass of lv (1 .. plan.levels) iterations from iteration `it`; the
// device lock must be held until it is done. With `check`, partials[block]
// receives each work-group's sum of |err| of the last iteration. The tags of
// the pass follow *tags, which it advances (0: the inbox is new); when they start
// over, all of the inbox is cleared, the words of larger plans among it. `lost`: one
// of its work-groups is missing.
int slide_pass(mh_ctx *ctx, const SlidePlan &plan, const SlideFields &F, const int dims[3],
               const mh_cmf_params *prm, int lv, int it, bool check, int cur, bool lost,
               const SlideControl &C, float *partials, void *inbox, size_t inbox_bytes, unsigned *tags,
               hipStream_t s);

}  // namespace mh
