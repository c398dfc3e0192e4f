// Max-flow solves whose whole state stays on the chip (cmf_onchip.hip).
#pragma once

#include <vector>

#include "mh_common.h"

namespace mh {

// One solve of a set that shares dims, frames, capacities and parameters.
struct OnchipSolve {
    float *u;            // u0 on entry, the labelling on exit
    const float *alpha;
    int *stop, *ncrit;   // device: stop reason and number of criteria
    int *done;           // device: set to 1 when u holds the result
    float *crit_log;     // device: crit_max values
    int crit_max;
};

struct OnchipFields {
    const float *eigs;  // AoS x3 frames, or AoS x6 with pointwise eigenvalues
    const float *cs, *ct;
    const uint8_t *labels;
};

// How a volume is cut into bricks, one work-group each: v planes of b1 x b2
// voxels, nt1 x nt2 tiles in the plane, nz plane chunks. v = 0: does not fit.
struct OnchipPlan {
    int v = 0, b1 = 0, b2 = 0, nt1 = 0, nt2 = 0, nz = 0;
    int blocks() const { return nt1 * nt2 * nz; }
};

// The plan for `solves` solves of one volume on this context's device (kept by
// the context).
OnchipPlan onchip_plan(mh_ctx *ctx, const int dims[3], const mh_cmf_params *prm, int solves);

// Device bytes the solves need beside their fields.
int64_t onchip_work_bytes(const OnchipPlan &plan, int solves, int max_blocks);

// Enqueue the solves on `s` and wait for them. `ran`: every solve has its
// result. Otherwise (the device runs another on-chip solve, or could not hold
// every work-group at once) `finished`, empty or one flag per solve, says
// which have; u of the others is as it was. One solve may ask for `head`:
// head_bytes from its stop word on, its done word among them, come with the
// same transfer.
int onchip_run(mh_ctx *ctx, const OnchipPlan &plan, const OnchipSolve *solves, int nsolves,
               const OnchipFields &F, const int dims[3], const mh_cmf_params *prm, void *work,
               int64_t work_bytes, hipStream_t s, bool *ran,
               std::vector<int> *finished = nullptr, void *head = nullptr, size_t head_bytes = 0);

// Solves of several volumes side by side, eigenvalues (l0, l1, l1), no seeds: the
// plan that takes the least of the device for one of them (v = 0: none), and the
// launch of up to 8 whose plans' work-groups fit the device together.
constexpr size_t kOnchipMany = 8;
struct OnchipVolume {
    OnchipPlan plan;
    OnchipSolve solve;
    OnchipFields F;
    int dims[3];
    int64_t head_bytes;  // of its control words and criteria
};
OnchipPlan onchip_plan_many(mh_ctx *ctx, const int dims[3], const mh_cmf_params *prm);
// Enqueue and wait. `heads` (device) holds the volumes' control words and criteria
// one after another and comes to `host`. `ran`: every volume has its result, else
// every u is as it was.
int onchip_run_many(mh_ctx *ctx, const OnchipVolume *vols, int nvol, const mh_cmf_params *prm,
                    void *work, int64_t work_bytes, void *heads, hipStream_t s, std::vector<char> *host,
                    bool *ran);

}  // namespace mh
