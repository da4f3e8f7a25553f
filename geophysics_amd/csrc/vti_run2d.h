// vti_run2d.h — resident runs of 2D steps (vti_run2d.hip): the descriptor of
// a shot, a group of shots that advance together, and the queue that turns
// an RTM's one-step-at-a-time schedule into runs.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <vector>

#include "vti_internal.h"

namespace vti {

constexpr int kRun2dMax = 64;   // steps of one RTM run (kernel argument space)

// One side (source or receiver) of a 2D shot.
struct Run2dShot {
    int nnx, nnz, ldz, M;
    float *f[8];                // u w px pz qx qz P Q of the state that steps
    const float *vp, *ep, *de, *cth, *sth, *tab;
    float dtx, dtz;
    int sv, svR, cx, cz;
    const double *tap;
    int point, sx, sz;          // point source (load-time) or the 7x7 footprint in the stress update
    const double *gw;
    const float *amp;           // nt source gains
    float *rec;                 // [it][nrec], nullptr: no record
    int nrec, rec_kind, rz, rx0, rdx, rnx;
    // RTM: the injection row (receiver side) that keeps the split form, the
    // source state's P, interior images and their geometry
    int split_z, rzi;
    const float *srcP;
    float *img, *illum;
    int clamp, rillum, inp, inx, inz;
    // filled in by the plan: tiles, exchange planes
    int gx, gz, tile0;
    unsigned long long *xP, *xQ;   // two planes each, of (tag, float) words
    long long xstride;
};

// Shots that step together in one launch, their source sides and receiver
// sides in device memory.
struct Run2dGroup {
    int ok = 0;                 // 1: usable
    int ns = 0, ntile = 0, shape = 0;
    size_t lds = 0;
    bool us = false;
    std::vector<Run2dShot> side[2];
    Run2dShot *dev = nullptr;   // source sides, then receiver sides
    unsigned long long *xbuf = nullptr;
    unsigned base = 1;          // tag of the next run's first step; the planes start with tag 0
    int *dead = nullptr;        // pinned, mapped
};

// The forward side of a 2D context's shot on state s.
Run2dShot run2d_shot(vti_ctx *c, const VtiState &s);

// Most consecutive shots from `first` on that one group can hold (0: not
// even one; the per-step kernels run it).
int run2d_fit(const std::vector<Run2dShot> &shots, int first, int device);
// 1: made, 0: not available here, < 0: error
int run2d_group_make(Run2dGroup &g, const std::vector<Run2dShot> &src, const std::vector<Run2dShot> &rcv, bool us,
                     int device, hipStream_t s);
void run2d_group_free(Run2dGroup &g);
// role 1 / 2 of the kernel; 1: launched, 0: not available, < 0: error
int run2d_group_run(Run2dGroup &g, int role, int it0, int n, bool rec, bool illum, int image_every, const long long *off,
                    hipStream_t s);
int run2d_group_check(Run2dGroup &g);

// The RTM schedule asks for single steps; this holds them back until
// something else needs the state, so that consecutive ones run as one
// resident launch (single steps and pairs stay with the per-step kernels,
// whose launches cost less than a tile's load and store).
struct RtmQueue {
    // n forward steps from it0 (first: with record and illumination), P of
    // step k also to off[k]; n receiver steps from it0 down, source P at
    // off[k].  1: done, 0: not available, < 0: error
    std::function<int(bool first, int it0, int n, const long long *off)> run_forward;
    std::function<int(int it0, int n, const long long *off)> run_receive;
    // the same one step at a time
    std::function<int(bool first, int it)> step;
    std::function<int(long long off)> keep;   // P -> off
    std::function<int(int it, long long off)> receive;

    int forward(bool first, int it);
    int keep_last(long long off);             // P after the last forward step -> off
    int receiver(int it, long long off);
    int flush();

private:
    static constexpr int kMinRun = 4;
    int kind = 0;                             // 1 first sweep, 2 recomputation, 3 receiver
    int it0 = 0, n = 0;
    long long off[kRun2dMax];
};

}  // namespace vti
