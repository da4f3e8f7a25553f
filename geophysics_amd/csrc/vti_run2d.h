// vti_run2d.h — resident runs of 2D steps (vti_run2d.hip): the descriptor of
// a shot, a group of shots that advance together, and the program that an
// RTM's one-step-at-a-time schedule becomes.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <vector>

#include "vti_internal.h"

namespace vti {

// A 2D shot: its source side and, for RTM, its receiver side.
struct Run2dShot {
    int nnx, nnz, ldz, M;
    float *f[8];                // u w px pz qx qz P Q: the source side's state
    const float *vp, *ep, *de, *cth, *sth, *tab;
    float dtx, dtz;
    int sv, svR, cx, cz;
    const double *tap;
    int point, sx, sz;          // point source (load-time) or the 7x7 footprint in the stress update
    const double *gw;
    const float *amp;           // nt source gains
    float *rec;                 // [it][nrec], nullptr: no record
    int nrec, rec_kind, rz, rx0, rdx, rnx;
    // RTM: the receiver side's state, its taper switch, the injection row
    // (which keeps the split form), interior images and their geometry
    float *g[8];
    int svr, split_z, rzi;
    float *img, *illum;
    int clamp, rillum, inp, inx, inz;
    // checkpoints of the unsplit interior with packed split fields: u, w, P,
    // Q whole (pvol floats each), then px, pz, qx, qz (psplit each) of the
    // cells outside [pxlo, pxhi) x [pzlo, pzhi); otherwise a checkpoint has
    // the state's own layout
    int packed, pxlo, pxhi, pzlo, pzhi;
    long long pvol, psplit;
    // filled in by the plan: tiles, exchange planes
    int gx, gz, tile0;
    unsigned long long *xP, *xQ, *xU, *xW;   // two planes each, of (tag, float) words
    long long xstride;
};

// The forward side of a 2D context's shot on state s.
Run2dShot run2d_shot(vti_ctx *c, const VtiState &s);

// One operation of an RTM program.
struct Run2dOp {
    int kind;        // 1 forward steps, 2 receiver steps, 3 checkpoint, 4 restore, 5 zero state
    int it0, n;      // steps: first time index and number (receiver: descending)
    int first;       // forward: the first sweep (record, illumination)
    int link;        // forward: a later run goes on from this one's last step
    int off0;        // steps: one entry each of the offsets: forward: where P also goes (floats
                     // from the shot's own P, 0: nowhere); receiver: where the source P lies
    long long slot;  // 3, 4: floats from the state to the checkpoint (packed: from u to its start)
};

// The parts of a list of shots: consecutive ones step together in one launch.
struct Run2dPart {
    int first, n;               // shots
    int shape, ntile;
    size_t lds;
};
struct Run2dParts {
    std::vector<Run2dPart> part;   // empty: not available, the per-step kernels run all of them
    std::vector<int> gx, gz, tile0;
};

struct Run2dGroup {
    int ok = 0;                 // 1: usable
    bool refused = false;       // a launch was refused: no further one until run2d_group_set
    bool ran = false;           // a program has run since the last check
    bool us = false, entered = false;
    int device = 0;
    hipStream_t stream = nullptr;
    Run2dParts parts;
    void *mem = nullptr, *more = nullptr;   // more: a program larger than mem's share
    Run2dShot *dev = nullptr;
    void *prog = nullptr;
    size_t prog_bytes = 0, words = 0;       // words: exchange planes
    unsigned base = 1;          // tag before the next run's first exchange; the planes start with tag 0
    int *dead = nullptr;        // on the device: an exchange that never came
};

Run2dParts run2d_parts(const std::vector<Run2dShot> &shots, int device);
// 1: made, 0: not available here, < 0: error
int run2d_group_make(Run2dGroup &g, const Run2dParts &p, std::vector<Run2dShot> shots, bool us, int nt, hipStream_t s);
// other shots on the same grids (their pointers, source and receivers)
int run2d_group_set(Run2dGroup &g, std::vector<Run2dShot> shots, hipStream_t s);
void run2d_group_free(Run2dGroup &g);
// the program on every part; 1: launched, 0: not available, nothing launched
// (the states lie where the programs before it left them; their checkpoints
// have no border cells), 2: refused after some of the parts have run it, < 0:
// error
int run2d_group_run(Run2dGroup &g, const std::vector<Run2dOp> &ops, const std::vector<long long> &offs, int image_every,
                    hipStream_t s);
// waits for the stream; reports an exchange that never came, once
int run2d_group_check(Run2dGroup &g, hipStream_t s);

// Collects the operations that an RTM's schedule asks for one by one, so that
// flush() runs them as one resident launch: a launch loads and stores the grid
// and its coefficients besides, and a 600-step shot's schedule has ~90 runs of
// steps (one launch each took 17.9 ms a shot, two in all 14.6).
struct RtmProgram {
    // 1: done, 0: not available, < 0: error
    std::function<int(const std::vector<Run2dOp> &, const std::vector<long long> &)> run;
    // the same one operation at a time
    std::function<int(bool first, int it)> step;
    std::function<int(long long off)> keep;
    std::function<int(int it, long long off)> receive;
    std::function<int(int kind, long long slot)> move;

    int forward(bool first, int it) { return steps(1, first, it, 0); }
    int keep_last(long long off);             // P after the last forward step -> off
    int receiver(int it, long long off) { return steps(2, false, it, off); }
    int state(int kind, long long slot);      // checkpoint, restore, zero
    int flush();

private:
    int steps(int kind, bool first, int it, long long off);
    std::vector<Run2dOp> ops;
    std::vector<long long> offs;
};

}  // namespace vti
