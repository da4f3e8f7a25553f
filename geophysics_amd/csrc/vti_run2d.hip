// vti_run2d.hip — many 2D time steps in one launch, the grid resident on
// the chip.
//
// The 2D grids of this path are small: 440 x 440 cells are 0.8 MB a field,
// and a velocity or a stress launch of such a grid takes 3.5-4 us, nearly
// all of it launch, first-load and drain latency; at 2441 x 843 the two
// launches move 122 MB a step through the caches at 4.5 TB/s.  Here one
// workgroup per CU owns a tile of the updated region for all steps of the
// call: u, w, P, Q in LDS with the stencil's halo, the split fields (or P
// and Q, unsplit) and the per-cell coefficients in registers.  A step
// moves nothing but the halos of P and Q: the stress update publishes the
// tile's 7 outer rows of P and columns of Q as it writes them (TTI: both
// fields both ways), the next step starts by taking the neighbours'.  The
// velocities of the halo (4 + 3 rows and columns) are computed by both
// sides, so there is one exchange a step.  The exchange planes are
// double-buffered by the step's parity: a neighbour publishes step s + 1
// only after it has taken all of step s, so a plane is written again only
// when its last samples have been read.
//
// What bounds a step now: on small tiles the chain of exchange, barriers and
// LDS (60 x 50: wavefronts wait 72 % of their time, VALU 18 % busy), on large
// ones instructions (2401 x 803: VALU 72 % busy).  Measured (us a step, velocity
// + stress launches -> this): 60 x 50 with a 20-cell layer 5.8 -> 1.8, 400 x
// 400 7.2 -> 3.0, TTI 600 x 300 with a 50-cell layer 10.7 -> 5.0, 2401 x 803
// unsplit 27.9 -> 10.7.
//
// The arithmetic is vel2d_kernel's / stress2d_kernel's (and the TTI pair's)
// term by term; products that do not change from step to step are formed
// once in the same order, so every field and record is the same bit for bit
// (update_vel2d GPU_vti2dfd_kernels.cu:209-238, update_stress2d :240-299,
// CPU_vti2dfd_kernels.c:78-177, Toa_gpu_2dtti_fd_1orderfunction.cu:81-183).
//
// Launch: all workgroups get a place on the chip and no other resident launch
// is under way (Chip, below), or the per-step kernels run.  Every wait ends: a
// tile that misses a sample for kWaitTicks raises the error word and leaves its
// loop, and the others, which look at the word while they wait, follow it within
// milliseconds.
#include <hip/hip_runtime.h>

#include <sys/socket.h>
#include <sys/un.h>
#include <unistd.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <queue>
#include <string>

#include "vti_internal.h"
#include "vti_run2d.h"

namespace vti {
namespace {

__device__ __forceinline__ float cst(int m)
{
    return m == 0 ? 1.196289f : (m == 1 ? -0.0797526f : (m == 2 ? 0.009570313f : -0.0006975447f));
}

// 100 MHz ticks that a tile may wait for a neighbour's sample before the call is
// given up (20 s); and those after which it looks whether another thread or tile
// has (1 ms)
constexpr unsigned kWaitTicks = 2000000000u, kLookTicks = 100000u;

struct Run2dArgs {
    Run2dShot one;              // vti_step: the shot
    int it0, n;                 // its first time index and number of steps
    // RTM program: ns shots in device memory (tile0 ascending), the same
    // operations on each
    const Run2dShot *many;
    int ns;
    const Run2dOp *ops;
    int nops;
    const long long *offs;
    int image_every;
    unsigned base;              // tag before the call's first exchange
    unsigned wait;              // ticks that a sample may take
    int *dead;                  // error word
};

// an opaque copy: what is derived from it inside the step loop is not hoisted
// out of it (addresses and masks of every row: more registers than there are)
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// What a launch reads and nothing in it writes (the arguments, the shots, a
// program): scalar loads, again where they are used, instead of registers
// held through the step loop.
using CArgs = const __attribute__((address_space(4))) Run2dArgs;
using CShot = const __attribute__((address_space(4))) Run2dShot;
using COp = const __attribute__((address_space(4))) Run2dOp;
using COff = const __attribute__((address_space(4))) long long;

struct Tile {
    int x0, nx, z0, nz;         // first cell, rows; first z, cells (a multiple of 4)
};
__host__ __device__ inline Tile tile_of(int nnx, int nnz, int gx, int gz, int tx, int tz)
{
    const int ux = nnx - 8, uq = (nnz - 8 + 3) / 4;
    const int xa = (int)((long long)ux * tx / gx), xb = (int)((long long)ux * (tx + 1) / gx);
    const int qa = (int)((long long)uq * tz / gz), qb = (int)((long long)uq * (tz + 1) / gz);
    return Tile{4 + xa, xb - xa, 4 + 4 * qa, 4 * (qb - qa)};
}

constexpr int kMaxRows = 8;     // rows of a thread's strip, at most

// LDS layout in floats: the halos are 7 rows / 8 columns for P and Q (7 of
// them used), 4 + 3 rows / 4 columns for u and w; the VTI update needs P and
// u only along x and Q and w only along z, the TTI update all of them both
// ways.  Every pitch and start is a multiple of 4.
template <bool TTI>
struct Lds {
    int pp, p0, qp, q0, up, u0, wp, w0;   // pitch and position of cell (0, 0)
    int oq, ou, ow, oc, os, ot, total;    // array starts (P at 0), tables, size
    __host__ __device__ Lds(int nx, int nz)
    {
        pp = TTI ? nz + 16 : nz;
        qp = nz + 16;
        up = TTI ? nz + 8 : nz;
        wp = nz + 8;
        p0 = 7 * pp + (TTI ? 8 : 0);
        q0 = (TTI ? 7 * qp : 0) + 8;
        u0 = 4 * up + (TTI ? 4 : 0);
        w0 = (TTI ? 4 * wp : 0) + 4;
        oq = (nx + 14) * pp;
        ou = oq + (TTI ? nx + 14 : nx) * qp;
        ow = ou + (nx + 7) * up;
        oc = ow + (TTI ? nx + 7 : nx) * wp;
        os = oc + (TTI ? (nx + 7) * up : 0);
        ot = os + (TTI ? (nx + 7) * up : 0);
        // tables: z (two velocity, two stress), then x (two velocity, two stress)
        // and what a strip's loads may read past the last rows
        total = ot + 2 * (nz + 8) + 2 * nz + 2 * (nx + 7) + 2 * nx + kMaxRows * (nz + 8);
    }
};

__device__ __forceinline__ float4 ldg4(const float *p, int nnx, int ldz, int x, int z)
{
    if (x < 0 || x >= nnx || z < 0 || z >= ldz) return make_float4(0.f, 0.f, 0.f, 0.f);
    return *reinterpret_cast<const float4 *>(p + (long long)x * ldz + z);
}

// Exchange planes.  A sample travels as one 8-byte word, its float and the
// step's tag; the reader polls the words themselves until they carry the tag,
// so there is no flag to raise after the data and to fetch before it.  All
// accesses are agent-scope atomics: other XCDs' workgroups read the planes.
__device__ __forceinline__ void put(unsigned long long *p, float v, unsigned tag)
{
    __hip_atomic_store(p, (unsigned long long)tag << 32 | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long peek(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The wait for one word is over when it began too long ago or, looked at only
// after a while (at every poll it cost 0.14 us a step at 60 x 50), another
// thread of the tile or another tile has given up.
struct Wait {
    unsigned limit;
    int *dead;                  // the tile's (LDS)
    const int *gone;            // the launch's error word
    __device__ __forceinline__ bool over(unsigned t0) const
    {
        const unsigned d = (unsigned)wall_clock64() - t0;
        if (__builtin_expect(d < min(kLookTicks, limit), 1)) return false;
        if (d <= limit && !__hip_atomic_load(dead, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) &&
            !__hip_atomic_load(gone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))
            return false;
        *dead = 1;
        return true;
    }
};
// the word's sample once it carries the tag (w: an earlier look at it)
__device__ __forceinline__ float await(const unsigned long long *p, unsigned long long w, unsigned tag, const Wait &x)
{
    if ((unsigned)(w >> 32) != tag) {
        const unsigned t0 = (unsigned)wall_clock64();
        do {
            w = peek(p);
            if (x.over(t0)) break;   // asked while the load is on its way
        } while ((unsigned)(w >> 32) != tag);
    }
    return __uint_as_float((unsigned)w);
}

// the shot of a tile (tile0 ascending)
__device__ __forceinline__ int find_shot2d(CShot *s, int ns, int tile)
{
    int lo = 0, hi = ns - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s[mid].tile0 <= tile) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// k / n and k % n of 0 <= k < 2^20 by a reciprocal (exact: the rounding is
// far below the half added to k)
__device__ __forceinline__ void divmod(int k, int n, float inv, int &q, int &r)
{
    q = (int)(((float)k + 0.5f) * inv);
    r = k - q * n;
}

// sum_m c_m (f[i + 4 + m] - f[i + 3 - m]) of eight consecutive samples
__device__ __forceinline__ float diff8(const float *f)
{
    float r = 0.0f;
#pragma unroll
    for (int m = 0; m < 4; ++m) r += cst(m) * (f[4 + m] - f[3 - m]);
    return r;
}
// the same of p[-4 + S] .. p[3 + S], S = 1: velocity, 0: stress
template <int S>
__device__ __forceinline__ float diff_z(const float *p)
{
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = p[j - 4 + S];
    return diff8(f);
}

// Every thread owns a strip of NU consecutive rows at one z (lanes along z:
// LDS and global rows are read without conflicts and coalesced) and holds
// the x-stencil of the strip in registers, NU + 7 loads for NU cells.  US:
// the unsplit interior (s0, s1 hold P and Q of an undamped cell, the split
// fields of a damped one).  One cell a lane and 16 wavefronts a CU: four cells
// a lane (16-byte LDS accesses, 8 wavefronts) took 3.8 against 3.6 us a step
// at 400 x 400 and 14.9 against 14.1 at 2401 x 803.
// PROG false: vti_step (source and record of one shot).  PROG true: the
// schedule of an RTM as a program (Run2dOp), of many shots at once: forward
// steps (record and illumination in the first sweep, P into checkpoints),
// receiver steps backward in time (the records written into P and Q on the
// injection row before each step: only the velocity update reads them, the
// split form of that row rebuilds P and Q; image img += P_source * P and,
// where asked for, the receiver illumination), whole-state checkpoints.  The
// state that steps is on the chip, the other side's and the checkpoints are
// in memory; all of those are a tile's own cells, written and read by the
// same thread, so tiles meet only in the exchange.
template <bool TTI, bool US, bool PROG, int NT, int NU>
__global__ __launch_bounds__(NT) void run2d_kernel(Run2dArgs a)
{
    extern __shared__ float4 smem4[];
    float *sm = reinterpret_cast<float *>(smem4);
    __shared__ int s_dead;
    const int tid = threadIdx.x;
    CArgs *ka = (CArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    CShot *many = (CShot *)a.many;
    CShot &b = PROG ? many[find_shot2d(many, a.ns, blockIdx.x)] : ka->one;
    COp *ops = (COp *)a.ops;
    COff *offs = (COff *)a.offs;
    const int tile = blockIdx.x - (PROG ? b.tile0 : 0);
    const Tile t = tile_of(b.nnx, b.nnz, b.gx, b.gz, tile / b.gz, tile % b.gz);
    const int nx = t.nx, nz = t.nz, x0 = t.x0, z0 = t.z0;
    const Lds<TTI> L(nx, nz);
    const int ldz = b.ldz, zend = b.nnz - 4, xend = b.nnx - 4, M = b.M;
    float *sP = sm + L.p0, *sQ = sm + L.oq + L.q0, *sU = sm + L.ou + L.u0, *sW = sm + L.ow + L.w0;
    float *sC = sm + L.oc + L.u0, *sS = sm + L.os + L.u0;   // TTI only
    float *kz1 = sm + L.ot + 4, *kz2 = kz1 + nz + 8;        // cells -4 .. nz + 3
    float *az1 = kz2 + nz + 4, *az2 = az1 + nz;
    float *kx1 = az2 + nz + 4, *kx2 = kx1 + nx + 7;         // rows -4 .. nx + 2
    float *ax1 = kx2 + nx + 3, *ax2 = ax1 + nx;

    // ---- load the tile ----
    if (tid == 0) s_dead = 0;
    for (int k = 4 * tid; k < L.ou; k += 4 * NT) {   // P and Q rectangles
        const bool q = k >= L.oq;
        const int i = q ? k - L.oq : k, pitch = q ? L.qp : L.pp;
        const int r = i / pitch - (q ? (TTI ? 7 : 0) : 7), c = i % pitch - ((q || TTI) ? 8 : 0);
        *reinterpret_cast<float4 *>(sm + k) = ldg4(q ? b.f[7] : b.f[6], b.nnx, ldz, x0 + r, z0 + c);
    }
    for (int k = L.ou + 4 * tid; k < L.oc; k += 4 * NT) {   // u and w
        const bool q = k >= L.ow;
        const int i = q ? k - L.ow : k - L.ou, pitch = q ? L.wp : L.up;
        const int r = i / pitch - (q ? (TTI ? 4 : 0) : 4), c = i % pitch - ((q || TTI) ? 4 : 0);
        *reinterpret_cast<float4 *>(sm + k) = ldg4(q ? b.f[1] : b.f[0], b.nnx, ldz, x0 + r, z0 + c);
    }
    if (TTI)
        for (int k = L.oc + 4 * tid; k < L.ot; k += 4 * NT) {
            const bool q = k >= L.os;
            const int i = q ? k - L.os : k - L.oc;
            *reinterpret_cast<float4 *>(sm + k) = ldg4(q ? b.sth : b.cth, b.nnx, ldz, x0 + i / L.up - 4, z0 + i % L.up - 4);
        }
    auto tabv = [&](int row, int i) { return i >= 0 && i < M ? b.tab[(long long)row * M + i] : 0.0f; };
    // velocity tables: VTI: coff1 * dt/dx (the reference's first product), coff2; TTI: the factors themselves
    for (int k = tid; k < nx + 7; k += NT) {
        kx1[k - 4] = TTI ? tabv(0, x0 + k - 4) : tabv(0, x0 + k - 4) * b.dtx;
        kx2[k - 4] = tabv(1, x0 + k - 4);
    }
    for (int k = tid; k < nx; k += NT) {
        ax1[k] = tabv(6, x0 + k);
        ax2[k] = tabv(7, x0 + k);
    }
    for (int k = tid; k < nz + 8; k += NT) {
        kz1[k - 4] = TTI ? tabv(4, z0 + k - 4) : tabv(4, z0 + k - 4) * b.dtz;
        kz2[k - 4] = tabv(5, z0 + k - 4);
    }
    for (int k = tid; k < nz; k += NT) {
        az1[k] = tabv(10, z0 + k);
        az2[k] = tabv(11, z0 + k);
    }
    __syncthreads();

    // ---- this thread's strip ----
    float s0[NU], s1[NU], s2[NU], s3[NU], c0[NU], c1[NU], c2[NU], c3[NU];
    const float inv_z = 1.0f / nz, inv_z8 = 1.0f / (nz + 8), inv_14 = 1.0f / 14.0f, inv_z14 = 1.0f / (nz + 14);
    int row0, col0;
    divmod(tid, nz, inv_z, row0, col0);
    row0 *= NU;
    const int r0 = row0, c = col0;
    const bool mine = r0 < nx, live = mine && z0 + c < zend;   // live: cells of the updated region
    const int rows = mine ? min(NU, nx - r0) : 0;
    int und = 0;             // rows of the undamped interior (US)
    int recs = 0, krec = 0;  // rows with a receiver, the first one's index
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        s0[i] = s1[i] = s2[i] = s3[i] = c0[i] = c1[i] = c2[i] = c3[i] = 0.0f;
        if (!live || i >= rows) continue;
        const int x = x0 + r0 + i, z = z0 + c;
        const long long g = (long long)x * ldz + z;
        if (!PROG) {
            s0[i] = b.f[2][g];
            s1[i] = b.f[4][g];
            s2[i] = b.f[3][g];
            s3[i] = b.f[5][g];
        }
        if (US && ax1[r0 + i] == 1.0f && ax2[r0 + i] == 1.0f && az1[c] == 1.0f && az2[c] == 1.0f) {
            und |= 1 << i;
            if (!PROG) {
                s0[i] = sP[(r0 + i) * L.pp + c];
                s1[i] = sQ[(r0 + i) * L.qp + c];
            }
        }
        if (b.rec && z == b.rz) {
            const int k = x - b.rx0;
            if (k >= 0 && k % b.rdx == 0 && k / b.rdx < b.rnx) {
                if (!recs) krec = k / b.rdx;
                recs |= 1 << i;
            }
        }
    }
    // the strip's coefficients, with the SV taper or without
    auto coefficients = [&](bool sv) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            if (!live || i >= rows) continue;
            const int x = x0 + row0 + i, z = z0 + col0;
            const long long g = (long long)x * ldz + z;
            const float v = b.vp[g];
            float ee = b.ep[g], dd = b.de[g];
            const float tx1 = ax1[row0 + i], tx2 = ax2[row0 + i], tz1 = az1[col0], tz2 = az2[col0];
            if (sv) {   // SV taper (GPU_vti2dfd_kernels.cu:260-278)
                const int rx = x - b.cx, rz = z - b.cz, r2 = rx * rx + rz * rz;
                if (r2 <= b.svR * b.svR) {
                    const double f = b.tap[r2];
                    ee = (float)(f * (double)ee);
                    dd = (float)(f * (double)dd);
                }
            }
            const float e2 = 1.0f + 2.0f * ee;
            const float sd = sqrtf(1.0f + 2.0f * dd);
            if (TTI) {   // the cos/sin terms carry dt/dx: g1 vp vp (1+2e), g1 vp vp sqrt(1+2d), g1 vp vp
                const float g1 = tx1 * tz1;
                c0[i] = g1 * v * v * e2;
                c1[i] = g1 * v * v * sd;
                c2[i] = g1 * v * v;
                c3[i] = tx2 * tz2;
            } else {
                c0[i] = tx1 * v * v * e2 * b.dtx;
                c1[i] = tx1 * v * v * sd * b.dtx;
                c2[i] = tz1 * v * v * sd * b.dtz;
                c3[i] = tz1 * v * v * b.dtz;
            }
        }
    };
    if (!PROG) coefficients(b.sv != 0);

    // images: interior cell (r0 + i, c) at img[io + i * inz]
    const bool inz_ok = PROG && live && z0 + c >= b.inp && z0 + c < b.inp + b.inz;
    const long long io = (long long)(x0 + row0 - b.inp) * b.inz + (z0 + col0 - b.inp);
    int inn = 0;                               // rows of the strip in the interior
    float il[PROG ? NU : 1], im[PROG ? NU : 1];
    if (PROG) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int jx = x0 + row0 + i - b.inp;
            il[i] = im[i] = 0.0f;
            if (!inz_ok || i >= rows || jx < 0 || jx >= b.inx) continue;
            inn |= 1 << i;
            il[i] = b.illum[io + (long long)i * b.inz];
            im[i] = b.img[io + (long long)i * b.inz];
        }
#pragma unroll
        for (int i = 0; i < NU; ++i) asm volatile("" : "+v"(il[i]), "+v"(im[i]));
    }
    // receiver samples of this lane's row of the injection row (tile and halo)
    const int zi = PROG ? b.rzi - z0 : 0;
    const bool inj_p = PROG && zi >= 0 && zi < nz, inj_q = PROG && zi >= -8 && zi < nz + 8;
    int kinj = -1;
    if (inj_q && tid < nx + 14) {
        const int k = x0 + tid - 7 - b.rx0;
        if (k >= 0 && k % b.rdx == 0 && k / b.rdx < b.rnx) kinj = k / b.rdx;
    }
    const int srow = b.sx - x0, scol = b.sz - z0;
    const bool src_p = b.point && srow >= -7 && srow < nx + 7 && scol >= (TTI ? -8 : 0) && scol < nz + (TTI ? 8 : 0);
    const bool src_q = b.point && srow >= (TTI ? -7 : 0) && srow < nx + (TTI ? 7 : 0) && scol >= -8 && scol < nz + 8;

    // the strip is in registers before the step loop, whose waits would
    // otherwise count these loads as possibly still on their way
#pragma unroll
    for (int i = 0; i < NU; ++i)
        asm volatile("" : "+v"(s0[i]), "+v"(s1[i]), "+v"(s2[i]), "+v"(s3[i]), "+v"(c0[i]), "+v"(c1[i]), "+v"(c2[i]), "+v"(c3[i]));
    if (US) __syncthreads();   // P and Q are in s0 and s1 before the source is added to them in LDS
    float amps = 0.0f;   // lane k: the gain of step k of the current 64
    unsigned tag = a.base;
    int cur = PROG ? 0 : 1;   // whose state is on the chip: 1 source, 2 receiver
    bool fresh = false;       // PROG: the halos are not those of the state on the chip
    const int nops = PROG ? a.nops : 1;
    for (int o = 0; o < nops; ++o) {
    Run2dOp op{};
    if (PROG) {
        op.kind = ops[o].kind;
        op.it0 = ops[o].it0;
        op.n = ops[o].n;
        op.first = ops[o].first;
        op.link = ops[o].link;
        op.off0 = ops[o].off0;
        op.slot = ops[o].slot;
    } else {
        op.kind = 1;
        op.first = 1;
        op.it0 = a.it0;
        op.n = a.n;
    }
    const bool rcv = PROG && op.kind == 2;
    if (PROG) {
        const int role = rcv ? 2 : 1;
        const bool sw = cur != role;
        // cell (row0 + i, col0) of a packed checkpoint's split fields
        auto packed = [&](int i) {
            const int x = x0 + row0 + i, z = z0 + col0;
            const bool whole = x < b.pxlo || x >= b.pxhi;
            const long long full = (long long)min(x, b.pxlo) + max(0, x - b.pxhi);
            return full * b.nnz + (x - full) * (long long)(b.pzlo + b.nnz - b.pzhi) +
                   (whole || z < b.pzlo ? z : b.pzlo + (z - b.pzhi));
        };
        if ((sw && cur) || op.kind == 3) {   // the state on the chip to its home, or to a checkpoint
            const bool pk = op.kind == 3 && b.packed;
            const long long off = op.kind == 3 ? op.slot : 0;
            float *F[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) F[k] = (cur == 2 ? b.g[k] : b.f[k]) + off;
            if (pk) {
                F[0] = b.f[0] + off;
                F[1] = F[0] + b.pvol; F[6] = F[1] + b.pvol; F[7] = F[6] + b.pvol;
                F[2] = F[7] + b.pvol; F[3] = F[2] + b.psplit; F[4] = F[3] + b.psplit; F[5] = F[4] + b.psplit;
            }
            const int ub = cur == 2 && z0 + col0 == b.split_z ? 0 : und;
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                asm volatile("" ::: "memory");
                if (!live || i >= rows) continue;
                const int r = row0 + i, c = col0;
                const long long g = (long long)(x0 + r) * ldz + z0 + c;
                F[0][g] = sU[r * L.up + c];
                F[1][g] = sW[r * L.wp + c];
                F[6][g] = sP[r * L.pp + c];
                F[7][g] = sQ[r * L.qp + c];
                if (US && (ub >> i & 1)) continue;
                const long long h = pk ? packed(i) : g;
                F[2][h] = s0[i];
                F[4][h] = s1[i];
                F[3][h] = s2[i];
                F[5][h] = s3[i];
            }
        }
        if (sw || op.kind >= 4) {            // another state onto the chip: a home, a checkpoint, zero
            const bool pk = op.kind == 4 && b.packed;
            const long long off = op.kind == 4 ? op.slot : 0;
            const float *F[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) F[k] = (rcv ? b.g[k] : b.f[k]) + off;
            if (pk) {
                F[0] = b.f[0] + off;
                F[1] = F[0] + b.pvol; F[6] = F[1] + b.pvol; F[7] = F[6] + b.pvol;
                F[2] = F[7] + b.pvol; F[3] = F[2] + b.psplit; F[4] = F[3] + b.psplit; F[5] = F[4] + b.psplit;
            }
            const bool zero = op.kind == 5;
            const int ub = rcv && z0 + col0 == b.split_z ? 0 : und;
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                asm volatile("" ::: "memory");
                if (!live || i >= rows) continue;
                const int r = row0 + i, c = col0;
                const long long g = (long long)(x0 + r) * ldz + z0 + c;
                const float P = zero ? 0.0f : F[6][g], Q = zero ? 0.0f : F[7][g];
                sU[r * L.up + c] = zero ? 0.0f : F[0][g];
                sW[r * L.wp + c] = zero ? 0.0f : F[1][g];
                sP[r * L.pp + c] = P;
                sQ[r * L.qp + c] = Q;
                if (US && (ub >> i & 1)) {
                    s0[i] = P;
                    s1[i] = Q;
                    continue;
                }
                const long long h = pk ? packed(i) : g;
                s0[i] = zero ? 0.0f : F[2][h];
                s1[i] = zero ? 0.0f : F[4][h];
                s2[i] = zero ? 0.0f : F[3][h];
                s3[i] = zero ? 0.0f : F[5][h];
            }
            if (sw) coefficients(rcv ? b.svr != 0 : b.sv != 0);
#pragma unroll
            for (int i = 0; i < NU; ++i)
                asm volatile("" : "+v"(s0[i]), "+v"(s1[i]), "+v"(s2[i]), "+v"(s3[i]), "+v"(c0[i]), "+v"(c1[i]), "+v"(c2[i]), "+v"(c3[i]));
            cur = role;
            fresh = true;
            __syncthreads();
        }
        if (op.kind >= 3) continue;
    }
    const bool lit = PROG && (rcv ? b.rillum != 0 : op.first != 0), clamp = PROG && !rcv && b.clamp;
    for (int s = 0; s < op.n; ++s) {
        const int it = rcv ? op.it0 - s : op.it0 + s;
        if (!rcv && (s & 63) == 0) {
            amps = b.amp[op.it0 + min(s + (tid & 63), op.n - 1)];
            // taken here: waited for at the top of each step, the load would
            // hold the step until the stores before it are acknowledged too
            asm volatile("" : "+v"(amps));
        }
        const float amp = rcv ? 0.0f : __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(amps), s & 63));
        const int vt = opaque(tid), r0 = opaque(row0), c = opaque(col0);
        // what this step reads from memory: its latency passes behind the exchange
        float inj = 0.0f, sp[PROG ? NU : 1];
        const bool imaged = rcv && it % a.image_every == 0;
        if (rcv) {
            if (kinj >= 0) inj = b.rec[(long long)it * b.nrec + kinj];
            const float *src = b.f[6] + offs[op.off0 + s] + (long long)(x0 + r0) * ldz + z0 + c;
#pragma unroll
            for (int i = 0; i < NU; ++i) sp[i] = imaged && (inn >> i & 1) ? src[(long long)i * ldz] : 0.0f;
        }
        if (PROG && fresh) {
            // ---- a state just put on the chip: its outer rows and columns of
            // all four fields to the neighbours, theirs taken ----
            ++tag;
            const long long par = (tag & 1) * b.xstride;
            unsigned long long *gP = b.xP + par, *gQ = b.xQ + par, *gU = b.xU + par, *gW = b.xW + par;
            if (live) {
#pragma unroll
                for (int i = 0; i < NU; ++i) {
                    if (i >= rows) continue;
                    const int r = r0 + i;
                    const long long g = (long long)(x0 + r) * ldz + z0 + c;
                    if (r < 7 || r >= nx - 7) put(gP + g, sP[r * L.pp + c], tag);
                    if (c < 7 || c >= nz - 7) put(gQ + g, sQ[r * L.qp + c], tag);
                    if (r < 4 || r >= nx - 4) put(gU + g, sU[r * L.up + c], tag);
                    if (c < 4 || c >= nz - 4) put(gW + g, sW[r * L.wp + c], tag);
                }
            }
            const Wait wait{a.wait, &s_dead, a.dead};
            for (int k = vt; k < 21 * nz + 21 * nx; k += NT) {
                const bool q = k >= 21 * nz;
                int r, cc;
                if (!q) divmod(k, nz, inv_z, r, cc);
                else divmod(k - 21 * nz, 21, 1.0f / 21.0f, r, cc);
                int &w = q ? cc : r;            // 0-13: P (Q), 14-20: u (w)
                const int n = q ? nz : nx;
                const bool vel = w >= 14;
                w = vel ? (w < 18 ? w - 18 : n + w - 18) : (w < 7 ? w - 7 : n + w - 7);
                const int x = x0 + r, z = z0 + cc;
                if (x < 4 || x >= xend || z < 4 || z >= zend) continue;
                const unsigned long long *p = (q ? (vel ? gW : gQ) : (vel ? gU : gP)) + (long long)x * ldz + z;
                float *d = q ? (vel ? sW + r * L.wp + cc : sQ + r * L.qp + cc) : (vel ? sU + r * L.up + cc : sP + r * L.pp + cc);
                *d = await(p, peek(p), tag, wait);
            }
            fresh = false;
            __syncthreads();
            if (s_dead) {
                if (tid == 0) __hip_atomic_store(a.dead, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                return;
            }
        } else if (PROG || s > 0) {
            // ---- the neighbours' outer rows and columns of the last step ----
            ++tag;
            const unsigned long long *gP = b.xP + (tag & 1) * b.xstride, *gQ = b.xQ + (tag & 1) * b.xstride;
            const int nrow = 14 * nz;
            const int wide = 14 * (nz + 14), nget = (TTI ? wide : nrow) + 14 * nx;
            const int total = TTI ? 2 * nget : nget;
            const Wait wait{a.wait, &s_dead, a.dead};
            constexpr int B = NU == 1 && !TTI ? 1 : (NU < 4 ? 2 : 4);   // words looked at before the first wait
            for (int k0 = vt; k0 < total; k0 += B * NT) {
                const unsigned long long *p[B];
                unsigned long long w[B];
                int at[B];
#pragma unroll
                for (int j = 0; j < B; ++j) {
                    const int k = k0 + j * NT;
                    const bool second = TTI && k >= nget;
                    const int i = second ? k - nget : k;
                    int r, c;
                    if (i < (TTI ? wide : nrow)) {
                        divmod(i, TTI ? nz + 14 : nz, TTI ? inv_z14 : inv_z, r, c);
                        r = r < 7 ? r - 7 : nx + r - 7;
                        if (TTI) c -= 7;
                    } else {
                        divmod(i - (TTI ? wide : nrow), 14, inv_14, r, c);
                        c = c < 7 ? c - 7 : nz + c - 7;
                    }
                    const bool q = TTI ? second : i >= nrow;
                    const int x = x0 + r, z = z0 + c;
                    const bool on = k < total && x >= 4 && x < xend && z >= 4 && z < zend;
                    at[j] = !on ? -1 : (q ? L.oq + L.q0 + r * L.qp + c : L.p0 + r * L.pp + c);
                    p[j] = (q ? gQ : gP) + (long long)x * ldz + z;
                    if (on) w[j] = peek(p[j]);
                }
#pragma unroll
                for (int j = 0; j < B; ++j)
                    if (at[j] >= 0) sm[at[j]] = await(p[j], w[j], tag, wait);
            }
            __syncthreads();
            if (s_dead) {   // the same for every thread: written before the barrier only
                if (tid == 0) __hip_atomic_store(a.dead, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                return;
            }
        }
        if (rcv && inj_q) {   // shot_record(load) Toa_gpu2DvtiFdRtmAdcigsLaplace.cu:525-528
            if (kinj >= 0) {
                const int r = tid - 7;
                if (inj_p) sP[r * L.pp + zi] = inj;
                if (r >= 0 && r < nx) sQ[r * L.qp + zi] = inj;
            }
            __syncthreads();
        }
        if (amp != 0.0f && (src_p || src_q)) {   // P[src] += amp, Q[src] += amp before the update (add_source2d :204-205)
            if (tid == 0) {
                if (src_p) sP[srow * L.pp + scol] += amp;
                if (src_q) sQ[srow * L.qp + scol] += amp;
            }
            __syncthreads();
        }

        // ---- velocity update of the tile and its halo, strips of NU rows ----
        {
            const int ns = (nx + 7 + NU - 1) / NU;               // strips of rows -4 .. nx + 2
            const int nu = ns * (TTI ? nz + 8 : nz), nup = TTI ? nu : (nu + 63) & ~63;
            const int total = TTI ? nu : nup + (nx + NU - 1) / NU * (nz + 8);
            for (int k = vt; k < total; k += NT) {
                int r, cc;
                if (TTI || k < nup) {
                    // u (TTI: u and w)
                    divmod(k, TTI ? nz + 8 : nz, TTI ? inv_z8 : inv_z, r, cc);
                    if (TTI) cc -= 4;
                    r = r * NU - 4;
                    const int z = z0 + cc, last = nx + 2;
                    if (r > last || z < 4 || z >= zend) continue;   // r > last: the items that pad nu
                    const float *p = sP + r * L.pp + cc, *q = sQ + r * L.qp + cc;
                    float f[NU + 7], h[TTI ? NU + 7 : 1];
#pragma unroll
                    for (int i = 0; i < NU + 7; ++i) {   // past the last row: other cells of LDS, not used
                        f[i] = p[(i - 3) * L.pp];
                        if (TTI) h[i] = q[(i - 3) * L.qp];
                    }
                    const float z1 = TTI ? kz1[cc] : 0.0f, z2 = TTI ? kz2[cc] : 0.0f;
#pragma unroll
                    for (int i = 0; i < NU; ++i) {
                        const int x = x0 + r + i;
                        const bool on = r + i <= last && x >= 4 && x < xend;
                        float *pu = sU + (r + i) * L.up + cc;
                        const float k1 = kx1[r + i], k2 = kx2[r + i];
                        const float d = diff8(f + i);
                        if (!TTI) {
                            const float u = k2 * *pu - k1 * d;
                            if (on) *pu = u;
                        } else {
                            float *pw = sW + (r + i) * L.wp + cc;
                            const float cs = sC[(r + i) * L.up + cc], sn = sS[(r + i) * L.up + cc];
                            const float Pz = diff_z<1>(p + i * L.pp), Qx = diff8(h + i), Qz = diff_z<1>(q + i * L.qp);
                            const float g2 = k2 * z2, g1 = k1 * z1;
                            const float u = g2 * *pu - g1 * (cs * b.dtx * d - sn * b.dtz * Pz);
                            const float w = g2 * *pw - g1 * (sn * b.dtx * Qx + cs * b.dtz * Qz);
                            if (on) {
                                *pu = u;
                                *pw = w;
                            }
                        }
                    }
                } else {
                    // w, from the next wavefront on: a small tile's two kinds run side by side
                    divmod(k - nup, nz + 8, inv_z8, r, cc);
                    cc -= 4;
                    r *= NU;
                    const int z = z0 + cc;
                    if (z < 4 || z >= zend) continue;
                    const float k1 = kz1[cc], k2 = kz2[cc];
#pragma unroll
                    for (int i = 0; i < NU; ++i) {
                        float *pw = sW + (r + i) * L.wp + cc;
                        const float w = k2 * *pw - k1 * diff_z<1>(sQ + (r + i) * L.qp + cc);
                        if (NU == 1 || r + i < nx) *pw = w;
                    }
                }
            }
        }
        __syncthreads();

        // ---- stress update of the tile ----
        if (live) {
            const int nr = opaque(rows), rb = opaque(recs), in_ = PROG ? opaque(inn) : 0;
            const int ub = opaque(rcv && z0 + c == b.split_z ? 0 : und);
            float *keep = nullptr;
            if (PROG && !rcv) {
                const long long off = offs[op.off0 + s];
                if (off) keep = b.f[6] + off;
            }
            const bool foot = !PROG && !b.point && amp != 0.0f, more = s + 1 < op.n || op.link, note = !rcv && op.first;
            const unsigned next = tag + 1;
            unsigned long long *gP = b.xP + (next & 1) * b.xstride, *gQ = b.xQ + (next & 1) * b.xstride;
            const bool ez = c < 7 || c >= nz - 7;
            const float *pu = sU + r0 * L.up + c, *pw = sW + r0 * L.wp + c;
            float f[NU + 7], h[TTI ? NU + 7 : 1];
#pragma unroll
            for (int i = 0; i < NU + 7; ++i) {
                f[i] = pu[(i - 4) * L.up];
                if (TTI) h[i] = pw[(i - 4) * L.wp];
            }
            const float tz2 = az2[c];
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                asm volatile("" ::: "memory");   // one row's z-stencil loads at a time
                const int r = r0 + i;
                float xx = diff8(f + i), zz = diff_z<0>(pw + i * L.wp);
                if (TTI) {   // the rotated x derivative of u and z derivative of w
                    const float uz = diff_z<0>(pu + i * L.up), wx = diff8(h + i);
                    const float cs = sC[r * L.up + c], sn = sS[r * L.up + c];
                    xx = cs * b.dtx * xx - sn * b.dtz * uz;
                    zz = sn * b.dtx * wx + cs * b.dtz * zz;
                }
                float Pn, Qn;
                if (US && (ub >> i & 1)) {
                    Pn = s0[i] -= c0[i] * xx + c2[i] * zz;
                    Qn = s1[i] -= c1[i] * xx + c3[i] * zz;
                } else {
                    const float fx = TTI ? c3[i] : ax2[r], fz = TTI ? c3[i] : tz2;
                    s0[i] = fx * s0[i] - c0[i] * xx;
                    s2[i] = fz * s2[i] - (TTI ? c1[i] : c2[i]) * zz;
                    s1[i] = fx * s1[i] - c1[i] * xx;
                    s3[i] = fz * s3[i] - (TTI ? c2[i] : c3[i]) * zz;
                    Pn = s0[i] + s2[i];
                    Qn = s1[i] + s3[i];
                    if (foot) {   // P = px+pz+s (CPU_vti2dfd_kernels.c:173-174), 7x7 footprint
                        const int fdx = x0 + r - b.sx, fdz = z0 + c - b.sz;
                        if (fdx >= -3 && fdx <= 3 && fdz >= -3 && fdz <= 3) {
                            const float sc = (float)((double)amp * b.gw[(fdx + 3) * 7 + (fdz + 3)]);
                            Pn = Pn + sc;
                            Qn = Qn + sc;
                        }
                    }
                }
                if (NU > 1 && i >= nr) continue;
                sP[r * L.pp + c] = Pn;
                sQ[r * L.qp + c] = Qn;
                if (more) {   // the outer 7 rows and columns, to the neighbours
                    const bool ex = r < 7 || r >= nx - 7;
                    const long long g = (long long)(x0 + r) * ldz + z0 + c;
                    if (ex || (TTI && ez)) put(gP + g, Pn, next);
                    if (ez || (TTI && ex)) put(gQ + g, Qn, next);
                }
                if (PROG && (in_ >> i & 1)) {
                    if (lit) {   // cal_illumination :654-677
                        il[i] += Pn * Pn + Qn * Qn;
                        if (clamp && il[i] <= 0.0f) il[i] = 1.0f;
                    }
                    if (imaged) im[i] += sp[i] * Pn;   // cal_migration :679-698
                }
                if (PROG && keep) keep[(long long)(x0 + r) * ldz + z0 + c] = Pn;
                if (note && (rb >> i & 1)) {
                    const int k = krec + __popc(rb & ((1 << i) - 1));
                    b.rec[(long long)it * b.nrec + k] = b.rec_kind == 0 ? Pn : (b.rec_kind == 1 ? Pn + Pn : Pn + Qn);
                }
            }
        }
        __syncthreads();
    }
    }   // operations

    // ---- write the tile back (n >= 2: every neighbour has loaded its halo;
    // PROG: none reads another's cells in memory) ----
    // the field pointers come from memory again: held through the loop they
    // would cost the registers that it needs
    CShot *bm = &b;
    asm volatile("" : "+s"(bm));
    float *gf[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) gf[k] = cur == 2 ? bm->g[k] : bm->f[k];
    const int ub = cur == 2 && z0 + c == b.split_z ? 0 : und;
    if (!live) return;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        if (i >= rows) continue;
        const int r = r0 + i;
        const long long g = (long long)(x0 + r) * ldz + z0 + c;
        gf[0][g] = sU[r * L.up + c];
        gf[1][g] = sW[r * L.wp + c];
        gf[6][g] = sP[r * L.pp + c];
        gf[7][g] = sQ[r * L.qp + c];
        if (PROG && (inn >> i & 1)) {
            b.illum[io + (long long)i * b.inz] = il[i];
            b.img[io + (long long)i * b.inz] = im[i];
        }
        if (US && (ub >> i & 1)) continue;   // no split fields there
        gf[2][g] = s0[i];
        gf[4][g] = s1[i];
        gf[3][g] = s2[i];
        gf[5][g] = s3[i];
    }
}

// ---- host side --------------------------------------------------------------
constexpr size_t kStaticLds = 64;   // s_dead, rounded up

using KernelFn = void (*)(Run2dArgs);
// Launch shapes: threads, rows a strip.
struct Shape2d {
    int nt, nu;
};
constexpr Shape2d kShapes[] = {{512, 1}, {1024, 1}, {1024, 2}, {1024, 3}, {1024, 4}, {1024, 6}, {1024, 8}};
constexpr int kNumShapes = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
constexpr int kRtmShapes = kNumShapes - 1;   // the RTM program's images leave no registers for strips of 8

template <bool TTI, bool US, bool PROG>
KernelFn kernel_of(int shape)
{
    switch (shape) {
    case 0: return run2d_kernel<TTI, US, PROG, 512, 1>;
    case 1: return run2d_kernel<TTI, US, PROG, 1024, 1>;
    case 2: return run2d_kernel<TTI, US, PROG, 1024, 2>;
    case 3: return run2d_kernel<TTI, US, PROG, 1024, 3>;
    case 4: return run2d_kernel<TTI, US, PROG, 1024, 4>;
    case 5: return run2d_kernel<TTI, US, PROG, 1024, 6>;
    default: return run2d_kernel<TTI, US, PROG, 1024, PROG ? 6 : 8>;
    }
}

// Tiles of one grid: at least 7 rows and 8 columns (a halo never reaches past
// the next tile), small enough for LDS and for one strip per thread.  cost:
// the estimated cycles of the largest tile's step: instructions at one
// wavefront instruction a cycle and CU (about 20 a velocity cell, 26 with its
// z-stencil, 50 a stress cell; the TTI update twice that), or, where few
// wavefronts leave the CU waiting, the rounds of strips by their latency;
// and the exchanged words.
struct Cut {
    int gx, gz, tiles;
    size_t lds;
    double cost;
};
// out: by ascending tiles, each cheaper than all with fewer
void cuts_of(int nnx, int nnz, bool tti, int shape, int cus, int lds_max, std::vector<Cut> &out)
{
    out.clear();
    const int ux = nnx - 8, uq = (nnz - 8 + 3) / 4;
    if (uq < 2) return;
    const int nt = kShapes[shape].nt, nu = kShapes[shape].nu;
    std::vector<Cut> best(cus + 1, Cut{0, 0, 0, 0, 1e300});   // by tiles
    // more columns or rows of tiles of the same height or width never pay: go
    // on to the next smaller one
    auto next = [](int n, int g) {
        const int size = (n + g - 1) / g;
        return size > 1 ? std::max(g + 1, (n + size - 2) / (size - 1)) : n + 1;
    };
    for (int gx = 1; gx <= std::min(cus, std::max(1, ux / 7)); gx = next(ux, gx)) {
        const int nx = (ux + gx - 1) / gx, rows = (nx + nu - 1) / nu;
        if (nx + 14 > nt || 8 * rows > nt) continue;
        const int widest = nt / rows / 4;   // units of 4 columns that leave a thread one strip
        for (int gz = (uq + widest - 1) / widest; gz <= std::min(cus / gx, std::max(1, uq / 2)); gz = next(uq, gz)) {
            const int nz = 4 * ((uq + gz - 1) / gz);
            const int strips = rows * nz;
            const size_t b = 4 * (size_t)(tti ? Lds<true>(nx, nz).total : Lds<false>(nx, nz).total);
            if (b + kStaticLds > (size_t)lds_max) continue;
            const int us = (nx + 7 + nu - 1) / nu * (tti ? nz + 8 : nz), ws = tti ? 0 : rows * (nz + 8);
            const double f = tti ? 2.0 : 1.0;
            const double issue = f * nu * (20.0 * us + 26.0 * ws + 50.0 * strips) / 64.0;
            const double wait = f * ((us + ws + nt - 1) / nt * (350.0 + 60.0 * nu) + 300.0 + 90.0 * nu);
            const double words = (tti ? 2.0 : 1.0) * 14.0 * (nx + nz + (tti ? 14 : 0));
            const double cost = std::max(issue, wait) + 0.25 * words;
            if (cost < best[gx * gz].cost) best[gx * gz] = Cut{gx, gz, gx * gz, b, cost};
        }
    }
    double least = 1e300;
    for (const Cut &c : best)
        if (c.cost < least) {
            least = c.cost;
            out.push_back(c);
        }
}

struct Device2d {
    int cus = 0, lds = 0;
};
bool device_2d(int device, Device2d &d)
{
    if (hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        hipDeviceGetAttribute(&d.lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// One tile per CU for one shot: the shape and the cut with the least cost.
struct Plan2d {
    double cost = 1e300;
    int shape = 0;
    std::vector<Cut> cut;
};
Plan2d plan_one(const Run2dShot &s, bool tti, const Device2d &d)
{
    Plan2d best;
    std::vector<Cut> cuts;
    for (int k = 0; k < kNumShapes; ++k) {
        cuts_of(s.nnx, s.nnz, tti, k, d.cus, d.lds, cuts);
        if (!cuts.empty() && cuts.back().cost < best.cost) best = Plan2d{cuts.back().cost, k, {cuts.back()}};
    }
    return best;
}

// One tile per CU for shots together, with one launch shape: the least cost of
// the slowest tile, every shot cut into the fewest tiles within it.  Shots are
// added one by one: the cost only rises then, and a shot's tiles only get fewer
// (planned anew for every number of shots, 256 shots took 30 ms).
struct PartPlan {
    using Cuts = std::vector<Cut>;      // of one grid: ascending tiles, descending cost
    double cost = 0.0;
    int tiles = 0;
    bool fits = true;
    std::vector<const Cuts *> cuts;     // by shot
    std::vector<int> pick;
    std::priority_queue<std::pair<double, int>, std::vector<std::pair<double, int>>, std::greater<>> next;   // cost of
                                                                                       // the next fewer tiles, shot
    void take(int s)                    // the fewest tiles within the cost
    {
        const Cuts &c = *cuts[s];
        if (pick[s] >= 0) tiles -= c[pick[s]].tiles;
        pick[s] = (int)(std::partition_point(c.begin(), c.end(), [&](const Cut &x) { return x.cost > cost; }) - c.begin());
        tiles += c[pick[s]].tiles;
        if (pick[s]) next.push({c[pick[s] - 1].cost, s});
    }
    void relax()
    {
        while (!next.empty() && next.top().first <= cost) {
            const int s = next.top().second;
            next.pop();
            take(s);
        }
    }
    void add(const Cuts &c, int cus)
    {
        fits = fits && !c.empty();
        if (!fits) return;
        cuts.push_back(&c);
        pick.push_back(-1);
        cost = std::max(cost, c.back().cost);
        relax();
        take((int)cuts.size() - 1);
        while (tiles > cus && !next.empty()) {
            cost = next.top().first;
            relax();
        }
        fits = tiles <= cus;
    }
};

size_t plane_of(const Run2dShot &s) { return (size_t)s.ldz * s.nnx; }

// words of the exchange planes, two a field
size_t plane_words(const Run2dShot *shots, int n, int nfield)
{
    size_t w = 0;
    for (int k = 0; k < n; ++k) w += 2 * nfield * plane_of(shots[k]);
    return w;
}
void place_planes(Run2dShot *shots, int n, int nfield, unsigned long long *p)
{
    for (int k = 0; k < n; ++k) {
        Run2dShot &b = shots[k];
        b.xstride = (long long)plane_of(b);
        b.xP = p;
        b.xQ = p + 2 * plane_of(b);
        b.xU = nfield > 2 ? p + 4 * plane_of(b) : nullptr;
        b.xW = nfield > 2 ? p + 6 * plane_of(b) : nullptr;
        p += 2 * nfield * plane_of(b);
    }
}

// Allocations that leave alone a capture of another stream, which the default
// mode would end.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// a context's exchange planes, zeroed, and its host-visible error word
bool alloc_plan(const Run2dShot &shot, unsigned long long *&xbuf, int *&dead, hipStream_t s)
{
    const size_t n = plane_words(&shot, 1, 2);
    const RelaxedCapture relaxed;
    if (hipMalloc(&xbuf, n * sizeof(unsigned long long)) != hipSuccess) xbuf = nullptr;
    else if (hipHostMalloc(&dead, sizeof(int), hipHostMallocMapped) != hipSuccess) dead = nullptr;
    else if (launch_zero(reinterpret_cast<float *>(xbuf), 2 * n, s) == hipSuccess) {
        *dead = 0;
        return true;
    }
    (void)hipFree(xbuf);
    (void)hipHostFree(dead);
    xbuf = nullptr;
    dead = nullptr;
    (void)hipGetLastError();
    return false;
}

bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone;
}

thread_local long long t_launches = 0;   // vti_resident_launches
thread_local long long t_left = -1;      // vti_resident_limit
thread_local unsigned t_wait = kWaitTicks;   // vti_resident_wait

// The resident launches on one device.  The workgroups of a launch wait for
// each other, one a CU at most: they all get a place once the kernels before
// them and beside them end, unless another resident launch holds some of the
// places and waits for the rest.  So no two are ever under way at once: those of
// this process follow each other (one stream's by themselves, those of several
// streams by events), and a process has the device's resident launches to itself
// while an object that makes them lives (a name in the abstract socket
// namespace, which the kernel takes back when the process ends); the others run
// the per-step kernels.
// A cooperative launch promises the same, on a hardware queue of its own, the
// fifth of a process with four.  Two queues then share a pipe, and while both
// have work every launch on either takes ~25 us instead of 3, also long after
// the cooperative one: gradients of 60 x 50, 200 steps, in 8 threads took 20 ms
// before the process's first cooperative launch and 73 after it.
struct Chip {
    std::mutex m;
    std::string id;                      // of the device, the same in every process
    int name = -1;                       // the socket bound to it
    std::map<hipStream_t, int> streams;  // of the objects that launch here
    hipStream_t last = nullptr;          // of the latest launch that may be under way
    hipEvent_t done = nullptr;           // after it, where there are several streams
};
Chip &chip_of(int device)
{
    static std::mutex m;
    static auto *all = new std::map<int, Chip>;   // outlives every thread
    const std::lock_guard<std::mutex> l(m);
    return (*all)[device];
}

bool take_device(Chip &c, int device)
{
    if (c.name >= 0) return true;
    if (c.id.empty()) {
        char pci[32] = "";
        hipUUID u{};
        hipDevice_t d;
        if (hipDeviceGetPCIBusId(pci, sizeof pci, device) != hipSuccess || hipDeviceGet(&d, device) != hipSuccess ||
            hipDeviceGetUuid(&u, d) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        c.id = std::string("vti-resident-") + pci + "-";
        for (const char b : u.bytes) {
            c.id += "0123456789abcdef"[b >> 4 & 15];
            c.id += "0123456789abcdef"[b & 15];
        }
    }
    sockaddr_un a{};
    a.sun_family = AF_UNIX;   // sun_path[0] stays 0: no file
    c.id.copy(a.sun_path + 1, sizeof a.sun_path - 1);
    const size_t n = offsetof(sockaddr_un, sun_path) + 1 + std::min(c.id.size(), sizeof a.sun_path - 1);
    const int fd = socket(AF_UNIX, SOCK_STREAM | SOCK_CLOEXEC, 0);
    if (fd < 0) return false;
    if (bind(fd, reinterpret_cast<sockaddr *>(&a), (socklen_t)n)) {
        close(fd);
        return false;
    }
    c.name = fd;
    return true;
}

// the latest launch, waited for by events from here on, or here
void note(Chip &c)
{
    if (!c.last) return;
    const RelaxedCapture relaxed;
    if ((!c.done && hipEventCreateWithFlags(&c.done, hipEventDisableTiming) != hipSuccess) ||
        hipEventRecord(c.done, c.last) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipStreamSynchronize(c.last);
        c.last = nullptr;
    }
}

// A short call does not wait for another stream's launch: the per-step kernels
// run beside it.  ms for 400 steps of a context, 8 threads, per-step kernels /
// waiting / this rule, in calls of 8, 16, 24, 32 steps: 60 x 50 0.97, 1.29, 0.86 /
// 0.96, 1.00, 0.89 / 0.96, 0.91, 0.91 / 0.96, 0.86, 0.87; 400 x 400 1.65, 2.04,
// 1.60 / 1.65, 1.64, 1.59 / 1.65, 1.52, 1.50 / 1.66, 1.45, 1.43.
constexpr int kShareSteps = 24;
bool under_way(const Chip &c)
{
    const RelaxedCapture relaxed;
    const bool yes = hipEventQuery(c.done) == hipErrorNotReady;
    (void)hipGetLastError();
    return yes;
}

// An object that launches on s: false: not on this stream (one that may not use
// all CUs), or not now.
bool chip_enter(int device, hipStream_t s)
{
    Device2d d;
    if (!device_2d(device, d)) return false;
    uint32_t mask[64] = {};
    if (hipExtStreamGetCUMask(s, 64, mask) == hipSuccess) {
        int n = 0;
        for (const uint32_t w : mask) n += __builtin_popcount(w);
        if (n < d.cus) return false;
    } else {
        (void)hipGetLastError();
    }
    Chip &c = chip_of(device);
    const std::lock_guard<std::mutex> l(c.m);
    const bool second = c.streams.size() == 1 && !c.streams.count(s);
    // an event recorded there now would belong to the graph that is captured
    if (second && c.last && capturing(c.last)) return false;
    ++c.streams[s];
    if (second) note(c);
    return true;
}
// its launches have been waited for
void chip_leave(int device, hipStream_t s)
{
    Chip &c = chip_of(device);
    const std::lock_guard<std::mutex> l(c.m);
    const auto i = c.streams.find(s);
    if (i == c.streams.end() || --i->second) return;
    c.streams.erase(i);
    if (c.last == s) c.last = nullptr;
    if (c.streams.empty() && c.name >= 0) {
        close(c.name);
        c.name = -1;
    }
}

hipError_t launch_resident(int device, KernelFn k, int grid, int nt, size_t lds, Run2dArgs &a, int steps, hipStream_t s)
{
    if (t_left == 0) return hipErrorOutOfMemory;
    a.wait = t_wait;
    void *args[] = {&a};
    // The function's own limit, which its callers in all threads share: always
    // the same value, what a workgroup can have, never this launch's need.
    static const int lds_max = [] {
        int device = 0, n = 0;
        if (hipGetDevice(&device) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
            (void)hipGetLastError();
        return n;
    }();
    Chip &c = chip_of(device);
    const std::lock_guard<std::mutex> l(c.m);
    if (!take_device(c, device)) return hipErrorNotReady;
    hipError_t e = hipSuccess;
    if (c.last && c.last != s) {
        if (steps < kShareSteps && under_way(c)) return hipErrorNotReady;
        e = hipStreamWaitEvent(s, c.done, 0);
    }
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                std::max((int)lds, lds_max - (int)kStaticLds));
    if (e == hipSuccess) e = hipLaunchKernel(reinterpret_cast<const void *>(k), dim3(grid), dim3(nt), args, lds, s);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return e;
    }
    c.last = s;
    if (c.streams.size() > 1) note(c);
    ++t_launches;
    if (t_left > 0) --t_left;
    return e;
}

}  // namespace

struct Run2dPlan {
    int device = 0;
    bool entered = false;       // on this stream
    hipStream_t stream = nullptr;
    int ok = 0;                 // 1: usable, 0: not planned yet, -1: this grid or device takes the per-step kernels
    std::vector<Run2dShot> shot;   // one: the plan's share of it
    int shape = 0, ntile = 0;
    size_t lds = 0;
    bool tti = false;
    unsigned long long *xbuf = nullptr;
    unsigned base = 1;
    int *dead = nullptr;
};

void run2d_free(vti_ctx *c)
{
    if (!c->run2d) return;
    (void)hipFree(c->run2d->xbuf);   // waits for the device
    (void)hipHostFree(c->run2d->dead);
    run2d_leave(c);
    delete c->run2d;
    c->run2d = nullptr;
}

void run2d_leave(vti_ctx *c)
{
    if (!c->run2d || !c->run2d->entered) return;
    chip_leave(c->run2d->device, c->run2d->stream);
    c->run2d->entered = false;
}

// The forward side of a context's shot on state s.
Run2dShot run2d_shot(vti_ctx *c, const VtiState &s)
{
    Run2dShot a{};
    a.nnx = c->g.nnx; a.nnz = c->g.nnz; a.ldz = c->g.ldz; a.M = c->nnmax;
    static const int kF[8] = {VTI_F_U, VTI_F_W, VTI_F_PX, VTI_F_PZ, VTI_F_QX, VTI_F_QZ, VTI_F_P, VTI_F_Q};
    for (int k = 0; k < 8; ++k) a.f[k] = s.f[kF[k]];
    a.vp = c->vp; a.ep = c->ep; a.de = c->de;
    a.cth = c->tti;
    a.sth = c->tti ? c->tti + c->nvol : nullptr;
    a.tab = c->tab;
    a.dtx = c->cfg.dt / c->cfg.dx; a.dtz = c->cfg.dt / c->cfg.dz;
    a.sv = c->cfg.sv != 0; a.svR = c->cfg.sv_R; a.cx = c->shot.sv_cx; a.cz = c->shot.sv_cz;
    a.tap = c->dtap;
    a.point = c->cfg.mode == VTI_MODE_GPU_REF;
    a.sx = c->shot.sx; a.sz = c->shot.sz;
    a.gw = c->dgw;
    a.amp = c->damp;
    a.rec = c->nrec > 0 ? c->rec : nullptr;
    a.nrec = c->nrec; a.rec_kind = c->cfg.rec_kind;
    a.rz = c->shot.rec_z; a.rx0 = c->shot.rec_x0; a.rdx = c->shot.rec_dx; a.rnx = c->shot.rec_nx;
    a.split_z = a.rzi = -1;
    a.inp = c->cfg.npml; a.inx = c->cfg.nx; a.inz = c->cfg.nz;
    return a;
}

// n steps from it0 of the main state, when one resident launch applies:
// 1 launched, 0 not applicable (the caller runs the per-step kernels), < 0
// an error.
int run2d_steps(vti_ctx *c, int it0, int n)
{
    // Two steps let the write-back start after every neighbour has loaded.
    // Eight are the fewest that were measured, and faster: us a call of 8 / 10 /
    // 16 steps among others, per-step kernels and resident, 200 x 150 46, 24 /
    // 58, 27 / 91, 39; 400 x 400 58, 36 / 72, 42 / 114, 60; 2401 x 803 222, 122 /
    // 281, 143 / 460, 205.
    if (c->cfg.ndim != 2 || c->cfg.mode == VTI_MODE_OMP_REF || capturing(c->stream)) return 0;
    // The plan and its memory cost a context's first such call 60 to 400 us, a
    // step saves 4 to 18: us of a fresh context's first call of 16 / 24 / 32
    // steps, per-step kernels and resident, 200 x 150 106, 108 / 149, 130 / 197,
    // 132; 400 x 400 126, 155 / 183, 189 / 240, 207; 1401 x 503 254, 457 / 370,
    // 226 / 488, 270; 2401 x 803 532, 630 / 782, 475 / 1033, 535.
    if (!c->run2d) c->asked2d += n;
    if (n < 8 || (!c->run2d && c->asked2d < 24)) return 0;
    const bool tti = c->tti != nullptr;
    if (!c->run2d) c->run2d = new (std::nothrow) Run2dPlan();
    if (!c->run2d) return 0;
    Run2dPlan &p = *c->run2d;
    if (!p.ok || p.tti != tti) {   // both forms use the planes alike
        p.tti = tti;
        p.ok = -1;
        Device2d d;
        p.shot.assign(1, run2d_shot(c, main_state(c)));
        if (!device_2d(c->device, d)) return 0;
        const Plan2d one = plan_one(p.shot[0], tti, d);
        if (one.cut.empty() || (!p.xbuf && !alloc_plan(p.shot[0], p.xbuf, p.dead, c->stream))) return 0;
        place_planes(p.shot.data(), 1, 2, p.xbuf);
        p.shape = one.shape;
        p.lds = one.cut[0].lds;
        p.ntile = one.cut[0].tiles;
        p.shot[0].gx = one.cut[0].gx;
        p.shot[0].gz = one.cut[0].gz;
        p.ok = 1;
    }
    if (p.ok != 1) return 0;
    Run2dArgs a{};
    const Run2dShot &t = p.shot[0];
    a.one = run2d_shot(c, main_state(c));
    a.one.gx = t.gx; a.one.gz = t.gz;
    a.one.xP = t.xP; a.one.xQ = t.xQ; a.one.xstride = t.xstride;
    a.ns = 1;
    a.it0 = it0; a.n = n;
    a.base = p.base;
    a.dead = p.dead;
    const bool us = c->unsplit && c->cfg.mode == VTI_MODE_GPU_REF && !tti;
    const KernelFn k = tti ? kernel_of<true, false, false>(p.shape)
                           : (us ? kernel_of<false, true, false>(p.shape) : kernel_of<false, false, false>(p.shape));
    if (!p.entered && !chip_enter(c->device, c->stream)) return 0;
    p.entered = true;
    p.device = c->device;
    p.stream = c->stream;
    // another process has the device, no memory: the next call tries again
    if (launch_resident(p.device, k, p.ntile, kShapes[p.shape].nt, p.lds, a, n, c->stream) != hipSuccess) return 0;
    p.base += (unsigned)n;
    if (us) c->us_dirty = true;
    return 1;
}

static int dead_check(int *dead, int &ok)
{
    if (!dead || !*dead) return VTI_OK;
    *dead = 0;
    ok = -1;          // later steps take the per-step kernels
    return fail(VTI_ERR_HIP, "resident 2D steps: a tile's exchange did not arrive");
}

// after the context's stream has been waited for: an exchange that never came
int run2d_check(vti_ctx *c) { return c->run2d ? dead_check(c->run2d->dead, c->run2d->ok) : VTI_OK; }

// ---- groups of shots (RTM) ---------------------------------------------------
// Consecutive shots to a part while that lowers the time a cell: the slowest
// tile's cost and what a step costs besides (exchange, barriers: ~2 us).
Run2dParts run2d_parts(const std::vector<Run2dShot> &shots, int device)
{
    Run2dParts r;
    Device2d d;
    if (!device_2d(device, d)) return r;
    const int ns = (int)shots.size();
    // one list of cuts a shape and grid
    std::map<std::pair<int, int>, int> grids;
    std::vector<int> grid(ns);
    std::vector<PartPlan::Cuts> cuts[kRtmShapes];
    for (int k = 0; k < ns; ++k) {
        const auto g = grids.insert({{shots[k].nnx, shots[k].nnz}, (int)grids.size()});
        grid[k] = g.first->second;
        for (int j = 0; g.second && j < kRtmShapes; ++j) {
            cuts[j].emplace_back();
            cuts_of(shots[k].nnx, shots[k].nnz, false, j, d.cus, d.lds, cuts[j].back());
        }
    }
    // strips of 6 spill ~80 registers with the images: for shots that fit no
    // other way (24 shots of 0.1 to 1 M cells: 46 ms in parts of strips of 6
    // taken at their plain cost, 39 with parts of 4)
    for (auto &c : cuts[kRtmShapes - 1])
        for (Cut &x : c) x.cost *= 2.0;
    for (int first = 0; first < ns;) {
        Plan2d best;
        PartPlan plan[kRtmShapes];
        double rate = 1e300, cells = 0.0;
        for (int n = 1; first + n <= ns; ++n) {
            cells += (double)shots[first + n - 1].nnx * shots[first + n - 1].nnz;
            int least = -1;
            for (int j = 0; j < kRtmShapes; ++j) {
                plan[j].add(cuts[j][grid[first + n - 1]], d.cus);
                if (plan[j].fits && (least < 0 || plan[j].cost < plan[least].cost)) least = j;
            }
            if (least < 0) break;
            const PartPlan &p = plan[least];
            if ((p.cost + 4000.0) / cells >= rate) continue;
            rate = (p.cost + 4000.0) / cells;
            best = Plan2d{p.cost, least, {}};
            for (int k = 0; k < n; ++k) best.cut.push_back((*p.cuts[k])[p.pick[k]]);
        }
        if (best.cut.empty()) return Run2dParts{};
        Run2dPart q{first, (int)best.cut.size(), best.shape, 0, 0};
        for (const Cut &c : best.cut) {
            r.gx.push_back(c.gx);
            r.gz.push_back(c.gz);
            r.tile0.push_back(q.ntile);
            q.ntile += c.tiles;
            q.lds = std::max(q.lds, c.lds);
        }
        r.part.push_back(q);
        first += q.n;
    }
    return r;
}

// one allocation: exchange planes (tag 0; the parts run one after the other
// and share them), error word, shots, program
int run2d_group_make(Run2dGroup &g, const Run2dParts &p, std::vector<Run2dShot> shots, bool us, int nt, hipStream_t s)
{
    g.ok = 0;
    if (p.part.empty() || capturing(s)) return 0;
    if (hipGetDevice(&g.device) != hipSuccess) return fail(VTI_ERR_HIP, "run2d: device");
    if (!chip_enter(g.device, s)) return 0;
    g.entered = true;
    g.stream = s;
    g.parts = p;
    g.us = us;
    g.words = 0;
    for (const Run2dPart &q : p.part) g.words = std::max(g.words, plane_words(&shots[q.first], q.n, 4));
    const size_t head = (g.words + 32) * 8, desc = (shots.size() * sizeof(Run2dShot) + 255) / 256 * 256;
    g.prog_bytes = 128 * (size_t)nt + 65536;
    if (hipMalloc(&g.mem, head + desc + g.prog_bytes) != hipSuccess) {
        (void)hipGetLastError();
        g.mem = nullptr;
        return 0;
    }
    char *m = static_cast<char *>(g.mem);
    g.dead = reinterpret_cast<int *>(m + g.words * 8);
    g.dev = reinterpret_cast<Run2dShot *>(m + head);
    g.prog = m + head + desc;
    if (launch_zero(static_cast<float *>(g.mem), head / 4, s) != hipSuccess) return fail(VTI_ERR_HIP, "run2d: planes");
    const int e = run2d_group_set(g, std::move(shots), s);
    if (e) return e;
    g.ok = 1;
    return 1;
}

int run2d_group_set(Run2dGroup &g, std::vector<Run2dShot> shots, hipStream_t s)
{
    g.refused = false;
    const Run2dParts &p = g.parts;
    for (size_t k = 0; k < shots.size(); ++k) {
        shots[k].gx = p.gx[k];
        shots[k].gz = p.gz[k];
        shots[k].tile0 = p.tile0[k];
    }
    for (const Run2dPart &q : p.part) place_planes(&shots[q.first], q.n, 4, static_cast<unsigned long long *>(g.mem));
    if (hipMemcpyAsync(g.dev, shots.data(), shots.size() * sizeof(Run2dShot), hipMemcpyHostToDevice, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return fail(VTI_ERR_HIP, "run2d: descriptors");
    return VTI_OK;
}

void run2d_group_free(Run2dGroup &g)
{
    (void)hipFree(g.mem);   // waits for the device
    (void)hipFree(g.more);
    if (g.entered) chip_leave(g.device, g.stream);
    g = Run2dGroup{};
}

// prog: the operations, then the offsets
int run2d_group_run(Run2dGroup &g, const std::vector<Run2dOp> &ops, const std::vector<long long> &offs, int image_every,
                    hipStream_t s)
{
    if (g.ok != 1 || g.refused) return 0;
    const size_t nb = ops.size() * sizeof(Run2dOp), need = nb + std::max<size_t>(offs.size(), 1) * sizeof(long long);
    if (need > g.prog_bytes) {
        if (hipStreamSynchronize(s) != hipSuccess) return fail(VTI_ERR_HIP, "run2d: sync");
        (void)hipFree(g.more);
        g.more = nullptr;
        if (hipMalloc(&g.more, 2 * need) != hipSuccess) {
            (void)hipGetLastError();
            g.more = nullptr;
            g.prog_bytes = 0;
            g.refused = true;
            return 0;
        }
        g.prog = g.more;
        g.prog_bytes = 2 * need;
    }
    static_assert(sizeof(Run2dOp) % sizeof(long long) == 0, "the offsets follow the operations");
    char *p = static_cast<char *>(g.prog);
    if (hipMemcpyAsync(p, ops.data(), nb, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(p + nb, offs.data(), offs.size() * sizeof(long long), hipMemcpyHostToDevice, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return fail(VTI_ERR_HIP, "run2d: program");
    for (const Run2dPart &q : g.parts.part) {
        Run2dArgs a{};
        a.many = g.dev + q.first;
        a.ns = q.n;
        a.ops = reinterpret_cast<const Run2dOp *>(p);
        a.nops = (int)ops.size();
        a.offs = reinterpret_cast<const long long *>(p + nb);
        a.image_every = image_every;
        a.base = g.base;
        a.dead = g.dead;
        const KernelFn k = g.us ? kernel_of<false, true, true>(q.shape) : kernel_of<false, false, true>(q.shape);
        if (launch_resident(g.device, k, q.ntile, kShapes[q.shape].nt, q.lds, a, kShareSteps, s) != hipSuccess) {
            g.refused = true;
            return &q == &g.parts.part.front() ? 0 : 2;
        }
        g.ran = true;
        g.base += (unsigned)(offs.size() + 2);   // one exchange a step
    }
    return 1;
}

int run2d_group_check(Run2dGroup &g, hipStream_t s)
{
    if (!g.ran) return VTI_OK;
    g.ran = false;
    int dead = 0;
    if (hipMemcpyAsync(&dead, g.dead, sizeof dead, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return fail(VTI_ERR_HIP, "run2d: check");
    if (dead && launch_zero(reinterpret_cast<float *>(g.dead), 1, s) != hipSuccess) return fail(VTI_ERR_HIP, "run2d: check");
    return dead_check(&dead, g.ok);
}

int RtmProgram::steps(int kind, bool first, int it, long long off)
{
    const int d = kind == 2 ? -1 : 1;
    if (!ops.empty()) {
        Run2dOp &l = ops.back();
        if (l.kind == kind && l.first == (int)first && it == l.it0 + d * l.n) {
            ++l.n;
            offs.push_back(off);
            return VTI_OK;
        }
    }
    // the run goes on from the state on the chip, a forward one over checkpoints
    for (size_t k = ops.size(); k-- > 0;) {
        if (kind == 1 && ops[k].kind == 3) continue;
        if (ops[k].kind == kind) ops[k].link = 1;
        break;
    }
    ops.push_back(Run2dOp{kind, it, 1, (int)first, 0, (int)offs.size(), 0});
    offs.push_back(off);
    return VTI_OK;
}

int RtmProgram::keep_last(long long off)
{
    if (ops.empty() || ops.back().kind != 1 || offs.back()) return fail(VTI_ERR_STATE, "RTM program: no step to keep");
    offs.back() = off;
    return VTI_OK;
}

int RtmProgram::state(int kind, long long slot)
{
    // a checkpoint is written from the chip
    if (kind == 3 && (ops.empty() || ops.back().kind != 1)) return fail(VTI_ERR_STATE, "RTM program: no step to store");
    ops.push_back(Run2dOp{kind, 0, 0, 0, 0, 0, slot});
    return VTI_OK;
}

int RtmProgram::flush()
{
    std::vector<Run2dOp> o;
    std::vector<long long> f;
    o.swap(ops);
    f.swap(offs);
    if (o.empty()) return VTI_OK;
    int e = run(o, f);
    if (e) return e < 0 ? e : VTI_OK;
    for (const Run2dOp &op : o) {
        if (op.kind >= 3) e = move(op.kind, op.slot);
        else
            for (int k = 0; k < op.n && !e; ++k) {
                if (op.kind == 2) e = receive(op.it0 - k, f[op.off0 + k]);
                else if (!(e = step(op.first != 0, op.it0 + k)) && f[op.off0 + k]) e = keep(f[op.off0 + k]);
            }
        if (e) return e;
    }
    return VTI_OK;
}

}  // namespace vti

extern "C" long long vti_resident_launches(void) { return vti::t_launches; }

extern "C" void vti_resident_limit(long long n) { vti::t_left = n < 0 ? -1 : n; }

extern "C" void vti_resident_wait(long long us)
{
    vti::t_wait = us < 0 ? vti::kWaitTicks : (unsigned)std::min(us, (long long)vti::kWaitTicks / 100) * 100;
}
