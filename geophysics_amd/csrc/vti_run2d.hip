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
// What bounds a step now: the exchange, ~0.8 us from one XCD's store to
// another's load, then LDS latency and instruction issue.  Measured (us a
// step, velocity + stress launches -> this): 60 x 50 with a 20-cell layer
// 5.8 -> 1.9, 400 x 400 7.2 -> 2.8, TTI 600 x 300 with a 50-cell layer
// 10.7 -> 5.2, 2401 x 803 unsplit 27.9 -> 11.3.
//
// The arithmetic is vel2d_kernel's / stress2d_kernel's (and the TTI pair's)
// term by term; products that do not change from step to step are formed
// once in the same order, so every field and record is the same bit for bit
// (update_vel2d GPU_vti2dfd_kernels.cu:209-238, update_stress2d :240-299,
// CPU_vti2dfd_kernels.c:78-177, Toa_gpu_2dtti_fd_1orderfunction.cu:81-183).
//
// Launch: cooperative (all workgroups resident, or the launch fails and the
// per-step kernels run).  Every wait ends: a sample that does not come within
// kWaitTicks raises the error word and the workgroup leaves its loop.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>

#include "vti_internal.h"

namespace vti {
namespace {

__device__ __forceinline__ float cst(int m)
{
    return m == 0 ? 1.196289f : (m == 1 ? -0.0797526f : (m == 2 ? 0.009570313f : -0.0006975447f));
}

// 100 MHz ticks a neighbour's sample may take before the call is given up (20 s)
constexpr unsigned long long kWaitTicks = 2000000000ull;

struct Run2dArgs {
    int nnx, nnz, ldz, M;
    float *u, *w, *px, *pz, *qx, *qz, *P, *Q;
    const float *vp, *ep, *de, *cth, *sth, *tab;
    float dtx, dtz;
    int sv, svR, cx, cz;
    const double *tap;
    int point, sx, sz;          // point source (load-time) or the 7x7 footprint in the stress update
    const double *gw;
    const float *amp;           // nt source gains
    float *rec;                 // [it][nrec], nullptr: no record
    int nrec, rec_kind, rz, rx0, rdx, rnx;
    int it0, n;
    int gx, gz;                 // tiles in x and z
    unsigned long long *xP, *xQ;   // exchange planes, two each, of (tag, float) words
    long long xstride;
    unsigned base;              // tag of the call's first step
    int *dead;                  // host-visible error word
};

// an opaque copy: what is derived from it inside the step loop is not hoisted
// out of it (addresses and masks of every row: more registers than there are)
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

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
// the word's sample once it carries the tag (w: an earlier look at it)
__device__ __forceinline__ float await(const unsigned long long *p, unsigned long long w, unsigned tag, int *dead)
{
    if ((unsigned)(w >> 32) != tag) {
        const unsigned long long t0 = wall_clock64();
        do {
            w = peek(p);
            if (wall_clock64() - t0 > kWaitTicks) {
                *dead = 1;
                break;
            }
        } while ((unsigned)(w >> 32) != tag);
    }
    return __uint_as_float((unsigned)w);
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
template <bool TTI, bool US, int NT, int NU>
__global__ __launch_bounds__(NT) void run2d_kernel(Run2dArgs a)
{
    extern __shared__ float4 smem4[];
    float *sm = reinterpret_cast<float *>(smem4);
    __shared__ int s_dead;
    const int tid = threadIdx.x;
    const Tile t = tile_of(a.nnx, a.nnz, a.gx, a.gz, blockIdx.x / a.gz, blockIdx.x % a.gz);
    const int nx = t.nx, nz = t.nz, x0 = t.x0, z0 = t.z0;
    const Lds<TTI> L(nx, nz);
    const int ldz = a.ldz, zend = a.nnz - 4, xend = a.nnx - 4, M = a.M;
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
        *reinterpret_cast<float4 *>(sm + k) = ldg4(q ? a.Q : a.P, a.nnx, ldz, x0 + r, z0 + c);
    }
    for (int k = L.ou + 4 * tid; k < L.oc; k += 4 * NT) {   // u and w
        const bool q = k >= L.ow;
        const int i = q ? k - L.ow : k - L.ou, pitch = q ? L.wp : L.up;
        const int r = i / pitch - (q ? (TTI ? 4 : 0) : 4), c = i % pitch - ((q || TTI) ? 4 : 0);
        *reinterpret_cast<float4 *>(sm + k) = ldg4(q ? a.w : a.u, a.nnx, ldz, x0 + r, z0 + c);
    }
    if (TTI)
        for (int k = L.oc + 4 * tid; k < L.ot; k += 4 * NT) {
            const bool q = k >= L.os;
            const int i = q ? k - L.os : k - L.oc;
            *reinterpret_cast<float4 *>(sm + k) = ldg4(q ? a.sth : a.cth, a.nnx, ldz, x0 + i / L.up - 4, z0 + i % L.up - 4);
        }
    auto tabv = [&](int row, int i) { return i >= 0 && i < M ? a.tab[(long long)row * M + i] : 0.0f; };
    // velocity tables: VTI: coff1 * dt/dx (the reference's first product), coff2; TTI: the factors themselves
    for (int k = tid; k < nx + 7; k += NT) {
        kx1[k - 4] = TTI ? tabv(0, x0 + k - 4) : tabv(0, x0 + k - 4) * a.dtx;
        kx2[k - 4] = tabv(1, x0 + k - 4);
    }
    for (int k = tid; k < nx; k += NT) {
        ax1[k] = tabv(6, x0 + k);
        ax2[k] = tabv(7, x0 + k);
    }
    for (int k = tid; k < nz + 8; k += NT) {
        kz1[k - 4] = TTI ? tabv(4, z0 + k - 4) : tabv(4, z0 + k - 4) * a.dtz;
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
        const float v = a.vp[g];
        float ee = a.ep[g], dd = a.de[g];
        s0[i] = a.px[g];
        s1[i] = a.qx[g];
        s2[i] = a.pz[g];
        s3[i] = a.qz[g];
        const float tx1 = ax1[r0 + i], tx2 = ax2[r0 + i], tz1 = az1[c], tz2 = az2[c];
        if (a.sv) {   // SV taper (GPU_vti2dfd_kernels.cu:260-278)
            const int rx = x - a.cx, rz = z - a.cz, r2 = rx * rx + rz * rz;
            if (r2 <= a.svR * a.svR) {
                const double f = a.tap[r2];
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
            c0[i] = tx1 * v * v * e2 * a.dtx;
            c1[i] = tx1 * v * v * sd * a.dtx;
            c2[i] = tz1 * v * v * sd * a.dtz;
            c3[i] = tz1 * v * v * a.dtz;
        }
        if (US && tx1 == 1.0f && tx2 == 1.0f && tz1 == 1.0f && tz2 == 1.0f) {
            und |= 1 << i;
            s0[i] = sP[(r0 + i) * L.pp + c];
            s1[i] = sQ[(r0 + i) * L.qp + c];
        }
        if (a.rec && z == a.rz) {
            const int k = x - a.rx0;
            if (k >= 0 && k % a.rdx == 0 && k / a.rdx < a.rnx) {
                if (!recs) krec = k / a.rdx;
                recs |= 1 << i;
            }
        }
    }

    const int srow = a.sx - x0, scol = a.sz - z0;
    const bool src_p = a.point && srow >= -7 && srow < nx + 7 && scol >= (TTI ? -8 : 0) && scol < nz + (TTI ? 8 : 0);
    const bool src_q = a.point && srow >= (TTI ? -7 : 0) && srow < nx + (TTI ? 7 : 0) && scol >= -8 && scol < nz + 8;

    // the strip is in registers before the step loop, whose waits would
    // otherwise count these loads as possibly still on their way
#pragma unroll
    for (int i = 0; i < NU; ++i)
        asm volatile("" : "+v"(s0[i]), "+v"(s1[i]), "+v"(s2[i]), "+v"(s3[i]), "+v"(c0[i]), "+v"(c1[i]), "+v"(c2[i]), "+v"(c3[i]));
    if (US) __syncthreads();   // P and Q are in s0 and s1 before the source is added to them in LDS
    float amps = 0.0f;   // lane k: the gain of step k of the current 64
    for (int s = 0; s < a.n; ++s) {
        const int it = a.it0 + s;
        if ((s & 63) == 0) {
            amps = a.amp[a.it0 + min(s + (tid & 63), a.n - 1)];
            // taken here: waited for at the top of each step, the load would
            // hold the step until the stores before it are acknowledged too
            asm volatile("" : "+v"(amps));
        }
        const float amp = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(amps), s & 63));
        const int vt = opaque(tid), r0 = opaque(row0), c = opaque(col0);
        if (s > 0) {
            // ---- the neighbours' outer rows and columns of the last step ----
            const unsigned tag = a.base + s;
            const unsigned long long *gP = a.xP + (s & 1) * a.xstride, *gQ = a.xQ + (s & 1) * a.xstride;
            const int nrow = 14 * nz;
            const int wide = 14 * (nz + 14), nget = (TTI ? wide : nrow) + 14 * nx;
            const int total = TTI ? 2 * nget : nget;
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
                    if (at[j] >= 0) sm[at[j]] = await(p[j], w[j], tag, &s_dead);
            }
            __syncthreads();
            if (s_dead) {   // the same for every thread: written before the barrier only
                if (tid == 0) *a.dead = 1;
                return;
            }
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
                            const float u = g2 * *pu - g1 * (cs * a.dtx * d - sn * a.dtz * Pz);
                            const float w = g2 * *pw - g1 * (sn * a.dtx * Qx + cs * a.dtz * Qz);
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
            const int nr = opaque(rows), ub = opaque(und), rb = opaque(recs);
            const bool foot = !a.point && amp != 0.0f, more = s + 1 < a.n;
            unsigned long long *gP = a.xP + ((s + 1) & 1) * a.xstride, *gQ = a.xQ + ((s + 1) & 1) * a.xstride;
            const unsigned tag = a.base + s + 1;
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
                    xx = cs * a.dtx * xx - sn * a.dtz * uz;
                    zz = sn * a.dtx * wx + cs * a.dtz * zz;
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
                        const int fdx = x0 + r - a.sx, fdz = z0 + c - a.sz;
                        if (fdx >= -3 && fdx <= 3 && fdz >= -3 && fdz <= 3) {
                            const float sc = (float)((double)amp * a.gw[(fdx + 3) * 7 + (fdz + 3)]);
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
                    if (ex || (TTI && ez)) put(gP + g, Pn, tag);
                    if (ez || (TTI && ex)) put(gQ + g, Qn, tag);
                }
                if (rb >> i & 1) {
                    const int k = krec + __popc(rb & ((1 << i) - 1));
                    a.rec[(long long)it * a.nrec + k] = a.rec_kind == 0 ? Pn : (a.rec_kind == 1 ? Pn + Pn : Pn + Qn);
                }
            }
        }
        __syncthreads();
    }

    // ---- write the tile back (n >= 2: every neighbour has loaded its halo) ----
    // the field pointers come from the argument segment again: held through
    // the loop they would cost the registers that it needs
    using KArgs = const __attribute__((address_space(4))) Run2dArgs;
    KArgs *b = (KArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(b));
    float *gu = b->u, *gw = b->w, *gP = b->P, *gQ = b->Q, *gpx = b->px, *gqx = b->qx, *gpz = b->pz, *gqz = b->qz;
    if (!live) return;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        if (i >= rows) continue;
        const int r = r0 + i;
        const long long g = (long long)(x0 + r) * ldz + z0 + c;
        gu[g] = sU[r * L.up + c];
        gw[g] = sW[r * L.wp + c];
        gP[g] = sP[r * L.pp + c];
        gQ[g] = sQ[r * L.qp + c];
        if (US && (und >> i & 1)) continue;   // no split fields there
        gpx[g] = s0[i];
        gqx[g] = s1[i];
        gpz[g] = s2[i];
        gqz[g] = s3[i];
    }
}

// ---- host side --------------------------------------------------------------
using KernelFn = void (*)(Run2dArgs);
// Launch shapes: threads, rows a strip.
struct Shape2d {
    int nt, nu;
};
constexpr Shape2d kShapes[] = {{512, 1}, {1024, 1}, {1024, 2}, {1024, 3}, {1024, 4}, {1024, 6}, {1024, 8}};
constexpr int kNumShapes = (int)(sizeof(kShapes) / sizeof(kShapes[0]));

template <bool TTI, bool US>
KernelFn kernel_of(int shape)
{
    switch (shape) {
    case 0: return run2d_kernel<TTI, US, 512, 1>;
    case 1: return run2d_kernel<TTI, US, 1024, 1>;
    case 2: return run2d_kernel<TTI, US, 1024, 2>;
    case 3: return run2d_kernel<TTI, US, 1024, 3>;
    case 4: return run2d_kernel<TTI, US, 1024, 4>;
    case 5: return run2d_kernel<TTI, US, 1024, 6>;
    default: return run2d_kernel<TTI, US, 1024, 8>;
    }
}

}  // namespace

struct Run2dPlan {
    int ok = 0;                 // 1: usable, -1: this grid or device takes the per-step kernels
    int gx = 0, gz = 0, shape = 0;
    size_t lds = 0;
    bool tti = false;
    unsigned long long *xbuf = nullptr;   // xP[2], xQ[2]
    unsigned base = 1;          // the planes start with tag 0
    int *dead = nullptr;        // pinned, mapped
};

void run2d_free(vti_ctx *c)
{
    if (!c->run2d) return;
    (void)hipFree(c->run2d->xbuf);
    (void)hipHostFree(c->run2d->dead);
    delete c->run2d;
    c->run2d = nullptr;
}

namespace {

// Tiles: at most one per CU, at least 7 rows and 8 columns (a halo never
// reaches past the next tile), small enough for LDS and for one strip per
// thread.  Among those the least estimated cycles of the largest tile's step:
// instructions at one wavefront instruction a cycle and CU (about 20 a
// velocity cell, 26 with its z-stencil, 50 a stress cell; the TTI update
// twice that), or, where few wavefronts leave the CU waiting, the rounds of
// strips by their latency; and the exchanged words.
bool plan_tiles(int nnx, int nnz, bool tti, int cus, int lds_max, Run2dPlan &p)
{
    const int ux = nnx - 8, uq = (nnz - 8 + 3) / 4;
    double best = 1e300;
    if (uq < 2) return false;
    for (int gx = 1; gx <= std::min(cus, std::max(1, ux / 7)); ++gx)
        for (int gz = 1; gz <= std::min(cus / gx, std::max(1, uq / 2)); ++gz) {
            const int nx = (ux + gx - 1) / gx, nz = 4 * ((uq + gz - 1) / gz);
            const size_t b = 4 * (size_t)(tti ? Lds<true>(nx, nz).total : Lds<false>(nx, nz).total);
            if (b + 64 > (size_t)lds_max) continue;
            for (int k = 0; k < kNumShapes; ++k) {
                const int nt = kShapes[k].nt, nu = kShapes[k].nu;
                const int strips = (nx + nu - 1) / nu * nz;
                if (strips > nt) continue;
                const int us = (nx + 7 + nu - 1) / nu * (tti ? nz + 8 : nz), ws = tti ? 0 : (nx + nu - 1) / nu * (nz + 8);
                const double f = tti ? 2.0 : 1.0;
                const double issue = f * nu * (20.0 * us + 26.0 * ws + 50.0 * strips) / 64.0;
                const double wait = f * ((us + ws + nt - 1) / nt * (350.0 + 60.0 * nu) + 300.0 + 90.0 * nu);
                const double words = (tti ? 2.0 : 1.0) * 14.0 * (nx + nz + (tti ? 14 : 0));
                const double cost = std::max(issue, wait) + 0.25 * words;
                if (cost < best) {
                    best = cost;
                    p.gx = gx;
                    p.gz = gz;
                    p.lds = b;
                    p.shape = k;
                }
            }
        }
    return best < 1e300;
}

}  // namespace

// n steps from it0 of the main state, when one resident launch applies:
// 1 launched, 0 not applicable (the caller runs the per-step kernels), < 0
// an error.
int run2d_steps(vti_ctx *c, int it0, int n)
{
    // Two steps let the write-back start after every neighbour has loaded.
    // Below eight the call's fixed cost (a cooperative launch, the tile's
    // coefficients, load and store) is more than the per-step kernels take
    // (5.8 us a step and up).
    if (c->cfg.ndim != 2 || n < 8 || c->cfg.mode == VTI_MODE_OMP_REF || !c->damp) return 0;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return 0;
    const bool tti = c->tti != nullptr;
    if (c->run2d && c->run2d->tti != tti) {
        if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(VTI_ERR_HIP, "run2d: sync");
        run2d_free(c);
    }
    if (!c->run2d) {
        c->run2d = new (std::nothrow) Run2dPlan();
        if (!c->run2d) return 0;
        Run2dPlan &p = *c->run2d;
        p.tti = tti;
        p.ok = -1;
        int coop = 0, cus = 0, lds = 0;
        if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, c->device) != hipSuccess || !coop ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess ||
            hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device) != hipSuccess) {
            (void)hipGetLastError();
            return 0;
        }
        if (!plan_tiles(c->g.nnx, c->g.nnz, tti, cus, lds, p)) return 0;
        if (hipMalloc(&p.xbuf, 4 * c->nvol * sizeof(unsigned long long)) != hipSuccess ||
            hipHostMalloc(&p.dead, sizeof(int), hipHostMallocMapped) != hipSuccess) {
            (void)hipGetLastError();
            return 0;
        }
        *p.dead = 0;
        if (launch_zero(reinterpret_cast<float *>(p.xbuf), 8 * c->nvol, c->stream) != hipSuccess)
            return fail(VTI_ERR_HIP, "run2d: exchange planes");
        p.ok = 1;
    }
    Run2dPlan &p = *c->run2d;
    if (p.ok != 1) return 0;
    const VtiState s = main_state(c);
    Run2dArgs a{};
    a.nnx = c->g.nnx; a.nnz = c->g.nnz; a.ldz = c->g.ldz; a.M = c->nnmax;
    a.u = s.f[VTI_F_U]; a.w = s.f[VTI_F_W];
    a.px = s.f[VTI_F_PX]; a.pz = s.f[VTI_F_PZ]; a.qx = s.f[VTI_F_QX]; a.qz = s.f[VTI_F_QZ];
    a.P = s.f[VTI_F_P]; a.Q = s.f[VTI_F_Q];
    a.vp = c->vp; a.ep = c->ep; a.de = c->de;
    a.cth = c->tti;
    a.sth = tti ? c->tti + c->nvol : nullptr;
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
    a.it0 = it0; a.n = n;
    a.gx = p.gx; a.gz = p.gz;
    a.xP = p.xbuf; a.xQ = p.xbuf + 2 * c->nvol;
    a.xstride = (long long)c->nvol;
    a.base = p.base;
    a.dead = p.dead;
    const bool us = c->unsplit && c->cfg.mode == VTI_MODE_GPU_REF && !tti;
    const KernelFn k = tti ? kernel_of<true, false>(p.shape)
                           : (us ? kernel_of<false, true>(p.shape) : kernel_of<false, false>(p.shape));
    void *args[] = {&a};
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds) !=
            hipSuccess ||
        hipLaunchCooperativeKernel(reinterpret_cast<const void *>(k), dim3(p.gx * p.gz), dim3(kShapes[p.shape].nt), args,
                                   (unsigned)p.lds, c->stream) != hipSuccess) {
        (void)hipGetLastError();
        p.ok = -1;
        return 0;
    }
    p.base += (unsigned)n;
    if (us) c->us_dirty = true;
    return 1;
}

// after the context's stream has been waited for: an exchange that never came
int run2d_check(vti_ctx *c)
{
    if (!c->run2d || !c->run2d->dead || !*c->run2d->dead) return VTI_OK;
    *c->run2d->dead = 0;
    c->run2d->ok = -1;          // later steps take the per-step kernels
    return fail(VTI_ERR_HIP, "resident 2D steps: a tile's exchange did not arrive");
}

}  // namespace vti
