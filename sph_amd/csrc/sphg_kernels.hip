// sphg_kernels.hip -- gfx950 kernels of the SPH solver step.
//
// Every kernel takes a scene table and a chunk table; a block works on one
// chunk (kBlock = 256 particles or kCellChunk = 1024 cells of one scene) or,
// with 4 lanes a particle, on one 64-particle group of a chunk; which one
// follows from the table, or without one from the block's number (chunk_at,
// part_at).  Sums of a scene are formed in a fixed order: a butterfly inside
// each wavefront, wave results combined in index order, one partial per chunk
// or group, and then the partials added in chunk order, by k_finalize (one
// block per scene, launched after the sweep) or, for a lone scene, by every
// block of the next sweep (loop_over) or k_loop_end.  Results therefore do not
// depend on scheduling.
//
// Reference algorithm: josemanuel28v/SPH src/SPHSolver.cpp,
// src/DFSPHSolver.cpp, src/WCSPHSolver.cpp, src/PCISPHSolver.cpp, the kernel
// headers and the force headers; each kernel names the lines it restates.

#include "sphg_internal.h"
#include "sphg_kernels.h"
#include "sphg_roots.h"

#include <type_traits>

namespace sphg {

// ------------------------------------------------------------ utilities

// f(integral_constant<int, I>) for I = 0 .. N-1, unrolled at compile time
template <int N, int I = 0, class F>
__device__ inline void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// Global-memory access.  The arrays come out of the scene table, so the
// compiler cannot prove their address space; these casts make it emit
// global (not flat) loads and stores.
typedef float v4f __attribute__((ext_vector_type(4)));
template <class T> using gptr = __attribute__((address_space(1))) T*;
__device__ inline float4 ld4(const float4* p, size_t i) {
    const v4f t = ((gptr<const v4f>)p)[i];
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ inline void st4(float4* p, size_t i, float4 v) {
    v4f t;
    t.x = v.x; t.y = v.y; t.z = v.z; t.w = v.w;
    ((gptr<v4f>)p)[i] = t;
}
template <class T> __device__ inline T ldg(const T* p, size_t i) { return ((gptr<const T>)p)[i]; }
// p as a global-address-space pointer, for p[i] and p->field of scalar types
template <class T> __device__ inline gptr<T> G(T* p) { return (gptr<T>)p; }
// Element j of a float4 array of fewer than 2^28 elements: the 32-bit byte
// offset lets the load take the uniform-base + 32-bit-offset address form
// (no 64-bit address arithmetic per element).
__device__ inline float4 ld4o(const float4* p, uint32_t j) {
    const v4f t = *(gptr<const v4f>)((gptr<const char>)p + (j << 4));
    return make_float4(t.x, t.y, t.z, t.w);
}
typedef float v2f __attribute__((ext_vector_type(2)));
__device__ inline float2 ld2o(const float2* p, uint32_t j) {
    const v2f t = *(gptr<const v2f>)((gptr<const char>)p + (j << 3));
    return make_float2(t.x, t.y);
}
// The xyz of element j of a float4 array: a 12-byte load.  (Measured on
// gfx950: slightly faster for the list build's survivors, slower than the
// 16-byte load for the solver sweeps' gathers.)
typedef float v3f __attribute__((ext_vector_type(3)));
__device__ inline float4 ld3o(const float4* p, uint32_t j) {
    const v3f t = *(gptr<const v3f>)((gptr<const char>)p + (j << 4));
    return make_float4(t.x, t.y, t.z, 0.0f);
}
template <class T> __device__ inline void stg(T* p, size_t i, T v) { ((gptr<T>)p)[i] = v; }
template <class T> __device__ inline void stg(T* p, uint32_t i, T v) {
    *(gptr<T>)((gptr<char>)p + (size_t)(i * (uint32_t)sizeof(T))) = v;
}


// The block's chunk: entry blockIdx.x of the chunk table, or, for a launch
// over one scene (no table), chunk number times `unit`.  Blocks go round-robin
// to the 8 XCDs, and XCD x gets the x-th contiguous part of the chunks, as the
// tables have it.  Without the table a block's first load is its scene's
// entry, not the chunk and then the scene: one memory round trip (0.5-0.8 us)
// less in each of a small step's launches.
__device__ inline Chunk chunk_at(const Chunk* C, int unit, int b, int nchunks) {
    if (C) return C[b];
    const int x = b & 7, per = nchunks >> 3, more = nchunks & 7;
    return Chunk{0, (x * per + min(x, more) + (b >> 3)) * unit};
}
__device__ inline Chunk chunk_at(const Chunk* C, int unit) { return chunk_at(C, unit, blockIdx.x, gridDim.x); }

// Kernels that give a particle Q = 4 lanes: a block of 4 wavefronts holds one
// 64-particle group, lane 4 q + u of wavefront w works on the group's particle
// 16 w + q, and a chunk's groups run on one XCD, like the chunk.  Q = 1: a
// block holds a chunk.  The block's first particle goes to i0, the thread's to
// i; false: there is no such chunk.
template <int Q>
__device__ inline bool part_at(const Chunk* C, int nchunks, Chunk& c, int& i0, int& i) {
    if (Q == 1) {
        c = chunk_at(C, kBlock);
        i0 = c.begin;
        i = i0 + threadIdx.x;
        return true;
    }
    const int g = (int)blockIdx.x >> 3, slot = (g / kWaves) * 8 + (int)(blockIdx.x & 7);
    if (slot >= nchunks) return false;
    c = chunk_at(C, kBlock, slot, nchunks);
    i0 = c.begin + (g % kWaves) * kGroup;
    i = i0 + (threadIdx.x >> 2);
    return true;
}
template <int Q> constexpr int kPartBlock = Q == 1 ? kBlock : 256;

// What the wavefront's lanes wrote before it is there for all of them, and none
// goes on before the others have come here.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// x of lane V of the quad
template <int V>
__device__ inline int quad_lane(int x) {
    return __builtin_amdgcn_update_dpp(0, x, V * 0x55, 0xf, 0xf, true);
}
template <int V>
__device__ inline double quad_lane(double x) {
    return __hiloint2double(quad_lane<V>(__double2hiint(x)), quad_lane<V>(__double2loint(x)));
}
// N doubles that go from lane to lane together
template <int N>
struct Terms {
    double v[N];
};
template <int V, int N>
__device__ inline Terms<N> quad_lane(const Terms<N>& t) {
    Terms<N> o;
#pragma unroll
    for (int k = 0; k < N; ++k) o.v[k] = quad_lane<V>(t.v[k]);
    return o;
}

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ inline double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}
// Result valid in every thread; the wave results are added in wave order.
// BT: the block's threads; sh: BT / 64 doubles of shared memory.
template <int BT = kBlock>
__device__ inline double block_sum(double v, double* sh) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    double r = sh[0];
#pragma unroll
    for (int k = 1; k < BT / 64; ++k) r += sh[k];
    __syncthreads();
    return r;
}
template <int BT = kBlock>
__device__ inline double block_max(double v, double* sh) {
    v = wave_max(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    double r = sh[0];
#pragma unroll
    for (int k = 1; k < BT / 64; ++k) r = fmax(r, sh[k]);
    __syncthreads();
    return r;
}

// Sum (or max) of one scene's chunk partials in chunk order.
// Each thread combines partials t, t + kBlock, t + 2 kBlock, ... in that order; the
// loads of 4096 / kBlock of them are issued before the first is used, so
// the loop waits on memory once for up to 4096 partials (a 1M-particle
// scene's chunks) instead of once per partial.
// Every kernel that forms a scene's sum adds in the same order, so a block of
// more than kBlock threads leaves it to the first kBlock.  (One of fewer has at
// most one partial a thread, which is that order: in the builds with blocks of
// 512 the launches with 4 lanes a particle have up to 192 chunks.)
constexpr int kPartU = 4096 / kBlock;
template <int BT> constexpr int kSumThreads = BT < kBlock ? BT : kBlock;
static_assert(kBlock <= 256 || kQuadSweepChunks <= kBlock, "at most 256 chunks, one partial a thread");
template <int BT = kBlock>
__device__ inline double scene_partial_sum(const double* partial, int n, double* sh) {
    constexpr int kT = kSumThreads<BT>;
    double acc = 0.0;
    if (kT == BT || threadIdx.x < kT)
        for (int b = threadIdx.x; b < n; b += kT * kPartU) {
            double v[kPartU];
#pragma unroll
            for (int u = 0; u < kPartU; ++u) v[u] = (b + u * kT < n) ? ldg(partial, (size_t)(b + u * kT)) : 0.0;
#pragma unroll
            for (int u = 0; u < kPartU; ++u) acc += v[u];
        }
    return block_sum<BT>(acc, sh);
}
// The same over n chunks whose 64-particle groups have a partial each (the
// kernels with 4 lanes a particle): a chunk's sum is formed as block_sum forms
// it.
template <int BT = kBlock>
__device__ inline double scene_group_sum(const double* partial, int n, double* sh) {
    constexpr int kT = kSumThreads<BT>;
    double acc = 0.0;
    if (kT == BT || threadIdx.x < kT)
        for (int b = threadIdx.x; b < n; b += kT) {
            double v[kWaves];
#pragma unroll
            for (int k = 0; k < kWaves; ++k) v[k] = ldg(partial, (size_t)b * kWaves + k);
            double r = v[0];
#pragma unroll
            for (int k = 1; k < kWaves; ++k) r += v[k];
            acc += r;
        }
    return block_sum<BT>(acc, sh);
}
template <int BT = kBlock>
__device__ inline double scene_partial_max(const double* partial, int n, double* sh) {
    double acc = -1e300;
    for (int b = threadIdx.x; b < n; b += BT * kPartU) {
        double v[kPartU];
#pragma unroll
        for (int u = 0; u < kPartU; ++u) v[u] = (b + u * BT < n) ? ldg(partial, (size_t)(b + u * BT)) : -1e300;
#pragma unroll
        for (int u = 0; u < kPartU; ++u) acc = fmax(acc, v[u]);
    }
    return block_max<BT>(acc, sh);
}

// ------------------------------------------------ loop control
//
// A solver loop goes on while (err > eta or it < minIt) and it < maxIt, where
// err is the scene's reduction over the last error sweep's chunk partials.
// For a lone scene of at most kFusedLoopChunks chunks every block of the next
// sweep forms that reduction itself, in the order k_finalize has, and decides:
// a launch less per iteration (~3 us), and no wait of the host (run_lone): a
// DFSPH step of 4,096 particles 197 -> 148 us, of 262,144 346 -> 309.  With
// 3,907 chunks (1M particles) a block would read 31 KB of partials, about what
// the finalize launch costs, so above the limit that stays.  The block
// that holds the scene's first chunk writes the outcome: done = idx + 1, where
// idx grows from launch to launch.  A launch takes only the ends that earlier
// launches wrote (ended_before) and forms its own decision otherwise, so all
// wavefronts of a block take the same branch, whenever they read the flag.

// The decision after `it` iterations with error err.
template <int KIND>
__device__ inline bool loop_goes_on(const DevScene& S, const Scalars* ss, int it, double err) {
    const double eta = KIND == LOOP_DIV ? S.etaV / ss->dt : S.eta;
    return ((err > eta) || (it < (KIND == LOOP_DIV ? S.minItV : S.minIt))) && (it < S.maxIt);
}
// Records the end of a loop (one thread).
template <int KIND>
__device__ inline void loop_ended(Scalars* ss, int it, double err, int idx) {
    if (KIND == LOOP_DENS) { ss->avgErr = err; ss->done = idx + 1; ss->sumIt += (unsigned)it; }
    if (KIND == LOOP_DIV) { ss->avgErrV = err; ss->doneV = idx + 1; ss->sumItV += (unsigned)it; }
    if (KIND == LOOP_PCI) { ss->maxDensErr = err; ss->done = idx + 1; ss->sumIt += (unsigned)it; }
}
__device__ inline bool ended_before(int done, int idx) { return done != 0 && done <= idx; }
constexpr int kLoopLast = 1 << 30;   // idx of the launches behind a loop
// The PCISPH loop's partials of iteration `it`: two buffers in turn, because
// its density sweep decides and writes partials in one launch.  The second is
// the sort's scratch, which the loop does not need.
__device__ inline double* pci_partial(const DevScene& S, int it) { return (it & 1) ? (double*)S.perm : S.partial; }
// Partials of 64-particle groups (kernels with 4 lanes a particle), one of two
// buffers in the sort's scratch: 0 also holds the partials of the errors
// before the DFSPH loops, 1 those of their iterations; the PCISPH loop uses
// both in turn.
__device__ inline double* group_partial(const DevScene& S, int buffer) {
    return (double*)S.perm + (size_t)buffer * S.nChunks * kWaves;
}
// The largest squared predicted displacement of each 64-particle group over a
// PCISPH step's iterations, behind the partials in the scratch; the next
// step's start reads it, before the sort.  (One atomic maximum per block
// into the scene's scalars was free with 1,371 blocks, but with the 4 times as
// many of 4 lanes a particle it took the step of 350,835 particles from 461 to
// 1,434 us.)
__device__ inline float* pci_displacements(const DevScene& S) {
    return (float*)((double*)S.perm + (size_t)2 * S.nChunks * kWaves);
}
// Whether the loop has ended, decided by every block alike (block-uniform;
// called where ended_before(done, idx) is false).
template <int KIND, int BT = kBlock>
__device__ inline bool loop_over(const DevScene& S, Scalars* ss, bool firstChunk, int idx, double* sh, bool large = false) {
    // too many partials for every block: k_loop_end decides
    if (!large && S.nChunks > kFusedLoopChunks) return false;
    const int it = KIND == LOOP_DIV ? ss->itV : ss->it;
    // below the minimum the error does not matter
    if (it < (KIND == LOOP_DIV ? S.minItV : S.minIt) && it < S.maxIt) return false;
    double err;
    if (KIND != LOOP_PCI)
        err = (quad_sweep(S.nChunks) ? scene_group_sum<BT>(group_partial(S, 1), S.nChunks, sh)
                                             : scene_partial_sum<BT>(S.partial, S.nChunks, sh)) / (double)S.n;
    else if (up_to(kQuadPciChunks, S.nChunks)) err = scene_partial_max<BT>(group_partial(S, (it - 1) & 1), S.nChunks * kWaves, sh);
    else err = scene_partial_max<BT>(pci_partial(S, it - 1), S.nChunks, sh);
    if (loop_goes_on<KIND>(S, ss, it, err)) return false;
    if (firstChunk && threadIdx.x == 0) loop_ended<KIND>(ss, it, err, idx);
    return true;
}

// A group's sum of e (in the first lane of each of 64 quads), formed as a wavefront
// that holds the 64 particles forms it.
__device__ inline void group_error(const DevScene& S, int buffer, int i0, double e) {
    __shared__ double se[kGroup];
    if (threadIdx.x < 256 && (threadIdx.x & 3) == 0) se[threadIdx.x >> 2] = e;
    __syncthreads();
    if (threadIdx.x < 64) {
        const double es = wave_sum(se[threadIdx.x]);
        if (threadIdx.x == 0) group_partial(S, buffer)[i0 >> 6] = es;
    }
}

// CFL time step (src/DFSPHSolver.cpp:827-870) from the scene's largest
// sqrt(|v + (a + g) dt|).
struct NextDt {
    double dt, maxVel, cflTs;
};
__device__ inline NextDt next_dt(const DevScene& S, double ts, int it, double red) {
    NextDt o;
    o.maxVel = fmax(0.1, red);
    o.cflTs = S.cfl * 0.4 * 2.0 * S.r / o.maxVel;
    double nts;
    if (o.cflTs < ts) nts = o.cflTs;
    else if (it > 3) nts = ts * 0.99;
    else nts = ts * 1.001;
    nts = fmax(nts, S.dtMin);
    o.dt = fmin(nts, S.dtMax);
    return o;
}

// ------------------------------------------------ SPH kernels (FP64 math)
//
// State is FP32 in HBM; every neighbor sum is formed in FP64.  On CDNA3/4
// an FP64 FMA issues at the rate of an unpacked FP32 FMA, and the FP32 sums
// lose the small differences the solvers run on (rho* - rho0 of a density
// near 1000).  1/|r| is an FP32 rsqrt refined by one FP64 Newton step
// (relative error ~1e-14), so no FP64 transcendental is issued.

// 1/sqrt(r2), zero for r2 <= 1e-30 (coincident points contribute no gradient).
// The seed is the hardware FP32 reciprocal square root: every r2 it is kept
// for is a normal float (1e-30 > 2^-126), where rsqrtf is that same
// instruction without its subnormal rescaling.
__device__ inline double rsqrt_d(double r2) {
    const double y = (double)__builtin_amdgcn_rsqf((float)r2);
    const double z = y * (1.5 - 0.5 * r2 * y * y);
    return (r2 > 1e-30) ? z : 0.0;
}
__device__ inline double sel(bool c, double a, double b) { return c ? a : b; }

struct Pair {
    double dx, dy, dz, r2, rl, inv, q;
};
__device__ inline Pair pair_of(double xi, double yi, double zi, float4 b, const KCoefD& k) {
    Pair p;
    p.dx = xi - (double)b.x;
    p.dy = yi - (double)b.y;
    p.dz = zi - (double)b.z;
    p.r2 = p.dx * p.dx + p.dy * p.dy + p.dz * p.dz;
    p.inv = rsqrt_d(p.r2);
    p.rl = p.r2 * p.inv;
    p.q = p.rl * k.invh;
    return p;
}
// Cubic spline W (src/CubicSpline.h:29-48); W_in for q <= 1.
__device__ inline double W_in(double q, const KCoefD& k) {
    const double om = 1.0 - q;
    const double w1 = k.ck * ((6.0 * q - 6.0) * q * q + 1.0);
    const double w2 = 2.0 * k.ck * om * om * om;
    return sel(q <= 0.5, w1, w2);
}
__device__ inline double W_d(double q, const KCoefD& k) { return sel(q <= 1.0, W_in(q, k), 0.0); }
// Cubic spline gradient factor: gradW(r) = g r, zero for |r| <= 1e-5 or
// q > 1 (src/CubicSpline.h:55-73).  For q <= 1/2 the reference's
// l q (3q-2) / (|r| h) equals l (3q-2) / h^2.  G_in for |r| > 1e-5, q <= 1.
__device__ inline double G_in(const Pair& p, const KCoefD& k) {
    const double om = 1.0 - p.q;
    const double g1 = k.clh2 * (3.0 * p.q - 2.0);
    const double g2 = -k.clh * om * om * p.inv;
    return sel(p.q <= 0.5, g1, g2);
}
__device__ inline double G_d(const Pair& p, const KCoefD& k) {
    return sel(p.rl > 1e-5 && p.q <= 1.0, G_in(p, k), 0.0);
}
// Cubic gradient factor of a neighbor-list member for the solver sweeps.
// List members have q <= 1 by construction and the padding entries are the
// particle itself (r = 0), so the q <= 1 test of G_d is dropped, and 1/r is
// the raw FP32 rsqrt refined by one FP64 Newton step with no guard: r = 0
// gives rl = NaN, which fails rl > 1e-5 and selects 0, as G_d does.
struct PairG {
    double dx, dy, dz, g;
    bool apart;   // |r| > 1e-5; otherwise the gradient is zero and g undefined
};
__device__ inline PairG pairg_of(double xi, double yi, double zi, float4 b, const KCoefD& k) {
    PairG p;
    p.dx = xi - (double)b.x;
    p.dy = yi - (double)b.y;
    p.dz = zi - (double)b.z;
    const double r2 = p.dx * p.dx + p.dy * p.dy + p.dz * p.dz;
    const double y = (double)__builtin_amdgcn_rsqf((float)r2);
    const double e = fma(-r2 * y, y, 1.0);          // 1 - r2 y^2
    const double inv = fma(0.5 * y, e, y);          // one Newton step
    const double rl = r2 * inv;
    // with q = r/h: g = clh2 (3q - 2) = gA r + gB for q <= 1/2, else
    // -clh (1 - q)^2 / r
    const double om = fma(-k.invh, rl, 1.0);
    const double g1 = fma(k.gA, rl, k.gB);
    const double g2 = (-k.clh * inv) * (om * om);
    p.g = sel(rl <= k.hHalf, g1, g2);
    p.apart = rl > 1e-5;
    return p;
}

// Spiky gradient factor (src/Spiky.h:44-55): -45/(pi h^6) (h-r)^2 / r.
__device__ inline double Gs_d(const Pair& p, const KCoefD& k) {
    const double d = k.h - p.rl;
    const double g = -k.spg * d * d * p.inv;
    return sel(p.r2 > 0.0 && p.rl <= k.h, g, 0.0);
}
// Cohesion C(r) (src/Cohesion.h:29-40) for 0 < r <= h; `outer` is the
// branch test 2r > h.  As written there the h^6/64 offset is not scaled by
// 32/(pi h^9), so C jumps at r = h/2 and the branch is decided exactly by
// the caller near that point.
__device__ inline double C_d(double rl, bool outer, const KCoefD& k) {
    const double d = k.h - rl;
    const double t = d * d * d * rl * rl * rl;
    return outer ? k.co1 * t : k.co1 * 2.0 * t - k.co2;
}
// Adhesion A(r) (src/Adhesion.h:24-35): (-4r^2/h + 6r - 2h)^(1/4) on
// (h/2, h], evaluated as ((2/h)(2r-h)(h-r))^(1/4), the same polynomial in a
// form that cannot round below zero.
__device__ inline double A_d(double rl, const KCoefD& k) {
    if (!(2.0 * rl > k.h && rl <= k.h)) return 0.0;
    const double v = (2.0 * k.invh) * (2.0 * rl - k.h) * (k.h - rl);
    return sqrt(sqrt(fmax(v, 0.0)));
}

// Exact FP64 distance test, operation for operation the reference's
// length(ri - rj) / h on FP32 positions promoted to FP64
// (src/CubicSpline.h:55-60, glm dot summed left to right).
struct Exact {
    double rl, q;
};
__device__ inline Exact exact_q(float4 a, float4 b, double h) {
    const double dx = __dsub_rn((double)a.x, (double)b.x);
    const double dy = __dsub_rn((double)a.y, (double)b.y);
    const double dz = __dsub_rn((double)a.z, (double)b.z);
    const double d2 = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
    Exact e;
    e.rl = __dsqrt_rn(d2);
    e.q = __ddiv_rn(e.rl, h);
    return e;
}
// Whether the reference's FP64 gradient is nonzero (its neighbor count of
// src/DFSPHSolver.cpp:446-447).
__device__ inline bool grad_nonzero64(const Exact& e) {
    if (!(e.rl > 1.0e-5 && e.q <= 1.0)) return false;
    if (e.q <= 0.5) return __dmul_rn(e.q, __dsub_rn(__dmul_rn(3.0, e.q), 2.0)) != 0.0;
    const double f = __dsub_rn(1.0, e.q);
    return __dmul_rn(f, f) != 0.0;
}

// List layout inside a 64-particle group: blocks of 4 slots, lane-major
// within a block, so slot s of lane l is element (s/4 * 64 + l) * 4 + s%4
// of the group's maxNbr * 64 entries, and a lane reads its next 4 slots
// with one 16-byte load (a wavefront reads 1 KB contiguous).
__device__ inline uint32_t slot_of(int s) { return (uint32_t)(((s >> 2) * kGroup) << 2) + (uint32_t)(s & 3); }
// Element offset of lane (i & 63)'s first slot (maxNbr is a multiple of 4).
__device__ inline uint32_t lane_base(const DevScene& S, int i) {
    return (uint32_t)(i >> 6) * (uint32_t)S.maxNbr * (uint32_t)kGroup + ((uint32_t)(i & 63) << 2);
}
__device__ inline const uint32_t* list_of(const DevScene& S, int i) { return S.nbr + lane_base(S, i); }
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
// slots 4b .. 4b+3 of a lane
__device__ inline v4u ld_block(const uint32_t* L, int b) { return ((gptr<const v4u>)L)[(size_t)b * kGroup]; }
// The group's padded list length, uniform across the wavefront (a
// wavefront is one 64-particle group: chunks start at multiples of 256).
__device__ inline int group_count(const DevScene& S, int i) {
    return __builtin_amdgcn_readfirstlane((int)ldg(S.gcnt, (size_t)(i >> 6)));
}

// Visit particle i's padded neighbor list four entries at a time: the four
// indices are loaded, then the four neighbors' data (load(j)), then the
// four terms are evaluated (body(j, data)), so every lane has several
// loads in flight.  The trip count is uniform across the wavefront.
template <class Load, class Body>
__device__ inline void sweep4(const DevScene& S, int i, Load&& load, Body&& body) {
    const uint32_t* L = list_of(S, i);
    const int gc = group_count(S, i);
    if (gc == 0) return;
    // the indices of the next 4 entries are requested before the neighbor
    // data of the current 4 is used, so the list stream (HBM) and the
    // neighbor loads (mostly L2) overlap instead of forming one chain
    v4u jn = ld_block(L, 0);
    for (int q = 0; q < gc; q += 4) {
        const uint32_t jj[4] = {jn.x, jn.y, jn.z, jn.w};
        decltype(load(0u)) dd[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) dd[u] = load(jj[u]);
        // unconditional (the last pass re-reads its own entries), so the
        // wait for this pass's data leaves the 4 index loads in flight
        const int qn = (q + 4 < gc) ? q + 4 : q;
        jn = ld_block(L, qn >> 2);
        // keeps the compiler from sinking these loads into the next pass
        asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < 4; ++u) body(jj[u], dd[u]);
    }
}

// A particle's list with Q lanes: term(data) of every entry, added in list
// order (add).  Q = 1 is sweep4.  With 4 lanes a lane takes every 4th entry,
// two at a time, and every lane adds the quad's terms one after the other, so
// the sums are the same bit for bit.  A small launch has a wavefront or so a
// SIMD, whose chain of gathers and FP64 math bounds it: a DFSPH sweep of 4,096
// particles 8 -> 5.3 us, the WCSPH forces of 2,197 15.8 -> 6.3.
template <int Q, class Load, class Term, class Add>
__device__ inline void sweep(const DevScene& S, int i, Load&& load, Term&& term, Add&& add) {
    if constexpr (Q == 1) {
        sweep4(S, i, load, [&](uint32_t, const auto& d) { add(term(d)); });
    } else {
        const uint32_t* const L = list_of(S, i) + (threadIdx.x & 3);
        const int nb = group_count(S, i) >> 2;
        if (nb == 0) return;
        auto at = [&](int b) { return ldg(L, (size_t)slot_of(4 * min(b, nb - 1))); };
        uint32_t jn[2] = {at(0), at(1)};
        for (int q = 0; q < nb; q += 2) {
            decltype(load(0u)) d[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) d[h] = load(jn[h]);
            jn[0] = at(q + 2);
            jn[1] = at(q + 3);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (h == 1 && q + 1 >= nb) break;
                const auto t = term(d[h]);
                static_for<4>([&](auto vc) { add(quad_lane<decltype(vc)::value>(t)); });
            }
        }
    }
}

struct XV {
    float4 x, v;
};
// x (with v_x in w) and (v_y, v_z) of a neighbor: 24 B, against 32 for x and v
struct XVP {
    float4 xv;
    float2 yz;
};
// the density solve's first error sweep: x (with u_x in w), v0 and (u_y, u_z)
struct XVU {
    float4 x, v;
    float2 yz;
};
struct NbF {
    float4 x, v, n;
    float d;
};
__device__ inline uint32_t* list_of_w(const DevScene& S, int i) { return S.nbr + lane_base(S, i); }

// Linear cell of a position: key floor(x/h) in FP64 (src/HashTable.h:81),
// clamped into the padded grid.  Clamping keeps any two particles closer
// than h in adjacent cells, so the 27-cell walk still sees every neighbor.
__device__ inline int cell_of(const DevScene& S, float4 p) {
    double fx = floor(__ddiv_rn((double)p.x, S.hD));
    double fy = floor(__ddiv_rn((double)p.y, S.hD));
    double fz = floor(__ddiv_rn((double)p.z, S.hD));
    fx = (fx == fx) ? fx : (double)S.kx0;
    fy = (fy == fy) ? fy : (double)S.ky0;
    fz = (fz == fz) ? fz : (double)S.kz0;
    const int ix = (int)fmin(fmax(fx - (double)S.kx0 + 1.0, 1.0), (double)(S.nx - 2));
    const int iy = (int)fmin(fmax(fy - (double)S.ky0 + 1.0, 1.0), (double)(S.ny - 2));
    const int iz = (int)fmin(fmax(fz - (double)S.kz0 + 1.0, 1.0), (double)(S.nz - 2));
    return ix + S.nx * (iy + S.ny * iz);
}

// Walk the 27 cells around cell c as 9 x-rows of 3 contiguous cells.
template <class F>
__device__ inline void walk27(const int* __restrict__ start, int c, int nx, int nxny, F&& f) {
#pragma unroll 1
    for (int dz = -1; dz <= 1; ++dz) {
#pragma unroll 1
        for (int dy = -1; dy <= 1; ++dy) {
            const int base = c + dy * nx + dz * nxny;
            const int s = start[base - 1];
            const int e = start[base + 2];
            for (int j = s; j < e; ++j) f(j);
        }
    }
}

// walk27 with the data of four candidates loaded before any is visited
// (`load(j)` then `visit(j, data)`, in walk order), so a lane has four
// independent loads in flight instead of one chain.
template <class Load, class Visit>
__device__ inline void walk27x4(const int* __restrict__ start, int c, int nx, int nxny, Load&& load, Visit&& visit) {
#pragma unroll 1
    for (int dz = -1; dz <= 1; ++dz) {
#pragma unroll 1
        for (int dy = -1; dy <= 1; ++dy) {
            const int base = c + dy * nx + dz * nxny;
            const int s = start[base - 1];
            const int e = start[base + 2];
            for (int j0 = s; j0 < e; j0 += 4) {
                decltype(load(0)) d[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) d[u] = load(min(j0 + u, e - 1));
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (j0 + u < e) visit(j0 + u, d[u]);
            }
        }
    }
}

// PCISPH shell width: 2.5 times the largest predicted displacement of the
// previous step (so a step's displacements may grow by 25%), at least
// 0.05 h.  The same for every kernel of a step (the previous step's maximum
// is copied at the step's start).
__device__ inline float pci_skin(const DevScene& S) {
    const float md = sqrtf(__uint_as_float(S.ss->maxD2Prev));
    return fmaxf(0.05f * S.kc.h, 2.5f * md);
}
// A predicted displacement longer than half the skin lets two particles
// outside each other's list and shell come within h, so the step's
// predicted densities take the 27-cell walk.
__device__ inline void shell_guard(const DevScene& S, double dx, double dy, double dz) {
    if (!S.pciShell) return;
    const double half = 0.5 * (double)pci_skin(S);
    if (dx * dx + dy * dy + dz * dz > half * half) atomicOr(&S.ss->shellBad, 1u);
}

// Poly6 W (src/Poly6.h:31-42) of a squared distance.
__device__ inline double P6_d(double r2, const KCoefD& k) {
    const double d = k.h2 - r2;
    return sel(r2 <= k.h2, k.p6v * d * d * d, 0.0);
}

// The collision projection of PCISPHBoundaryModel (src/PCISPHBoundaryModel.
// cpp:219-309, 385-439) for one fluid particle at position (px, py, pz):
// boundary candidates of the position's cell (none when no particle was
// ever inserted in that cell: the reference's hash table has no entry for
// it) with |x - r_b| < h/2 weigh w = max(0, (h/2 - |q_b|) / (h/2)), q_b =
// (qx, qy, qz) - r_b; returns n = glm::normalize(sum w n_b) (NaN for a zero
// sum) and the shift (1 / sum w)(sum w (h/2 - |q_b|)), applied when sum w > 0.
struct PbHit {
    double nx, ny, nz, s;
    bool hit;
};
__device__ inline PbHit pb_project(const DevScene& S, double px, double py, double pz, float4 pf, double qx, double qy,
                                   double qz) {
    const KCoefD k = S.kd;
    const double R = 0.5 * k.h;
    double ax = 0.0, ay = 0.0, az = 0.0, ws = 0.0, w2 = 0.0;
    const int cl = cell_of(S, pf);
    if (S.everOcc[cl]) {
        walk27(S.bCellStart, cl, S.nx, S.nx * S.ny, [&](int b) {
            const float4 y = S.xb[b];
            const double dx = px - (double)y.x, dy = py - (double)y.y, dz = pz - (double)y.z;
            if (sqrt(dx * dx + dy * dy + dz * dz) < R) {
                const double ex = qx - (double)y.x, ey = qy - (double)y.y, ez = qz - (double)y.z;
                const double lq = sqrt(ex * ex + ey * ey + ez * ez);
                const double w = fmax(0.0, (R - lq) / R);
                ws += w;
                w2 += w * (R - lq);
                const float4 nb = S.bn[b];
                ax += w * (double)nb.x;
                ay += w * (double)nb.y;
                az += w * (double)nb.z;
            }
        });
    }
    const double inv = 1.0 / sqrt(ax * ax + ay * ay + az * az);
    PbHit h;
    h.nx = ax * inv;
    h.ny = ay * inv;
    h.nz = az * inv;
    h.hit = ws > 0.0;
    h.s = h.hit ? (1.0 / ws) * w2 : 0.0;
    return h;
}
// correctVelocities (src/PCISPHBoundaryModel.cpp:311-383): where |n| > 0
// (false for NaN), v = tangentialFct (u - (u.n) n) - normalFct (u.n) n.
__device__ inline bool pb_velocity(const DevScene& S, double nx, double ny, double nz, double& ux, double& uy,
                                   double& uz) {
    if (!(sqrt(nx * nx + ny * ny + nz * nz) > 0.0)) return false;
    const double d = ux * nx + uy * ny + uz * nz;
    const double nvx = d * nx, nvy = d * ny, nvz = d * nz;
    ux = S.pbTf * (ux - nvx) - S.pbNf * nvx;
    uy = S.pbTf * (uy - nvy) - S.pbNf * nvy;
    uz = S.pbTf * (uz - nvz) - S.pbNf * nvz;
    return true;
}


// ================================================================ grid

// Cell key + histogram (src/HashTable.h:79-86 insertion, as a count).
// Adds SIGN = 1 to counter[key] for every lane with key >= 0 and returns the
// counter's value before this lane's unit, a slot unique to the lane; SIGN =
// -1 takes one away and returns the value after it.  The
// particles of a wavefront are in the previous step's cell order and most
// keep their cell, so runs of consecutive lanes share a key: each run adds
// its length with one atomic (a dense fluid has ~8 lanes per run), and its
// lanes take consecutive slots.  Every lane of the wavefront calls it; lanes
// with nothing to count pass -1 and must all come after the counting ones.
template <int SIGN = 1>
__device__ inline int wave_count_add(int* counter, int key) {
    const int lane = threadIdx.x & 63;
    const int prev = __shfl_up(key, 1);
    const bool head = (lane == 0) || (key != prev);
    const uint64_t heads = __ballot(head);
    const uint64_t upto = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);   // lanes 0 .. lane
    const int first = 63 - __clzll((long long)(heads & upto));             // this lane's run head
    const uint64_t later = heads & ~upto;
    const int end = later ? __ffsll((long long)later) - 1 : 64;             // one past the run
    int base = 0;
    if (head && key >= 0) {
        const int len = end - lane;
        base = __hip_atomic_fetch_add(G(counter) + key, SIGN * len, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (SIGN < 0) base -= len;
    }
    base = __shfl(base, first);
    return base + (lane - first);
}

// The start of a WCSPH or PCISPH step: the scene's step counters, and for
// PCISPH zero pressures and pressure accelerations and the pressure loop's
// start (src/PCISPHSolver.cpp:21-50); `active` counts the scenes whose loop
// runs.
__device__ inline void step_begin(const DevScene& S, const Chunk& c, int i, int* active) {
    if (S.method == PCISPH && i < S.n) {
        S.p[i] = 0.0f;
        S.pacc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (c.begin != 0) return;
    Scalars* ss = S.ss;
    // the previous step's largest predicted displacement (none if no
    // iteration of it ran)
    double d2 = 0.0;
    const bool moved = S.pciShell && ss->moved;
    __syncthreads();   // every thread has read the flag before it is set
    if (moved) {
        __shared__ double sh[kWaves];
        float m = 0.f;
        const float* const disp = pci_displacements(S);
        for (int t = threadIdx.x; t < S.nChunks * kWaves; t += kBlock * 16) {
            float q[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) q[u] = (t + u * kBlock < S.nChunks * kWaves) ? ldg(disp, (size_t)(t + u * kBlock)) : 0.f;
#pragma unroll
            for (int u = 0; u < 16; ++u) m = fmaxf(m, q[u]);
        }
        d2 = block_max((double)m, sh);
    }
    if (threadIdx.x == 0) {
        ss->steps += 1u;
        ss->shellBad = 0u;
        ss->maxD2Prev = __float_as_uint((float)d2);
        if (S.method == PCISPH) {
            ss->it = 0;
            const bool run = (ss->maxDensErr > S.eta || 0 < S.minIt) && 0 < S.maxIt;
            ss->moved = run ? 1u : 0u;
            ss->done = run ? 0 : 1;
            if (run) atomicAdd(active, 1);
        }
    }
}

// Cell key of each particle and its count in its cell; with BEGIN also the
// start of a WCSPH or PCISPH step (one launch fewer per step).
template <bool BEGIN>
__global__ __launch_bounds__(kBlock) void k_keys(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                 int* active) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    const int i = c.begin + threadIdx.x;
    if (BEGIN) step_begin(S, c, i, active);
    // the lists about to be built start without an overflow
    if (c.begin == 0 && threadIdx.x == 0) G(S.ss)->listOver = 0u;
    int cl = -1;
    if (i < S.n) {
        cl = cell_of(S, ld4(S.x, (size_t)i));
        G(S.cellU)[i] = cl;
    }
    (void)wave_count_add(S.cellCount, cl);
}

// DFSPH with the loops decided in the sweeps: the error before the density
// loop, for the log, from the partials its sweep left in the sort's scratch
// (one block, before the scatter overwrites them).
__device__ inline void density_error0(const DevScene& S) {
    __shared__ double sh[kWaves];
    const double avg0 = (quad_sweep(S.nChunks) ? scene_group_sum(group_partial(S, 0), S.nChunks, sh)
                                                       : scene_partial_sum(group_partial(S, 0), S.nChunks, sh)) / (double)S.n;
    if (threadIdx.x == 0) S.ss->avgErr0 = avg0;
}
// The first launch behind a DFSPH density loop whose end the position update
// has decided (`tables` not null: a lone scene whose iterations were launched
// ahead): whether it had ended.  If not, nothing behind this launch runs.
// (`tables` are the tables that the kernel reads as T: its T is not restrict,
// and what it needs of the scene it reads before its own stores.)
__device__ inline bool sort_runs(const DevScene& S, const Chunk& c, const Tables& tables, int fused) {
    if (tables.a && !S.ss->done) {
        if (c.begin == 0 && threadIdx.x == 0) tables.a->stall = tables.b->stall = 1;
        return false;
    }
    if (fused && c.begin == 0) density_error0(S);
    return true;
}

// Per cell chunk: total count.
__global__ __launch_bounds__(kBlock) void k_scan_sum(const DevScene* T, const Chunk* __restrict__ C,
                                                     Tables tables, int fused) {
    const Chunk c = chunk_at(C, kCellChunk);
    const DevScene& S = T[c.scene];
    const int ncells = S.ncells;
    int *const cellCount = S.cellCount, *const cellChunkSum = S.cellChunkSum;
    if (S.stall || !sort_runs(S, c, tables, fused)) return;
    __shared__ double sh[kWaves];
    int acc = 0;
    const int c0 = c.begin + threadIdx.x * kCellPerThread;
#pragma unroll
    for (int u = 0; u < kCellPerThread; ++u) {
        const int cc = c0 + u;
        if (cc < ncells) acc += ldg(cellCount, (size_t)cc);
    }
    const double tot = block_sum((double)acc, sh);
    if (threadIdx.x == 0) G(cellChunkSum)[c.begin / kCellChunk] = (int)tot;
}

__device__ inline int wave_incl_scan(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o);
        if (lane >= o) v += t;
    }
    return v;
}

// One block per scene: exclusive scan of the chunk totals, in place, kBlock
// totals per pass with the running total carried between passes.
__global__ __launch_bounds__(kBlock) void k_scan_offsets(const DevScene* __restrict__ T, int nscenes) {
    const int s = blockIdx.x;
    if (s >= nscenes) return;
    const DevScene& S = T[s];
    if (S.stall) return;
    __shared__ int wsum[kWaves];
    __shared__ int carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    const int n = S.nCellChunks;
    for (int b = 0; b < n; b += kBlock) {
        const int t = b + threadIdx.x;
        const int v = (t < n) ? ldg(S.cellChunkSum, (size_t)t) : 0;
        const int incl = wave_incl_scan(v);
        const int w = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 63) wsum[w] = incl;
        __syncthreads();
        int off = carry;
        for (int q = 0; q < w; ++q) off += wsum[q];
        if (t < n) G(S.cellChunkSum)[t] = off + incl - v;
        __syncthreads();
        if (threadIdx.x == kBlock - 1) carry = off + incl;
        __syncthreads();
    }
}

// Final scan: cellStart[c] = exclusive prefix of counts.  What comes before
// the block's chunk:
//   SCAN_ONE     the counts themselves, added up by the block (no other launch
//                of the scan runs): grids of up to kScanOneChunks chunks, where
//                the last block reads 31 K counts in ~2 us and a launch costs
//                ~3 (2k-particle WCSPH step 84.2 -> 82.7 us)
//   SCAN_TOTALS  the chunk totals of k_scan_sum, added up by the block
//   SCAN_OFFSETS the chunk offsets of k_scan_offsets
// Integer sums, so all give the same offsets.
enum ScanKind { SCAN_ONE, SCAN_TOTALS, SCAN_OFFSETS };
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_scan_final(const DevScene* T, const Chunk* __restrict__ C,
                                                       Tables tables, int fused) {
    const Chunk c = chunk_at(C, kCellChunk);
    const DevScene& S = T[c.scene];
    const int ncells = S.ncells, n = S.n;
    int *const cellCount = S.cellCount, *const cellChunkSum = S.cellChunkSum, *const cellStart = S.cellStart;
    if (S.stall || !sort_runs(S, c, tables, fused)) return;
    __shared__ int wsum[kWaves];
    __shared__ int base;
    const int chunk = c.begin / kCellChunk;
    if (KIND != SCAN_OFFSETS) {
        int acc = 0;
        if (KIND == SCAN_ONE) {
            constexpr int kU = 8;
            typedef int v4i __attribute__((ext_vector_type(4)));
            const gptr<const v4i> cnt = (gptr<const v4i>)cellCount;
            for (int t = threadIdx.x; t < c.begin / 4; t += kBlock * kU) {
                v4i q[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) q[u] = (t + u * kBlock < c.begin / 4) ? cnt[t + u * kBlock] : (v4i)0;
#pragma unroll
                for (int u = 0; u < kU; ++u) acc += q[u].x + q[u].y + q[u].z + q[u].w;
            }
        } else {
            for (int t = threadIdx.x; t < chunk; t += kBlock) acc += ldg(cellChunkSum, (size_t)t);
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o);
        if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            int b = 0;
#pragma unroll
            for (int q = 0; q < kWaves; ++q) b += wsum[q];
            base = b;
        }
        __syncthreads();
    }
    const int c0 = c.begin + threadIdx.x * kCellPerThread;
    int vals[kCellPerThread];
    int local = 0;
#pragma unroll
    for (int u = 0; u < kCellPerThread; ++u) {
        const int cc = c0 + u;
        vals[u] = (cc < ncells) ? ldg(cellCount, (size_t)cc) : 0;
        local += vals[u];
    }
    const int incl = wave_incl_scan(local);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) wsum[w] = incl;
    __syncthreads();
    int woff = 0;
    for (int q = 0; q < w; ++q) woff += wsum[q];
    int run = (KIND != SCAN_OFFSETS ? base : ldg(cellChunkSum, (size_t)chunk)) + woff + incl - local;
#pragma unroll
    for (int u = 0; u < kCellPerThread; ++u) {
        const int cc = c0 + u;
        if (cc < ncells) G(cellStart)[cc] = run;
        run += vals[u];
    }
    // the chunk table covers ncells + 1 entries: the last one is the end
    if (c0 <= ncells && ncells < c0 + kCellPerThread) G(cellStart)[ncells] = n;
}

// Scatter the particle ids into their cells' slots (arrival order).  Each
// cell's count goes back to zero for the next step's.
__global__ __launch_bounds__(kBlock) void k_scatter(const DevScene* __restrict__ T, const Chunk* __restrict__ C) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    const int i = c.begin + threadIdx.x;
    const int cl = (i < S.n) ? ldg(S.cellU, (size_t)i) : -1;
    const int r = wave_count_add<-1>(S.cellCount, cl);
    if (i < S.n) G(S.perm)[ldg(S.cellStart, (size_t)cl) + r] = ldg(S.id, (size_t)i);
}

// Final slot of each particle = cell start + number of particles of its
// cell with a smaller id, so every bucket lists its particles in ascending
// id, the reference's insertion order (src/SPHSolver.cpp:188-191,
// src/HashTable.h:79-86).  The state is written straight to that slot (the
// other half of each double buffer).
__global__ __launch_bounds__(kBlock) void k_rank_reorder(const DevScene* __restrict__ T, const Chunk* __restrict__ C) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    const int i = c.begin + threadIdx.x;
    if (i >= S.n) return;
    const int cl = ldg(S.cellU, (size_t)i);
    const int s = ldg(S.cellStart, (size_t)cl), e = ldg(S.cellStart, (size_t)cl + 1);
    const uint32_t me = ldg(S.id, (size_t)i);
    // the particle's data is loaded before the rank loop and before any
    // store (a wait for a load also waits for the stores issued before it)
    const float4 xo = ld4(S.x, (size_t)i), vo = ld4(S.v, (size_t)i);
    const bool df = S.method == DFSPH;
    const float ko = df ? ldg(S.k, (size_t)i) : 0.f, kvo = df ? ldg(S.kv, (size_t)i) : 0.f;
    const float4 no = (df && S.pbOn) ? ld4(S.pbn, (size_t)i) : make_float4(0.f, 0.f, 0.f, 0.f);
    // rank within the cell: the ids of its first 8 members are loaded
    // together (a fluid cell holds ~8; the cell holds this particle, so
    // e > s and the clamped index stays in it), the rest one at a time
    uint32_t q8[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) q8[u] = ldg(S.perm, (size_t)min(s + u, e - 1));
    int rank = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) rank += ((s + u < e) & (q8[u] < me)) ? 1 : 0;
    for (int q = s + 8; q < e; ++q) rank += (ldg(S.perm, (size_t)q) < me) ? 1 : 0;
    const int d = s + rank;
    st4(S.x2, (size_t)d, xo);
    st4(S.v2, (size_t)d, vo);
    stg(S.id2, (size_t)d, me);
    stg(S.cell, (size_t)d, cl);
    if (df) {
        stg(S.k2, (size_t)d, ko);
        stg(S.kv2, (size_t)d, kvo);
        if (S.pbOn) st4(S.pbn2, (size_t)d, no);
    }
    if (S.pbOn) stg(S.everOcc, (size_t)cl, (uint8_t)1);
}

// =========================================================== boundary

// Akinci boundary volume V_b = 1 / sum_b' W(x_b - x_b'), self included
// (src/AkinciBoundayModel.cpp:11-40).  One scene per launch; bvol sorted.
__global__ __launch_bounds__(kBlock) void k_bvolume(const DevScene* __restrict__ T, int scene, float* __restrict__ bvol) {
    const DevScene& S = T[scene];
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b >= S.nb) return;
    const float4 xb = S.xb[b];
    const int cb = cell_of(S, xb);
    const KCoefD k = S.kd;
    const double bx = xb.x, by = xb.y, bz = xb.z;
    double sum = 0.0;
    walk27(S.bCellStart, cb, S.nx, S.nx * S.ny, [&](int j) {
        const Pair p = pair_of(bx, by, bz, S.xb[j], k);
        sum += W_d(p.q, k);
    });
    bvol[b] = (float)(1.0 / sum);
}
__global__ __launch_bounds__(kBlock) void k_bvolume_pack(const DevScene* __restrict__ T, int scene, const float* __restrict__ bvol) {
    const DevScene& S = T[scene];
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b >= S.nb) return;
    S.xb[b].w = bvol[b];
}

// ================================================ neighbor list + density

// Per particle: walk the 27 cells, keep the fluid neighbors with
// |r|/h <= 1 decided exactly in FP64 (the reference's W and gradW vanish
// beyond h, so its sums over the whole bucket equal sums over this list),
// and in the same pass form
//   rho_i   = m W(0) + sum_j m W_ij + sum_b rho0 V_b W_ib   (src/SPHSolver.cpp:60-89)
//   alpha_i = rho_i / (|sum_j m gradW_ij + sum_b rho0 V_b gradW_ib|^2 + sum_j |m gradW_ij|^2)
//             or 0 when that is <= 1e-5                     (src/DFSPHSolver.cpp:139-186)
//   gb_i    = (sum_b rho0 V_b gradW_ib, sum_b rho0 V_b W_ib)
// plus, per method, the pressure of the Tait EOS (src/WCSPHSolver.cpp:93),
// the Spiky boundary sum used by PCISPH (src/PCISPHSolver.cpp:342-353) and
// the adhesion sum (src/AdhesionForce.h:46-59).
// Fluid neighbors of particle i in two passes.  Pass 1 walks the 27 cells
// with an FP32 distance test whose bound is 1e-5 above h^2 (FP32 rounding of
// |x_i - x_j|^2 is ~1e-7 relative) and keeps the survivors in the list's
// memory.  Pass 2 runs the FP64 test and sums over those survivors only and
// writes the list in place.  Pass 2 thus iterates ~1.1x the neighbor count on
// every lane of a wavefront, instead of running the FP64 path for every
// candidate that any lane of the wavefront accepts.  A particle with more
// survivors than list slots takes the one-pass walk over all candidates.
//
// Both passes read positions from LDS.  The particles of a block are sorted by
// cell, so they span one cell range [cF, cL], and each of a lane's 9 candidate
// rows (cells c-1..c+1 of row (dy, dz)) lies inside that row's range
// cF-1..cL+1 for the whole block.  The block copies those 9 particle ranges
// (~2,450 positions in a dense fluid, 12 B each) into LDS once; rows past the
// stage are read from global memory.
//
// FP64 math (~45 instructions a survivor, half of the vector instructions) and
// pass 1's FP32 tests bound it, with 4 wavefronts a SIMD to cover LDS and the
// velocity gathers.  With a stage a wavefront, a store for every candidate
// step that some lane accepted (28 M write requests to L2 in a scene of 1M
// particles, now 18 M) and pass 2's positions gathered from memory, it took
// 255 us for 1M DFSPH particles, 166 for 600k WCSPH and 111 for 350k PCISPH;
// now 207, 123 and 91.  5 wavefronts a SIMD (96 registers) spill in DFSPH: +85.
// Candidates staged by a block: 9 rows of its own particles and two cells on
// each side.  With 256 particles 31.9 KB, which leaves room for 5 blocks a
// compute unit.  A row is read kScan candidates at a time, so up to kScan - 1
// entries past its end.
constexpr int kScan = 8;   // 32 a multiple of it: a row's tests fill a mask
constexpr int kBuildStage = 9 * (kBlock + 38), kBuildPad = kScan - 1;
static_assert(32 % kScan == 0, "whole masks");

// FP64 test of a candidate: whether the reference's sums hold it, its W and
// gradient factor, and whether its gradient is nonzero.
// 1e-9 <= r2 < hlo2: |r| > 1e-5 and q < 1, where W and the gradient take
// their inner forms and the gradient is nonzero.  The reference's gradient
// (src/CubicSpline.h:55-73) vanishes only at |r| <= 1e-5 and q = 1; near those
// two, and near q = 1 for the list membership, the test is repeated
// operation-exact in FP64.
__device__ inline bool member_of(const Pair& p, const float4& xi, const float4& xj, double hD, const KCoefD& k, double& g,
                                 double& wq, bool& gnz) {
    if (!(p.r2 <= k.hhi2)) return false;
    g = G_in(p, k);
    wq = W_in(p.q, k);
    gnz = true;
    if (p.r2 >= k.hlo2 || p.r2 < 1e-9) {
        const Exact e = exact_q(xi, xj, hD);
        if (!(e.q <= 1.0)) return false;
        gnz = grad_nonzero64(e);
        g = G_d(p, k);
        wq = W_d(p.q, k);
    }
    return true;
}

// A particle's sums over its neighbors and boundary neighbors.
struct BuildSums {
    double ws = 0.0, sgx = 0.0, sgy = 0.0, sgz = 0.0, ssq = 0.0;
    double dv = 0.0;                             // DFSPH: sum_j g_ij (v_i - v_j).(x_i - x_j)
    double bw = 0.0, bgx = 0.0, bgy = 0.0, bgz = 0.0;
    double sx2 = 0.0, sy2 = 0.0, sz2 = 0.0;      // spiky boundary sum (PCISPH)
    double ax = 0.0, ay = 0.0, az = 0.0;         // adhesion sum
};

// What a particle's list and sums give, stored: `cnt` members, `own` of them
// in the list; nearBound (PCISPH): its cells hold boundary particles.  Returns
// its share of the average divergence error (DFSPH).
template <int M>
__device__ inline double build_finish(const DevScene& S, const KCoefD& k, int i, const float4& xi, const float4& vi,
                                      const BuildSums& b, int cnt, int own, int ngr, bool nearBound) {
    const double rho0 = S.rho0D, m = S.mD;
    if (cnt > S.maxNbr) {
        atomicMax(&S.ss->overflow, (unsigned)cnt);
        atomicMax(&S.ss->listOver, (unsigned)cnt);
    }
    stg(S.nnb, (size_t)i, (uint16_t)own);
    stg(S.ngrad, (size_t)i, (uint8_t)min(ngr, 255));
    const double drho = (m * (k.ck + b.ws) + b.bw) - rho0;
    const double rho = rho0 + drho;
    stg(S.drho, (size_t)i, (float)drho);
    st4(S.gb, i, make_float4((float)b.bgx, (float)b.bgy, (float)b.bgz, (float)b.bw));
    if (S.flags & F_ADH) st4(S.adh, i, make_float4((float)b.ax, (float)b.ay, (float)b.az, 0.f));
    if (M == DFSPH) {
        const double tx = m * b.sgx + b.bgx, ty = m * b.sgy + b.bgy, tz = m * b.sgz + b.bgz;
        const double den = tx * tx + ty * ty + tz * tz + m * m * b.ssq;
        const float alpha = (fabs(den) > 1e-5) ? (float)(rho / den) : 0.0f;
        stg(S.alpha, (size_t)i, alpha);
        // initial divergence error of the step's divergence solve
        // (computeDivergenceError, src/DFSPHSolver.cpp:408-492, and kappa_v,
        // :531), from the pairs above; stored values are read back as the
        // later sweeps read them (FP32 gb, delta rho, alpha)
        const float4 gbf = make_float4((float)b.bgx, (float)b.bgy, (float)b.bgz, (float)b.bw);
        const double ux = vi.x, uy = vi.y, uz = vi.z;
        const double dc = m * b.dv + (ux * (double)gbf.x + uy * (double)gbf.y + uz * (double)gbf.z);
        const double de = (ngr < 20) ? 0.0 : fmax(dc, 0.0);
        const double rhof = rho0 + (double)(float)drho;
        // the divergence of the velocities: the next step's D0 unless a
        // divergence iteration replaces it
        ((gptr<double>)S.d0)[i] = dc;
        stg(S.divErr, (size_t)i, (float)de);
        st4(S.xk, i, make_float4(xi.x, xi.y, xi.z, (float)(de * (double)alpha / (S.ss->dt * rhof))));
        return de / rho0;
    }
    if (M == WCSPH) {
        // p = max(0, kappa rho0/gamma ((rho/rho0)^gamma - 1)), written
        // (1+x)^g - 1 = expm1(g log1p(x)) with x = (rho - rho0)/rho0
        const double x = drho / rho0;
        const double pr = fmax(0.0, (double)S.stiffness * rho0 / (double)S.gammaEos * expm1((double)S.gammaEos * log1p(x)));
        stg(S.p, (size_t)i, (float)pr);
        st4(S.xk, i, make_float4(xi.x, xi.y, xi.z, (float)(pr / (rho * rho))));
        const float4 v = ld4(S.v, i);
        st4(S.aux, i, make_float4(v.x, v.y, v.z, (float)(m / rho)));
    } else {
        st4(S.gbs, i, make_float4((float)b.sx2, (float)b.sy2, (float)b.sz2, nearBound ? 1.f : 0.f));
    }
    return 0.0;
}

// The end of a DFSPH list build: the chunks' shares of the error before the
// divergence loop (only the log has it; k_build_quad: the groups') go to the
// sort's scratch, and one thread of a scene starts the divergence loop
// (`fused`: no finalize kernel does).
__device__ inline void build_starts_divergence(const DevScene& S, int fused) {
    Scalars* const ss = S.ss;
    ss->d0Valid = 1u;
    if (fused) {
        ss->itV = 0;
        ss->time += ss->dt;
        ss->doneV = loop_goes_on<LOOP_DIV>(S, ss, 0, 0.0) ? 0 : 1;
    }
}

template <int M>
__global__ __launch_bounds__(kBlock) void k_build(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                  int fused) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    __shared__ float2 sxy[kBuildStage + kBuildPad];
    __shared__ float sz[kBuildStage + kBuildPad];
    __shared__ int sd[9];
    const int i = c.begin + threadIdx.x;
    if (c.begin >= S.n) {
        // past the active particles, of which a scene with emitters may have
        // none: there is no cell to take the row ranges from
        if (M == DFSPH && threadIdx.x == 0) {
            group_partial(S, 0)[c.begin / kBlock] = 0.0;
            if (c.begin == 0) build_starts_divergence(S, fused);
        }
        return;
    }
    const bool valid = i < S.n;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const KCoefD k = S.kd;
    const float hh = S.kc.hhi2 * (1.0f + 1e-5f);   // conservative FP32 pre-filter
    const float4 xi = valid ? ld4(S.x, i) : make_float4(0.f, 0.f, 0.f, 0.f);
    const double xx = xi.x, xy = xi.y, xz = xi.z;
    const int ci = valid ? ldg(S.cell, (size_t)i) : 0;
    const int nx = S.nx, nxny = S.nx * S.ny;

    // the block's 9 row ranges: first particle and offset in the stage
    int rfirst = 0, rcnt = 0;
    if (lane < 9) {
        const int cF = ldg(S.cell, (size_t)c.begin), cL = ldg(S.cell, (size_t)min(c.begin + kBlock - 1, S.n - 1));
        const int off = (lane % 3 - 1) * nx + (lane / 3 - 1) * nxny;
        rfirst = ldg(S.cellStart, (size_t)(cF - 1 + off));
        rcnt = ldg(S.cellStart, (size_t)(cL + 2 + off)) - rfirst;
    }
    int incl = rcnt;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        const int t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    int first[9], base[10];
    base[0] = 0;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        first[r] = __builtin_amdgcn_readlane(rfirst, r);
        base[r + 1] = __builtin_amdgcn_readlane(incl, r);
    }
    // the leading rows that fit are staged (all 9 in a dense fluid); the
    // others are read from global memory
    int nStaged = 0;
#pragma unroll
    for (int r = 0; r < 9; ++r)
        if (base[r + 1] <= kBuildStage) nStaged = r + 1;
    if (lane < 9 && w == 0) sd[lane] = incl - rcnt - rfirst;
    {
        // 4 loads per lane in flight before the first is written to LDS
        const int tot = base[nStaged];
        for (int t0 = threadIdx.x; t0 < tot; t0 += 4 * kBlock) {
            float4 p[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = t0 + kBlock * u;
                int o = first[0];
#pragma unroll
                for (int q = 1; q < 9; ++q)
                    if (t >= base[q]) o = first[q] - base[q];
                if (t < tot) p[u] = ld3o(S.x, (uint32_t)(o + t));
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = t0 + kBlock * u;
                if (t < tot) {
                    sxy[t] = make_float2(p[u].x, p[u].y);
                    sz[t] = p[u].z;
                }
            }
        }
    }
    __syncthreads();

    uint32_t* L = list_of_w(S, valid ? i : (i & ~63));
    const int maxN = S.maxNbr;
    // Pass 1's survivors go to the group's list memory (a uniform base, so
    // each store takes the base + 32-bit offset form; a group's list is maxN
    // KB): slot by slot, 64 lanes' entries in a row, so a store touches a few
    // 64 B lines, until pass 2, which has read a block of 4 slots in all lanes
    // before it writes that KB as 16 B a lane.  PCISPH has the shells of other
    // lanes there and stores where the list has its slots.
    char* const Lw = (char*)(S.nbr + (size_t)__builtin_amdgcn_readfirstlane(i >> 6) * (size_t)maxN * kGroup);
    constexpr bool kRows = M != PCISPH;
    // where all rows are staged a survivor is kept as its place in the stage
    // and its row, and pass 2 reads its position there
    const bool codes = nStaged == 9;
    const uint32_t lane4 = (uint32_t)lane << 2, lane16 = (uint32_t)lane << 4;
    auto putAt = [&](uint32_t at, uint32_t j) { *(gptr<uint32_t>)((gptr<char>)Lw + at) = j; };
    auto putSlot = [&](int s, uint32_t j) { putAt((slot_of(s) << 2) | lane16, j); };
    // PCISPH: the shell, candidates within h + skin that are not in the
    // list, fills the slots from the last one down; it stands in for the
    // 27-cell walk of the predicted densities while it fits beside the list
    float hsk = 0.f;
    if (M == PCISPH && S.pciShell) {
        const float hs = S.kc.h + pci_skin(S);
        hsk = hs * hs * (1.0f + 1e-4f);
    }
    int ns = 0;
    bool shellLost = false;
    int cnt = 0, ngr = 0;
    BuildSums b;
    const float4 vi = (M == DFSPH && valid) ? ld4(S.v, i) : make_float4(0.f, 0.f, 0.f, 0.f);
    const double ux = vi.x, uy = vi.y, uz = vi.z;
    // FP64 test and sums of one candidate that passed the FP32 test
    int nc = 0;   // FP32 survivors of pass 1
    // a survivor the FP64 test rejects goes to the shell (PCISPH)
    auto toShell = [&](uint32_t j) {
        if (M != PCISPH) return;
        if (ns < maxN - nc) stg(L, (size_t)slot_of(maxN - 1 - ns), j);
        else shellLost = true;
        ++ns;
    };
    auto visit = [&](uint32_t j, const float4& xj, const float4& vj) {
        const Pair p = pair_of(xx, xy, xz, xj, k);
        double g, wq;
        bool gnz;
        if (!member_of(p, xi, xj, S.hD, k, g, wq, gnz)) {
            toShell(j);
            return false;
        }
        ++cnt;
        ngr += gnz ? 1 : 0;
        b.ws += wq;
        b.sgx += g * p.dx;
        b.sgy += g * p.dy;
        b.sgz += g * p.dz;
        b.ssq += g * g * p.r2;
        if (M == DFSPH) b.dv += g * ((ux - (double)vj.x) * p.dx + (uy - (double)vj.y) * p.dy + (uz - (double)vj.z) * p.dz);
        return true;
    };
    auto vel = [&](uint32_t j) { return (M == DFSPH) ? ld3o(S.v, j) : make_float4(0.f, 0.f, 0.f, 0.f); };
    // Pass 1 over the 27 cells as 9 rows (walk27 order), up to 32 candidates
    // of a row at a time: their tests go to the bits of a mask, kScan
    // candidates' loads before the first test, and the survivors are then taken
    // from it.  Candidates past the row's end are read (staged rows: at most
    // kScan - 1, inside the padded stage) and dropped with the mask's last bits.
    // fetch(j): position of candidate j; self: the row may hold particle i;
    // survivor j is kept as j + code
    auto scanRow = [&](int s0, int e0, bool self, int code, auto&& fetch) {
        for (int c0 = s0; c0 < e0; c0 += 32) {
            const int nv = min(e0 - c0, 32);
            uint32_t mo = 0, ms = 0;
            int k0 = 0;
            for (; k0 < nv; k0 += kScan) {
                float3 p[kScan];
#pragma unroll
                for (int u = 0; u < kScan; ++u) p[u] = fetch(c0 + k0 + u);
#pragma unroll
                for (int u = 0; u < kScan; ++u) {
                    const float fx = xi.x - p[u].x, fy = xi.y - p[u].y, fz = xi.z - p[u].z;
                    if (M == PCISPH) {
                        const float d2 = fx * fx + fy * fy + fz * fz;
                        mo = mo + mo + (d2 <= hh ? 1u : 0u);
                        ms = ms + ms + (d2 <= hsk ? 1u : 0u);
                    } else {
                        // the sign of d2 - hh
                        mo = __builtin_amdgcn_alignbit(mo, __float_as_uint(fmaf(fz, fz, fmaf(fy, fy, fmaf(fx, fx, -hh)))), 31);
                    }
                }
            }
            // bit b: candidate jb + b
            const int jb = c0 + nv - 32;
            mo = __builtin_bitreverse32(mo >> (k0 - nv));
            if (self && (uint32_t)(i - c0) < (uint32_t)nv) mo &= ~(1u << (i - jb));
            if (M == PCISPH) {
                ms = __builtin_bitreverse32(ms >> (k0 - nv)) & ~mo;
                if (self && (uint32_t)(i - c0) < (uint32_t)nv) ms &= ~(1u << (i - jb));
            }
            // past the last slot the particle takes the one-pass walk
            if (nc + __popc(mo) > maxN) {
                nc = maxN + 1;
                mo = 0;
            }
            uint32_t at = lane4 + (uint32_t)nc * 256u;
            nc += __popc(mo);
            int s = nc - __popc(mo);
            while (mo) {
                const uint32_t j = (uint32_t)(jb + code + __builtin_ctz(mo));
                mo &= mo - 1u;
                if (kRows) {
                    putAt(at, j);
                    at += 256u;
                } else {
                    putSlot(s++, j);
                }
            }
            if (M == PCISPH)
                while (ms) {
                    const uint32_t j = (uint32_t)(jb + __builtin_ctz(ms));
                    ms &= ms - 1u;
                    // below the list's slots only (list writes that later
                    // reach the shell are caught by nc + ns > maxN)
                    if (nc + ns < maxN) putSlot(maxN - 1 - ns, j);
                    else shellLost = true;
                    ++ns;
                }
        }
    };
    if (valid) {
        // the 9 rows' ranges are loaded before pass 1's first list store:
        // a wait for a load also waits for every store issued before it
        int rs[9], re[9];
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int off = (r % 3 - 1) * nx + (r / 3 - 1) * nxny;
            rs[r] = ldg(S.cellStart, (size_t)(ci - 1 + off));
            re[r] = ldg(S.cellStart, (size_t)(ci + 2 + off));
        }
        static_for<9>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            // particle i can only lie in row 4 (cells ci-1..ci+1): the other
            // rows are offset by at least nx >= 3 cells
            if (r < nStaged) {
                const int d = base[r] - first[r];
                scanRow(rs[r], re[r], r == 4, codes ? d + (r << 16) : 0, [&](int j) {
                    const float2 a = sxy[j + d];
                    return make_float3(a.x, a.y, sz[j + d]);
                });
            } else {
                const int last = re[r] - 1;
                scanRow(rs[r], re[r], r == 4, 0, [&](int j) {
                    const float4 p = ld4(S.x, (size_t)min(j, last));
                    return make_float3(p.x, p.y, p.z);
                });
            }
        });
    }
    if (M == PCISPH && nc + ns > maxN) shellLost = true;
    // the lanes' survivors lie in common rows, and pass 2 writes lists over
    // them: it starts after every lane's pass 1
    wave_sync();
    if (valid && nc <= maxN) {
        // 4 survivors per pass, their list entries and positions loaded
        // first; visit writes slots <= the one it reads, so entries
        // already loaded are not overwritten before use, and the next
        // block of entries is requested before this pass's data is used
        auto entries = [&](int q0) {
            if (!kRows) return ld_block(L, q0 >> 2);
            v4u e;
#pragma unroll
            for (int u = 0; u < 4; ++u) e[u] = *(gptr<const uint32_t>)((gptr<char>)Lw + (lane4 + (uint32_t)(q0 + u) * 256u));
            return e;
        };
        const uint32_t own0 = (uint32_t)i + (codes ? (uint32_t)(base[4] - first[4] + (4 << 16)) : 0u);
        v4u bn = entries(0);
        for (int q0 = 0; q0 < nc; q0 += 4) {
            // one block of 4 slots; those past the last survivor hold
            // stale values and are replaced by the particle itself
            v4u jj = bn;
#pragma unroll
            for (int u = 0; u < 4; ++u) jj[u] = q0 + u < nc ? jj[u] : own0;
            float4 xj[4], vj[4];
            if (codes) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t t = jj[u] & 0xFFFFu;
                    const float2 a = sxy[t];
                    xj[u] = make_float4(a.x, a.y, sz[t], 0.f);
                    jj[u] = t - (uint32_t)sd[jj[u] >> 16];
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) xj[u] = ld3o(S.x, jj[u]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) vj[u] = vel(jj[u]);
            bn = entries(q0 + 4 < nc ? q0 + 4 : q0);
            asm volatile("" ::: "memory");
            // every lane has read this block's rows before one writes there
            __builtin_amdgcn_wave_barrier();
            const int c0 = cnt;
            bool in[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) in[u] = q0 + u < nc && visit(jj[u], xj[u], vj[u]);
            // where the FP64 test has rejected none so far the whole block
            // goes out, past the last survivor the particle itself
            if (c0 == q0 && cnt - c0 == min(4, nc - q0)) {
                *(gptr<v4u>)((gptr<char>)Lw + ((uint32_t)q0 * 256u + lane16)) = jj;
            } else {
                int to = c0;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (in[u]) putSlot(to++, jj[u]);
            }
        }
    }
    // (after every lane's pass 2: a walk writes its list where the others'
    // survivors were)
    wave_sync();
    const bool walk = valid && nc > maxN;
    if (walk) {
        shellLost = true;
        ns = maxN;   // toShell writes nothing from here on
        walk27(S.cellStart, ci, nx, nxny, [&](int j) {
            const float4 xj = ld4(S.x, j);
            const float fx = xi.x - xj.x, fy = xi.y - xj.y, fz = xi.z - xj.z;
            if (!(fx * fx + fy * fy + fz * fz <= hh) || j == i) return;
            if (visit((uint32_t)j, xj, vel((uint32_t)j)) && cnt <= maxN) putSlot(cnt - 1, (uint32_t)j);
        });
    }
    // pad the list with the particle itself up to the group's longest list
    // rounded to 4 (a self term is exactly zero in every sweep)
    const int own = min(cnt, maxN);
    int pad = min((own + 3) & ~3, maxN);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pad = max(pad, __shfl_xor(pad, o));
    double e = 0.0;   // DFSPH: this particle's share of the average divergence error
    if (valid) {
    const bool wantAdh = (S.flags & F_ADH) != 0;
    const double rho0 = S.rho0D;
    // boundary sums, in two passes like the fluid: FP32 survivors go to the
    // free list slots past the fluid list, then the FP64 pass runs over them
    auto bvisit = [&](const float4& y) {
        const Pair p = pair_of(xx, xy, xz, y, k);
        if (!(p.q <= 1.0)) return;
        const double cb = rho0 * (double)y.w;
        b.bw += cb * W_d(p.q, k);
        const double g = cb * G_d(p, k);
        b.bgx += g * p.dx;
        b.bgy += g * p.dy;
        b.bgz += g * p.dz;
        if (M == PCISPH) {
            const double gs = cb * Gs_d(p, k);
            b.sx2 += gs * p.dx;
            b.sy2 += gs * p.dy;
            b.sz2 += gs * p.dz;
        }
        if (wantAdh && p.r2 > 0.0) {
            const double sa = cb * A_d(p.rl, k) * p.inv;
            b.ax += sa * p.dx;
            b.ay += sa * p.dy;
            b.az += sa * p.dz;
        }
    };
    // the boundary survivors use the free slots between the list's blocks and
    // the shell
    const int free0 = (own + 3) & ~3;
    const int room = max(0, maxN - free0 - ((M == PCISPH && !shellLost) ? ns : 0));
    int nbc = 0;
    bool nearBound = false;
    {
        // the 9 rows' ranges first, then 4 candidates' loads at a time: a
        // wait for a load also waits for the survivor stores before it
        int bs[9], be[9];
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int off = (r % 3 - 1) * nx + (r / 3 - 1) * nxny;
            bs[r] = ldg(S.bCellStart, (size_t)(ci - 1 + off));
            be[r] = ldg(S.bCellStart, (size_t)(ci + 2 + off));
        }
        if (M == PCISPH) {
#pragma unroll
            for (int r = 0; r < 9; ++r) nearBound |= be[r] > bs[r];
        }
#pragma unroll 1
        for (int r = 0; r < 9; ++r) {
            for (int b0 = bs[r]; b0 < be[r]; b0 += 4) {
                float4 y[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] = ld4(S.xb, min(b0 + u, be[r] - 1));
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float fx = xi.x - y[u].x, fy = xi.y - y[u].y, fz = xi.z - y[u].z;
                    if ((b0 + u < be[r]) & (fx * fx + fy * fy + fz * fz <= hh)) {
                        if (nbc < room) putSlot(free0 + nbc, (uint32_t)(b0 + u));
                        ++nbc;
                    }
                }
            }
        }
    }
    if (nbc <= room) {
        for (int q0 = 0; q0 < nbc; q0 += 4) {
            float4 yb[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                yb[u] = ld4(S.xb, ldg((const uint32_t*)L, (size_t)slot_of(free0 + min(q0 + u, nbc - 1))));
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (q0 + u < nbc) bvisit(yb[u]);
        }
    } else {
        walk27(S.bCellStart, ci, nx, nxny, [&](int jb) {
            const float4 y = ld4(S.xb, jb);
            const float fx = xi.x - y.x, fy = xi.y - y.y, fz = xi.z - y.z;
            if (fx * fx + fy * fy + fz * fz <= hh) bvisit(y);
        });
    }
    // pad the list with the particle itself up to the group's longest list
    // (overwrites the boundary survivors' slots); pass 2 has filled the last
    // block unless the FP64 test rejected a survivor
    if (cnt != nc)
        for (int q = own; q < free0; ++q) putSlot(q, (uint32_t)i);
    const uint32_t self = (uint32_t)i;
    for (int q = free0; q < pad; q += 4) *(gptr<v4u>)((gptr<char>)Lw + ((uint32_t)q * 256u + lane16)) = v4u{self, self, self, self};
    if (M == PCISPH) {
        if (pad + ns > maxN) shellLost = true;   // the padding reached the shell
        stg(S.nsh, (size_t)i, (uint16_t)(shellLost ? 0xFFFF : ns));
    }
    if ((i & 63) == 0) stg(S.gcnt, (size_t)(i >> 6), (uint16_t)pad);
    e = build_finish<M>(S, k, i, xi, vi, b, cnt, own, ngr, nearBound);
    }
    if (M == DFSPH) {
        __shared__ double sh[kWaves];
        const double bs = block_sum(e, sh);
        if (threadIdx.x == 0) group_partial(S, 0)[c.begin / kBlock] = bs;
        if (c.begin == 0 && threadIdx.x == 0) build_starts_divergence(S, fused);
    }
}

// The same build with 4 lanes a particle, for launches too small to fill the
// chip.  A block of 8 wavefronts holds one list group (part_at): in wavefronts
// 0-3 lane 4 q + u of wavefront w works on the fluid candidates 4 k + u of
// particle 16 w + q, in 4-7 likewise on the boundary's.  The tests' signs are
// shifted into a mask a lane, the quad's masks joined, so that every lane knows
// the place of its survivors in the list; up to 126 of a particle wait in LDS,
// as their place in the stage and their row.  The four lanes' FP64 terms are
// added one after the other in list order, in every lane alike, so the sums are
// k_build's bit for bit.
//
// A lone wavefront a SIMD bounds it: ~2,000 instructions of ~10 cycles for the
// fluid, as many for the boundary of a particle in a corner, which ran one
// after the other (23 us for 2,197 particles, 13 of them in the slowest block's
// boundary, read from memory where the group's row ranges, with the walls
// between two rows of fluid, exceeded the stage).  Side by side 14 us.  A step:
// WCSPH 2,197 particles 83 -> 37 us (one lane 64), 32,768 71 -> 42, PCISPH
// 4,845 154 -> 122, DFSPH 4,096 131 -> 94, 9,261 125 -> 100 (one lane -> 4).
// DFSPH takes one survivor a lane at a time: two at once need 184 registers,
// which leaves one block a compute unit (35,805 particles 164 us, now 152).
constexpr int kQuadStage = 1024;   // fluid candidates staged (12 B each); ~800 are usual, more where a group goes on to the next row
constexpr int kQuadBound = 512;    // boundary candidates staged (16 B each)
constexpr int kQuadPad = 32;       // reads past a row's end
// survivors of a particle kept in LDS, of the fluid (2 B each) and of the
// boundary (4 B); odd numbers of dwords a particle
constexpr int kQuadList = 126, kQuadBoundList = 45;
// a particle's boundary sums (see BuildSums) from the wavefronts that form them
struct BoundSums {
    double bw, gx, gy, gz, sx, sy, sz, ax, ay, az;
    int near;
};

template <int M>
__global__ __launch_bounds__(512, 4) void k_build_quad(const DevScene* __restrict__ T, const Chunk* __restrict__ C, int nchunks,
                                                    int fused) {
    Chunk c;
    int g0, i;   // the group's first particle and the lane's
    if (!part_at<4>(C, nchunks, c, g0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    __shared__ float2 sxy[kQuadStage + kQuadPad];
    __shared__ float sz[kQuadStage + kQuadPad];
    __shared__ float4 sb[kQuadBound + kQuadPad];
    __shared__ uint16_t sl[kGroup * kQuadList];
    __shared__ uint32_t sbl[kGroup * kQuadBoundList];
    __shared__ BoundSums sbs[kGroup];
    __shared__ int sd[9];
    __shared__ int spad[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, u = lane & 3;
    const bool fluid = w < 4;                // wavefronts 0-3: the fluid, 4-7: the boundary
    const int pl = (tid & 255) >> 2;         // the lane's particle in the group
    i = g0 + pl;
    if (g0 >= S.n) {
        if (M == DFSPH && tid == 0) group_partial(S, 0)[g0 >> 6] = 0.0;
        return;
    }
    const bool valid = i < S.n;
    const int il = min(i, S.n - 1);
    const KCoefD k = S.kd;
    const float hh = S.kc.hhi2 * (1.0f + 1e-5f);   // conservative FP32 pre-filter
    const float4 xi = ld4(S.x, (size_t)il);
    const int ci = ldg(S.cell, (size_t)il);
    const int cF = ldg(S.cell, (size_t)g0), cL = ldg(S.cell, (size_t)min(g0 + kGroup - 1, S.n - 1));
    const float4 vi = (M == DFSPH) ? ld4(S.v, (size_t)il) : make_float4(0.f, 0.f, 0.f, 0.f);
    const double xx = xi.x, xy = xi.y, xz = xi.z;
    const double ux = vi.x, uy = vi.y, uz = vi.z;
    const int nx = S.nx, nxny = S.nx * S.ny;
    // the particle's 9 fluid or boundary rows, and the group's 9 fluid (lanes
    // 0..8) and boundary (lanes 16..24) rows with their offsets in the stages
    const int* const rows = fluid ? S.cellStart : S.bCellStart;
    int rs[9], re[9];
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const int off = (r % 3 - 1) * nx + (r / 3 - 1) * nxny;
        rs[r] = ldg(rows, (size_t)(ci - 1 + off));
        re[r] = ldg(rows, (size_t)(ci + 2 + off));
    }
    int rfirst = 0, rcnt = 0;
    const int lr = lane & 15;
    if (lane < 32 && lr < 9) {
        const int off = (lr % 3 - 1) * nx + (lr / 3 - 1) * nxny;
        const int* const tab = lane < 16 ? S.cellStart : S.bCellStart;
        rfirst = ldg(tab, (size_t)(cF - 1 + off));
        rcnt = ldg(tab, (size_t)(cL + 2 + off)) - rfirst;
    }
    int incl = rcnt;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        const int t = __shfl_up(incl, o);
        if (lr >= o) incl += t;
    }
    int first[9], base[10], bfirst[9], bbase[10];
    base[0] = bbase[0] = 0;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        first[r] = __builtin_amdgcn_readlane(rfirst, r);
        base[r + 1] = __builtin_amdgcn_readlane(incl, r);
        bfirst[r] = __builtin_amdgcn_readlane(rfirst, 16 + r);
        bbase[r + 1] = __builtin_amdgcn_readlane(incl, 16 + r);
    }
    // the leading fluid rows that fit are staged, and the boundary rows where
    // all of them fit; what is not staged is read from memory
    int nStaged = 0;
#pragma unroll
    for (int r = 0; r < 9; ++r)
        if (base[r + 1] <= kQuadStage) nStaged = r + 1;
    const int tot = base[nStaged];
    const bool staged = nStaged == 9;
    if (tid < 9) sd[tid] = incl - rcnt - rfirst;
    const bool bStaged = bbase[9] <= kQuadBound;
    const int btot = bStaged ? bbase[9] : 0;
    {
        auto at = [&](int t, const int* f, const int* bs) {
            int o = f[0];
#pragma unroll
            for (int q = 1; q < 9; ++q)
                if (t >= bs[q]) o = f[q] - bs[q];
            return o + t;
        };
        float4 p[2], y;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (tid + 512 * q < tot) p[q] = ld3o(S.x, (uint32_t)at(tid + 512 * q, first, base));
        if (tid < btot) y = ld4o(S.xb, (uint32_t)at(tid, bfirst, bbase));
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (tid + 512 * q < tot) {
                sxy[tid + 512 * q] = make_float2(p[q].x, p[q].y);
                sz[tid + 512 * q] = p[q].z;
            }
        if (tid < btot) sb[tid] = y;
    }
    __syncthreads();

    uint32_t* const L = list_of_w(S, g0 + pl);
    const int maxN = S.maxNbr;
    const uint32_t below = (1u << u) - 1u;
    const int qshift = lane & ~3;
    // the quad's 4 flags, lane u in bit u
    auto quad_bits = [&](bool f) { return (uint32_t)(__ballot(f) >> qshift) & 15u; };
    float hsk = 0.f;
    if (M == PCISPH && S.pciShell) {
        const float hs = S.kc.h + pci_skin(S);
        hsk = hs * hs * (1.0f + 1e-4f);
    }
    int nc = 0, ns = 0;
    bool shellLost = false;
    // up to 32 candidates c0.. of a row, every 4th of them a lane's: the sign
    // of each test is shifted into bits 31, 27, .. of m.  Makes bit b stand for
    // candidate c0 + b, of nv; m: the lane's own, returns the quad's
    auto joined = [&](uint32_t& m, int nv) {
        m = __builtin_bitreverse32((m & 0x88888888u) >> u);
        if (nv < 32) m &= (1u << nv) - 1u;
        uint32_t f = m | (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xF, 0xF, true);
        return f | (uint32_t)__builtin_amdgcn_mov_dpp((int)f, 0x4E, 0xF, 0xF, true);
    };
    auto test = [&](float fx, float fy, float fz, float bound) {
        return __float_as_uint(fmaf(fz, fz, fmaf(fy, fy, fmaf(fx, fx, -bound))));
    };
    uint16_t* const mine = sl + pl * kQuadList;
    uint32_t* const bmine = sbl + pl * kQuadBoundList;
    // the lane's survivors m of f, kept as code + bit from place n of the list on
    auto keep = [&](uint32_t m, uint32_t f, int n, uint32_t code, auto* list, int most) {
        while (m) {
            const int b = __builtin_ctz(m);
            m &= m - 1u;
            const int to = n + __popc(f & ((1u << b) - 1u));
            if (to < most) list[to] = (std::remove_pointer_t<decltype(list)>)(code + b);
        }
    };
    // pass 1: this lane's candidate j at squared distance d2 (in: it is one)
    auto scan = [&](bool in, uint32_t j, float d2) {
        const bool ok = in & (d2 <= hh);
        const uint32_t okb = quad_bits(ok);
        if (M == PCISPH) {
            const bool sh = in & (d2 > hh) & (d2 <= hsk);
            const uint32_t shb = quad_bits(sh);
            const int sn = ns + __popc(shb & below);
            if (sh) {
                // below the list's slots only (list writes that later reach
                // the shell are caught by nc + ns > maxN)
                if (nc + __popc(okb & below) + sn < maxN) stg(L, (size_t)slot_of(maxN - 1 - sn), j);
                else shellLost = true;
            }
            ns += __popc(shb);
        }
        // past the last slot the particle takes the walk over all candidates,
        // which rewrites its list: the store is clamped to the last slot
        if (ok) stg(L, (size_t)slot_of(min(nc + __popc(okb & below), maxN - 1)), j);
        nc += __popc(okb);
    };
    bool lds = staged;
    if (fluid && valid && lds) {
        static_for<9>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            const int d = base[r] - first[r];
            for (int c0 = rs[r]; c0 < re[r]; c0 += 32) {
                const int nv = min(re[r] - c0, 32);
                const float2* const pxy = sxy + c0 + d + u;
                const float* const pz = sz + c0 + d + u;
                uint32_t m = 0, ms = 0;
                auto half = [&](int k0) {
                    float2 a[4];
                    float z[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        a[k] = pxy[k0 + 4 * k];
                        z[k] = pz[k0 + 4 * k];
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float fx = xi.x - a[k].x, fy = xi.y - a[k].y, fz = xi.z - z[k];
                        if (M == PCISPH) {
                            const float d2 = fx * fx + fy * fy + fz * fz;
                            m = (m << 4) | (d2 <= hh ? 8u : 0u);
                            ms = (ms << 4) | (d2 <= hsk ? 8u : 0u);
                        } else {
                            m = __builtin_amdgcn_alignbit(m, test(fx, fy, fz, hh), 28);
                        }
                    }
                };
                half(0);
                if (nv > 16) {
                    half(16);
                } else {
                    m <<= 16;
                    ms <<= 16;
                }
                uint32_t f = joined(m, nv);
                // particle i itself can only lie in row 4
                const uint32_t other = (r == 4 && (uint32_t)(i - c0) < 32u) ? ~(1u << (i - c0)) : ~0u;
                f &= other;
                m &= other;
                keep(m, f, nc, (uint32_t)(c0 + d + (r << 12)), mine, kQuadList);
                nc += __popc(f);
                if (M == PCISPH) {
                    uint32_t fs = joined(ms, nv);
                    fs &= other & ~f;
                    ms &= fs;
                    while (ms) {
                        const int b = __builtin_ctz(ms);
                        ms &= ms - 1u;
                        const int sn = ns + __popc(fs & ((1u << b) - 1u));
                        // below the list's slots only (list writes that later
                        // reach the shell are caught by nc + ns > maxN)
                        if (nc + sn < maxN) stg(L, (size_t)slot_of(maxN - 1 - sn), (uint32_t)(c0 + b));
                        else shellLost = true;
                    }
                    ns += __popc(fs);
                }
            }
        });
    }
    // survivors that LDS does not hold, like those of rows that are not
    // staged, go through the list's memory
    if (fluid && lds && __any(nc > kQuadList && nc <= maxN)) {
        lds = false;
        nc = ns = 0;
        shellLost = false;
    }
    if (fluid && valid && !lds) {
        static_for<9>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            const int s0 = rs[r], e0 = re[r];
            if (r < nStaged) {
                const int t0 = base[r] - first[r] + u;
                for (int j0 = s0; j0 < e0; j0 += 8) {
                    float d2[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const float2 a = sxy[t0 + j0 + 4 * h];
                        const float fx = xi.x - a.x, fy = xi.y - a.y, fz = xi.z - sz[t0 + j0 + 4 * h];
                        d2[h] = fx * fx + fy * fy + fz * fz;
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int j = j0 + 4 * h + u;
                        // particle i itself can only lie in row 4
                        scan((j < e0) & (r != 4 || j != i), (uint32_t)j, d2[h]);
                    }
                }
            } else {
                for (int j0 = s0; j0 < e0; j0 += 4) {
                    const int j = j0 + u;
                    const float4 a = ld4(S.x, (size_t)min(j, e0 - 1));
                    const float fx = xi.x - a.x, fy = xi.y - a.y, fz = xi.z - a.z;
                    scan((j < e0) & (j != i), (uint32_t)j, fx * fx + fy * fy + fz * fz);
                }
            }
        });
    }
    shellLost = quad_bits(shellLost) != 0u;
    int cnt = 0, ngr = 0;
    BuildSums b;
    if (M == PCISPH && nc + ns > maxN) shellLost = true;
    if (fluid && valid && nc <= maxN) {
        // pass 2, kH survivors a lane at a time
        constexpr int kH = M == DFSPH ? 1 : 2;
        auto sums = [&](int q0, const uint32_t* j, const float4* xj, const float4* vj) {
#pragma unroll
            for (int h = 0; h < kH; ++h) {
                const int pos = q0 + 4 * h + u;
                const Pair p = pair_of(xx, xy, xz, xj[h], k);
                double g = 0.0, wq = 0.0;
                bool gnz = false;
                const bool cand = pos < nc;
                const bool in = cand && member_of(p, xi, xj[h], S.hD, k, g, wq, gnz);
                const uint32_t inb = quad_bits(in);
                if (M == PCISPH) {
                    // what the FP64 test rejects goes to the shell
                    const uint32_t rj = quad_bits(cand && !in);
                    const int sn = ns + __popc(rj & below);
                    if (cand && !in) {
                        if (sn < maxN - nc) stg(L, (size_t)slot_of(maxN - 1 - sn), j[h]);
                        else shellLost = true;
                    }
                    ns += __popc(rj);
                }
                // an entry is written only where the compaction moves it
                const int to = cnt + __popc(inb & below);
                if (in && (lds || to != pos)) stg(L, (size_t)slot_of(to), j[h]);
                cnt += __popc(inb);
                ngr += __popc(quad_bits(in && gnz));
                // in list order; a lane without a member adds zeros, which
                // change no sum (all factors: a rejected candidate's position
                // or velocity may be infinite or NaN)
                if (!in) g = wq = 0.0;
                const double gg = g * g;
                double dx = p.dx, dy = p.dy, dz = p.dz, r2 = p.r2;
                double dot = (M == DFSPH) ? (ux - (double)vj[h].x) * p.dx + (uy - (double)vj[h].y) * p.dy +
                                                (uz - (double)vj[h].z) * p.dz
                                          : 0.0;
                if (!in) dx = dy = dz = r2 = dot = 0.0;
                static_for<4>([&](auto vc) {
                    constexpr int v = decltype(vc)::value;
                    b.ws += quad_lane<v>(wq);
                    if (M == DFSPH) {
                        const double gv = quad_lane<v>(g);
                        b.sgx = fma(gv, quad_lane<v>(dx), b.sgx);
                        b.sgy = fma(gv, quad_lane<v>(dy), b.sgy);
                        b.sgz = fma(gv, quad_lane<v>(dz), b.sgz);
                        b.ssq = fma(quad_lane<v>(gg), quad_lane<v>(r2), b.ssq);
                        b.dv = fma(gv, quad_lane<v>(dot), b.dv);
                    }
                });
            }
        };
        if (lds) {
            // the next survivors' velocities are requested before the current
            // ones' sums; past the last survivor the particle itself
            const uint32_t own0 = (uint32_t)(i + base[4] - first[4] + (4 << 12));
            uint32_t e[kH], jn[kH];
            float4 vn[kH];
            auto next = [&](int q0) {
#pragma unroll
                for (int h = 0; h < kH; ++h) {
                    const int pos = q0 + 4 * h + u;
                    e[h] = pos < nc ? (uint32_t)mine[pos] : own0;
                    jn[h] = (e[h] & 0xFFFu) - (uint32_t)sd[e[h] >> 12];
                    vn[h] = (M == DFSPH) ? ld3o(S.v, jn[h]) : make_float4(0.f, 0.f, 0.f, 0.f);
                }
            };
            next(0);
            for (int q0 = 0; q0 < nc; q0 += 4 * kH) {
                float4 xj[kH], vj[kH];
                uint32_t j[kH];
#pragma unroll
                for (int h = 0; h < kH; ++h) {
                    const uint32_t t = e[h] & 0xFFFu;
                    const float2 a = sxy[t];
                    xj[h] = make_float4(a.x, a.y, sz[t], 0.f);
                    vj[h] = vn[h];
                    j[h] = jn[h];
                }
                next(q0 + 4 * kH);
                asm volatile("" ::: "memory");
                sums(q0, j, xj, vj);
            }
        } else {
            const uint32_t* const Lu = L + u;
            uint32_t jn[kH];
#pragma unroll
            for (int h = 0; h < kH; ++h) jn[h] = ldg(Lu, (size_t)slot_of(min(4 * h, maxN - 4)));
            for (int q0 = 0; q0 < nc; q0 += 4 * kH) {
                uint32_t j[kH];
                float4 xj[kH], vj[kH];
#pragma unroll
                for (int h = 0; h < kH; ++h) {
                    j[h] = (q0 + 4 * h + u < nc) ? jn[h] : (uint32_t)i;   // past the last: a valid index
                    xj[h] = ld3o(S.x, j[h]);
                    vj[h] = (M == DFSPH) ? ld3o(S.v, j[h]) : make_float4(0.f, 0.f, 0.f, 0.f);
                }
                // maxN is a multiple of 4: the block after the last is re-read
#pragma unroll
                for (int h = 0; h < kH; ++h) jn[h] = ldg(Lu, (size_t)slot_of(q0 + 4 * kH + 4 * h < nc ? q0 + 4 * kH + 4 * h : q0));
                asm volatile("" ::: "memory");
                sums(q0, j, xj, vj);
            }
        }
    } else if (fluid && valid) {
        // more survivors than slots: all candidates one after the other, the
        // four lanes alike
        shellLost = true;
        walk27(S.cellStart, ci, nx, nxny, [&](int j) {
            const float4 xj = ld4(S.x, j);
            const float fx = xi.x - xj.x, fy = xi.y - xj.y, fz = xi.z - xj.z;
            if (!(fx * fx + fy * fy + fz * fz <= hh) || j == i) return;
            const Pair p = pair_of(xx, xy, xz, xj, k);
            double g, wq;
            bool gnz;
            if (!member_of(p, xi, xj, S.hD, k, g, wq, gnz)) return;
            if (cnt < maxN && u == 0) stg(L, (size_t)slot_of(cnt), (uint32_t)j);
            ++cnt;
            ngr += gnz ? 1 : 0;
            b.ws += wq;
            if (M == DFSPH) {
                const float4 vj = ld3o(S.v, (uint32_t)j);
                b.sgx = fma(g, p.dx, b.sgx);
                b.sgy = fma(g, p.dy, b.sgy);
                b.sgz = fma(g, p.dz, b.sgz);
                b.ssq = fma(g * g, p.r2, b.ssq);
                b.dv = fma(g, (ux - (double)vj.x) * p.dx + (uy - (double)vj.y) * p.dy + (uz - (double)vj.z) * p.dz, b.dv);
            }
        });
    }
    const bool wantAdh = (S.flags & F_ADH) != 0;
    const double rho0 = S.rho0D;
    // boundary sums, 4 survivors of the FP32 test at a time
    bool nearBound = false;
    if (!fluid && bbase[9] > 0 && valid) {
#pragma unroll
        for (int r = 0; r < 9; ++r) nearBound |= re[r] > rs[r];
        // one boundary candidate a lane
        auto bsums = [&](bool ok, const float4& y) {
            const Pair p = pair_of(xx, xy, xz, y, k);
            const bool in = ok && p.q <= 1.0;
            const double cb = in ? rho0 * (double)y.w : 0.0;
            const double wq = in ? W_d(p.q, k) : 0.0;
            const double g = in ? cb * G_d(p, k) : 0.0;
            const double gs = (M == PCISPH && in) ? cb * Gs_d(p, k) : 0.0;
            const double sa = (wantAdh && in && p.r2 > 0.0) ? cb * A_d(p.rl, k) * p.inv : 0.0;
            // (every factor of a candidate that is none is zero)
            const double px = in ? p.dx : 0.0, py = in ? p.dy : 0.0, pz = in ? p.dz : 0.0;
            static_for<4>([&](auto vc) {
                constexpr int v = decltype(vc)::value;
                const double dx = quad_lane<v>(px), dy = quad_lane<v>(py), dz = quad_lane<v>(pz);
                b.bw = fma(quad_lane<v>(cb), quad_lane<v>(wq), b.bw);
                const double gv = quad_lane<v>(g);
                b.bgx = fma(gv, dx, b.bgx);
                b.bgy = fma(gv, dy, b.bgy);
                b.bgz = fma(gv, dz, b.bgz);
                if (M == PCISPH) {
                    const double gsv = quad_lane<v>(gs);
                    b.sx2 = fma(gsv, dx, b.sx2);
                    b.sy2 = fma(gsv, dy, b.sy2);
                    b.sz2 = fma(gsv, dz, b.sz2);
                }
                if (wantAdh) {
                    const double sav = quad_lane<v>(sa);
                    b.ax = fma(sav, dx, b.ax);
                    b.ay = fma(sav, dy, b.ay);
                    b.az = fma(sav, dz, b.az);
                }
            });
        };
        int nb = 0;
        // (survivors as places in the stage or in the boundary table)
        static_for<9>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            const int d = bStaged ? bbase[r] - bfirst[r] : 0;
            for (int c0 = rs[r]; c0 < re[r]; c0 += 32) {
                const int nv = min(re[r] - c0, 32);
                uint32_t m = 0;
                auto half = [&](int k0) {
                    float4 y[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int t = c0 + u + k0 + 4 * k;
                        if (bStaged) y[k] = sb[t + d];
                        else y[k] = ld4(S.xb, (size_t)min(t, re[r] - 1));
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        m = __builtin_amdgcn_alignbit(m, test(xi.x - y[k].x, xi.y - y[k].y, xi.z - y[k].z, hh), 28);
                };
                half(0);
                if (nv > 16) half(16);
                else m <<= 16;
                const uint32_t f = joined(m, nv);
                keep(m, f, nb, (uint32_t)(c0 + d), bmine, kQuadBoundList);
                nb += __popc(f);
            }
        });
        if (!__any(nb > kQuadBoundList)) {
            for (int q0 = 0; q0 < nb; q0 += 4) {
                const int pos = q0 + u;
                const uint32_t t = bmine[min(pos, nb - 1)];
                float4 y;
                if (bStaged) y = sb[t];
                else y = ld4(S.xb, (size_t)t);
                bsums(pos < nb, y);
            }
        } else {
            static_for<9>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                for (int b0 = rs[r]; b0 < re[r]; b0 += 4) {
                    const int t = min(b0 + u, re[r] - 1);
                    const float4 y = ld4(S.xb, (size_t)t);
                    const float fx = xi.x - y.x, fy = xi.y - y.y, fz = xi.z - y.z;
                    const bool ok = (b0 + u < re[r]) & (fx * fx + fy * fy + fz * fz <= hh);
                    if (__any(ok)) bsums(ok, y);
                }
            });
        }
    }
    if (!fluid && u == 0) sbs[pl] = BoundSums{b.bw, b.bgx, b.bgy, b.bgz, b.sx2, b.sy2, b.sz2, b.ax, b.ay, b.az, nearBound ? 1 : 0};
    // the list is padded with the particle itself up to the group's longest
    // list rounded to 4
    const int own = min(cnt, maxN);
    int pad = min((own + 3) & ~3, maxN);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pad = max(pad, __shfl_xor(pad, o));
    if (lane == 0 && fluid) spad[w] = pad;
    __syncthreads();
    pad = max(max(spad[0], spad[1]), max(spad[2], spad[3]));
    double e = 0.0;
    if (M == PCISPH) {
        if (pad + ns > maxN) shellLost = true;   // the padding reached the shell
        shellLost = quad_bits(shellLost) != 0u;
    }
    if (fluid && valid) {
        for (int q = own + u; q < pad; q += 4) stg(L, (size_t)slot_of(q), (uint32_t)i);
        if (u == 0) {
            if (M == PCISPH) stg(S.nsh, (size_t)i, (uint16_t)(shellLost ? 0xFFFF : ns));
            if (pl == 0) stg(S.gcnt, (size_t)(i >> 6), (uint16_t)pad);
            const BoundSums& f = sbs[pl];
            b.bw = f.bw;
            b.bgx = f.gx;
            b.bgy = f.gy;
            b.bgz = f.gz;
            b.sx2 = f.sx;
            b.sy2 = f.sy;
            b.sz2 = f.sz;
            b.ax = f.ax;
            b.ay = f.ay;
            b.az = f.az;
            nearBound = f.near != 0;
            e = build_finish<M>(S, k, i, xi, vi, b, cnt, own, ngr, nearBound);
        }
    }
    if (M == DFSPH) {
        group_error(S, 0, g0, e);
        if (g0 == 0 && tid == 0) build_starts_divergence(S, fused);
    }
}

// ======================================================= non-pressure

// Akinci surface normals n_i = h sum_j (m/rho_j) gradW_ij
// (src/SurfaceTensionAkinci.h:46-61).  nrm.w carries rho_i - rho0 for pass 2.
template <int Q>
__global__ __launch_bounds__(kPartBlock<Q>) void k_normals(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                           int nchunks) {
    Chunk c;
    int i0, i;
    if (!part_at<Q>(C, nchunks, c, i0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    // a batch may hold scenes without surface tension, which have no normals
    if (i >= S.n || !(S.flags & F_ST)) return;
    const KCoefD k = S.kd;
    const float4 xi = ld4(S.x, i);
    const double xx = xi.x, xy = xi.y, xz = xi.z;
    const double m = S.mD, rho0 = S.rho0D;
    double nx = 0.0, ny = 0.0, nz = 0.0;
    sweep<Q>(S, i, [&](uint32_t j) { XV r; r.x = ld4(S.x, j); r.v.x = ldg(S.drho, j); return r; },
             [&](const XV& d) {
                 const Pair p = pair_of(xx, xy, xz, d.x, k);
                 return Terms<4>{{G_d(p, k) * div_n(m, rho0 + (double)d.v.x), p.dx, p.dy, p.dz}};
             },
             [&](const Terms<4>& t) {
                 nx = fma(t.v[0], t.v[1], nx);
                 ny = fma(t.v[0], t.v[2], ny);
                 nz = fma(t.v[0], t.v[3], nz);
             });
    if (Q > 1 && (threadIdx.x & 3) != 0) return;
    const double h = k.h;
    st4(S.nrm, i, make_float4((float)(nx * h), (float)(ny * h), (float)(nz * h), ldg(S.drho, i)));
}

// The end of a WCSPH or PCISPH step: time += dt (src/WCSPHSolver.cpp:77,
// src/PCISPHSolver.cpp:80), and which predicted-density path a PCISPH step
// took.
__device__ inline void advance_time(const DevScene& S) {
    Scalars* ss = S.ss;
    ss->time += ss->dt;
    if (S.method == PCISPH) {
        if (S.pciShell && ss->shellBad == 0u) ss->shellSteps += 1u;
        else ss->walkSteps += 1u;
    }
}
// Whether the step's last kernel (the WCSPH forces, the PCISPH integration)
// advances the time, one launch fewer per step: not when the cube clamp, the
// PCISPH boundary projection or an emitter runs after it (the emitters read
// the step's start time); k_time_advance does it then.
__device__ inline bool time_in_last_kernel(const DevScene& S) { return !(S.cubeOn || S.pbOn || S.nEmit > 0); }

// Non-pressure accelerations (and, for WCSPH, the pressure force and the
// explicit integration).
//   pressure  src/WCSPHSolver.cpp:152-186
//   XSPH      src/XSPHViscosity.h:45-67
//   standard viscosity   src/StandardViscosityForce.h:37-74:
//     a_i += nu/rho0 sum_j m (v_j - v_i)/rho_j lapl(r_ij)
//          + nu_b/rho0 sum_b rho0 V_b (-v_i)/rho_i lapl(r_ib),
//     lapl(r) = 45/(pi h^6) (h - r) (src/ViscoK.h:28-35)
//   artificial viscosity src/ArtificialViscosity.h:40-81:
//     a_i += sum_j k_ij nu (m/rho_j) (v_i - v_j).r_ij/(r^2 + 0.01 h^2) gradW_ij
//          + sum_b nu_b (rho0 V_b/rho_i) v_i.r_ib/(r^2 + 0.01 h^2) gradW_ib,
//     k_ij = 2 rho0/(rho_i + rho_j); the reference's factor 10 * 0.1 is 1
//   (boundary terms only when nu_b != 0, walked here over the boundary cells)
//   cohesion  src/SurfaceTensionAkinci.h:66-96
//   adhesion  src/AdhesionForce.h:38-61
//   integrate src/SPHSolver.cpp:154-167
// M = WCSPH reads neighbor positions from xk and velocities from aux (both
// written by k_build) because it updates x and v in place.  M = PCISPH also
// predicts v*, x* for the first pressure iteration (pacc = 0,
// src/PCISPHSolver.cpp:139-146).
// FL: the forces (Flags, F_ADH aside) every scene of the launch has, known at
// compile time, or -1.  The kernel is bound by its FP64 pair math, and by how
// many wavefronts hide its gathers: with every force compiled in it holds 166
// to 190 registers, 2 wavefronts a SIMD, with one of XSPH and cohesion 90 to
// 118, with both 124 to 146.  XSPH alone, WCSPH, 599,169 particles: 99.8 ->
// 78.4 us; XSPH and cohesion, DFSPH, 35,805 particles: 30.4 -> 15 us.
template <int M, int FL, int Q>
__global__ __launch_bounds__(kPartBlock<Q>) void k_forces(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                          int nchunks) {
    Chunk c;
    int i0, i;
    if (!part_at<Q>(C, nchunks, c, i0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    if ((M == WCSPH) && i0 == 0 && threadIdx.x == 0 && time_in_last_kernel(S)) advance_time(S);
    if (i >= S.n) return;
    const KCoefD k = S.kd;
    const double dt = S.ss->dt;
    const int fl = FL >= 0 ? FL : S.flags;
    const bool xs = (fl & F_XSPH) != 0, st = (fl & F_ST) != 0;
    const bool vstd = (fl & F_VSTD) != 0, vart = (fl & F_VART) != 0;
    const bool vel = xs || vstd || vart;
    const float4 xi = (M == WCSPH) ? ld4(S.xk, i) : ld4(S.x, i);
    const float4 vi = (M == WCSPH) ? ld4(S.aux, i) : ld4(S.v, i);
    const double xx = xi.x, xy = xi.y, xz = xi.z;
    const double vx0 = vi.x, vy0 = vi.y, vz0 = vi.z;
    const double m = S.mD, rho0 = S.rho0D;
    const double rhoi = rho0 + (double)ldg(S.drho, i);
    const float4 ni = st ? ld4(S.nrm, i) : make_float4(0.f, 0.f, 0.f, 0.f);
    const double pri = xi.w;
    double px = 0.0, py = 0.0, pz = 0.0;   // pressure part
    double vx = 0.0, vy = 0.0, vz = 0.0;   // XSPH part (before nu/dt)
    double sx = 0.0, sy = 0.0, sz = 0.0;   // surface tension part (before gamma)
    double wx = 0.0, wy = 0.0, wz = 0.0;   // standard / artificial viscosity part
    auto load = [&](uint32_t j) {
        NbF r;
        r.x = (M == WCSPH) ? ld4(S.xk, j) : ld4(S.x, j);
        if (vel) r.v = (M == WCSPH) ? ld4(S.aux, j) : ld4(S.v, j);
        // rho_j: XSPH under WCSPH takes m/rho_j from aux.w instead
        if ((vel && M != WCSPH) || vstd || vart) r.d = ldg(S.drho, j);
        if (st) r.n = ld4(S.nrm, j);
        return r;
    };
    auto pressure_of = [&](const Pair& p, const NbF& d) { return G_d(p, k) * m * (pri + (double)d.x.w); };
    auto xsph_of = [&](const Pair& p, const NbF& d) {
        const double mj = (M == WCSPH) ? (double)d.v.w : div_n(m, rho0 + (double)d.d);
        return mj * W_d(p.q, k);
    };
    // list members satisfy |r| <= h exactly (FP64), the reference's test at
    // src/SurfaceTensionAkinci.h:88
    auto kij_of = [&](const NbF& d) { return div_n(2.0 * rho0, rhoi + (rho0 + (double)d.n.w)); };
    auto cohesion_of = [&](const Pair& p, const NbF& d) {
        bool outer = 2.0 * p.rl > k.h;
        if (fabs(2.0 * p.rl - k.h) < 1e-9 * k.h) outer = 2.0 * exact_q(xi, d.x, S.hD).rl > S.hD;
        return -m * C_d(p.rl, outer, k) * p.inv;
    };
    if constexpr (Q == 1) {
        sweep4(S, i, load, [&](uint32_t, const NbF& d) {
            const Pair p = pair_of(xx, xy, xz, d.x, k);
            if (M == WCSPH) {
                const double g = pressure_of(p, d);
                px -= g * p.dx;
                py -= g * p.dy;
                pz -= g * p.dz;
            }
            if (xs) {
                const double w = xsph_of(p, d);
                vx += w * ((double)d.v.x - vx0);
                vy += w * ((double)d.v.y - vy0);
                vz += w * ((double)d.v.z - vz0);
            }
            if (vstd) {
                // m/rho_j lapl(r) (v_j - v_i); list members have r <= h
                const double w = (m / (rho0 + (double)d.d)) * (k.vl * (k.h - p.rl));
                wx += w * ((double)d.v.x - vx0);
                wy += w * ((double)d.v.y - vy0);
                wz += w * ((double)d.v.z - vz0);
            }
            if (vart) {
                const double rhoj = rho0 + (double)d.d;
                const double kij = 2.0 * rho0 / (rhoi + rhoj);
                const double dot = (vx0 - (double)d.v.x) * p.dx + (vy0 - (double)d.v.y) * p.dy + (vz0 - (double)d.v.z) * p.dz;
                const double f = kij * (m / rhoj) * dot / (p.rl * p.rl + 0.01 * k.h2) * G_d(p, k);
                wx += f * p.dx;
                wy += f * p.dy;
                wz += f * p.dz;
            }
            if (st && p.r2 > 0.0) {
                const double kij = kij_of(d);
                const double cs = cohesion_of(p, d);
                sx += kij * (cs * p.dx - ((double)ni.x - (double)d.n.x));
                sy += kij * (cs * p.dy - ((double)ni.y - (double)d.n.y));
                sz += kij * (cs * p.dz - ((double)ni.z - (double)d.n.z));
            }
        });
    } else {
        // (pressure g, d), (XSPH w, v_j - v_i), (cohesion K_ij and its vector)
        constexpr int kX = M == WCSPH ? 4 : 0, kS = kX + ((FL & F_XSPH) ? 4 : 0), kN = kS + ((FL & F_ST) ? 4 : 0);
        if constexpr (kN > 0)
            sweep<Q>(S, i, load,
                     [&](const NbF& d) {
                         const Pair p = pair_of(xx, xy, xz, d.x, k);
                         Terms<kN> t;
                         if constexpr (M == WCSPH) {
                             t.v[0] = pressure_of(p, d);
                             t.v[1] = p.dx;
                             t.v[2] = p.dy;
                             t.v[3] = p.dz;
                         }
                         if constexpr ((FL & F_XSPH) != 0) {
                             t.v[kX] = xsph_of(p, d);
                             t.v[kX + 1] = (double)d.v.x - vx0;
                             t.v[kX + 2] = (double)d.v.y - vy0;
                             t.v[kX + 3] = (double)d.v.z - vz0;
                         }
                         if constexpr ((FL & F_ST) != 0) {
                             const bool on = p.r2 > 0.0;
                             const double cs = cohesion_of(p, d);
                             t.v[kS] = on ? kij_of(d) : 0.0;
                             t.v[kS + 1] = on ? fma(cs, p.dx, -((double)ni.x - (double)d.n.x)) : 0.0;
                             t.v[kS + 2] = on ? fma(cs, p.dy, -((double)ni.y - (double)d.n.y)) : 0.0;
                             t.v[kS + 3] = on ? fma(cs, p.dz, -((double)ni.z - (double)d.n.z)) : 0.0;
                         }
                         return t;
                     },
                     [&](const Terms<kN>& t) {
                         if constexpr (M == WCSPH) {
                             px = fma(-t.v[0], t.v[1], px);
                             py = fma(-t.v[0], t.v[2], py);
                             pz = fma(-t.v[0], t.v[3], pz);
                         }
                         if constexpr ((FL & F_XSPH) != 0) {
                             vx = fma(t.v[kX], t.v[kX + 1], vx);
                             vy = fma(t.v[kX], t.v[kX + 2], vy);
                             vz = fma(t.v[kX], t.v[kX + 3], vz);
                         }
                         if constexpr ((FL & F_ST) != 0) {
                             sx = fma(t.v[kS], t.v[kS + 1], sx);
                             sy = fma(t.v[kS], t.v[kS + 2], sy);
                             sz = fma(t.v[kS], t.v[kS + 3], sz);
                         }
                     });
        if ((threadIdx.x & 3) != 0) return;
    }
    double ax = 0.0, ay = 0.0, az = 0.0;
    if (M == WCSPH) {
        const float4 gb = S.gb[i];
        ax = px - pri * (double)gb.x;
        ay = py - pri * (double)gb.y;
        az = pz - pri * (double)gb.z;
        if (S.pbOn) {
            // the boundary particles' own pressure term m_b p_b / rho_b^2
            // gradW of the PCISPH method (src/WCSPHSolver.cpp:160-172)
            walk27(S.bCellStart, ldg(S.cell, (size_t)i), S.nx, S.nx * S.ny, [&](int b) {
                const float4 y = ld4(S.xb, b);
                const Pair p = pair_of(xx, xy, xz, y, k);
                const double g = S.rho0D * (double)y.w * (double)S.bpr[b] * G_d(p, k);
                ax -= g * p.dx;
                ay -= g * p.dy;
                az -= g * p.dz;
            });
        }
    }
    if (xs) {
        const double f = (double)S.nu / dt;
        ax += f * vx;
        ay += f * vy;
        az += f * vz;
        if (S.nub != 0.0f) {
            const double fb = (double)S.nub * ((double)S.gb[i].w / rhoi) / dt;
            ax -= fb * vx0;
            ay -= fb * vy0;
            az -= fb * vz0;
        }
    }
    if (vstd || vart) {
        const double nu = S.nu, nub = S.nub;
        double bx = 0.0, by = 0.0, bz = 0.0;
        if (nub != 0.0) {
            walk27(S.bCellStart, ldg(S.cell, (size_t)i), S.nx, S.nx * S.ny, [&](int b) {
                const float4 y = ld4(S.xb, b);
                const Pair p = pair_of(xx, xy, xz, y, k);
                if (!(p.q <= 1.0)) return;
                const double cb = rho0 * (double)y.w;
                if (vstd) {
                    const double w = cb * (k.vl * (k.h - p.rl)) / rhoi;
                    bx -= w * vx0;
                    by -= w * vy0;
                    bz -= w * vz0;
                } else {
                    const double dot = vx0 * p.dx + vy0 * p.dy + vz0 * p.dz;
                    const double f = (cb / rhoi) * dot / (p.rl * p.rl + 0.01 * k.h2) * G_d(p, k);
                    bx += f * p.dx;
                    by += f * p.dy;
                    bz += f * p.dz;
                }
            });
        }
        const double fv = vstd ? nu / rho0 : nu, fb = vstd ? nub / rho0 : nub;
        ax += fv * wx + fb * bx;
        ay += fv * wy + fb * by;
        az += fv * wz + fb * bz;
    }
    if (st) {
        ax += (double)S.stCoef * sx;
        ay += (double)S.stCoef * sy;
        az += (double)S.stCoef * sz;
    }
    if (S.flags & F_ADH) {
        const float4 ad = S.adh[i];
        ax -= (double)S.adhBeta * (double)ad.x;
        ay -= (double)S.adhBeta * (double)ad.y;
        az -= (double)S.adhBeta * (double)ad.z;
    }
    S.a[i] = make_float4((float)ax, (float)ay, (float)az, 0.f);
    if (M == WCSPH) {
        const double nvx = vx0 + (ax + (double)S.gx) * dt;
        const double nvy = vy0 + (ay + (double)S.gy) * dt;
        const double nvz = vz0 + (az + (double)S.gz) * dt;
        S.v[i] = make_float4((float)nvx, (float)nvy, (float)nvz, 0.f);
        S.x[i] = make_float4((float)(xx + nvx * dt), (float)(xy + nvy * dt), (float)(xz + nvz * dt), 0.f);
    } else if (M == PCISPH) {
        const double wx = vx0 + (ax + (double)S.gx) * dt;
        const double wy = vy0 + (ay + (double)S.gy) * dt;
        const double wz = vz0 + (az + (double)S.gz) * dt;
        S.xs[i] = make_float4((float)(wx * dt), (float)(wy * dt), (float)(wz * dt), 0.f);
        if (S.pbOn) S.pv[i] = make_float4((float)wx, (float)wy, (float)wz, 0.f);
        shell_guard(S, wx * dt, wy * dt, wz * dt);
    }
}

// ================================================================ DFSPH

// CFL time step (src/DFSPHSolver.cpp:827-870): maxVel = max(0.1, max_i
// sqrt(|v_i + (a_i + g) dt|)); dt' = cfl if cfl < dt, else 0.99 dt after
// more than 3 density iterations, else 1.001 dt; clamped to [min, max].
__global__ __launch_bounds__(kBlock) void k_dt(const DevScene* __restrict__ T, const Chunk* __restrict__ C) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    const gptr<const Scalars> ss = G((const Scalars*)S.ss);
    __shared__ double sh[kWaves];
    const int i = c.begin + threadIdx.x;
    const double dt = ss->dt;
    double val = 0.0;
    if (i < S.n) {
        const float4 v = ld4(S.v, (size_t)i);
        double ax = S.gx, ay = S.gy, az = S.gz;
        if (S.flags & F_FORCES) {
            const float4 a = ld4(S.a, (size_t)i);
            ax = (double)a.x + ax;
            ay = (double)a.y + ay;
            az = (double)a.z + az;
        }
        const double cx = v.x + ax * dt, cy = v.y + ay * dt, cz = v.z + az * dt;
        val = sqrt(sqrt(cx * cx + cy * cy + cz * cz));
    }
    const double bm = block_max(val, sh);
    if (threadIdx.x == 0) G(S.partial)[c.begin / kBlock] = bm;
}

// The density solve (predict, warm start, density iterations) keeps the
// velocity of the step's start, v0, unchanged in v and accumulates the
// step's change u = v - v0 in x.w and vyz, the slots its error sweeps
// gather; the position update forms v = v0 + u.  The predicted density is
// rho + dt (D0 + U): D0, the sum over v0, is formed once per step in FP64,
// and U, the sum over u, in every iteration.  Velocities rounded to FP32
// after every sweep would put their rounding (~1e-7 of |v|) into rho*, which
// kappa = (rho* - rho0) alpha / (dt^2 rho) amplifies; u is the size of the
// step's corrections, so its FP32 rounding is far below that.
__device__ inline void store_u(const DevScene& S, int i, double ux, double uy, double uz) {
    ((gptr<float>)S.x)[4 * (size_t)i + 3] = (float)ux;
    ((gptr<v2f>)S.vyz)[i] = v2f{(float)uy, (float)uz};
}

// predictVelocities (src/DFSPHSolver.cpp:191-214) fused with the first loop
// of densityWarmStart (:602-613): k_i <- min(k_i/rho_i, 1e-9)/dt^2, staged
// in xk.w for the warm-start sweep.  The predicted velocity is kept as
// u = (a + g) dt beside v0 (and, with the PCISPH boundary method, the change
// of its velocity correction).
// `fused`: the time step from k_dt's partials is formed here, by every block.
__global__ __launch_bounds__(kBlock) void k_df_predict(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                       int fused) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    __shared__ double sh[kWaves];
    const int i = c.begin + threadIdx.x;
    double dt = G(S.ss)->dt;
    if (fused && S.nChunks <= kFusedLoopChunks) {
        const NextDt d = next_dt(S, dt, G(S.ss)->it, scene_partial_max(S.partial, S.nChunks, sh));
        dt = d.dt;
        if (c.begin == 0 && threadIdx.x == 0) {
            const gptr<Scalars> ss = G(S.ss);
            ss->dtNew = d.dt;
            ss->maxVel = d.maxVel;
            ss->cflTs = d.cflTs;
            ss->steps += 1u;
        }
    }
    if (i >= S.n) return;
    const float4 v = ld4(S.v, (size_t)i);
    double ax = S.gx, ay = S.gy, az = S.gz;
    if (S.flags & F_FORCES) {
        const float4 a = ld4(S.a, (size_t)i);
        ax = (double)a.x + ax;
        ay = (double)a.y + ay;
        az = (double)a.z + az;
    }
    double ux = ax * dt, uy = ay * dt, uz = az * dt;
    if (S.pbOn) {
        // correctVelocities with the normals of the last step's projection
        // (src/DFSPHSolver.cpp:51-58)
        const float4 n = ld4(S.pbn, (size_t)i);
        double wx = (double)v.x + ux, wy = (double)v.y + uy, wz = (double)v.z + uz;
        if (pb_velocity(S, n.x, n.y, n.z, wx, wy, wz)) {
            ux = wx - (double)v.x;
            uy = wy - (double)v.y;
            uz = wz - (double)v.z;
        }
    }
    const double rho = S.rho0D + (double)ldg(S.drho, (size_t)i);
    const double kw = -fmax(-(double)ldg(S.k, (size_t)i) / rho, -1.0e-9) / (dt * dt);
    const float4 x = ld4(S.x, (size_t)i);
    st4(S.xk, (size_t)i, make_float4(x.x, x.y, x.z, (float)kw));
    store_u(S, i, ux, uy, uz);
}

// Velocity correction sweep shared by the warm start (src/DFSPHSolver.cpp:
// 622-677), the density solve (:335-395) and the divergence solve
// (:520-579):  v_i -= dt (sum_j m (s_i + s_j) gradW_ij [|s_i+s_j| > eps]
//                         + c s_i gb_i [|c s_i| > eps])
// with s = xk.w, c = 2 for the warm start, 1 otherwise.  MODE 0 = warm start
// (then k_i = 0, :679-689), 1 = density (k_i += (rho*_i - rho0) alpha_i,
// :349), 2 = divergence (kv_i += divErr_i alpha_i, :534).
// `fused`: the sweep decides whether its iteration runs (loop_over); the warm
// start makes the new time step dt and starts the density loop.  FP64 math, 36
// instructions a neighbor, bounds it (1M particles 50 us at 1.9-2.1 GHz); one
// zeroing for both conditions on a term, of its size and of the distance, is 2
// fewer (a step of 1M 918 -> 914 us, a batch of 825k 1222 -> 1215, 4,096 94 -> 92).
template <int MODE, int Q>
__global__ __launch_bounds__(kPartBlock<Q>) void k_df_vel(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                          int nchunks, int iter, int fused) {
    Chunk c;
    int i0, i;
    if (!part_at<Q>(C, nchunks, c, i0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    Scalars* ss = S.ss;
    if (MODE == 1 && ended_before(ss->done, iter + 1)) return;
    if (MODE == 2 && ended_before(ss->doneV, iter + 1)) return;
    double dt = ss->dt;
    if (fused) {
        if (MODE == 0) {
            // (a large scene's finalize kernel has written dt itself)
            if (S.nChunks <= kFusedLoopChunks) dt = ss->dtNew;
            if (i0 == 0 && threadIdx.x == 0) {
                if (S.nChunks <= kFusedLoopChunks) ss->dt = dt;
                ss->it = 0;
                ss->done = loop_goes_on<LOOP_DENS>(S, ss, 0, 0.0) ? 0 : 1;
            }
        } else {
            __shared__ double sh[kPartBlock<Q> / 64];
            if (loop_over<MODE == 1 ? LOOP_DENS : LOOP_DIV, kPartBlock<Q>>(S, ss, i0 == 0, iter + 1, sh)) return;
        }
    }
    if (i >= S.n) return;
    const KCoefD k = S.kd;
    const double eps = 1.0e-5;
    const float4 xi = ld4(S.xk, i);
    const double xx = xi.x, xy = xi.y, xz = xi.z;
    const double si = xi.w;
    const double m = S.mD;
    double sx = 0.0, sy = 0.0, sz = 0.0;
    sweep<Q>(S, i, [&](uint32_t j) { return ld4o(S.xk, j); },
             [&](const float4& xj) {
                 const double ks = si + (double)xj.w;
                 const PairG p = pairg_of(xx, xy, xz, xj, k);
                 return Terms<4>{{sel((fabs(ks) > eps) & p.apart, m * ks * p.g, 0.0), p.dx, p.dy, p.dz}};
             },
             [&](const Terms<4>& t) {
                 sx = fma(t.v[0], t.v[1], sx);
                 sy = fma(t.v[0], t.v[2], sy);
                 sz = fma(t.v[0], t.v[3], sz);
             });
    if (Q > 1 && (threadIdx.x & 3) != 0) return;
    // every load of the epilogue is issued before its first store: a wait
    // for a load also waits for the stores issued before it
    const float4 gb = S.gb[i];
    float kold = 0.f, kerr = 0.f, kal = 0.f;
    if (MODE == 1) { kold = S.k[i]; kerr = S.drhoS[i]; kal = S.alpha[i]; }
    if (MODE == 2) { kold = S.kv[i]; kerr = S.divErr[i]; kal = S.alpha[i]; }
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    float uxf = 0.f;
    float2 uyz = make_float2(0.f, 0.f);
    if (MODE <= 1) {
        uxf = ((gptr<const float>)S.x)[4 * (size_t)i + 3];
        uyz = ld2o(S.vyz, (uint32_t)i);
    } else {
        v = S.v[i];
    }
    const double cb = (MODE == 0) ? 2.0 * si : si;
    if (fabs(cb) > eps) {
        sx += cb * (double)gb.x;
        sy += cb * (double)gb.y;
        sz += cb * (double)gb.z;
    }
    if (MODE <= 1) {
        // the density solve: the change u (x.w, vyz; no kernel gathers x
        // during this sweep) takes the correction, v keeps v0
        store_u(S, i, (double)uxf - dt * sx, (double)uyz.x - dt * sy, (double)uyz.y - dt * sz);
    } else {
        v.x = (float)((double)v.x - dt * sx);
        v.y = (float)((double)v.y - dt * sy);
        v.z = (float)((double)v.z - dt * sz);
        S.v[i] = v;
        // copies for the error sweep's gathers: v_x into the unused x.w (no
        // kernel gathers x during this sweep), (v_y, v_z) into vyz
        ((gptr<float>)S.x)[4 * (size_t)i + 3] = v.x;
        ((gptr<v2f>)S.vyz)[i] = v2f{v.y, v.z};
    }
    if (MODE == 0) S.k[i] = 0.0f;
    if (MODE == 1) S.k[i] = (float)((double)kold + (double)kerr * (double)kal);
    if (MODE == 2) S.kv[i] = (float)((double)kold + (double)kerr * (double)kal);
}

// Density or divergence error sweep with the scene reduction and the loop
// test.  MODE 0/1: predictDensities (src/DFSPHSolver.cpp:238-309),
//   rho*_i = max(rho_i + dt (sum_j m (v_i - v_j).gradW_ij + v_i.gb_i), rho0),
//   kappa_i = (rho*_i - rho0) alpha_i / (dt^2 rho_i)   (:346)
// MODE 3: computeDivergenceError (:408-492),
//   e_i = sum_j m (v_i - v_j).gradW_ij + v_i.gb_i, 0 below 20 nonzero-gradient
//   neighbors, else max(e_i, 0);  kappa_v_i = e_i alpha_i / (dt rho_i) (:531)
// MODE 0 is the call before the density loop, whose error starts at 0 (:326;
// before the divergence loop, :511, the list build forms the error); 1 and 3
// are the calls at the end of an iteration.  Loop test
// (:327, :512; the divergence loop is bounded by maxIterations):
//   continue while (err > eta (eta_V/dt) or it < minIt) and it < maxIt.
template <int MODE, int Q>
__global__ __launch_bounds__(kPartBlock<Q>) void k_df_err(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                          int nchunks, int fused) {
    Chunk c;
    int i0, i;
    if (!part_at<Q>(C, nchunks, c, i0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    Scalars* ss = S.ss;
    constexpr bool DENS = (MODE <= 1);
    if (MODE == 1 && ss->done) return;
    if (MODE == 3 && ss->doneV) return;
    // `fused`: no finalize kernel counts the iteration
    if (fused && MODE != 0 && i0 == 0 && threadIdx.x == 0) {
        if (DENS) ss->it += 1;
        else ss->itV += 1;
    }
    const KCoefD k = S.kd;
    const double dt = ss->dt;
    double e = 0.0;
    if (i < S.n) {
        const float4 xi = ld4(S.x, i);
        const double xx = xi.x, xy = xi.y, xz = xi.z;
        const float4 gb = S.gb[i];
        // loaded before any store (a wait for a load also waits for the
        // stores issued before it)
        const float drhof = S.drho[i], alf = S.alpha[i];
        const int ngr = DENS ? 20 : (int)S.ngrad[i];
        // sum_j g_ij (u_i - u_j).(x_i - x_j), u_j in x.w and vyz
        auto change = [&](double ux, double uy, double uz, double& sum) {
            sweep<Q>(S, i, [&](uint32_t j) { XVP r; r.xv = ld4o(S.x, j); r.yz = ld2o(S.vyz, j); return r; },
                     [&](const XVP& d) {
                         const PairG p = pairg_of(xx, xy, xz, d.xv, k);
                         return Terms<2>{{sel(p.apart, p.g, 0.0), (ux - (double)d.xv.w) * p.dx + (uy - (double)d.yz.x) * p.dy + (uz - (double)d.yz.y) * p.dz}};
                     },
                     [&](const Terms<2>& t) { sum = fma(t.v[0], t.v[1], sum); });
        };
        double dc;
        if (DENS) {
            // the density solve: x.w and vyz hold u, v holds v0 (see store_u)
            const float2 yz = ld2o(S.vyz, (uint32_t)i);
            const double ux = xi.w, uy = yz.x, uz = yz.y;
            double su = 0.0;
            if (MODE == 0 && !ss->d0Valid) {
                // the constant part D0 over v0, once per step (unless the
                // previous divergence sweep left it: see d0Valid)
                const float4 vi = ld4(S.v, i);
                const double wx = vi.x, wy = vi.y, wz = vi.z;
                double s0 = 0.0;
                sweep<Q>(S, i,
                         [&](uint32_t j) { XVU r; r.x = ld4o(S.x, j); r.v = ld4o(S.v, j); r.yz = ld2o(S.vyz, j); return r; },
                         [&](const XVU& d) {
                             const PairG p = pairg_of(xx, xy, xz, d.x, k);
                             return Terms<3>{{sel(p.apart, p.g, 0.0),
                                              (wx - (double)d.v.x) * p.dx + (wy - (double)d.v.y) * p.dy + (wz - (double)d.v.z) * p.dz,
                                              (ux - (double)d.x.w) * p.dx + (uy - (double)d.yz.x) * p.dy + (uz - (double)d.yz.y) * p.dz}};
                         },
                         [&](const Terms<3>& t) {
                             s0 = fma(t.v[0], t.v[1], s0);
                             su = fma(t.v[0], t.v[2], su);
                         });
                const double d0 = S.mD * s0 + (wx * (double)gb.x + wy * (double)gb.y + wz * (double)gb.z);
                if (Q == 1 || (threadIdx.x & 3) == 0) ((gptr<double>)S.d0)[i] = d0;
                dc = d0;
                // (d0Valid stays 0 until the next divergence sweep: other
                // blocks of this launch test it)
            } else {
                change(ux, uy, uz, su);
                dc = ((gptr<const double>)S.d0)[i];
            }
            dc += S.mD * su + (ux * (double)gb.x + uy * (double)gb.y + uz * (double)gb.z);
        } else {
            const float4 vi = ld4(S.v, i);
            const double ux = vi.x, uy = vi.y, uz = vi.z;
            dc = 0.0;
            // the velocity sweep before this one wrote x.w and vyz
            change(ux, uy, uz, dc);
            dc = S.mD * dc + (ux * (double)gb.x + uy * (double)gb.y + uz * (double)gb.z);
            // the divergence of the current velocities: the next step's D0
            if (Q == 1 || (threadIdx.x & 3) == 0) ((gptr<double>)S.d0)[i] = dc;
        }
        if (Q == 1 || (threadIdx.x & 3) == 0) {
            const double drho = (double)drhof;
            const double rho = S.rho0D + drho;
            const double al = alf;
            double s;
            if (DENS) {
                const double drs = fmax(drho + dc * dt, 0.0);
                S.drhoS[i] = (float)drs;
                s = drs * al / (dt * dt * rho);
                e = drs / S.rho0D;
            } else {
                const double de = (ngr < 20) ? 0.0 : fmax(dc, 0.0);
                S.divErr[i] = (float)de;
                s = de * al / (dt * rho);
                e = de / S.rho0D;
            }
            S.xk[i] = make_float4(xi.x, xi.y, xi.z, (float)s);
        }
    }
    // `fused`: the error before the loop, which only the log has, waits in
    // the sort's scratch for the cell scan to add it up
    const bool log = fused && MODE == 0;
    if constexpr (Q == 1) {
        __shared__ double sh[kWaves];
        const double bs = block_sum(e, sh);
        if (threadIdx.x == 0) (log ? group_partial(S, 0) : S.partial)[i0 / kBlock] = bs;
    } else {
        group_error(S, log ? 0 : 1, i0, e);
    }
}

// updatePositions (src/DFSPHSolver.cpp:216-236) fused with the cell key and
// histogram of the grid rebuild.
// Also clears the loop counters (scenes iterating, largest count) for the
// divergence solve, which the list build's finalize starts counting.
// `ahead`: the host has launched the density iterations of a lone scene
// without asking; if the loop has not ended, nothing from here on runs (the
// cell scan behind it tells the later launches).
__global__ __launch_bounds__(kBlock) void k_df_positions(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                         int* active, int ahead) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    if (ahead && !ended_before(S.ss->done, kLoopLast)) {
        __shared__ double sh[kWaves];
        if (!loop_over<LOOP_DENS>(S, S.ss, c.begin == 0, kLoopLast, sh)) return;
    }
    if (blockIdx.x == 0 && threadIdx.x < 2) active[threadIdx.x] = 0;
    // the lists about to be built start without an overflow
    if (c.begin == 0 && threadIdx.x == 0) G(S.ss)->listOver = 0u;
    const int i = c.begin + threadIdx.x;
    int cl = -1;
    if (i < S.n) {
        const double dt = G(S.ss)->dt;
        float4 x = ld4(S.x, (size_t)i);
        // the density solve's velocity: v0 + u (see store_u)
        const float4 v0 = ld4(S.v, (size_t)i);
        const float2 uyz = ld2o(S.vyz, (uint32_t)i);
        const float4 v = make_float4((float)((double)v0.x + (double)x.w), (float)((double)v0.y + (double)uyz.x),
                                     (float)((double)v0.z + (double)uyz.y), 0.f);
        st4(S.v, (size_t)i, v);
        x.x = (float)((double)x.x + (double)v.x * dt);
        x.y = (float)((double)x.y + (double)v.y * dt);
        x.z = (float)((double)x.z + (double)v.z * dt);
        st4(S.x, (size_t)i, x);
        if (!S.pbOn) {
            cl = cell_of(S, x);
            G(S.cellU)[i] = cl;
        }
    }
    // with the PCISPH boundary method the projection moves the particle
    // first, then counts its cell (a scene-uniform branch)
    if (!S.pbOn) (void)wave_count_add(S.cellCount, cl);
}

// =============================================================== PCISPH

// Predicted densities at x* with the candidate cells of x
// (src/PCISPHSolver.cpp:164-212; every candidate of the 27 cells, self
// included), then updatePressure (:249-295): p_i += delta max(0, rho_i -
// rho0); the scene's max relative error decides the loop (:365), counting
// this iteration as done (its pressure acceleration always follows).
// The nine rows of a particle's boundary (or fluid) candidates.
struct Rows {
    int s[9], e[9];
};
__device__ inline Rows rows_of(const int* start, int c, int nx, int nxny) {
    Rows o;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const int off = (r % 3 - 1) * nx + (r / 3 - 1) * nxny;
        o.s[r] = ldg(start, (size_t)(c - 1 + off));
        o.e[r] = ldg(start, (size_t)(c + 2 + off));
    }
    return o;
}
// x* = x + d with d = v* dt held separately: x*_i - x*_j = (x_i - x_j) +
// (d_i - d_j) keeps FP64 accuracy from FP32 storage.
struct Predicted {
    double px, py, pz, ex, ey, ez;
};
// W at the predicted distance to a particle at y + d, zero past h.
__device__ inline double predicted_w(const Predicted& a, const float4& y, const float4& d, const KCoefD& k) {
    const double dx = (a.px - (double)y.x) + (a.ex - (double)d.x);
    const double dy = (a.py - (double)y.y) + (a.ey - (double)d.y);
    const double dz = (a.pz - (double)y.z) + (a.ez - (double)d.z);
    const double r2 = dx * dx + dy * dy + dz * dz;
    return r2 <= k.hhi2 ? W_d(sqrt_n(r2) * k.invh, k) : 0.0;
}
// The same to a boundary particle.
__device__ inline double predicted_wb(const Predicted& a, const float4& y, const KCoefD& k) {
    const double dx = (a.px - (double)y.x) + a.ex, dy = (a.py - (double)y.y) + a.ey, dz = (a.pz - (double)y.z) + a.ez;
    const double r2 = dx * dx + dy * dy + dz * dz;
    return r2 <= k.hhi2 ? W_d(sqrt_n(r2) * k.invh, k) : 0.0;
}
// What the sums give: the density, p_i and p_i / rho_i^2; returns the error.
__device__ inline double pci_pressure(const DevScene& S, int i, const float4& xi, double ws, double bw) {
    const double rho0 = S.rho0D;
    const double drho = (S.mD * ws + rho0 * bw) - rho0;
    const double rho = rho0 + drho;
    S.drho[i] = (float)drho;
    const double err = fmax(0.0, drho);
    const double pr = (double)S.p[i] + S.pciDeltaD * err;
    S.p[i] = (float)pr;
    S.xk[i] = make_float4(xi.x, xi.y, xi.z, (float)(pr / (rho * rho)));
    return err / rho0;
}

// A group's largest squared displacement, kept over the step's iterations (one
// lane of each wavefront of the group stores it).
__device__ inline void store_displacement(const DevScene& S, int group, double d2, int iter) {
    if ((threadIdx.x & 63) != 0) return;
    float* const p = pci_displacements(S) + group;
    *p = iter == 0 ? (float)d2 : fmaxf(*p, (float)d2);
}

// Every candidate of the 27 cells that can come within h at x* is the
// particle itself, a list member (|x_i - x_j| <= h) or a shell member (<= h +
// skin): the walk's terms in another order.  Shell member s is in slot maxN -
// 1 - s.  ~60 FP64 instructions a term (a square root among them) bound it in
// a large scene; the next entries are requested before the current ones' data
// is used, and particles whose cells hold no boundary skip its 9 rows.
// `fused`: the sweep decides whether its iteration runs (loop_over).
__global__ __launch_bounds__(kBlock) void k_pci_density(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                        int iter, int fused) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    Scalars* ss = S.ss;
    if (ended_before(ss->done, iter + 1)) return;
    __shared__ double sh[kWaves];
    if (fused && loop_over<LOOP_PCI>(S, ss, c.begin == 0, iter + 1, sh)) return;
    double* const part = fused ? pci_partial(S, ss->it) : S.partial;
    const int i = c.begin + threadIdx.x;
    const KCoefD k = S.kd;
    const bool useShell = S.pciShell && ss->shellBad == 0u;
    double e = 0.0;
    double dd = 0.0;   // squared predicted displacement, for the next step's shell width
    if (i < S.n) {
        const float4 xi = ld4(S.x, (size_t)i);
        const float4 di = ld4(S.xs, (size_t)i);
        const int ci = ldg(S.cell, (size_t)i);
        const float nearBound = ldg(&S.gbs[i].w, 0);
        const int nx = S.nx, nxny = S.nx * S.ny;
        dd = (double)(di.x * di.x + di.y * di.y + di.z * di.z);
        const Predicted a{xi.x, xi.y, xi.z, di.x, di.y, di.z};
        double ws = 0.0;
        auto xv = [&](uint32_t j) { XV r; r.x = ld4o(S.x, j); r.v = ld4o(S.xs, j); return r; };
        const int nsi = useShell ? (int)ldg(S.nsh, (size_t)i) : 0xFFFF;
        if (nsi != 0xFFFF) {
            ws = W_d(0.0, k);
            const uint32_t* L = list_of(S, i);
            // `count` entries in list order, from the first slot up or the
            // last one down
            auto run = [&](int count, bool down) {
                const int last = (S.maxNbr >> 2) - 1;
                if (count == 0) return;
                v4u bn = ld_block(L, down ? last : 0);
                for (int q0 = 0; q0 < count; q0 += 4) {
                    const uint32_t j0 = down ? bn.w : bn.x;
                    const uint32_t jj[4] = {j0, q0 + 1 < count ? (down ? bn.z : bn.y) : j0,
                                            q0 + 2 < count ? (down ? bn.y : bn.z) : j0,
                                            q0 + 3 < count ? (down ? bn.x : bn.w) : j0};
                    XV d[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) d[u] = xv(jj[u]);
                    const int nb = (q0 + 4 < count ? q0 + 4 : q0) >> 2;
                    bn = ld_block(L, down ? last - nb : nb);
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (q0 + u < count) ws += predicted_w(a, d[u].x, d[u].v, k);
                }
            };
            run((int)ldg(S.nnb, (size_t)i), false);
            run(nsi, true);
        } else {
            walk27x4(S.cellStart, ci, nx, nxny, [&](int j) { return xv((uint32_t)j); },
                     [&](int, const XV& q) { ws += predicted_w(a, q.x, q.v, k); });
        }
        double bw = 0.0;
        if (nearBound != 0.f)
            walk27x4(S.bCellStart, ci, nx, nxny, [&](int b) { return ld4(S.xb, b); },
                     [&](int, const float4& y) { bw += (double)y.w * predicted_wb(a, y, k); });
        e = pci_pressure(S, i, xi, ws, bw);
    }
    const double bm = block_max(e, sh);
    if (threadIdx.x == 0) part[c.begin / kBlock] = bm;
    if (S.pciShell) store_displacement(S, i >> 6, wave_max(dd), iter);
}

// The same with 4 lanes a particle, a block per list group, for small
// launches (see k_build_quad): a lane takes every 4th entry and the terms are
// added in list order.  PCISPH, 4,845 particles: 28 -> 13 us a launch, the step
// 204 -> 144; then with a conservative FP32 test before the FP64 terms of the
// boundary's candidates, most of which lie beyond h, and in the smallest
// launches the boundary in 4 more wavefronts, the step 122 -> 110.
template <int V>
__device__ inline double quad_sum(double s, double t) {
    s += quad_lane<V>(t);
    if constexpr (V < 3) return quad_sum<V + 1>(s, t);
    else return s;
}
template <bool SIDE>
__global__ __launch_bounds__(SIDE ? 512 : 256) void k_pci_density_quad(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                          int nchunks, int iter, int fused) {
    Chunk c;
    int g0, i;
    if (!part_at<4>(C, nchunks, c, g0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    Scalars* ss = S.ss;
    if (ended_before(ss->done, iter + 1)) return;
    constexpr int kBT = SIDE ? 512 : 256;
    __shared__ double sh[kBT / 64], sbw[kGroup];
    const int tid = threadIdx.x, lane = tid & 63, u = lane & 3;
    // SIDE: wavefronts 0-3 work on the fluid, 4-7 on the boundary
    const bool fluid = !SIDE || tid < 256, bound = !SIDE || tid >= 256;
    const int pl = (tid & 255) >> 2;
    i = g0 + pl;
    if (fused && loop_over<LOOP_PCI, kBT>(S, ss, g0 == 0, iter + 1, sh)) return;
    double* const part = group_partial(S, fused ? ss->it & 1 : 0);
    if (g0 >= S.n) {
        // past the active particles, of which a scene with emitters may have
        // none: there is no particle to read
        if (tid == 0) {
            part[g0 >> 6] = 0.0;
            if (S.pciShell) store_displacement(S, g0 >> 6, 0.0, iter);
        }
        return;
    }
    const int il = min(i, S.n - 1);
    const KCoefD k = S.kd;
    const float hh = S.kc.hhi2 * (1.0f + 1e-5f);   // conservative FP32 test
    const bool useShell = S.pciShell && ss->shellBad == 0u;
    double e = 0.0, dd = 0.0, ws = 0.0;
    const float4 xi = ld4(S.x, (size_t)il);
    if (i < S.n) {
        const float4 di = ld4(S.xs, (size_t)il);
        const int ci = ldg(S.cell, (size_t)il);
        const int nx = S.nx, nxny = S.nx * S.ny;
        dd = (double)(di.x * di.x + di.y * di.y + di.z * di.z);
        const Predicted a{xi.x, xi.y, xi.z, di.x, di.y, di.z};
        const int nsi = useShell && fluid ? (int)ldg(S.nsh, (size_t)i) : 0xFFFF;
        if (bound) {
            const Rows br = rows_of(S.bCellStart, ci, nx, nxny);
            double bw = 0.0;
            static_for<9>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                for (int b0 = br.s[r]; b0 < br.e[r]; b0 += 8) {
                    float4 y[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) y[h] = ld4(S.xb, (size_t)min(b0 + 4 * h + u, br.e[r] - 1));
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const float fx = (xi.x - y[h].x) + di.x, fy = (xi.y - y[h].y) + di.y, fz = (xi.z - y[h].z) + di.z;
                        const bool ok = (b0 + 4 * h + u < br.e[r]) & (fx * fx + fy * fy + fz * fz <= hh);
                        if (!__any(ok)) continue;
                        const double w = predicted_wb(a, y[h], k), vb = ok ? y[h].w : 0.f;   // (w is finite)
                        static_for<4>([&](auto vc) {
                            constexpr int v = decltype(vc)::value;
                            bw = fma(quad_lane<v>(vb), quad_lane<v>(w), bw);
                        });
                    }
                }
            });
            if (u == 0) sbw[pl] = bw;
        }
        if (fluid && nsi != 0xFFFF) {
            ws = W_d(0.0, k);
            const uint32_t* const L = list_of(S, i);
            const int maxN = S.maxNbr;
            // two entries a lane at a time
            auto run = [&](int count, bool down) {
                auto at = [&](int q) {
                    const int t = q < count ? q : (q & 3) < count ? (q & 3) : 0;
                    return ldg(L, (size_t)slot_of(down ? maxN - 1 - t : t));
                };
                if (count == 0) return;
                uint32_t jn[2] = {at(u), at(4 + u)};
                for (int q0 = 0; q0 < count; q0 += 8) {
                    float4 x[2], d[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        x[h] = ld4o(S.x, jn[h]);
                        d[h] = ld4o(S.xs, jn[h]);
                    }
                    jn[0] = at(q0 + 8 + u);
                    jn[1] = at(q0 + 12 + u);
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        ws = quad_sum<0>(ws, q0 + 4 * h + u < count ? predicted_w(a, x[h], d[h], k) : 0.0);
                }
            };
            run((int)ldg(S.nnb, (size_t)i), false);
            run(nsi, true);
        } else if (fluid) {
            const Rows fr = rows_of(S.cellStart, ci, nx, nxny);
            static_for<9>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                for (int j0 = fr.s[r]; j0 < fr.e[r]; j0 += 4) {
                    const uint32_t j = (uint32_t)min(j0 + u, fr.e[r] - 1);
                    const float4 x = ld4o(S.x, j), d = ld4o(S.xs, j);
                    ws = quad_sum<0>(ws, j0 + u < fr.e[r] ? predicted_w(a, x, d, k) : 0.0);
                }
            });
        }
    }
    __syncthreads();
    if (fluid && i < S.n && u == 0) e = pci_pressure(S, i, xi, ws, sbw[pl]);
    // one partial a group
    e = wave_max(e);
    dd = wave_max(dd);
    __shared__ double sm[8];
    if (lane == 0 && fluid) {
        sm[tid >> 6] = e;
        sm[4 + (tid >> 6)] = dd;
    }
    __syncthreads();
    if (tid == 0) {
        part[g0 >> 6] = fmax(fmax(sm[0], sm[1]), fmax(sm[2], sm[3]));
        if (S.pciShell) store_displacement(S, g0 >> 6, fmax(fmax(sm[4], sm[5]), fmax(sm[6], sm[7])), iter);
    }
}

// Pressure acceleration with the Spiky gradient at the current positions and
// predicted densities (src/PCISPHSolver.cpp:297-358), then the prediction of
// the next iteration (:122-149).  Runs after every k_pci_density, including
// the one that ended the loop.
template <int Q>
__global__ __launch_bounds__(kPartBlock<Q>) void k_pci_pacc(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                            int nchunks, int iter, int fused) {
    Chunk c;
    int i0, i;
    if (!part_at<Q>(C, nchunks, c, i0, i)) return;
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    Scalars* ss = S.ss;
    // this scene finished before this iteration (the finalize kernel counts
    // the iteration; with `fused` the density sweep sets done instead, and the
    // iteration is counted here)
    if (fused ? ss->done : ss->it <= iter) return;
    if (fused && i0 == 0 && threadIdx.x == 0) ss->it += 1;
    if (i >= S.n) return;
    const KCoefD k = S.kd;
    const double dt = ss->dt;
    const float4 xi = S.xk[i];
    const double xx = xi.x, xy = xi.y, xz = xi.z;
    const double pri = xi.w;
    const double m = S.mD;
    double ax = 0.0, ay = 0.0, az = 0.0;
    sweep<Q>(S, i, [&](uint32_t j) { return ld4(S.xk, j); },
             [&](const float4& xj) {
                 const Pair p = pair_of(xx, xy, xz, xj, k);
                 return Terms<4>{{m * (pri + (double)xj.w) * Gs_d(p, k), p.dx, p.dy, p.dz}};
             },
             [&](const Terms<4>& t) {
                 ax = fma(-t.v[0], t.v[1], ax);
                 ay = fma(-t.v[0], t.v[2], ay);
                 az = fma(-t.v[0], t.v[3], az);
             });
    if (Q > 1 && (threadIdx.x & 3) != 0) return;
    const float4 gs = S.gbs[i];
    ax -= pri * (double)gs.x;
    ay -= pri * (double)gs.y;
    az -= pri * (double)gs.z;
    if (S.pbOn) {
        // m_b p_b / rho_b^2 Spiky gradW of the PCISPH method
        // (src/PCISPHSolver.cpp:330-340)
        walk27(S.bCellStart, S.cell[i], S.nx, S.nx * S.ny, [&](int b) {
            const float4 y = S.xb[b];
            const Pair p = pair_of(xx, xy, xz, y, k);
            const double g = S.rho0D * (double)y.w * (double)S.bpr[b] * Gs_d(p, k);
            ax -= g * p.dx;
            ay -= g * p.dy;
            az -= g * p.dz;
        });
    }
    S.pacc[i] = make_float4((float)ax, (float)ay, (float)az, 0.f);
    const float4 a = S.a[i];
    const float4 v = S.v[i];
    const double wx = (double)v.x + (((double)a.x + ax) + (double)S.gx) * dt;
    const double wy = (double)v.y + (((double)a.y + ay) + (double)S.gy) * dt;
    const double wz = (double)v.z + (((double)a.z + az) + (double)S.gz) * dt;
    S.xs[i] = make_float4((float)(wx * dt), (float)(wy * dt), (float)(wz * dt), 0.f);
    if (S.pbOn) S.pv[i] = make_float4((float)wx, (float)wy, (float)wz, 0.f);
    shell_guard(S, wx * dt, wy * dt, wz * dt);
}

// PCISPH integrate (src/PCISPHSolver.cpp:444-474): a += g + pacc.
// `ahead`: as in k_df_positions; the launch behind this one tells the rest.
__global__ __launch_bounds__(kBlock) void k_pci_integrate(const DevScene* __restrict__ T, const Chunk* __restrict__ C,
                                                          int ahead) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (S.stall) return;
    if (ahead && !ended_before(S.ss->done, kLoopLast)) {
        __shared__ double sh[kWaves];
        if (!loop_over<LOOP_PCI>(S, S.ss, c.begin == 0, kLoopLast, sh)) return;
    }
    const int i = c.begin + threadIdx.x;
    if (c.begin == 0 && threadIdx.x == 0 && time_in_last_kernel(S)) advance_time(S);
    if (i >= S.n) return;
    const double dt = S.ss->dt;
    const float4 a = S.a[i], pa = S.pacc[i];
    const float4 v0 = S.v[i];
    const float4 x0 = S.x[i];
    if (S.pbOn) S.x0s[i] = x0;
    const double vx = (double)v0.x + ((double)a.x + ((double)S.gx + (double)pa.x)) * dt;
    const double vy = (double)v0.y + ((double)a.y + ((double)S.gy + (double)pa.y)) * dt;
    const double vz = (double)v0.z + ((double)a.z + ((double)S.gz + (double)pa.z)) * dt;
    S.v[i] = make_float4((float)vx, (float)vy, (float)vz, 0.f);
    S.x[i] = make_float4((float)((double)x0.x + vx * dt), (float)((double)x0.y + vy * dt),
                         (float)((double)x0.z + vz * dt), 0.f);
}

// =========================================================== finalize

// Scene reductions and loop control, one block per scene, after the sweep
// that wrote the chunk partials: the partials are added (or maxed) in chunk
// order, so the result does not depend on scheduling.
//   FIN_DT    CFL time step (src/DFSPHSolver.cpp:827-870): maxVel =
//             max(0.1, max_i sqrt(|v_i + (a_i + g) dt|)); dt' = cfl if
//             cfl < dt, else 0.99 dt after more than 3 density iterations,
//             else 1.001 dt; clamped to [min, max].
//   FIN_DENS0 / FIN_DENS   density loop of src/DFSPHSolver.cpp:320-398
//   FIN_DIV0 / FIN_DIV     divergence loop of src/DFSPHSolver.cpp:505-582
//             (bounded by maxIterations, :512; time += dt at its start)
//   FIN_PCI   PCISPH loop test after updatePressure (src/PCISPHSolver.cpp:365)
// The *0 kinds follow the call before the loop, whose error only feeds the
// log: the loop's error starts at 0 (:326, :511).  active[0] counts the
// scenes still iterating, active[1] is the largest iteration count reached.
enum FinKind { FIN_DT = 0, FIN_DENS0, FIN_DENS, FIN_DIV0, FIN_DIV, FIN_PCI };

// wide: the kernel that wrote the partials gave a particle 4 lanes, so they are
// one a group
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_finalize(const DevScene* __restrict__ T, int nscenes, int* active, int wide) {
    const int sc = blockIdx.x;
    if (sc >= nscenes) return;
    const DevScene& S = T[sc];
    if (S.stall) return;
    const gptr<Scalars> ss = G(S.ss);
    if ((KIND == FIN_DENS || KIND == FIN_PCI) && ss->done) return;
    if (KIND == FIN_DIV && ss->doneV) return;
    __shared__ double sh[kWaves];
    const double* const part = (KIND == FIN_PCI && wide) || KIND == FIN_DIV0 ? group_partial(S, 0)
                               : wide ? group_partial(S, 1) : S.partial;
    const double red = (KIND == FIN_DT || KIND == FIN_PCI) ? scene_partial_max(part, wide ? S.nChunks * kWaves : S.nChunks, sh)
                       : wide ? scene_group_sum(part, S.nChunks, sh)
                              : scene_partial_sum(part, S.nChunks, sh);
    if (threadIdx.x != 0) return;
    if (KIND == FIN_DT) {
        // the density solve's loop counters start here (counted by FIN_DENS0)
        if (sc == 0) {
            active[0] = 0;
            active[1] = 0;
        }
        const NextDt d = next_dt(S, ss->dt, ss->it, red);
        ss->dt = d.dt;
        ss->maxVel = d.maxVel;
        ss->cflTs = d.cflTs;
        ss->steps += 1u;
    } else if (KIND == FIN_PCI) {
        ss->maxDensErr = red;
        const int it = ++ss->it;
        const bool more = ((red > S.eta) || (it < S.minIt)) && (it < S.maxIt);
        if (!more) {
            ss->done = 1;
            ss->sumIt += (unsigned)it;
            atomicSub(active, 1);
            atomicMax(active + 1, it);
        }
    } else {
        const double avg = (S.n == 0) ? 0.0 : red / (double)S.n;
        const bool dens = (KIND == FIN_DENS0 || KIND == FIN_DENS);
        const bool first = (KIND == FIN_DENS0 || KIND == FIN_DIV0);
        int it;
        double err;
        if (first) {
            it = 0;
            err = 0.0;
            if (dens) {
                ss->avgErr0 = avg;
                ss->it = 0;
            } else {
                ss->avgErrV0 = avg;
                ss->itV = 0;
                ss->time += ss->dt;
            }
        } else {
            err = avg;
            if (dens) {
                it = ++ss->it;
                ss->avgErr = avg;
            } else {
                it = ++ss->itV;
                ss->avgErrV = avg;
            }
        }
        const bool more = dens ? (((err > S.eta) || (it < S.minIt)) && (it < S.maxIt))
                               : (((err > S.etaV / ss->dt) || (it < S.minItV)) && (it < S.maxIt));
        if (dens) ss->done = more ? 0 : 1;
        else ss->doneV = more ? 0 : 1;
        if (first && more) atomicAdd(active, 1);
        if (!first && !more) atomicSub(active, 1);
        if (!more) atomicMax(active + 1, it);
        if (!more) {
            if (dens) ss->sumIt += (unsigned)it;
            else ss->sumItV += (unsigned)it;
        }
    }
}

// Where a lone scene's loop stands, for the host (one block): after the
// iterations launched of the density loop (LOOP_DENS), the PCISPH loop, or the
// divergence loop.  END: the end of a step.  With `tables` the host has not
// asked after the step's loops and the next step's launches wait behind this
// one: they return at once if a loop has not ended.
// Without `rec` it only decides, for a scene whose sweeps leave that to it;
// idx: see loop_over.
template <int KIND, bool END>
__global__ __launch_bounds__(kBlock) void k_loop_end(const DevScene* T, Tables tables, StepRec* rec,
                                                     unsigned seq, int idx) {
    const DevScene& S = T[0];
    Scalars* ss = S.ss;
    int stall = S.stall;
    __shared__ double sh[kWaves];
    if (!stall) {
        bool over = (KIND == LOOP_DIV ? ss->doneV : ss->done) != 0;
        __syncthreads();   // every thread has read the flag before it is set
        // (the PCISPH integration has decided where the sweeps do)
        if (!over && !(END && KIND == LOOP_PCI)) over = loop_over<KIND>(S, ss, true, idx, sh, true);
        if (END && KIND == LOOP_DIV) {
            const double avg0 = (up_to(kQuadChunks, S.nChunks) ? scene_group_sum(group_partial(S, 0), S.nChunks, sh)
                                                          : scene_partial_sum(group_partial(S, 0), S.nChunks, sh)) / (double)S.n;
            if (threadIdx.x == 0) ss->avgErrV0 = avg0;
        }
        if (END && !over && tables.a) {
            stall = KIND == LOOP_PCI ? 1 : 2;
            if (threadIdx.x == 0) tables.a->stall = tables.b->stall = stall;
        }
        if (threadIdx.x == 0 && rec) rec->done = over ? 1 : 0;
    }
    if (threadIdx.x == 0 && rec) {
        rec->it = ss->it;
        rec->itV = ss->itV;
        rec->stall = stall;
        __hip_atomic_store(&rec->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
// A batch's loop counters for the host: the scenes still iterating (done) and
// the largest count reached (it).
__global__ void k_tell_active(const int* active, StepRec* rec, unsigned seq) {
    if (threadIdx.x == 0) {
        rec->done = active[0];
        rec->it = active[1];
        __hip_atomic_store(&rec->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
// The host has taken notice of a stall.
__global__ void k_clear_stall(Tables tables) {
    if (threadIdx.x == 0) tables.a->stall = tables.b->stall = 0;
}

// CubeBoundaryModel::correctPositionAndVelocity (src/CubeBoundaryModel.cpp:
// 16-94): per axis in x, y, z order, a position below the minimum (above
// the maximum) is set to it, the axis velocity is multiplied by -normalFct if
// it points out of the box, and the other two components by tangentialFct.
// The faces are the nearest FP32 values inside the box, so the set of
// clamped particles is the FP64 comparison's, and a particle left on a face
// is not clamped again on later steps (FP64 positions sit exactly on it).
__global__ __launch_bounds__(kBlock) void k_cube(const DevScene* __restrict__ T, const Chunk* __restrict__ C) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    const int i = c.begin + threadIdx.x;
    if (!S.cubeOn) return;
    // the clamp changes velocities after the divergence sweeps formed d0
    if (c.begin == 0 && threadIdx.x == 0 && S.method == DFSPH) S.ss->d0Valid = 0u;
    if (i >= S.n) return;
    const float4 xf = S.x[i], vf = S.v[i];
    float p[3] = {xf.x, xf.y, xf.z};
    double u[3] = {vf.x, vf.y, vf.z};
    const double nf = S.cubeNf, tf = S.cubeTf;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int b = (a + 1) % 3, e = (a + 2) % 3;
        bool hit = false;
        if (p[a] < S.cubeLo[a]) {
            p[a] = S.cubeLo[a];
            if (u[a] < 0.0) u[a] *= -nf;
            hit = true;
        } else if (p[a] > S.cubeHi[a]) {
            p[a] = S.cubeHi[a];
            if (u[a] > 0.0) u[a] *= -nf;
            hit = true;
        }
        if (hit) {
            u[b] *= tf;
            u[e] *= tf;
        }
    }
    S.x[i] = make_float4(p[0], p[1], p[2], xf.w);
    S.v[i] = make_float4((float)u[0], (float)u[1], (float)u[2], vf.w);
}

// Emitters (Simulation::emitParticles -> Emitter::emitParticles,
// src/Emitter.cpp:85-162), one block per scene, emitters in order: an
// emitter whose next emission time has come (time >= next) and whose budget
// holds a whole group appends the group at slots n, n+1, ... (ids equal to
// the slots, continuing the active count): velocity (0, 0, vel) and
// position group + t (velocity + g t), t = time - next, both rotated by the
// quaternion as glm evaluates it (u = (q.x, q.y, q.z):
// v + ((u x v) w + u x (u x v)) 2), the position then offset by the
// emitter origin.  Warm-start values start at zero.  With `cells`, the new
// particles' cells are counted for the grid sort that follows (DFSPH emits
// between its position update and the grid rebuild).  Tc is the table whose
// buffers are current at the call (before or after the step's sort), To
// the other; the new count goes to both and to the scalars.
__device__ inline void quat_rotate(const double q[4], double& x, double& y, double& z) {
    const double ux = q[1], uy = q[2], uz = q[3];
    const double cx = uy * z - y * uz, cy = uz * x - z * ux, cz = ux * y - x * uy;      // u x v
    const double dx = uy * cz - cy * uz, dy = uz * cx - cz * ux, dz = ux * cy - cx * uy;  // u x (u x v)
    x = x + ((cx * q[0]) + dx) * 2.0;
    y = y + ((cy * q[0]) + dy) * 2.0;
    z = z + ((cz * q[0]) + dz) * 2.0;
}

__global__ __launch_bounds__(kBlock) void k_emit(DevScene* __restrict__ Tc, DevScene* __restrict__ To, int nscenes,
                                                 int cells) {
    const int sc = blockIdx.x;
    if (sc >= nscenes) return;
    const DevScene& S = Tc[sc];
    if (S.nEmit == 0) return;
    Scalars* ss = S.ss;
    const double time = ss->time;
    const int n0 = S.n;
    int n = n0;
    for (int e = 0; e < S.nEmit; ++e) {
        EmitterDev* E = S.emit + e;
        const int gs = E->groupSize;
        const bool fire = (time >= E->next) && (E->remaining >= (unsigned)gs) && (n + gs <= S.cap);
        if (fire) {
            const double t = time - E->next;
            double q[4] = {E->q[0], E->q[1], E->q[2], E->q[3]};
            for (int g = threadIdx.x; g < gs; g += blockDim.x) {
                const double* lp = S.emitGroup + 3 * (size_t)(E->group + g);
                double vx = 0.0, vy = 0.0, vz = E->vel;
                double px = lp[0] + (vx + (double)S.gx * t) * t;
                double py = lp[1] + (vy + (double)S.gy * t) * t;
                double pz = lp[2] + (vz + (double)S.gz * t) * t;
                quat_rotate(q, px, py, pz);
                quat_rotate(q, vx, vy, vz);
                px += E->pos[0];
                py += E->pos[1];
                pz += E->pos[2];
                const int slot = n + g;
                const float4 xp = make_float4((float)px, (float)py, (float)pz, 0.f);
                S.x[slot] = xp;
                S.v[slot] = make_float4((float)vx, (float)vy, (float)vz, 0.f);
                S.id[slot] = (uint32_t)slot;
                if (S.k) {
                    S.k[slot] = 0.f;
                    S.kv[slot] = 0.f;
                }
                if (cells) {
                    const int cl = cell_of(S, xp);
                    S.cellU[slot] = cl;
                    atomicAdd(&S.cellCount[cl], 1);
                }
            }
            n += gs;
        }
        __syncthreads();   // every thread has read this emitter's state
        if (fire && threadIdx.x == 0) {
            E->remaining -= (unsigned)gs;
            E->next += E->interval;
        }
    }
    if (threadIdx.x == 0 && n != n0) {
        Tc[sc].n = n;
        To[sc].n = n;
        ss->nActive = (unsigned)n;
    }
}

// ===================================================== PCISPH boundary method

// The boundary particles' sums over the (static) boundary, m_b W and m_b
// Poly6 with the boundary candidates of the particle's cell
// (src/SPHSolver.cpp:115-120, src/PCISPHSolver.cpp:239-244).  One scene.
__global__ __launch_bounds__(kBlock) void k_pb_bself(const DevScene* __restrict__ T, int scene) {
    const DevScene& S = T[scene];
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b >= S.nb) return;
    const KCoefD k = S.kd;
    const float4 yb = S.xb[b];
    const double px = yb.x, py = yb.y, pz = yb.z;
    double wc = 0.0, wp = 0.0;
    walk27(S.bCellStart, cell_of(S, yb), S.nx, S.nx * S.ny, [&](int c) {
        const float4 y = S.xb[c];
        const Pair p = pair_of(px, py, pz, y, k);
        const double mb = S.rho0D * (double)y.w;
        wc += mb * W_d(p.q, k);
        wp += mb * P6_d(p.r2, k);
    });
    S.bself[2 * b] = wc;
    S.bself[2 * b + 1] = wp;
}

// Boundary densities and pressures (one scene).  PRED = 0, WCSPH
// (src/SPHSolver.cpp:93-121, src/WCSPHSolver.cpp:97-114): rho_b = sum over
// the fluid candidates of the particle's cell of m W(r_b - x_j) plus the
// boundary sum, p_b = max(0, kappa rho0/gamma ((rho_b/rho0)^gamma - 1)).
// PRED = 1, PCISPH loop (src/PCISPHSolver.cpp:214-247, :276-293): Poly6
// with the predicted fluid positions, p_b += delta max(0, rho_b - rho0),
// from zero at the first iteration.  Both store p_b / rho_b^2 for the
// fluid's pressure sums.  In the loop it runs after the finalize of
// iteration `iter`, for scenes that ran that iteration.
template <int PRED>
__global__ __launch_bounds__(kBlock) void k_pb_bdensity(const DevScene* __restrict__ T, int scene, int iter) {
    const DevScene& S = T[scene];
    if (PRED && S.ss->it <= iter) return;
    const int first = iter == 0;
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b >= S.nb) return;
    const KCoefD k = S.kd;
    const float4 yb = S.xb[b];
    const double px = yb.x, py = yb.y, pz = yb.z;
    const double m = S.mD, rho0 = S.rho0D;
    double s = 0.0;
    walk27(S.cellStart, cell_of(S, yb), S.nx, S.nx * S.ny, [&](int j) {
        const float4 xj = S.x[j];
        if (PRED) {
            const float4 dj = S.xs[j];
            const double dx = (px - (double)xj.x) - (double)dj.x;
            const double dy = (py - (double)xj.y) - (double)dj.y;
            const double dz = (pz - (double)xj.z) - (double)dj.z;
            s += m * P6_d(dx * dx + dy * dy + dz * dz, k);
        } else {
            const Pair p = pair_of(px, py, pz, xj, k);
            s += m * W_d(p.q, k);
        }
    });
    const double rho = s + S.bself[2 * b + PRED];
    double pr;
    if (PRED) {
        pr = (first ? 0.0 : (double)S.bpres[b]) + S.pciDeltaD * fmax(0.0, rho - rho0);
    } else {
        const double x = (rho - rho0) / rho0;
        pr = fmax(0.0, (double)S.stiffness * rho0 / (double)S.gammaEos * expm1((double)S.gammaEos * log1p(x)));
    }
    S.bdens[b] = (float)rho;
    S.bpres[b] = (float)pr;
    S.bpr[b] = (float)(pr / (rho * rho));
}

// Position (and velocity) projection after the step's position update.
// MODE 0, DFSPH (src/DFSPHSolver.cpp:65-75): q = x; the particle's cell is
// then counted for the grid rebuild.  MODE 1, WCSPH (src/WCSPHSolver.cpp:
// 62-73): q = x, then the velocity.  MODE 2, PCISPH (src/PCISPHSolver.cpp:
// 65-76): q = the loop's last corrected predicted position, and the velocity
// correction starts from its predicted velocity.
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_pb_correct(const DevScene* __restrict__ T, const Chunk* __restrict__ C) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (!S.pbOn) return;
    const int i = c.begin + threadIdx.x;
    if (i >= S.n) return;
    float4 xf = S.x[i];
    const double px = xf.x, py = xf.y, pz = xf.z;
    double qx = px, qy = py, qz = pz;
    if (MODE == 2) {
        const float4 x0 = S.x0s[i], d = S.prS[i];
        qx = (double)x0.x + (double)d.x;
        qy = (double)x0.y + (double)d.y;
        qz = (double)x0.z + (double)d.z;
    }
    const PbHit h = pb_project(S, px, py, pz, xf, qx, qy, qz);
    S.pbn[i] = make_float4((float)h.nx, (float)h.ny, (float)h.nz, 0.f);
    if (h.hit) {
        xf.x = (float)(px + h.s * h.nx);
        xf.y = (float)(py + h.s * h.ny);
        xf.z = (float)(pz + h.s * h.nz);
        S.x[i] = xf;
    }
    if (MODE == 0) {
        const int cl = cell_of(S, xf);
        S.cellU[i] = cl;
        atomicAdd(&S.cellCount[cl], 1);
    } else {
        double ux, uy, uz;
        if (MODE == 1) {
            const float4 v = S.v[i];
            ux = v.x; uy = v.y; uz = v.z;
        } else {
            const float4 v = S.pvS[i];
            ux = v.x; uy = v.y; uz = v.z;
        }
        if (pb_velocity(S, h.nx, h.ny, h.nz, ux, uy, uz)) S.v[i] = make_float4((float)ux, (float)uy, (float)uz, 0.f);
    }
}

// correctPredPositions (src/PCISPHBoundaryModel.cpp:385-439), each PCISPH
// loop iteration after the prediction: collision test with the current
// position, weights and shift on the predicted one (x + d), d corrected.
// Keeps the corrected d and the predicted velocity for the projection after
// the integration.
__global__ __launch_bounds__(kBlock) void k_pb_predcorrect(const DevScene* __restrict__ T, const Chunk* __restrict__ C) {
    const Chunk c = chunk_at(C, kBlock);
    const DevScene& S = T[c.scene];
    if (!S.pbOn || S.ss->done) return;
    const int i = c.begin + threadIdx.x;
    if (i >= S.n) return;
    const float4 xf = S.x[i];
    float4 d = S.xs[i];
    const double px = xf.x, py = xf.y, pz = xf.z;
    const PbHit h = pb_project(S, px, py, pz, xf, px + (double)d.x, py + (double)d.y, pz + (double)d.z);
    S.pbn[i] = make_float4((float)h.nx, (float)h.ny, (float)h.nz, 0.f);
    if (h.hit) {
        d.x = (float)((double)d.x + h.s * h.nx);
        d.y = (float)((double)d.y + h.s * h.ny);
        d.z = (float)((double)d.z + h.s * h.nz);
        S.xs[i] = d;
    }
    S.prS[i] = d;
    S.pvS[i] = S.pv[i];
}

// WCSPH: time += dt after the integration (src/WCSPHSolver.cpp:77).
__global__ void k_time_advance(const DevScene* __restrict__ T, int nscenes) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nscenes || time_in_last_kernel(T[s])) return;
    advance_time(T[s]);
}

// The neighbor-overflow maximum of every scene of a batch starts each step
// call at the overflow of the lists the call starts with -- DFSPH's first
// sweeps use the lists of the previous call's last rebuild (or of init /
// set_state); WCSPH and PCISPH build theirs at the start of each step -- so
// it reports the lists of that call's steps only.
__global__ void k_clear_overflow(const DevScene* __restrict__ T, int nscenes) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nscenes) T[s].ss->overflow = (T[s].method == DFSPH) ? T[s].ss->listOver : 0u;
}

// ============================================================ utilities

__global__ void k_fill_int(int* p, int v, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Sorted -> particle-id order.
__global__ void k_unsort_f4(const float4* __restrict__ src, const uint32_t* __restrict__ id, float* __restrict__ dst, int n, int comps) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const float4 v = src[s];
    float* d = dst + (size_t)id[s] * comps;
    d[0] = v.x;
    if (comps > 1) d[1] = v.y;
    if (comps > 2) d[2] = v.z;
    if (comps > 3) d[3] = v.w;
}
__global__ void k_unsort_f1(const float* __restrict__ src, const uint32_t* __restrict__ id, float* __restrict__ dst, int n,
                            double offset) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    dst[id[s]] = (float)(offset + (double)src[s]);
}
__global__ void k_unsort_i1(const int* __restrict__ src, const uint32_t* __restrict__ id, int* __restrict__ dst, int n) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    dst[id[s]] = src[s];
}
// Reference keys floor(x/h) of each particle, in id order.
__global__ void k_keys3(const DevScene* __restrict__ T, int scene, int* __restrict__ dst) {
    const DevScene& S = T[scene];
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S.n) return;
    const float4 p = S.x[s];
    int* d = dst + (size_t)S.id[s] * 3;
    d[0] = (int)floor(__ddiv_rn((double)p.x, S.hD));
    d[1] = (int)floor(__ddiv_rn((double)p.y, S.hD));
    d[2] = (int)floor(__ddiv_rn((double)p.z, S.hD));
}
// Id-ordered upload -> working arrays (identity order until the first sort).
__global__ void k_load_state(const DevScene* __restrict__ T, int scene, const float* __restrict__ xyz, const float* __restrict__ vel,
                             const float* __restrict__ kk, const float* __restrict__ kkv) {
    const DevScene& S = T[scene];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.n) return;
    S.x[i] = make_float4(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], 0.f);
    S.v[i] = vel ? make_float4(vel[3 * i], vel[3 * i + 1], vel[3 * i + 2], 0.f) : make_float4(0.f, 0.f, 0.f, 0.f);
    S.id[i] = (uint32_t)i;
    if (S.a) S.a[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (S.k) S.k[i] = kk ? kk[i] : 0.0f;
    if (S.kv) S.kv[i] = kkv ? kkv[i] : 0.0f;
}

// ============================================================ launchers

// a kernel with 4 lanes a particle over n chunks, with 4 wavefronts or BT
// threads a block
#define LAUNCH_QUAD_BT(kern, BT, n, stream, ...) \
    hipLaunchKernelGGL(kern, dim3((n + 7) / 8 * 8 * kWaves), dim3(BT), 0, stream, __VA_ARGS__)
#define LAUNCH_QUAD(kern, n, stream, ...) LAUNCH_QUAD_BT(kern, 256, n, stream, __VA_ARGS__)
#define LAUNCH(kern, grid, stream, ...) hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, stream, __VA_ARGS__)

void launch_keys(hipStream_t st, const DevScene* T, const Chunk* C, int n, int* begin_active) {
    if (!n) return;
    if (begin_active) LAUNCH(k_keys<true>, n, st, T, C, begin_active);
    else LAUNCH(k_keys<false>, n, st, T, C, nullptr);
}
void launch_scan(hipStream_t st, const DevScene* T, const Chunk* CC, int ncc, int nscenes, int maxChunks, Tables tables,
                 int fused) {
    if (!ncc) return;
    if (maxChunks <= kScanOneChunks) {
        LAUNCH(k_scan_final<SCAN_ONE>, ncc, st, T, CC, tables, fused);
        return;
    }
    LAUNCH(k_scan_sum, ncc, st, T, CC, tables, fused);
    if (maxChunks <= kScanFusedChunks) {
        LAUNCH(k_scan_final<SCAN_TOTALS>, ncc, st, T, CC, Tables{}, 0);
        return;
    }
    LAUNCH(k_scan_offsets, nscenes, st, T, nscenes);
    LAUNCH(k_scan_final<SCAN_OFFSETS>, ncc, st, T, CC, Tables{}, 0);
}
void launch_scatter(hipStream_t st, const DevScene* T, const Chunk* C, int n) { if (n) LAUNCH(k_scatter, n, st, T, C); }
void launch_rank_reorder(hipStream_t st, const DevScene* T, const Chunk* C, int n) { if (n) LAUNCH(k_rank_reorder, n, st, T, C); }
void launch_bvolume(hipStream_t st, const DevScene* T, int scene, int nb, float* tmp) {
    if (!nb) return;
    const int g = (nb + kBlock - 1) / kBlock;
    LAUNCH(k_bvolume, g, st, T, scene, tmp);
    LAUNCH(k_bvolume_pack, g, st, T, scene, (const float*)tmp);
}
void launch_build(hipStream_t st, int method, const DevScene* T, const Chunk* C, int n, int fused) {
    if (!n) return;
    // Up to where 4 lanes a particle are faster (us a step; one lane / four):
    // WCSPH 16 chunks 64 / 36, 128 62 / 42, 232 71 / 63, 311 78 / 76, 381 83 /
    // 87; PCISPH 16 136 / 105, 232 160 / 154, 311 180 / 180; DFSPH 16 123 / 94,
    // 232 157 / 152, 311 178 / 178.
    if (up_to(kQuadChunks, n)) {
        if (method == DFSPH) LAUNCH_QUAD_BT(k_build_quad<DFSPH>, 512, n, st, T, C, n, fused);
        else if (method == WCSPH) LAUNCH_QUAD_BT(k_build_quad<WCSPH>, 512, n, st, T, C, n, 0);
        else LAUNCH_QUAD_BT(k_build_quad<PCISPH>, 512, n, st, T, C, n, 0);
        return;
    }
    if (method == DFSPH) LAUNCH(k_build<DFSPH>, n, st, T, C, fused);
    else if (method == WCSPH) LAUNCH(k_build<WCSPH>, n, st, T, C, 0);
    else LAUNCH(k_build<PCISPH>, n, st, T, C, 0);
}
// The sweeps with 4 lanes a particle where a launch leaves SIMDs without a
// wavefront (us per step, one lane -> 4).  DFSPH without forces: 16 chunks 122
// -> 102, 128: 136 -> 123, 183: 144 -> 138, 198: 149 -> 152, 250: 158 -> 160,
// 290: 188 -> 177, 381: 203 -> 199, 432: 206 -> 212; the cohesion of DFSPH and
// PCISPH has its lines in the same places (154: 221 -> 219, 198: 253 -> 254,
// 333: 347 -> 346, 489: 398 -> 404).  Forces without cohesion, WCSPH: 16: 52
// -> 42, 128: 55 -> 49, 333: 81 -> 79, 489: 94 -> 94; with it 16: 57 -> 50,
// 128: 60 -> 58, 154: 68 -> 71 (128 registers and ~100 FP64 instructions a
// pair, 12 terms to exchange).  PCISPH pressure force: 16: 118.9 -> 114.7,
// 128: 125 -> 123, 141: 139 -> 140, 198: 152 -> 159.
void launch_normals(hipStream_t st, const DevScene* T, const Chunk* C, int n) {
    if (!n) return;
    if (quad_sweep(n)) LAUNCH_QUAD(k_normals<4>, n, st, T, C, n);
    else LAUNCH(k_normals<1>, n, st, T, C, n);
}
// The combinations of XSPH and cohesion get a kernel of their own; the two
// viscosity forces that read rho_j as well, and batches whose scenes differ,
// take the general one.
template <int M, int FL>
void launch_forces_f(hipStream_t st, const DevScene* T, const Chunk* C, int n) {
    const bool quad = !(FL & F_ST) ? up_to(kQuadForcesChunks, n) : M == WCSPH ? up_to(kQuadTensionChunks, n) : quad_sweep(n);
    if (quad) LAUNCH_QUAD((k_forces<M, FL, 4>), n, st, T, C, n);
    else LAUNCH((k_forces<M, FL, 1>), n, st, T, C, n);
}
template <int M>
void launch_forces_m(hipStream_t st, int flags, const DevScene* T, const Chunk* C, int n) {
    switch (flags < 0 ? -1 : flags & ~F_ADH) {
        case 0: launch_forces_f<M, 0>(st, T, C, n); break;
        case F_XSPH: launch_forces_f<M, F_XSPH>(st, T, C, n); break;
        case F_ST: launch_forces_f<M, F_ST>(st, T, C, n); break;
        case F_XSPH | F_ST: launch_forces_f<M, F_XSPH | F_ST>(st, T, C, n); break;
        default: LAUNCH((k_forces<M, -1, 1>), n, st, T, C, n);
    }
}
void launch_forces(hipStream_t st, int method, int flags, const DevScene* T, const Chunk* C, int n) {
    if (!n) return;
    if (method == DFSPH) launch_forces_m<DFSPH>(st, flags, T, C, n);
    else if (method == WCSPH) launch_forces_m<WCSPH>(st, flags, T, C, n);
    else launch_forces_m<PCISPH>(st, flags, T, C, n);
}
void launch_dt(hipStream_t st, const DevScene* T, const Chunk* C, int n) { if (n) LAUNCH(k_dt, n, st, T, C); }
void launch_df_predict(hipStream_t st, const DevScene* T, const Chunk* C, int n, int fused) {
    if (n) LAUNCH(k_df_predict, n, st, T, C, fused);
}
template <int MODE>
void launch_df_vel_m(hipStream_t st, const DevScene* T, const Chunk* C, int n, int iter, int fused) {
    if (quad_sweep(n)) LAUNCH_QUAD((k_df_vel<MODE, 4>), n, st, T, C, n, iter, fused);
    else LAUNCH((k_df_vel<MODE, 1>), n, st, T, C, n, iter, fused);
}
void launch_df_vel(hipStream_t st, int mode, const DevScene* T, const Chunk* C, int n, int iter, int fused) {
    if (!n) return;
    if (mode == 0) launch_df_vel_m<0>(st, T, C, n, iter, fused);
    else if (mode == 1) launch_df_vel_m<1>(st, T, C, n, iter, fused);
    else launch_df_vel_m<2>(st, T, C, n, iter, fused);
}
template <int MODE>
void launch_df_err_m(hipStream_t st, const DevScene* T, const Chunk* C, int n, int fused) {
    if (quad_sweep(n)) LAUNCH_QUAD((k_df_err<MODE, 4>), n, st, T, C, n, fused);
    else LAUNCH((k_df_err<MODE, 1>), n, st, T, C, n, fused);
}
void launch_df_err(hipStream_t st, int mode, const DevScene* T, const Chunk* C, int n, int fused) {
    if (!n) return;
    if (mode == 0) launch_df_err_m<0>(st, T, C, n, fused);
    else if (mode == 1) launch_df_err_m<1>(st, T, C, n, fused);
    else launch_df_err_m<3>(st, T, C, n, fused);
}
void launch_finalize(hipStream_t st, int kind, const DevScene* T, int nscenes, int* active, int nchunks) {
    if (!nscenes) return;
    switch (kind) {
        case FIN_DT: LAUNCH(k_finalize<FIN_DT>, nscenes, st, T, nscenes, active, 0); break;
        case FIN_DENS0: LAUNCH(k_finalize<FIN_DENS0>, nscenes, st, T, nscenes, active, quad_sweep(nchunks)); break;
        case FIN_DENS: LAUNCH(k_finalize<FIN_DENS>, nscenes, st, T, nscenes, active, quad_sweep(nchunks)); break;
        case FIN_DIV0: LAUNCH(k_finalize<FIN_DIV0>, nscenes, st, T, nscenes, active, up_to(kQuadChunks, nchunks) ? 1 : 0); break;
        case FIN_DIV: LAUNCH(k_finalize<FIN_DIV>, nscenes, st, T, nscenes, active, quad_sweep(nchunks)); break;
        default: LAUNCH(k_finalize<FIN_PCI>, nscenes, st, T, nscenes, active, up_to(kQuadPciChunks, nchunks) ? 1 : 0); break;
    }
}
void launch_df_positions(hipStream_t st, const DevScene* T, const Chunk* C, int n, int* active, int ahead) {
    if (n) LAUNCH(k_df_positions, n, st, T, C, active, ahead);
}
void launch_pci_density(hipStream_t st, const DevScene* T, const Chunk* C, int n, int iter, int fused) {
    if (!n) return;
    // (us a step, one lane / four: 64,000 particles 191 / 142, 97k 221 / 187, 195k
    // 283 / 269, 287k 308 / 308, 351k spheres 412 / 440; four lanes, boundary after
    // the fluid / beside it: 4,096 101 / 93, 51k 144 / 141, 59k 148.6 / 149.2, 64k
    // 142 / 149)
    if (up_to(kQuadSideChunks, n)) LAUNCH_QUAD_BT(k_pci_density_quad<true>, 512, n, st, T, C, n, iter, fused);
    else if (up_to(kQuadPciChunks, n)) LAUNCH_QUAD(k_pci_density_quad<false>, n, st, T, C, n, iter, fused);
    else LAUNCH(k_pci_density, n, st, T, C, iter, fused);
}
void launch_pci_pacc(hipStream_t st, const DevScene* T, const Chunk* C, int n, int iter, int fused) {
    if (!n) return;
    if (up_to(kQuadPaccChunks, n)) LAUNCH_QUAD(k_pci_pacc<4>, n, st, T, C, n, iter, fused);
    else LAUNCH(k_pci_pacc<1>, n, st, T, C, n, iter, fused);
}
void launch_pci_integrate(hipStream_t st, const DevScene* T, const Chunk* C, int n, int ahead) {
    if (n) LAUNCH(k_pci_integrate, n, st, T, C, ahead);
}
void launch_loop_end(hipStream_t st, int loop, int end, const DevScene* T, Tables t, StepRec* rec, unsigned seq, int iter) {
    const int idx = end ? kLoopLast : iter;
    if (loop == LOOP_PCI && end) LAUNCH((k_loop_end<LOOP_PCI, true>), 1, st, T, t, rec, seq, idx);
    else if (loop == LOOP_PCI) LAUNCH((k_loop_end<LOOP_PCI, false>), 1, st, T, t, rec, seq, idx);
    else if (loop == LOOP_DENS) LAUNCH((k_loop_end<LOOP_DENS, false>), 1, st, T, t, rec, seq, idx);
    else if (end) LAUNCH((k_loop_end<LOOP_DIV, true>), 1, st, T, t, rec, seq, idx);
    else LAUNCH((k_loop_end<LOOP_DIV, false>), 1, st, T, t, rec, seq, idx);
}
void launch_tell_active(hipStream_t st, const int* active, StepRec* rec, unsigned seq) {
    hipLaunchKernelGGL(k_tell_active, dim3(1), dim3(64), 0, st, active, rec, seq);
}
void launch_clear_stall(hipStream_t st, Tables t) { hipLaunchKernelGGL(k_clear_stall, dim3(1), dim3(64), 0, st, t); }
void launch_cube(hipStream_t st, const DevScene* T, const Chunk* C, int n) { if (n) LAUNCH(k_cube, n, st, T, C); }
void launch_pb_bself(hipStream_t st, const DevScene* T, int scene, int nb) {
    if (nb) hipLaunchKernelGGL(k_pb_bself, dim3((nb + kBlock - 1) / kBlock), dim3(kBlock), 0, st, T, scene);
}
void launch_pb_bdensity(hipStream_t st, int pred, const DevScene* T, int scene, int nb, int iter) {
    if (!nb) return;
    const dim3 g((nb + kBlock - 1) / kBlock), b(kBlock);
    if (pred) hipLaunchKernelGGL(k_pb_bdensity<1>, g, b, 0, st, T, scene, iter);
    else hipLaunchKernelGGL(k_pb_bdensity<0>, g, b, 0, st, T, scene, iter);
}
// dst[s] = src[id[s]] (an id-ordered float3 array into the working order).
__global__ void k_gather_f3(float4* __restrict__ dst, const float* __restrict__ src, const uint32_t* __restrict__ id,
                            int n) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const float* q = src + 3 * (size_t)id[s];
    dst[s] = make_float4(q[0], q[1], q[2], 0.f);
}
void launch_gather_f3(hipStream_t st, float4* dst, const float* src, const uint32_t* id, int n) {
    if (n) hipLaunchKernelGGL(k_gather_f3, dim3((n + 255) / 256), dim3(256), 0, st, dst, src, id, n);
}
void launch_pb_correct(hipStream_t st, int mode, const DevScene* T, const Chunk* C, int n) {
    if (!n) return;
    if (mode == 0) LAUNCH(k_pb_correct<0>, n, st, T, C);
    else if (mode == 1) LAUNCH(k_pb_correct<1>, n, st, T, C);
    else LAUNCH(k_pb_correct<2>, n, st, T, C);
}
void launch_pb_predcorrect(hipStream_t st, const DevScene* T, const Chunk* C, int n) {
    if (n) LAUNCH(k_pb_predcorrect, n, st, T, C);
}
void launch_emit(hipStream_t st, DevScene* Tc, DevScene* To, int nscenes, int cells) {
    if (nscenes) hipLaunchKernelGGL(k_emit, dim3(nscenes), dim3(kBlock), 0, st, Tc, To, nscenes, cells);
}
void launch_time_advance(hipStream_t st, const DevScene* T, int nscenes) {
    hipLaunchKernelGGL(k_time_advance, dim3((nscenes + 255) / 256), dim3(256), 0, st, T, nscenes);
}
void launch_clear_overflow(hipStream_t st, const DevScene* T, int nscenes) {
    hipLaunchKernelGGL(k_clear_overflow, dim3((nscenes + 255) / 256), dim3(256), 0, st, T, nscenes);
}
void launch_fill_int(hipStream_t st, int* p, int v, long n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_int, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, v, n);
}
void launch_unsort_f4(hipStream_t st, const float4* src, const uint32_t* id, float* dst, int n, int comps) {
    if (n) hipLaunchKernelGGL(k_unsort_f4, dim3((n + 255) / 256), dim3(256), 0, st, src, id, dst, n, comps);
}
void launch_unsort_f1(hipStream_t st, const float* src, const uint32_t* id, float* dst, int n, double offset) {
    if (n) hipLaunchKernelGGL(k_unsort_f1, dim3((n + 255) / 256), dim3(256), 0, st, src, id, dst, n, offset);
}
void launch_unsort_i1(hipStream_t st, const int* src, const uint32_t* id, int* dst, int n) {
    if (n) hipLaunchKernelGGL(k_unsort_i1, dim3((n + 255) / 256), dim3(256), 0, st, src, id, dst, n);
}
void launch_keys3(hipStream_t st, const DevScene* T, int scene, int n, int* dst) {
    if (n) hipLaunchKernelGGL(k_keys3, dim3((n + 255) / 256), dim3(256), 0, st, T, scene, dst);
}
void launch_load_state(hipStream_t st, const DevScene* T, int scene, int n, const float* xyz, const float* vel, const float* k, const float* kv) {
    if (n) hipLaunchKernelGGL(k_load_state, dim3((n + 255) / 256), dim3(256), 0, st, T, scene, xyz, vel, k, kv);
}

}  // namespace sphg
