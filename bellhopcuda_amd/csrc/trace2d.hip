// trace2d.hip -- MI355X (gfx950) kernels of the 2D ray/beam tracer and the
// device half of the C ABI (include/bhc_hip.h).
//
// Launch model (replaces FieldModesKernel, src/mode/fieldimpl.cu.in:29-64):
//  * persistent workgroups; every lane owns one ray for the ray's whole life
//    and pulls the next ray index from a device-side work counter as soon as
//    its ray terminates (one atomic per wavefront refill), so the lanes of a
//    wavefront stay busy although rays finish after very different numbers of
//    steps;
//  * the SSP knots / coefficients and the boundary nodes of the problem are
//    staged in LDS once per workgroup;
//  * after each step, every lane reduces its step segment to a descriptor
//    (SegDesc: the receiver range / depth window it can reach and the
//    interpolation constants of the influence) and appends it to a segment
//    buffer in HBM (one atomic per wavefront).
// A second phase scatters the segments' receiver work items:
//  * k_scatter2d: one wavefront per segment, descriptor in scalar registers,
//    the 64 lanes split its receivers, FP32 atomics into the field;
//  * tiled TL path: segments are counting-sorted into receiver-range bins
//    (k_bin_count / k_bin_scan / k_bin_fill); k_scatter_tile accumulates one
//    range tile of the field in LDS and flushes it with one atomic per
//    receiver, which keeps the dense grids' atomics out of L2.
// A full segment buffer ends the pass; the host splits the ray range and
// traces the rest in further passes (the field is only written by the
// scatter, so the split leaves the result unchanged).
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include <cstdarg>
#include <string>
#include <vector>
#include <algorithm>
#include <cmath>
#include <atomic>
#include <mutex>
#include <thread>

#include "../../include/bhc_hip.h"
#include "core2d.h"
#include "devpool.h"
#include "pack2d.h"
#include "nx2d.h"
#include "pack3d.h"

using namespace bhc2d;

namespace {

thread_local std::string g_last_error;

int fail(const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return -1;
}

#define HIPCHECK(x) \
    do { \
        hipError_t _e = (x); \
        if(_e != hipSuccess) return fail("%s failed: %s (%s:%d)", #x, hipGetErrorString(_e), __FILE__, __LINE__); \
    } while(0)

constexpr int MAXN = 100000;   // include/bhc/structs.hpp:66
constexpr int WAVE = 64;

// Arrival candidate: one raw AddArr call, ordered by (ray job, step).
struct ArrCand {
    long long key;
    double a, phase, dre, dim; // full precision: AddArr compares these before rounding
    float src, rcv;             // source / receiver declination (deg)
    float srcaz, rcvaz;         // source / receiver azimuth (deg; NaN in 2D)
    int32_t ntop, nbot;
};

// Stored step segment: the descriptor plus padding to a 16-byte multiple.
template<typename real> struct alignas(16) Seg {
    SegDesc<real> d;
};

// Segment buffer layout, structure of arrays: 16-byte word k of slot s's
// descriptor at segs + (k seg_cap + s) 16, so that a wavefront's 64 lanes
// store and load consecutive words (coalesced, one 16-byte access per lane
// and word). Words below SEG_NC hold the core (every field a Cartesian TL
// scatter reads); the rest (ray-centred geometry, arrival and eigen fields)
// is stored only where seg_full. A slot takes sizeof(Seg<real>) bytes of the
// buffer in all.
template<typename real> constexpr int SEG_NC = (int)((seg_core_bytes<real>() + 15) / 16);
template<typename real> constexpr int SEG_NW = (int)((sizeof(SegDesc<real>) + 15) / 16);
// Slots whose 16-byte words all lie within a 32-bit offset of the word's row.
constexpr size_t SEG_CAP_MAX = ((size_t)1 << 28) - 1;
static_assert(SEG_NW<double> * 16 <= sizeof(Seg<double>) && SEG_NW<float> * 16 <= sizeof(Seg<float>), "slot size");
template<typename real> union SegWords {
    SegDesc<real> d;
    unsigned long long w[2 * SEG_NW<real>];
};


// Finished-ray progress of a launch (completedRayCount / totalJobs,
// src/mode/fieldimpl.cpp.in:43,62-63): wavefronts add their finished rays to
// a device counter; each time the total crosses a multiple of PROG_QUANTUM it
// is also stored (plain system-scope store, no host atomics) to the
// context's pinned host word, which bhc_progress reads while kernels run.
// Stores may land out of order; the reader keeps the largest value seen.
constexpr unsigned long long PROG_QUANTUM = 256ull;
struct Progress {
    unsigned long long *dev;    // device counter (null: not counted)
    unsigned long long *host;   // pinned host mirror
};

__device__ inline void note_done(const Progress &G, bool fin)
{
    const unsigned long long m = __ballot(fin);
    if(!m || !G.dev) return;
    if((int)(threadIdx.x & (WAVE - 1)) == __ffsll(m) - 1) {
        const unsigned long long c = (unsigned long long)__popcll(m);
        const unsigned long long old = atomicAdd(G.dev, c);
        if((old + c) / PROG_QUANTUM != old / PROG_QUANTUM)
            __hip_atomic_store(G.host, old + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

struct DevOut {
    ArrCand *cand;
    int32_t *ncand;
    int32_t cand_cap;
    bhc_eigen_hit *hits;
    int32_t *neigen;
    int32_t eigen_memsize;
    int32_t *stats;             // [njobs][3] nsteps, ntop, nbot (or null)
    double *xend;               // [njobs][2]
    bhc_ray_pt2d *points;       // ray mode
    int32_t max_points;
    const int32_t *job_alpha;   // ray mode: explicit ray list (or null)
    const int32_t *job_sz;
    const int32_t *nsteps_in;   // eigen re-trace limits (or null)
    int32_t *nsteps_out;
    unsigned long long *counters; // [0] steps, [1] contributions, [2] candidate receivers (single problems)
    uint32_t *errw;             // err, warn, nerr, nwarn
    int32_t *work;              // ray work counter (relative to job_begin)
    int32_t job_begin, job_end; // ray range of this trace pass
    int32_t lanes;              // 2D / Nx2D trace: lanes of a wavefront that take rays (fan_lanes)
    void *segs;                 // segment buffer: seg_cap descriptor cores, then seg_cap rests (seg_core / seg_rest)
    uint32_t *seg_count;
    uint32_t seg_cap;
    int32_t seg_words;          // words of a descriptor that the buffer has rows for: SEG_NW, or SEG_NC (seg_slots)
    uint32_t *overflow;
    Progress prog;
};

// First 8 bytes of 16-byte word k of slot s.
__device__ inline unsigned long long *seg_word(const DevOut &O, int k, size_t s)
{
    return reinterpret_cast<unsigned long long *>(O.segs) + 2 * ((size_t)k * O.seg_cap + s);
}
template<typename real> __device__ inline int seg_nitems(const DevOut &O, size_t s)
{
    constexpr size_t off = offsetof(SegDesc<real>, nitems);
    return reinterpret_cast<const int32_t *>(seg_word(O, (int)(off / 16), s))[(off % 16) / 4];
}
template<typename real> __device__ inline void clear_seg(const DevOut &O, size_t s)
{
    constexpr size_t off = offsetof(SegDesc<real>, nitems);
    reinterpret_cast<int32_t *>(seg_word(O, (int)(off / 16), s))[(off % 16) / 4] = 0;
}
template<typename real> __device__ inline void load_seg_words(const DevOut &O, size_t s, int k0, int k1, SegWords<real> &u)
{
#pragma unroll
    for(int k = 0; k < SEG_NW<real>; ++k)
        if(k >= k0 && k < k1) {
            const uint4 v = *reinterpret_cast<const uint4 *>(seg_word(O, k, s));
            u.w[2 * k] = (unsigned long long)v.x | ((unsigned long long)v.y << 32);
            u.w[2 * k + 1] = (unsigned long long)v.z | ((unsigned long long)v.w << 32);
        }
}
template<typename real> __device__ inline void load_seg_core(const DevOut &O, size_t s, SegDesc<real> &d)
{
    SegWords<real> u;
    load_seg_words(O, s, 0, SEG_NC<real>, u);
    __builtin_memcpy(&d, &u, seg_core_bytes<real>());
}
template<typename real> __device__ inline void load_seg_rest(const DevOut &O, size_t s, SegDesc<real> &d)
{
    SegWords<real> u;
    constexpr size_t c = seg_core_bytes<real>();
    load_seg_words(O, s, (int)(c / 16), SEG_NW<real>, u);
    __builtin_memcpy(reinterpret_cast<char *>(&d) + c, reinterpret_cast<const char *>(&u) + c,
                     sizeof(SegDesc<real>) - c);
}

template<typename real> struct DevSink {
    static constexpr bool IN_LDS = false;
    const DevOut *O;
    const Prob2D<real> *P;
    unsigned long long nc;
    __device__ void add_field(const Prob2D<real> &Pp, size_t idx, float re, float im)
    {
        unsafeAtomicAdd(Pp.field + 2 * idx, re);
        unsafeAtomicAdd(Pp.field + 2 * idx + 1, im);
    }
    __device__ void add_arrival(size_t idx, real amp, real phase, cpx<real> delay, real src, real rcv, int ntop,
                                int nbot, int ialpha, int isz, int is)
    {
        int slot = atomicAdd(O->ncand + idx, 1);
        if(slot >= O->cand_cap) return;
        int job = (P->iSingle >= 1) ? isz : isz * P->Nalpha + ialpha;
        ArrCand c;
        c.key = ((long long)job << 17) | (long long)is;
        c.a = (double)amp;
        c.phase = (double)phase;
        c.dre = (double)delay.re;
        c.dim = (double)delay.im;
        c.src = (float)src;
        c.rcv = (float)rcv;
        c.srcaz = NAN;
        c.rcvaz = NAN;
        if(P->nx_ntheta) { // Nx2D: RcvrAzimAngle = SrcAzimAngle = the bearing (influence.hpp:122-135)
            float az = (float)((RL(180.0) / RC<real>::PI) * P->base[P->o_beta + isz % P->nx_ntheta]);
            c.srcaz = az;
            c.rcvaz = az;
        }
        c.ntop = ntop;
        c.nbot = nbot;
        O->cand[idx * (size_t)O->cand_cap + slot] = c;
    }
    __device__ void add_eigen(int is, int ir, int iz, int isz, int ialpha)
    {
        int mi = atomicAdd(O->neigen, 1);
        if(mi >= O->eigen_memsize) return;
        bhc_eigen_hit h;
        h.is = is;
        h.itheta = 0;
        h.ir = ir;
        h.iz = iz;
        h.isx = 0;
        h.isy = 0;
        h.isz = isz;
        h.ialpha = ialpha;
        h.ibeta = 0;
        if(P->nx_ntheta) { // Nx2D: itheta = ibeta (influence.hpp:439) and the source indices
            int r = isz / P->nx_ntheta;
            h.itheta = h.ibeta = isz - r * P->nx_ntheta;
            h.isy = r % P->nx_nsy;
            r /= P->nx_nsy;
            h.isx = r % P->nx_nsx;
            h.isz = r / P->nx_nsx;
        }
        O->hits[mi] = h;
    }
    __device__ void count() { ++nc; }
    __device__ void mark() {}
};

__device__ inline void flush_err(const Err &e, const DevOut &O)
{
    if(e.err) atomicOr(O.errw + 0, e.err);
    if(e.warn) atomicOr(O.errw + 1, e.warn);
    if(e.nerr) atomicAdd(O.errw + 2, e.nerr);
    if(e.nwarn) atomicAdd(O.errw + 3, e.nwarn);
}

// Segment slots are reserved SEG_BLOCK at a time per wavefront (one atomic per
// block instead of one per step). Slots of a block that stay unused are marked
// empty (nitems = 0) and skipped by the scatter phase.
constexpr uint32_t SEG_BLOCK = 256;

// The same pointer, marked as global memory: after inlining, the loads and
// stores through it become global_* instructions instead of flat_* ones,
// which the compiler must also count against LDS traffic (every wait for a
// flat load then drains outstanding LDS operations and vice versa).
template<typename T> __device__ inline T *as_global(T *p)
{
    return (T *)((__attribute__((address_space(1))) T *)p);
}

struct SegBlock {
    uint32_t base, used, cap;
};

template<typename real> __device__ inline void seal_block(const SegBlock &B, int lane, const DevOut &O)
{
    for(uint32_t k = B.used + (uint32_t)lane; k < B.cap; k += WAVE) {
        uint32_t slot = B.base + k;
        if(slot < O.seg_cap) clear_seg<real>(O, slot);
    }
}

// A slot of the segment buffer for this lane (if has), called by all lanes of
// the wavefront. A slot beyond the buffer sets the overflow flag: the host
// then discards the pass and splits the ray range.
template<typename real>
__device__ inline uint32_t reserve_seg(bool has, int lane, const DevOut &O, SegBlock &B)
{
    const unsigned long long m = __ballot(has);
    if(!m) return 0xFFFFFFFFu;
    const uint32_t cnt = (uint32_t)__popcll(m);
    if(B.used + cnt > B.cap) {
        seal_block<real>(B, lane, O);
        uint32_t base = 0;
        if(lane == 0) base = atomicAdd(O.seg_count, SEG_BLOCK);
        B.base = __builtin_amdgcn_readfirstlane(__shfl(base, 0));
        B.used = 0;
        B.cap = SEG_BLOCK;
    }
    const uint32_t slot = B.base + B.used + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    B.used += cnt;
    return slot;
}

// Store a descriptor in its slot: all of it, or its core when `full` is false
// (seg_full).
template<typename real>
__device__ inline void store_seg(const SegDesc<real> &d, uint32_t slot, const DevOut &O, bool full)
{
    if(slot >= O.seg_cap) {
        atomicOr(O.overflow, 1u);
        return;
    }
    // 16-byte stores through a global-memory pointer (global_store, counted
    // apart from LDS reads; a generic store would make every later LDS wait
    // wait for it too). Word k's address is a scalar base, advanced from word
    // to word, plus the slot's 32-bit offset: the empty asm keeps the compiler
    // from holding all the words' addresses from one step to the next.
    typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(1))) char gchar;
    typedef __attribute__((address_space(1))) u64x2 gu64x2;
    SegWords<real> u;
    u.d = d;
    const uint32_t off = slot * 16u;
    const unsigned long long stride = 16ull * (uint32_t)__builtin_amdgcn_readfirstlane((int)O.seg_cap);
    const unsigned long long at = (unsigned long long)O.segs;
    unsigned long long base = (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at)
        | ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32)) << 32);
    auto store = [&](int k) {
        *(gu64x2 *)((gchar *)base + off) = u64x2{u.w[2 * k], u.w[2 * k + 1]};
        base += stride;
        asm volatile("" : "+s"(base));
    };
#pragma unroll
    for(int k = 0; k < SEG_NC<real>; ++k) store(k);
    if(full) {
#pragma unroll
        for(int k = SEG_NC<real>; k < SEG_NW<real>; ++k) store(k);
    }
}

// Exclusive prefix sum of cnt over the wavefront; returns the total.
__device__ inline int wave_excl_scan(int cnt, int lane, int &excl)
{
    int incl = cnt;
    for(int off = 1; off < WAVE; off <<= 1) {
        int v = __shfl_up(incl, off);
        if(lane >= off) incl += v;
    }
    excl = incl - cnt;
    return __shfl(incl, WAVE - 1);
}

// Lane whose [excl, excl + cnt) holds flattened index t (excl non-decreasing).
__device__ inline int wave_owner(int excl, int t)
{
    int own = 0;
    for(int b = WAVE / 2; b >= 1; b >>= 1) {
        int probe = own + b < WAVE ? own + b : WAVE - 1;
        int e = __shfl(excl, probe);
        if(own + b < WAVE && e <= t) own += b;
    }
    return own;
}

// Ray-centred rows of up to this many receivers are walked by the row's own
// lane, without the prefix sum and the search per item, where the receivers lie
// in an LDS tile (20001-beam seamount field, tile scatter: 79.5 ms, 92.5 without).
// Atomics to global memory need the flattened order, which puts neighbouring
// receivers of a row on neighbouring lanes: a row per lane touches a line of
// memory per lane (2001 beams, 201 x 1001 receivers, one wavefront per segment:
// 7.4 ms a row per lane, 2.8 flattened; 1366 x 1001: 40.4 and 15.1).
constexpr int RAYCEN_DIRECT = 6;
// Scatter one segment's receivers with the 64 lanes of a wavefront (d is
// wavefront-uniform). Both geometries have rows of different lengths --
// Cartesian range columns with their depth bands, ray-centred depths with
// their range windows -- so the items of up to 64 rows are flattened over the
// lanes: a prefix sum of the row lengths, then each lane finds the row of its
// item by a binary search over the lanes' prefix values.
template<typename real, int RT, bool FAST, typename Sink>
__device__ inline void scatter_seg(const SegDesc<real> &d, const Prob2D<real> &P, Sink &sink, int lane)
{
    if(!P.isRayCen) {
        const int nr = (d.ir1 - d.ir0) * d.dir + 1;
        for(int g = 0; g < nr; g += WAVE) {
            int ir = 0, i0 = 0, i1 = -1;
            if(g + lane < nr) cart_column(d, g + lane, P, P.base, ir, i0, i1);
            const int cnt = i1 >= i0 ? i1 - i0 + 1 : 0;
            int excl;
            const int total = wave_excl_scan(cnt, lane, excl);
            for(int t0 = 0; t0 < total; t0 += WAVE) {
                const int t = t0 + lane;
                const int own = wave_owner(excl, t);
                const int oir = __shfl(ir, own), oi0 = __shfl(i0, own), oexcl = __shfl(excl, own);
                if(t < total) item_cart_at<real, RT, Sink, FAST>(d, oir, oi0 + (t - oexcl), P, P.base, P.Rz, sink);
            }
        }
        return;
    }
    const real *Rr = P.base + P.o_Rr;
    for(int g = 0; g < d.nz; g += WAVE) {
        const int iz = d.iz0 + g + lane;
        real nA = 0, rA = 0, nB = 0, rB = 1;
        int blo = 0, bhi = -1;
        if(g + lane < d.nz && !raycen_range(d, iz, P, Rr, P.Rz, nA, rA, nB, rB, blo, bhi)) bhi = blo - 1;
        const int cnt = bhi - blo + 1;
        if constexpr(Sink::IN_LDS) {
            if(!__any(cnt > RAYCEN_DIRECT || !sink.holds(d.isz))) {
                for(int k = 0; __any(k < cnt); ++k)
                    if(k < cnt) raycen_one<real, RT, Sink, FAST>(d, blo + k, iz, nA, rA, nB, rB, P, Rr, sink);
                continue;
            }
        }
        int excl;
        const int total = wave_excl_scan(cnt, lane, excl);
        for(int t0 = 0; t0 < total; t0 += WAVE) {
            const int t = t0 + lane;
            const int own = wave_owner(excl, t);
            const real onA = __shfl(nA, own), orA = __shfl(rA, own), onB = __shfl(nB, own), orB = __shfl(rB, own);
            const int oblo = __shfl(blo, own), oexcl = __shfl(excl, own), oiz = __shfl(iz, own);
            if(t < total) raycen_one<real, RT, Sink, FAST>(d, oblo + (t - oexcl), oiz, onA, orA, onB, orB, P, Rr, sink);
        }
    }
}

// One step of the wavefront's rays (RayUpdate and both influence updates of
// the ray loop, src/trace.hpp:525-589): p0 moves to the step's end, or past the
// reflection there. step(p0, p1) (which tells the boundary it ends on: 1 top, 2
// bottom) and reflect(p0, p1, top) are the ray's own; reserve(has) is called by
// all lanes and gives the lanes with a segment its slot; out(d, slot) takes the
// descriptor. The reflected point's segment has no length on Cartesian beams
// unless the beam is shifted: its influence update then changes nothing and is
// left out. Both segments run through one copy of the code, the descriptor is
// formed where it is stored, and the reflection is made after that, so that
// descriptor, reflection and the points between are not held in registers side
// by side.
template<typename real, bool WINDOW, typename StepF, typename ReflF, typename Reserve, typename Out>
__device__ inline void step_ray(bool active, RayPt<real> &p0, Infl<real> &I, int &is, const Prob2D<real> &P,
                                const real *RzT, const real *G, int isz, int ia, StepF step, ReflF reflect,
                                Reserve reserve, Out out)
{
    RayPt<real> p1;
    bool go = active;
    int refl = 0;
    if(go) refl = step(p0, p1);
#pragma unroll 1
    for(;;) {
        SegGeo<real> g;
        real lo, hi;
        const bool has = go && seg_begin(g, p0, p1, I, P, G, lo, hi);
        const uint32_t slot = reserve(has);
        if(has) {
            SegDesc<real> d;
            d.lo = lo;
            d.hi = hi;
            seg_fill<real, WINDOW>(d, g, p0, p1, I, is, P, RzT, isz, ia);
            out(d, slot);
        }
        if(go) {
            seg_end(g, p1, I, P);
            ++is;
            p0 = p1;
            go = false;
        }
        if(refl) {
            reflect(p0, p1, refl == 1);
            refl = 0;
            go = P.isRayCen || p1.x.x != p0.x.x || p1.x.y != p0.x.y;
            if(!go) {
                ++is;
                p0 = p1;
            }
        }
        if(!__any(go)) break;
    }
}

// Receivers that a segment's descriptor brackets, about (ray-centred: its
// depths by the ranges it spans).
template<typename real> __device__ inline unsigned candidates(const SegDesc<real> &d, const Prob2D<real> &P)
{
    if(!P.isRayCen) return (unsigned)d.nitems;
    const float span = fabsf((float)(d.xb.x - d.xa.x)) / (float)P.Delta_r;
    return (unsigned)((float)d.nitems * (1.0f + fminf(span, (float)P.NRr)));
}

// Trace kernel of the field modes (TL / arrivals / eigen): the ray loop of
// MainFieldModes (src/trace.hpp:525-589). Each step's influence state update
// is done here (prelude); the receiver work goes to the segment buffer.
// STAGED: the problem's tables are read from their LDS copy, through a pointer
// the compiler knows to be LDS; else from global memory, known to be global (a
// generic pointer's loads wait for LDS and for the descriptor stores alike).
template<typename real, char ST, bool STAGED>
__global__ void __launch_bounds__(WAVE) k_trace2d(Prob2D<real> P, DevOut O)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const real *G = as_global(P.base);
    const real *B;
    if constexpr(STAGED) {
        real *L = reinterpret_cast<real *>(lds_raw);
        for(int i = threadIdx.x; i < P.staged_reals; i += WAVE) L[i] = G[i];
        __syncthreads();
        B = L;
    } else {
        B = G;
    }
    const int lane = threadIdx.x;
    const int njobs = O.job_end - O.job_begin;
    const bool full = seg_full(P);
    int32_t *const stats = as_global(O.stats);
    double *const xend = as_global(O.xend);
    Err e = {0, 0, 0, 0};
    RayPt<real> p0;
    Trace<real> S;
    Infl<real> I;
    int job = 0, isz = 0, ia = 0, is = 0;
    bool active = false, exhausted = false;
    unsigned long long steps = 0, cand = 0;
    SegBlock blk{0u, 0u, 0u};
    for(int iter = 0;; ++iter) {
        if(!exhausted) {
            const bool want = !active && lane < O.lanes;
            const unsigned long long need = __ballot(want);
            if(need) {
                const int cnt = __popcll(need);
                const int leader = __ffsll(need) - 1;
                int base = 0;
                if(lane == leader) base = atomicAdd(O.work, cnt);
                base = __shfl(base, leader);
                if(base + cnt >= njobs) exhausted = true;
                bool init_fail = false;
                const int my = base + __popcll(need & ((1ull << lane) - 1ull));
                if(want && my < njobs) {
                    job = O.job_begin + my;
                    JobIndices(job, P, isz, ia);
                    is = 0;
                    active = RayInit<real, ST>(isz, ia, p0, S, I, P, B, G, e);
                    init_fail = !active;
                    if(!active && O.stats) {
                        stats[3 * job] = 0;
                        stats[3 * job + 1] = 0;
                        stats[3 * job + 2] = 0;
                        xend[2 * job] = 0.0;
                        xend[2 * job + 1] = 0.0;
                    }
                }
                note_done(O.prog, init_fail);
            }
        }
        if(!__any(active)) {
            if(exhausted) break;
            continue;
        }
        if((iter & 31) == 31) {
            // HasErrored (src/util/errors.hpp:48-51), polled every 32 steps and
            // made wavefront-uniform so that all lanes leave together; a full
            // segment buffer ends the pass the same way.
            if(e.err) atomicOr(O.errw + 0, e.err);
            uint32_t ge = __hip_atomic_load(O.errw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t of = __hip_atomic_load(O.overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if(__any(ge != 0u || e.err != 0u || of != 0u)) {
                exhausted = true;
                active = false;
                continue;
            }
        }
        step_ray<real, true>(
            active, p0, I, is, P, B + P.o_rzs, G, isz, ia,
            [&](const RayPt<real> &a, RayPt<real> &b) { return RayStep<real, ST>(a, b, S, P, B, e); },
            [&](const RayPt<real> &a, RayPt<real> &b, bool top) { RayReflect<real, ST>(a, b, top, S, P, B, G, e); },
            [&](bool has) { return reserve_seg<real>(has, lane, O, blk); },
            [&](const SegDesc<real> &d, uint32_t slot) {
                cand += candidates(d, P);
                store_seg(d, slot, O, full);
            });
        bool fin = false;
        if(active) {
            int t = RayTerminate(p0, is, S, MAXN, P, e);
            if(t) {
                active = false;
                fin = true;
                steps += (unsigned long long)is;
                if(O.stats) {
                    stats[3 * job] = is;
                    stats[3 * job + 1] = p0.NumTopBnc;
                    stats[3 * job + 2] = p0.NumBotBnc;
                    xend[2 * job] = (double)p0.x.x;
                    xend[2 * job + 1] = (double)p0.x.y;
                }
            }
        }
        note_done(O.prog, fin);
    }
    seal_block<real>(blk, lane, O);
    flush_err(e, O);
    for(int off = WAVE / 2; off > 0; off >>= 1) {
        steps += __shfl_xor(steps, off);
        cand += __shfl_xor(cand, off);
    }
    if(lane == 0) {
        atomicAdd(O.counters + 0, steps);
        atomicAdd(O.counters + 2, cand);
    }
}

// Scatter kernel: one wavefront per segment; the descriptor is wavefront-
// uniform (scalar loads) and the 64 lanes split its receiver work items
// (influence.hpp:1075-1187 ray-centred depths, :1298-1386 Cartesian ranges x
// depths).
template<typename real, int RT, bool FAST>
__global__ void __launch_bounds__(256) k_scatter2d(Prob2D<real> P, DevOut O)
{
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE));
    const int nwaves = gridDim.x * (blockDim.x / WAVE);
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    DevSink<real> sink{&O, &P, 0};
    for(uint32_t s = (uint32_t)wave; s < n; s += (uint32_t)nwaves) {
        SegDesc<real> d;
        load_seg_core(O, s, d);
        if(d.nitems <= 0) continue;
        if(seg_full(P)) load_seg_rest(O, s, d);
        scatter_seg<real, RT, FAST>(d, P, sink, lane);
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) sink.nc += __shfl_xor(sink.nc, off);
    if(lane == 0 && sink.nc) atomicAdd(O.counters + 1, sink.nc);
}

// ---------------------------------------------------------------------------
// Range-binned TL scatter with an LDS field tile.
//
// Segments are counting-sorted by the receiver-range column at their centre
// (bins of BIN_W columns). A workgroup takes a chunk of one bin and keeps the
// complex field of TILE_W columns around the bin (all NRz_per_range depths) in
// LDS; contributions inside the tile are added with LDS atomics, the rest go
// straight to the global field, and the tile is flushed once at the end. With
// ~10^3 contributions per receiver per field, this removes almost all global
// atomics.
// ---------------------------------------------------------------------------
// Single-problem scatter with one lane per segment (segments with few
// receivers each: hat beams on coarse depth windows).
template<typename real, int RT, bool FAST>
__global__ void __launch_bounds__(256) k_scatter2d_lanes(Prob2D<real> P, DevOut O)
{
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    DevSink<real> sink{&O, &P, 0};
    const uint32_t stride = gridDim.x * blockDim.x;
    for(uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += stride) {
        SegDesc<real> d;
        load_seg_core(O, s, d);
        if(d.nitems <= 0) continue;
        if(seg_full(P)) load_seg_rest(O, s, d);
        seg_items<real, RT, DevSink<real>, FAST>(d, P, P.base, P.Rz, sink);
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) sink.nc += __shfl_xor(sink.nc, off);
    if((threadIdx.x & (WAVE - 1)) == 0 && sink.nc) atomicAdd(O.counters + 1, sink.nc);
}

enum : int { SCATTER_AUTO = 0, SCATTER_TILED = 1, SCATTER_WAVE = 2, SCATTER_LANES = 3 };

struct BinCfg {
    int32_t nbins;              // range bins of one source; source isz's bins are isz nbins ..
    int32_t nsrc;               // sources with bins of their own; source isz from nsrc on goes into isz % nsrc's
    int32_t total;              // nbins nsrc
    int32_t bin_w, tile_w, tile_lo_off; // tile columns of range bin b = [b*bin_w - tile_lo_off, + tile_w)
    int32_t chunk;              // segments per workgroup
    int32_t *counts, *offsets, *cursor;
    int32_t *chunk_bin, *chunk_pos; // per chunk: its bin and its first position in idx
    uint32_t *idx;
    int32_t *nchunks;
};

template<typename real> __device__ inline int seg_bin(const SegDesc<real> &d, const Prob2D<real> &P, const BinCfg &C)
{
    int col;
    if(P.isRayCen) {
        double c = 0.5 * ((double)d.xb.x + (d.lastValid ? (double)d.xa.x : (double)d.xb.x));
        double t = (c - (double)P.base[P.o_Rr]) / (double)P.Delta_r;
        t = t < -1.0 ? -1.0 : (t > (double)P.NRr ? (double)P.NRr : t);
        col = (int)t;
    } else {
        col = (d.ir0 + d.ir1) / 2;
    }
    col = imax(0, imin(col, P.NRr - 1));
    return (d.isz < C.nsrc ? d.isz : d.isz % C.nsrc) * C.nbins + imin(col / C.bin_w, C.nbins - 1);
}

// The bin of stored segment s (its rest read for ray-centred segments only).
template<typename real> __device__ inline int seg_bin_at(const DevOut &O, size_t s, const Prob2D<real> &P, const BinCfg &C)
{
    SegDesc<real> d;
    load_seg_core(O, s, d);
    if(P.isRayCen) load_seg_rest(O, s, d);
    return seg_bin(d, P, C);
}

// Bin histogram: each workgroup owns a contiguous slice of the segments and
// counts it in LDS first (one global atomic per bin per workgroup).
template<typename real> __global__ void __launch_bounds__(256) k_bin_count(Prob2D<real> P, DevOut O, BinCfg C)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    int32_t *h = reinterpret_cast<int32_t *>(lds_raw);
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    uint32_t per = (n + gridDim.x - 1) / gridDim.x;
    uint32_t s0 = blockIdx.x * per, s1 = min(n, s0 + per);
    for(int b = threadIdx.x; b < C.total; b += blockDim.x) h[b] = 0;
    __syncthreads();
    for(uint32_t s = s0 + threadIdx.x; s < s1; s += blockDim.x)
        if(seg_nitems<real>(O, s) > 0) atomicAdd(h + seg_bin_at(O, s, P, C), 1);
    __syncthreads();
    for(int b = threadIdx.x; b < C.total; b += blockDim.x)
        if(h[b]) atomicAdd(C.counts + b, h[b]);
}

// Exclusive scan of the bin counts and of the per-bin chunk counts (one workgroup).
__global__ void __launch_bounds__(1024) k_bin_scan(BinCfg C)
{
    __shared__ int32_t wave_s[16], wave_c[16];
    const int t = threadIdx.x, lane = t & (WAVE - 1), w = t / WAVE, nb = C.total;
    const int per = (nb + 1023) / 1024;
    const int b0 = min(nb, t * per), b1 = min(nb, b0 + per);
    int ss = 0, sc = 0;
    for(int b = b0; b < b1; ++b) {
        ss += C.counts[b];
        sc += (C.counts[b] + C.chunk - 1) / C.chunk;
    }
    int is = ss, ic = sc; // inclusive over the wavefront
    for(int o = 1; o < WAVE; o <<= 1) {
        const int a = __shfl_up(is, o), c = __shfl_up(ic, o);
        if(lane >= o) {
            is += a;
            ic += c;
        }
    }
    if(lane == WAVE - 1) {
        wave_s[w] = is;
        wave_c[w] = ic;
    }
    __syncthreads();
    int ps = is - ss, pc = ic - sc;
    for(int k = 0; k < w; ++k) {
        ps += wave_s[k];
        pc += wave_c[k];
    }
    if(t == 1023) *C.nchunks = pc + sc;
    for(int b = b0; b < b1; ++b) {
        C.offsets[b] = ps;
        C.cursor[b] = ps;
        const int nc = (C.counts[b] + C.chunk - 1) / C.chunk;
        for(int k = 0; k < nc; ++k) {
            C.chunk_bin[pc + k] = b;
            C.chunk_pos[pc + k] = ps + k * C.chunk;
        }
        ps += C.counts[b];
        pc += nc;
    }
}

// Bin fill with the same slicing as k_bin_count: the workgroup reserves its
// range in every bin with one global atomic, then ranks its segments in LDS.
template<typename real> __global__ void __launch_bounds__(256) k_bin_fill(Prob2D<real> P, DevOut O, BinCfg C)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    int32_t *h = reinterpret_cast<int32_t *>(lds_raw);
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    uint32_t per = (n + gridDim.x - 1) / gridDim.x;
    uint32_t s0 = blockIdx.x * per, s1 = min(n, s0 + per);
    for(int b = threadIdx.x; b < C.total; b += blockDim.x) h[b] = 0;
    __syncthreads();
    for(uint32_t s = s0 + threadIdx.x; s < s1; s += blockDim.x)
        if(seg_nitems<real>(O, s) > 0) atomicAdd(h + seg_bin_at(O, s, P, C), 1);
    __syncthreads();
    for(int b = threadIdx.x; b < C.total; b += blockDim.x)
        if(h[b]) h[b] = atomicAdd(C.cursor + b, h[b]);
    __syncthreads();
    for(uint32_t s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
        if(seg_nitems<real>(O, s) <= 0) continue;
        int pos = atomicAdd(h + seg_bin_at(O, s, P, C), 1);
        C.idx[pos] = s;
    }
}

template<typename real> struct TileSink {
    static constexpr bool IN_LDS = true;
    float *tile;          // LDS [tile_w][nz] complex, of source isz0
    int col0, tile_w, nz, nrr, isz0;
    unsigned long long nc;
    // (the cell, not its index: an index would have to be divided back into
    // range and depth, several hundred instructions of 64-bit division)
    __device__ bool holds(int isz) const { return isz == isz0; }
    __device__ void add_cell(const Prob2D<real> &Pp, int isz, int iz, int ir, float re, float im)
    {
        const int c = ir - col0;
        if(c >= 0 && c < tile_w && isz == isz0) {
            int k = c * nz + iz; // real parts first, then imaginary parts (bank-conflict free)
            atomicAdd(tile + k, re);
            atomicAdd(tile + tile_w * nz + k, im);
        } else {
            const size_t idx = ((size_t)isz * nz + iz) * nrr + ir;
            unsafeAtomicAdd(Pp.field + 2 * idx, re);
            unsafeAtomicAdd(Pp.field + 2 * idx + 1, im);
        }
    }
    template<typename R2> __device__ void add_arrival(size_t, R2, R2, cpx<R2>, R2, R2, int, int, int, int, int) {}
    __device__ void add_eigen(int, int, int, int, int) {}
    __device__ void count() { ++nc; }
    __device__ void mark() {}
};

// One workgroup per chunk of a (source, range) bin (a source without bins of its
// own shares another's and adds to global memory), one wavefront per segment
// at a time. Latency bounds it (on the 20001-ray seamount field the SIMDs
// issue vector instructions in 45 % of their cycles), so the wavefront's next
// descriptor is on its way while it works on the current one: 64 segment
// numbers are read at a time, lane k loads word k of the next descriptor (one
// load instruction for all its words), and the words reach every lane through
// LDS.
constexpr int TILE_THREADS = 512;
constexpr int TILE_STAGE = (TILE_THREADS / WAVE) * SEG_NW<double> * 16; // bytes beside the tile

template<typename real, bool FAST>
__global__ void __launch_bounds__(TILE_THREADS, 4) k_scatter_tile(Prob2D<real> P, DevOut O, BinCfg C)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ uint4 stage_all[TILE_THREADS / WAVE][SEG_NW<real>];
    float *tile = reinterpret_cast<float *>(lds_raw);
    const int nchunks = *C.nchunks;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int nw = blockDim.x / WAVE;
    const int nz = P.NRz_per_range;
    const int words = seg_full(P) ? SEG_NW<real> : SEG_NC<real>;
    uint4 *stage = stage_all[wave];
    unsigned long long total = 0;
    for(int ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
        const int b = C.chunk_bin[ch], k0 = C.chunk_pos[ch];
        const int k1 = min(C.offsets[b] + C.counts[b], k0 + C.chunk);
        const int isz = b / C.nbins;
        const int col0 = (b - isz * C.nbins) * C.bin_w - C.tile_lo_off;
        const int ncol = C.tile_w;
        for(int i = threadIdx.x; i < 2 * ncol * nz; i += blockDim.x) tile[i] = 0.f;
        __syncthreads();
        TileSink<real> sink{tile, col0, ncol, nz, P.NRr, isz, 0};
        // this wavefront's segments: positions k0 + wave, + nw, ...
        const int mine = k1 - k0 - wave > 0 ? (k1 - k0 - wave + nw - 1) / nw : 0;
        uint32_t nums = 0;
        uint4 next = make_uint4(0u, 0u, 0u, 0u);
        auto fetch = [&](int j) { // the words of segment j, one per lane
            if((j & (WAVE - 1)) == 0) nums = C.idx[k0 + wave + nw * min(j + lane, mine - 1)];
            const uint32_t si = (uint32_t)__builtin_amdgcn_readlane((int)nums, j & (WAVE - 1));
            if(lane < words) next = *reinterpret_cast<const uint4 *>(seg_word(O, lane, si));
        };
        if(mine > 0) fetch(0);
        for(int j = 0; j < mine; ++j) {
            if(lane < words) stage[lane] = next;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            SegWords<real> u;
            if(words == SEG_NW<real>) __builtin_memcpy(&u, stage, SEG_NW<real> * 16);
            else __builtin_memcpy(&u, stage, SEG_NC<real> * 16);
            if(j + 1 < mine) fetch(j + 1);
            scatter_seg<real, RT_TL, FAST>(u.d, P, sink, lane);
            // the stage is rewritten for the next segment
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        __syncthreads();
        // flush: tile column c, depth iz -> the source's field
        float *field = P.field + 2 * (size_t)isz * nz * P.NRr;
        for(int i = threadIdx.x; i < ncol * nz; i += blockDim.x) {
            int c = i / nz, iz = i - c * nz;
            int ir = col0 + c;
            if(ir < 0 || ir >= P.NRr) continue;
            float re = tile[i], im = tile[ncol * nz + i];
            if(re != 0.f || im != 0.f) {
                size_t idx = (size_t)iz * P.NRr + ir;
                unsafeAtomicAdd(field + 2 * idx, re);
                unsafeAtomicAdd(field + 2 * idx + 1, im);
            }
        }
        __syncthreads();
        total += sink.nc;
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) total += __shfl_xor(total, off);
    if(lane == 0 && total) atomicAdd(O.counters + 1, total);
}

template<typename real> __device__ inline void store_pt(bhc_ray_pt2d *d, const RayPt<real> &s)
{
    bhc_ray_pt2d r;
    r.p[0] = s.p.x;
    r.p[1] = s.p.y;
    r.q[0] = s.q.x;
    r.q[1] = s.q.y;
    r.NumTopBnc = s.NumTopBnc;
    r.NumBotBnc = s.NumBotBnc;
    r.x[0] = s.x.x;
    r.x[1] = s.x.y;
    r.t[0] = s.t.x;
    r.t[1] = s.t.y;
    r.c = s.c;
    r.Amp = s.Amp;
    r.Phase = s.Phase;
    r.tau[0] = s.tau.re;
    r.tau[1] = s.tau.im;
    *d = r;
}

// Ray run type and eigenray re-trace: MainRayMode, src/trace.hpp:482-520.
// Bound by the serial chain of a ray's steps. A plot's few rays are spread over
// the wavefronts (O.lanes, as the field trace's), and the tables are read as
// there (STAGED, ST): 101 rays of a
// Munk fan with all their points, the call from 4.6 to 3.3 ms.
template<typename real, char ST, bool STAGED>
__global__ void __launch_bounds__(WAVE) k_ray2d(Prob2D<real> P, DevOut O)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const real *G = as_global(P.base);
    const real *B;
    if constexpr(STAGED) {
        real *L = reinterpret_cast<real *>(lds_raw);
        for(int i = threadIdx.x; i < P.staged_reals; i += WAVE) L[i] = G[i];
        __syncthreads();
        B = L;
    } else {
        B = G;
    }
    bhc_ray_pt2d *const points = as_global(O.points);
    const int first = threadIdx.x < O.lanes ? (int)(blockIdx.x * O.lanes + threadIdx.x) : O.job_end;
    Err e = {0, 0, 0, 0};
    const int M = O.max_points;
    for(int job = first; job < O.job_end; job += gridDim.x * O.lanes) {
        int isz, ia;
        if(O.job_alpha) {
            ia = O.job_alpha[job];
            isz = O.job_sz[job];
        } else {
            JobIndices(job, P, isz, ia);
        }
        bhc_ray_pt2d *ray = points + (size_t)job * M;
        RayPt<real> p0, p1, p2;
        Trace<real> S;
        Infl<real> I;
        int Nsteps = O.nsteps_in ? O.nsteps_in[job] : -1;
        bool ok = RayInit<real, ST>(isz, ia, p0, S, I, P, B, G, e);
        store_pt(ray, p0);
        if(!ok) {
            O.nsteps_out[job] = 1;
            continue;
        }
        int is = 0;
        for(;;) {
            if(e.err) break;
            bool two = RayUpdate<real, ST>(p0, p1, p2, S, P, B, G, e);
            store_pt(ray + is + 1, p1);
            if(two) store_pt(ray + is + 2, p2);
            if(Nsteps >= 0 && is >= Nsteps) {
                Nsteps = is + 2;
                break;
            }
            is += two ? 2 : 1;
            p0 = two ? p2 : p1;
            int t = RayTerminate(p0, is, S, M, P, e);
            if(t == 1) {
                Nsteps = is + 1;
                break;
            }
            if(t == 2) {
                Nsteps = is;
                break;
            }
        }
        O.nsteps_out[job] = Nsteps;
    }
    flush_err(e, O);
}

// Nx2D trace kernel: the ray loop of MainFieldModes (src/trace.hpp:525-589)
// with O3D && !R3D -- rays on the bearing planes of a 3D environment (nx2d.h),
// influence state and segment descriptors of the 2D beams, so that the 2D
// scatter kernels apply the receivers of every bearing plane. One wavefront
// per workgroup; the 3D environment stays in global memory (L2-resident).
template<typename real>
__global__ void __launch_bounds__(64) k_tracenx2d(Prob2D<real> P, bhc3d::Prob3D<real> N, DevOut O)
{
    using bhc3d::OrgNx;
    using bhc3d::Trace3;
    __shared__ real refl_lds[768];  // the reflection tables in LDS when they fit
    const real *tabs = bhc3d::stage_refl_tables(N, refl_lds, 768);
    const real *G = P.base;
    const int lane = threadIdx.x & (WAVE - 1);
    const int njobs = O.job_end - O.job_begin;
    Err e = {0, 0, 0, 0};
    RayPt<real> p0;
    Trace3<real> S;
    OrgNx<real> org;
    Infl<real> I;
    int job = 0, isf = 0, ia = 0, is = 0;
    const bool full = seg_full(P);
    bool active = false, exhausted = false, init_fail = false;
    unsigned long long steps = 0, cand = 0;
    SegBlock blk{0u, 0u, 0u};
    for(int iter = 0;; ++iter) {
        if(!exhausted) {
            const bool want = !active && lane < O.lanes;
            unsigned long long need = __ballot(want);
            if(need) {
                int cnt = __popcll(need);
                int leader = __ffsll((unsigned long long)need) - 1;
                int base = 0;
                if(lane == leader) base = atomicAdd(O.work, cnt);
                base = __shfl(base, leader);
                if(base + cnt >= njobs) exhausted = true;
                if(want) {
                    int my = base + __popcll(need & ((1ull << lane) - 1ull));
                    if(my < njobs) {
                        job = O.job_begin + my;
                        int ib, isx, isy, isz;
                        isf = bhc3d::JobIndicesNx(job, N, ia, ib, isx, isy, isz);
                        is = 0;
                        active = bhc3d::RayInitNx(ia, ib, isx, isy, isz, p0, S, org, I, P, N, e);
                        init_fail = !active;
                        if(!active && O.stats) {
                            O.stats[3 * job] = O.stats[3 * job + 1] = O.stats[3 * job + 2] = 0;
                            O.xend[3 * job] = O.xend[3 * job + 1] = O.xend[3 * job + 2] = 0.0;
                        }
                    }
                }
                note_done(O.prog, init_fail);
                init_fail = false;
            }
        }
        if(!__any(active)) {
            if(exhausted) break;
            continue;
        }
        if((iter & 31) == 31) {
            // HasErrored (src/util/errors.hpp:48-51) and a full segment buffer
            // end the pass for the whole wavefront
            if(e.err) atomicOr(O.errw + 0, e.err);
            uint32_t ge = __hip_atomic_load(O.errw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t of = __hip_atomic_load(O.overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if(__any(ge != 0u || e.err != 0u || of != 0u)) {
                exhausted = true;
                active = false;
                continue;
            }
        }
        step_ray<real, true>(
            active, p0, I, is, P, G + P.o_rzs, G, isf, ia,
            [&](const RayPt<real> &a, RayPt<real> &b) { return bhc3d::RayStepNx(a, b, S, org, N, e); },
            [&](const RayPt<real> &a, RayPt<real> &b, bool top) { bhc3d::RayReflectNx(a, b, top, S, org, N, P, e, tabs); },
            [&](bool has) { return reserve_seg<real>(has, lane, O, blk); },
            [&](const SegDesc<real> &d, uint32_t slot) {
                cand += candidates(d, P);
                store_seg(d, slot, O, full);
            });
        bool fin = false;
        if(active) {
            if(bhc3d::RayTerminateNx(p0, is, S, org, N, e, MAXN)) {
                active = false;
                fin = true;
                steps += (unsigned long long)is;
                if(O.stats) {
                    const bhc3d::v3<real> xe = bhc3d::RayToOceanX(p0.x, org);
                    O.stats[3 * job] = is;
                    O.stats[3 * job + 1] = p0.NumTopBnc;
                    O.stats[3 * job + 2] = p0.NumBotBnc;
                    O.xend[3 * job] = (double)xe.x;
                    O.xend[3 * job + 1] = (double)xe.y;
                    O.xend[3 * job + 2] = (double)xe.z;
                }
            }
        }
        note_done(O.prog, fin);
    }
    seal_block<real>(blk, lane, O);
    flush_err(e, O);
    for(int off = WAVE / 2; off > 0; off >>= 1) {
        steps += __shfl_xor(steps, off);
        cand += __shfl_xor(cand, off);
    }
    if(lane == 0) {
        atomicAdd(O.counters + 0, steps);
        atomicAdd(O.counters + 2, cand);
    }
}

// Nx2D ray run type: MainRayMode (src/trace.hpp:482-520) with O3D && !R3D.
// Points are in ray coordinates (range along the bearing, depth); org_out
// gets each ray's origin (xs.x, xs.y, cos beta, sin beta).
template<typename real>
__global__ void __launch_bounds__(256) k_raynx2d(Prob2D<real> P, bhc3d::Prob3D<real> N, DevOut O, double *org_out)
{
    Err e = {0, 0, 0, 0};
    const int M = O.max_points;
    for(int job = blockIdx.x * blockDim.x + threadIdx.x; job < O.job_end; job += gridDim.x * blockDim.x) {
        int ia, ib, isx, isy, isz;
        bhc3d::JobIndicesNx(job, N, ia, ib, isx, isy, isz);
        bhc_ray_pt2d *ray = O.points + (size_t)job * M;
        RayPt<real> p0, p1, p2;
        bhc3d::Trace3<real> S;
        bhc3d::OrgNx<real> org;
        Infl<real> I;
        int Nsteps = -1;
        bool ok = bhc3d::RayInitNx(ia, ib, isx, isy, isz, p0, S, org, I, P, N, e);
        store_pt(ray, p0);
        org_out[4 * job] = (double)org.xs.x;
        org_out[4 * job + 1] = (double)org.xs.y;
        org_out[4 * job + 2] = (double)org.tr.x;
        org_out[4 * job + 3] = (double)org.tr.y;
        if(!ok) {
            O.nsteps_out[job] = 1;
            continue;
        }
        int is = 0;
        for(;;) {
            if(e.err) break;
            bool two = bhc3d::RayUpdateNx(p0, p1, p2, S, org, N, P, e);
            store_pt(ray + is + 1, p1);
            if(two) store_pt(ray + is + 2, p2);
            is += two ? 2 : 1;
            p0 = two ? p2 : p1;
            int t = bhc3d::RayTerminateNx(p0, is, S, org, N, e, M);
            if(t == 1) {
                Nsteps = is + 1;
                break;
            }
            if(t == 2) {
                Nsteps = is;
                break;
            }
        }
        O.nsteps_out[job] = Nsteps;
    }
    flush_err(e, O);
}

// Deterministic arrivals: one thread per receiver sorts its candidates by
// (ray, step) -- the order of the reference's single-threaded run -- and
// replays AddArr (src/arrivals.hpp:45-130) on them.
__global__ void __launch_bounds__(256) k_arr_merge(const ArrCand *cand, const int32_t *ncand, int cand_cap,
                                                   bhc_arrival *arr, int32_t *narr, int max_narr, int nrcv,
                                                   int allow_merging, float omega_f, double omega_d, int fp64,
                                                   uint32_t *errw)
{
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if(r >= nrcv) return;
    int n = ncand[r];
    if(n > cand_cap) {
        atomicOr(errw + 1, 1u << BHC_WARN_RAYS_OUTOFMEMORY);
        atomicAdd(errw + 3, 1u);
        n = cand_cap;
    }
    ArrCand *c = const_cast<ArrCand *>(cand) + (size_t)r * cand_cap;
    // insertion sort: candidates arrive nearly sorted (rays are handed out in order)
    for(int i = 1; i < n; ++i) {
        ArrCand v = c[i];
        int j = i - 1;
        while(j >= 0 && c[j].key > v.key) {
            c[j + 1] = c[j];
            --j;
        }
        c[j + 1] = v;
    }
    bhc_arrival *A = arr + (size_t)r * max_narr;
    int Nt = 0;
    for(int i = 0; i < n; ++i) {
        const ArrCand &v = c[i];
        if(!allow_merging) {
            if(Nt >= max_narr) break;
            bhc_arrival &a = A[Nt++];
            a.a = (float)v.a;
            a.Phase = (float)v.phase;
            a.delay[0] = (float)v.dre;
            a.delay[1] = (float)v.dim;
            a.SrcDeclAngle = v.src;
            a.SrcAzimAngle = v.srcaz;
            a.RcvrDeclAngle = v.rcv;
            a.RcvrAzimAngle = v.rcvaz;
            a.NTopBnc = v.ntop;
            a.NBotBnc = v.nbot;
            continue;
        }
        // IsSecondStepOfPair, arrivals.hpp:31-39, in the run's real type
        bool second = false;
        if(Nt >= 1) {
            const float PhaseTol = 0.05f;
            const bhc_arrival &b = A[Nt - 1];
            if(fp64) {
                double dr = v.dre - (double)b.delay[0], di = v.dim - (double)b.delay[1];
                second = omega_d * hypot(dr, di) < (double)PhaseTol
                    && fabs((double)b.Phase - v.phase) < (double)PhaseTol;
            } else {
                float dr = (float)v.dre - b.delay[0], di = (float)v.dim - b.delay[1];
                second = omega_f * hypotf(dr, di) < PhaseTol && fabsf(b.Phase - (float)v.phase) < PhaseTol;
            }
        }
        if(!second) {
            int iArr;
            if(Nt >= max_narr) {
                iArr = -1;
                double weakest = v.a;
                for(int k = 0; k < max_narr; ++k)
                    if((double)A[k].a < weakest) {
                        weakest = A[k].a;
                        iArr = k;
                    }
                if(iArr < 0) continue;
            } else {
                iArr = Nt++;
            }
            bhc_arrival &a = A[iArr];
            a.a = (float)v.a;
            a.Phase = (float)v.phase;
            a.delay[0] = (float)v.dre;
            a.delay[1] = (float)v.dim;
            a.SrcDeclAngle = v.src;
            a.SrcAzimAngle = v.srcaz;
            a.RcvrDeclAngle = v.rcv;
            a.RcvrAzimAngle = v.rcvaz;
            a.NTopBnc = v.ntop;
            a.NBotBnc = v.nbot;
        } else {
            bhc_arrival &a = A[Nt - 1];
            float amp = (float)v.a;
            float AmpTot = a.a + amp;
            float w1 = a.a / AmpTot, w2 = amp / AmpTot;
            a.delay[0] = w1 * a.delay[0] + w2 * (float)v.dre;
            a.delay[1] = w1 * a.delay[1] + w2 * (float)v.dim;
            a.a = AmpTot;
            a.SrcDeclAngle = w1 * a.SrcDeclAngle + w2 * v.src;
            a.SrcAzimAngle = w1 * a.SrcAzimAngle + w2 * v.srcaz;
            a.RcvrDeclAngle = w1 * a.RcvrDeclAngle + w2 * v.rcv;
            a.RcvrAzimAngle = w1 * a.RcvrAzimAngle + w2 * v.rcvaz;
        }
    }
    narr[r] = Nt;
}

} // namespace

// ===========================================================================
// Host side of the C ABI
// ===========================================================================

// Device blocks of a context that its problems and runs gave back, for the
// next ones: a run allocates a dozen arrays, among them the arrivals'
// candidate slots (up to 16 GiB, for which hipMalloc waits until the driver
// has cleared as much memory: 249 ms for a 2121-receiver run whose kernels
// take 7 ms, 4 ms when cleared memory was at hand). At most BHC_POOL_MB
// (default 20 GiB) are kept; bhc_ctx_trim and destroying the context give them
// back to the device, and an allocation of the library that finds no memory
// first gives back those of every context. A block is put here only after the
// context's stream has been waited for, so an idle block is in no one's use.
constexpr size_t POOL_MB = 20480;
void bhc_give_back_pools();

// hipMalloc that gives the pools back before it gives up
hipError_t bhc_device_malloc(void **p, size_t n)
{
    hipError_t e = hipMalloc(p, n);
    if(e == hipSuccess) return e;
    (void)hipGetLastError();
    bhc_give_back_pools();
    return hipMalloc(p, n);
}

struct DevMem {
    static int alloc(void **p, size_t n) { return (int)bhc_device_malloc(p, n); }
    static void free(void *p) { (void)hipFree(p); }
};
struct DevPool;
std::mutex g_pools_mu;
std::vector<DevPool *> g_pools;                     // of every context
struct DevPool : BlockPool<DevMem> {
    DevPool() : BlockPool<DevMem>(POOL_MB << 20)
    {
        std::lock_guard<std::mutex> lk(g_pools_mu);
        g_pools.push_back(this);
    }
    ~DevPool()
    {
        std::lock_guard<std::mutex> lk(g_pools_mu);
        g_pools.erase(std::find(g_pools.begin(), g_pools.end(), this));
    }
};

void bhc_give_back_pools()
{
    std::lock_guard<std::mutex> lk(g_pools_mu);
    for(DevPool *p : g_pools) p->trim();
}

struct bhc_ctx {
    int device;
    hipStream_t stream;
    hipEvent_t ev0, ev1, evm;   // start, end, trace/scatter boundary of the first pass
    hipEvent_t pa, pb;          // per-pass phase brackets
    double ph_trace_ms, ph_scatter_ms; // trace / scatter kernel time summed over the last run's passes
    int num_cus;
    int lds_max;
    int tpb, bpc;
    char name[256];
    // segment buffer shared by all problems of the context (grown on demand)
    void *segs;
    size_t seg_bytes;
    uint32_t *d_seg_count, *d_overflow;
    uint32_t *d_bin_idx;        // binned segment order (seg capacity entries)
    int passes;                 // trace/scatter passes of the last launch
    int use_tiles;              // 0 disables the LDS-tiled TL scatter
    int exact_phasor;           // 1: TL phasor in the reference's full arithmetic
    size_t seg_mb;              // segment buffer size (MiB), allocated at first use
    double seg_per_ray3;        // 3D runs: largest segments-per-ray seen (sizes the first pass)
    int scatter3_map;           // 3D scatter mapping: 0 one wavefront per segment, 1 one lane per segment,
                                // 2 (default) segment groups flattened per wavefront
    // finished-ray progress of the current or last run (bhc_progress)
    unsigned long long *h_prog; // pinned, device-visible host word written by the trace kernels
    unsigned long long *d_prog; // device counter
    std::atomic<long long> prog_total{0}, prog_seen{0};
    std::atomic<int> prog_final{0};
    // non-blocking runs: one worker thread at a time per context
    std::thread worker;
    std::atomic<int> busy{0};
    int async_rc = 0;
    std::string async_msg;
    // device address of the static scratch array on this context's device
    void *scratch = nullptr;
    DevPool pool;
};

namespace {
// set on a context's worker thread: the run it performs may use the context
thread_local bool tl_async_worker = false;

// Entry points that use a context refuse while a non-blocking run holds it.
int check_idle(bhc_ctx *c, const char *who)
{
    if(!c) return fail("%s: null context", who);
    if(c->busy.load() && !tl_async_worker) return fail("%s: a non-blocking run is in flight on this context", who);
    return 0;
}

// Start of a run of `total` rays: the host word now, the device counter on the
// stream ahead of the run's kernels.
int prog_begin(bhc_ctx *c, long long total)
{
    c->prog_final = 0;
    c->prog_seen = 0;
    c->prog_total = total;
    __atomic_store_n(c->h_prog, 0ull, __ATOMIC_RELAXED);
    HIPCHECK(hipMemsetAsync(c->d_prog, 0, sizeof(unsigned long long), c->stream));
    return 0;
}

Progress prog_of(bhc_ctx *c) { return Progress{c->d_prog, c->h_prog}; }
} // namespace

struct bhc_dev_problem {
    bhc_ctx *ctx;
    int precision;
    char run0;
    int njobs, NSz, NRz_per_range, NRr;
    size_t nrcv;
    void *d_blob;
    float *d_Rz, *d_Sz;
    Prob2D<double> P64;
    Prob2D<float> P32;
    size_t lds_bytes;
    float *d_field;
    ArrCand *d_cand;
    int32_t *d_ncand;
    int cand_cap;
    bhc_arrival *d_arr;
    int32_t *d_narr;
    int max_narr, allow_merging;
    bhc_eigen_hit *d_hits;
    int32_t *d_neigen;
    int eigen_memsize;
    int32_t *d_stats;
    double *d_xend;
    unsigned long long *d_counters;
    uint32_t *d_errw;
    int32_t *d_work;
    int cleared;                // the outputs hold zeros or a launch's results (clear_outputs)
    double freq0;
    // range bins of the tiled TL scatter
    int nbins, bin_sources, total_bins, bin_w, tile_w, tile_lo_off, chunk, max_chunks;
    int scatter_mode;           // SCATTER_AUTO / _TILED / _WAVE / _LANES
    int32_t *d_bins;            // counts | offsets | cursor | chunk_start | nchunks
    // Nx2D runs: the 3D environment the trace kernel reads (P64 / P32 then view
    // the same blob as the receiver side), and 3 reals per ray end point
    int nx2d, xend_dim;
    bhc3d::Prob3D<double> N64;
    bhc3d::Prob3D<float> N32;
};

extern "C" const char *bhc_last_error(void) { return g_last_error.c_str(); }

extern "C" int bhc_device_info(int device, char *name, int name_len, int *num_cus, int *lds_bytes)
{
    hipDeviceProp_t prop;
    HIPCHECK(hipGetDeviceProperties(&prop, device));
    if(name && name_len > 0) snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    if(num_cus) *num_cus = prop.multiProcessorCount;
    if(lds_bytes) *lds_bytes = (int)prop.sharedMemPerBlock;
    return 0;
}

// Segment buffer of bhc_field_launch_noalloc: a file-scope device array, so
// that launch allocates nothing. Every GPU the library runs on holds its own
// copy until the process ends. In host code the array's name is not a device
// address: host code uses only the address hipGetSymbolAddress returns for
// the current device (kept per device, and in each context).
constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[MAX_DEVICES];

// Address of `scratch` on `device` (which must be current), looked up once.
int scratch_address(int device, void **ptr)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if(device < 0 || device >= MAX_DEVICES) return fail("scratch: device %d out of range", device);
    if(!g_scratch_ptr[device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if(e != hipSuccess || !p) return fail("scratch: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
        g_scratch_ptr[device] = p;
    }
    *ptr = g_scratch_ptr[device];
    return 0;
}
} // namespace

extern "C" int bhc_ctx_create(int device, bhc_ctx **out)
{
    *out = nullptr;
    int n = 0;
    HIPCHECK(hipGetDeviceCount(&n));
    if(device < 0 || device >= n) return fail("bhc_ctx_create: device %d not present (%d devices)", device, n);
    HIPCHECK(hipSetDevice(device));
    bhc_ctx *c = new bhc_ctx();
    c->device = device;
    hipDeviceProp_t prop;
    HIPCHECK(hipGetDeviceProperties(&prop, device));
    c->num_cus = prop.multiProcessorCount;
    c->lds_max = (int)prop.sharedMemPerBlock;
    snprintf(c->name, sizeof(c->name), "%s", prop.gcnArchName);
    c->tpb = 256;
    c->bpc = 2;
    c->use_tiles = 1;
    if(const char *e = getenv("BHC_TL_TILES")) c->use_tiles = atoi(e) != 0;
    c->exact_phasor = 0;
    if(const char *e = getenv("BHC_EXACT_PHASOR")) c->exact_phasor = atoi(e) != 0;
    c->seg_mb = 16384;
    c->scatter3_map = 2;
    if(const char *e = getenv("BHC_SCATTER3_MAP")) c->scatter3_map = std::min(std::max(atoi(e), 0), 2);
    if(const char *e = getenv("BHC_SEG_BUFFER_MB")) c->seg_mb = (size_t)std::max(16L, atol(e));
    if(const char *e = getenv("BHC_POOL_MB")) c->pool.set_limit((size_t)std::max(0L, atol(e)) << 20);
    HIPCHECK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIPCHECK(hipEventCreate(&c->ev0));
    HIPCHECK(hipEventCreate(&c->ev1));
    HIPCHECK(hipEventCreate(&c->evm));
    HIPCHECK(hipEventCreate(&c->pa));
    HIPCHECK(hipEventCreate(&c->pb));
    HIPCHECK(bhc_device_malloc((void **)&c->d_seg_count, sizeof(uint32_t)));
    HIPCHECK(bhc_device_malloc((void **)&c->d_overflow, sizeof(uint32_t)));
    HIPCHECK(bhc_device_malloc((void **)&c->d_prog, sizeof(unsigned long long)));
    HIPCHECK(hipHostMalloc((void **)&c->h_prog, 64, hipHostMallocMapped | hipHostMallocCoherent));
    *c->h_prog = 0ull;
    if(scratch_address(device, &c->scratch)) return -1;
    *out = c;
    return 0;
}

extern "C" void bhc_ctx_destroy(bhc_ctx *ctx)
{
    if(!ctx) return;
    if(ctx->worker.joinable()) {
        if(ctx->worker.get_id() == std::this_thread::get_id()) ctx->worker.detach();
        else ctx->worker.join();
    }
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipEventDestroy(ctx->ev0);
    (void)hipEventDestroy(ctx->ev1);
    (void)hipEventDestroy(ctx->evm);
    (void)hipEventDestroy(ctx->pa);
    (void)hipEventDestroy(ctx->pb);
    if(ctx->segs) (void)hipFree(ctx->segs);
    if(ctx->d_bin_idx) (void)hipFree(ctx->d_bin_idx);
    (void)hipFree(ctx->d_seg_count);
    (void)hipFree(ctx->d_overflow);
    (void)hipFree(ctx->d_prog);
    (void)hipHostFree(ctx->h_prog);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

extern "C" int bhc_progress(bhc_ctx *ctx, int64_t *done, int64_t *total)
{
    if(!ctx || !done || !total) return fail("bhc_progress: null argument");
    const long long t = ctx->prog_total.load();
    long long d = t;
    if(!ctx->prog_final.load()) {
        d = std::min((long long)__atomic_load_n(ctx->h_prog, __ATOMIC_RELAXED), t);
        long long seen = ctx->prog_seen.load();
        while(d > seen && !ctx->prog_seen.compare_exchange_weak(seen, d)) {
        }
        d = std::max(d, seen);
    }
    *done = d;
    *total = t;
    return 0;
}

extern "C" int bhc_ctx_set_launch(bhc_ctx *ctx, int threads_per_block, int blocks_per_cu)
{
    if(threads_per_block != 0 && threads_per_block != 256)
        return fail("bhc_ctx_set_launch: kernels are built for 256 threads per workgroup");
    if(blocks_per_cu < 0 || blocks_per_cu > 64) return fail("bhc_ctx_set_launch: blocks_per_cu out of range");
    ctx->bpc = blocks_per_cu ? blocks_per_cu : 2;
    return 0;
}

extern "C" int bhc_ctx_synchronize(bhc_ctx *ctx)
{
    HIPCHECK(hipStreamSynchronize(ctx->stream));
    return 0;
}

extern "C" int bhc_ctx_trim(bhc_ctx *ctx)
{
    if(!ctx) return fail("bhc_ctx_trim: null context");
    ctx->pool.trim();
    return 0;
}

namespace {
// Plain streaming copy (16 B per lane per iteration): the known-size kernel
// against which profiler byte counters (FETCH_SIZE, WRITE_SIZE) are scaled.
__global__ void __launch_bounds__(256) k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n)
{
    for(size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}
} // namespace

extern "C" int bhc_copy_calibrate(bhc_ctx *ctx, long long bytes, double *ms)
{
    if(check_idle(ctx, "bhc_copy_calibrate")) return -1;
    if(bytes < 16 || (bytes & 15)) return fail("bhc_copy_calibrate: bytes must be a positive multiple of 16");
    HIPCHECK(hipSetDevice(ctx->device));
    void *a = nullptr, *b = nullptr;
    HIPCHECK(bhc_device_malloc(&a, (size_t)bytes));
    if(bhc_device_malloc(&b, (size_t)bytes) != hipSuccess) {
        (void)hipFree(a);
        return fail("bhc_copy_calibrate: allocation failed");
    }
    int rc = 0;
    const size_t n = (size_t)bytes / 16;
    const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, (size_t)ctx->num_cus * 16);
    if(hipMemsetAsync(a, 1, (size_t)bytes, ctx->stream) != hipSuccess) rc = fail("bhc_copy_calibrate: memset failed");
    if(!rc) {
        (void)hipEventRecord(ctx->ev0, ctx->stream);
        hipLaunchKernelGGL(k_copy16, dim3(grid), dim3(256), 0, ctx->stream, (const uint4 *)a, (uint4 *)b, n);
        (void)hipEventRecord(ctx->ev1, ctx->stream);
        float f = 0.f;
        if(hipGetLastError() != hipSuccess || hipEventSynchronize(ctx->ev1) != hipSuccess
           || hipEventElapsedTime(&f, ctx->ev0, ctx->ev1) != hipSuccess)
            rc = fail("bhc_copy_calibrate: copy kernel failed");
        if(ms) *ms = f;
    }
    (void)hipFree(a);
    (void)hipFree(b);
    return rc;
}

extern "C" int bhc_last_phase_ms(bhc_ctx *ctx, double *trace_ms, double *scatter_ms, int *passes)
{
    HIPCHECK(hipEventSynchronize(ctx->ev1));
    *trace_ms = ctx->ph_trace_ms;
    *scatter_ms = ctx->ph_scatter_ms;
    *passes = ctx->passes;
    return 0;
}

// Per-pass phase timing: a trace (or scatter) launch is bracketed by pa / pb on
// the context's stream and its duration added once the pass has finished.
static int phase_add(bhc_ctx *c, double *acc)
{
    float ms = 0.f;
    HIPCHECK(hipEventSynchronize(c->pb));
    HIPCHECK(hipEventElapsedTime(&ms, c->pa, c->pb));
    *acc += ms;
    return 0;
}

extern "C" int bhc_last_kernel_ms(bhc_ctx *ctx, double *ms)
{
    float f = 0.f;
    HIPCHECK(hipEventSynchronize(ctx->ev1));
    HIPCHECK(hipEventElapsedTime(&f, ctx->ev0, ctx->ev1));
    *ms = f;
    return 0;
}

namespace {

template<typename T> int dalloc(T **p, size_t n)
{
    *p = nullptr;
    if(n == 0) return 0;
    HIPCHECK(bhc_device_malloc((void **)p, n * sizeof(T)));
    return 0;
}

// dalloc from the context's pool (given back with ctx->pool.put)
template<typename T> int palloc(bhc_ctx *c, T **p, size_t n)
{
    *p = nullptr;
    if(n == 0) return 0;
    HIPCHECK((hipError_t)c->pool.get((void **)p, n * sizeof(T)));
    return 0;
}

int check_problem(const bhc_problem2d *p)
{
    if(!p) return fail("null problem");
    if(p->precision != 64 && p->precision != 32) return fail("precision must be 32 or 64");
    if(p->NSz < 1 || p->NRz < 1 || p->NRr < 1 || p->Nalpha < 1) return fail("empty source/receiver/angle set");
    if(p->NRz_per_range != p->NRz && p->NRz_per_range != 1) return fail("bad NRz_per_range");
    if(p->RunType[4] == 'I' && p->NRz != p->NRr) return fail("irregular grid needs NRz == NRr");
    if(p->iSingle_alpha < 0 || p->iSingle_alpha > p->Nalpha) return fail("iSingle out of range");
    if(p->NSBPPts < 2) return fail("source beam pattern needs 2 points");
    if((long long)p->NSz * p->Nalpha >= (1ll << 31) / 2) return fail("too many rays");
    if(!(p->deltas > 0)) return fail("deltas must be positive after preprocessing");
    return 0;
}

} // namespace

extern "C" void bhc_problem_release(bhc_dev_problem *dp)
{
    if(!dp) return;
    (void)hipSetDevice(dp->ctx->device);
    (void)hipStreamSynchronize(dp->ctx->stream);
    void *ptrs[] = {dp->d_bins, dp->d_blob, dp->d_Rz,   dp->d_Sz,     dp->d_field,    dp->d_cand, dp->d_ncand,
                    dp->d_arr,  dp->d_narr, dp->d_hits,   dp->d_neigen,   dp->d_stats, dp->d_xend,
                    dp->d_counters, dp->d_errw, dp->d_work};
    for(void *p : ptrs) dp->ctx->pool.put(p);
    delete dp;
}

namespace {
int ensure_segs(bhc_ctx *c);
}

extern "C" int bhc_problem_upload2d(bhc_ctx *ctx, const bhc_problem2d *prob, const bhc_field_out *spec,
                                    bhc_dev_problem **out)
{
    *out = nullptr;
    if(check_problem(prob)) return -1;
    HIPCHECK(hipSetDevice(ctx->device));
    bhc_dev_problem *dp = new bhc_dev_problem();
    memset(dp, 0, sizeof(*dp));
    dp->ctx = ctx;
    dp->precision = prob->precision;
    dp->run0 = prob->RunType[0];
    dp->NSz = prob->NSz;
    dp->NRz_per_range = prob->NRz_per_range;
    dp->NRr = prob->NRr;
    dp->njobs = (prob->iSingle_alpha >= 1 ? 1 : prob->Nalpha) * prob->NSz;
    dp->nrcv = (size_t)prob->NSz * prob->NRz_per_range * prob->NRr;
    dp->freq0 = prob->freq0;
    dp->xend_dim = 2;
    int rc = 0;
    size_t blob_bytes = 0, staged = 0;
    if(prob->precision == 64) {
        std::vector<double> blob;
        std::string err;
        rc = pack<double>(prob, blob, dp->P64, err);
        if(rc) fail("%s", err.c_str());
        if(!rc) {
            blob_bytes = blob.size() * sizeof(double);
            staged = (size_t)dp->P64.staged_reals * sizeof(double);
            rc = palloc(ctx, (unsigned char **)&dp->d_blob, blob_bytes);
            if(!rc && hipMemcpy(dp->d_blob, blob.data(), blob_bytes, hipMemcpyHostToDevice) != hipSuccess)
                rc = fail("blob upload failed");
        }
    } else {
        std::vector<float> blob;
        std::string err;
        rc = pack<float>(prob, blob, dp->P32, err);
        if(rc) fail("%s", err.c_str());
        if(!rc) {
            blob_bytes = blob.size() * sizeof(float);
            staged = (size_t)dp->P32.staged_reals * sizeof(float);
            rc = palloc(ctx, (unsigned char **)&dp->d_blob, blob_bytes);
            if(!rc && hipMemcpy(dp->d_blob, blob.data(), blob_bytes, hipMemcpyHostToDevice) != hipSuccess)
                rc = fail("blob upload failed");
        }
    }
    if(rc) {
        bhc_problem_release(dp);
        return -1;
    }
    // Stage in LDS when the SSP + boundary tables fit the workgroup's LDS.
    dp->lds_bytes = (staged <= (size_t)std::min(ctx->lds_max, 65536)) ? staged : 0;
    if(!dp->lds_bytes) {
        dp->P64.staged_reals = 0;
        dp->P32.staged_reals = 0;
    }
    dp->P64.base = (const double *)dp->d_blob;
    dp->P32.base = (const float *)dp->d_blob;
    if(palloc(ctx, &dp->d_Rz, prob->NRz) || palloc(ctx, &dp->d_Sz, prob->NSz) || palloc(ctx, &dp->d_counters, 3)
       || palloc(ctx, &dp->d_errw, 4) || palloc(ctx, &dp->d_work, 1)) {
        bhc_problem_release(dp);
        return -1;
    }
    HIPCHECK(hipMemcpy(dp->d_Rz, prob->Rz, prob->NRz * sizeof(float), hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(dp->d_Sz, prob->Sz, prob->NSz * sizeof(float), hipMemcpyHostToDevice));
    dp->P64.Rz = dp->P32.Rz = dp->d_Rz;
    dp->P64.Sz = dp->P32.Sz = dp->d_Sz;
    char r0 = dp->run0;
    bool tl = (r0 == 'C' || r0 == 'S' || r0 == 'I');
    bool arr = (r0 == 'A' || r0 == 'a' || r0 == 'V' || r0 == 'v');
    bool eig = (r0 == 'E' || r0 == 'V' || r0 == 'v');
    if(!tl && !arr && !eig && r0 != 'R') {
        bhc_problem_release(dp);
        return fail("unknown run type '%c'", r0);
    }
    if(tl && palloc(ctx, &dp->d_field, 2 * dp->nrcv)) {
        bhc_problem_release(dp);
        return -1;
    }
    dp->P64.field = dp->P32.field = dp->d_field;
    dp->P64.njobs = dp->P32.njobs = dp->njobs;
    if(tl && prob->NRr > 1 && prob->Delta_r > 0) {
        // LDS tile of 64 KiB beside the descriptors' stage, so that a CU holds two
        // workgroups: tile_w range columns x all depths, complex float. (Taken
        // from the tile, the stage left fields of 1318 to 1365 depths without
        // one: 1340 x 1001 receivers of 2001 Gaussian beams, 43.9 instead of
        // 14.3 ms.)
        int nz = prob->NRz_per_range;
        int tile_w = (int)((size_t)std::min(65536, ctx->lds_max - TILE_STAGE) / ((size_t)nz * 2 * sizeof(float)));
        int margin = (int)std::ceil(prob->deltas / (2.0 * prob->Delta_r)) + 2;
        // at most 16384 bins (a workgroup's histogram in 64 KiB of LDS). Where the
        // sources would need more, Cartesian Gaussian beams, whose many atomics per
        // segment a tile saves, have them for as many sources as that allows; the
        // others go without (2001 beams, 2 x 1001 x 9001 receivers, bins for one
        // source and for none: Gaussian 467 and 506 ms, hat 16.8 and 15.6,
        // ray-centred Gaussian 98.9 and 93.8)
        const int bin_w = std::max(1, tile_w - 2 * margin), per_source = (prob->NRr + bin_w - 1) / bin_w;
        const bool some = prob->BeamType[0] == 'B';
        if(tile_w >= 6 && (some ? per_source : (long long)prob->NSz * per_source) <= 16384) {
            if(bin_w == 1) margin = (tile_w - 1) / 2;
            dp->tile_w = tile_w;
            dp->bin_w = bin_w;
            dp->tile_lo_off = margin;
            dp->nbins = per_source;
            dp->chunk = 2048;
            dp->bin_sources = std::min(prob->NSz, 16384 / per_source);
            dp->total_bins = dp->nbins * dp->bin_sources;
            if(ensure_segs(ctx)) {
                bhc_problem_release(dp);
                return -1;
            }
            size_t cap = ctx->seg_bytes / sizeof(Seg<float>);
            // chunks hold dp->chunk segments, or fewer when there are less than
            // two full ones per CU (run_passes): at most that many either way
            dp->max_chunks = (int)std::min<size_t>(
                std::max<size_t>(cap / dp->chunk, 2 * (size_t)ctx->num_cus) + dp->total_bins + 2, 0x3FFFFFFF);
            if(palloc(ctx, &dp->d_bins, 3 * (size_t)dp->total_bins + 1 + 2 * (size_t)dp->max_chunks)) {
                bhc_problem_release(dp);
                return -1;
            }
        }
    }
    if(arr) {
        dp->max_narr = spec ? spec->max_narr : 0;
        dp->allow_merging = spec ? spec->allow_merging : 1;
        if(dp->max_narr < 1) {
            bhc_problem_release(dp);
            return fail("arrivals run needs max_narr >= 1");
        }
        // candidate capacity per receiver from a 16 GiB budget, at least 8 x MaxNArr
        size_t budget = (size_t)16 << 30;
        size_t cap = budget / (dp->nrcv * sizeof(ArrCand));
        cap = std::min<size_t>(cap, 65536);
        cap = std::max<size_t>(cap, 8 * (size_t)dp->max_narr);
        dp->cand_cap = (int)cap;
        if(palloc(ctx, &dp->d_cand, dp->nrcv * cap) || palloc(ctx, &dp->d_ncand, dp->nrcv)
           || palloc(ctx, &dp->d_arr, dp->nrcv * dp->max_narr) || palloc(ctx, &dp->d_narr, dp->nrcv)) {
            bhc_problem_release(dp);
            return -1;
        }
    }
    if(eig) {
        dp->eigen_memsize = spec ? spec->eigen_memsize : 0;
        if(dp->eigen_memsize < 1) {
            bhc_problem_release(dp);
            return fail("eigenray run needs eigen_memsize >= 1");
        }
        if(palloc(ctx, &dp->d_hits, dp->eigen_memsize) || palloc(ctx, &dp->d_neigen, 1)) {
            bhc_problem_release(dp);
            return -1;
        }
    }
    if(spec && spec->ray_nsteps) {
        if(palloc(ctx, &dp->d_stats, 3 * (size_t)dp->njobs) || palloc(ctx, &dp->d_xend, 2 * (size_t)dp->njobs)) {
            bhc_problem_release(dp);
            return -1;
        }
    }
    *out = dp;
    return 0;
}

namespace {
DevOut make_out(bhc_dev_problem *dp)
{
    DevOut O;
    memset(&O, 0, sizeof(O));
    O.cand = dp->d_cand;
    O.ncand = dp->d_ncand;
    O.cand_cap = dp->cand_cap;
    O.hits = dp->d_hits;
    O.neigen = dp->d_neigen;
    O.eigen_memsize = dp->eigen_memsize;
    O.stats = dp->d_stats;
    O.xend = dp->d_xend;
    O.counters = dp->d_counters;
    O.errw = dp->d_errw;
    O.work = dp->d_work;
    O.job_begin = 0;
    O.job_end = dp->njobs;
    O.prog = prog_of(dp->ctx);
    return O;
}

// Slots of a segment buffer of `bytes`. A sweep that stores descriptor cores
// alone (full false) has slots of a core, so a pass holds 1.4 times as many and
// two wavefronts per SIMD leave it as many passes as one did; a single field
// fits in one or two passes either way. Never more than the binned order has
// entries (ensure_segs).
template<typename real> uint32_t seg_slots(size_t bytes, bool full)
{
    const size_t slot = std::max(full ? sizeof(Seg<real>) : (size_t)SEG_NC<real> * 16, sizeof(Seg<float>));
    return (uint32_t)std::min(bytes / slot, SEG_CAP_MAX);
}

size_t seg_size(int precision) { return precision == 64 ? sizeof(Seg<double>) : sizeof(Seg<float>); }

// Segment buffer: BHC_SEG_BUFFER_MB (default 16384 MiB) of HBM, allocated once per context.
int ensure_segs(bhc_ctx *c)
{
    if(c->segs) return 0;
    c->seg_bytes = c->seg_mb << 20;
    HIPCHECK(bhc_device_malloc(&c->segs, c->seg_bytes));
    size_t maxseg = c->seg_bytes / sizeof(Seg<float>);
    HIPCHECK(bhc_device_malloc((void **)&c->d_bin_idx, maxseg * sizeof(uint32_t)));
    return 0;
}

// Lanes of a wavefront that take rays: a fan smaller than the GPU's lanes is
// spread over one wavefront per SIMD (four SIMDs per CU) instead of filling few
// wavefronts. A wavefront walks the code of every case that one of its lanes
// meets in a step (reflection, profile knot, receiver range, refill), so
// fewer rays per wavefront make each step shorter.
// Every wavefront takes a slot block of its own, so a small segment buffer
// (slots; 0: none) bounds their number: together they may leave an eighth of it
// in partly used blocks. 2001 rays on 1001 wavefronts overflow the
// allocation-free launch's 64 MiB whatever they trace: over 5 km 2.75 ms in four
// passes, against 0.67 ms in one on the 113 wavefronts of this bound and 0.85 on
// 32 full ones.
int fan_lanes(int nrays, int num_cus, size_t slots)
{
    size_t waves = std::max(1, 4 * num_cus);
    if(slots) waves = std::min(waves, std::max<size_t>(1, slots / (8 * (size_t)SEG_BLOCK)));
    return (int)std::min<size_t>(WAVE, std::max<size_t>(1, ((size_t)nrays + waves - 1) / waves));
}

// The scatter mapping that a problem without a chosen one gets, per pass, from
// the candidate receivers its segments bracket per step (counted by the
// trace): below this many, one lane walks a segment alone, which for a few
// receivers costs less than a wavefront per segment, or range bins and tiles
// (2001 hat beams, 1.8 contributions per step: 0.28 ms against 0.71 and 0.68).
// Above, tiles (at 8.5 contributions per step 4.4 ms against 7.2 for lanes and
// 10.5 for wavefronts). A hat beam's bracket holds about three times the
// receivers that it reaches, a Gaussian's hardly more than those.
double sparse_items(bool gaussian) { return gaussian ? 6.0 : 16.0; }

template<typename real> const bhc3d::Prob3D<real> &nx_of(const bhc_dev_problem *dp);
template<> const bhc3d::Prob3D<double> &nx_of<double>(const bhc_dev_problem *dp) { return dp->N64; }
template<> const bhc3d::Prob3D<float> &nx_of<float>(const bhc_dev_problem *dp) { return dp->N32; }

// Trace / scatter passes over the problem's rays. segbuf == null: the
// context's segment buffer (allocated at first use); otherwise the given
// buffer of segbytes, with the scatter restricted to the mappings that need
// no range bins (the bins are allocated with the context's buffer).
template<typename real, int RT>
int run_passes(bhc_dev_problem *dp, const Prob2D<real> &P, DevOut O, void *segbuf = nullptr, size_t segbytes = 0)
{
    bhc_ctx *c = dp->ctx;
    hipStream_t s = c->stream;
    const bool own_buffer = segbuf != nullptr;
    if(!own_buffer) {
        if(ensure_segs(c)) return -1;
        segbuf = c->segs;
        segbytes = c->seg_bytes;
    }
    O.segs = segbuf;
    O.seg_count = c->d_seg_count;
    O.overflow = c->d_overflow;
    O.seg_cap = seg_slots<real>(segbytes, true);
    O.seg_words = SEG_NW<real>;
    std::vector<std::pair<int, int>> todo{{0, dp->njobs}};
    c->passes = 0;
    c->ph_trace_ms = c->ph_scatter_ms = 0.0;
    bool first = true;
    unsigned long long steps_done = 0, cand_done = 0;
    while(!todo.empty()) {
        auto r = todo.back();
        todo.pop_back();
        O.job_begin = r.first;
        O.job_end = r.second;
        HIPCHECK(hipMemsetAsync(c->d_seg_count, 0, sizeof(uint32_t), s));
        HIPCHECK(hipMemsetAsync(c->d_overflow, 0, sizeof(uint32_t), s));
        HIPCHECK(hipMemsetAsync(dp->d_work, 0, sizeof(int32_t), s));
        int nj = r.second - r.first;
        O.lanes = fan_lanes(nj, c->num_cus, O.seg_cap);
        // one wavefront per workgroup spreads the rays over all CUs (the trace
        // kernel is register-bound at one wavefront per SIMD)
        int tblocks = std::max(1, std::min((nj + O.lanes - 1) / O.lanes, c->num_cus * 4 * c->bpc));
        // error / warning words as the completed passes left them (stream
        // order: after the previous pass's scatter), restored if this trace
        // pass overflows and its rays are traced again
        uint32_t ew_start[4] = {0u, 0u, 0u, 0u};
        unsigned long long prog_start = 0;
        HIPCHECK(hipMemcpyAsync(ew_start, dp->d_errw, sizeof(ew_start), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipMemcpyAsync(&prog_start, c->d_prog, sizeof(prog_start), hipMemcpyDeviceToHost, s));
        if(first) HIPCHECK(hipEventRecord(c->ev0, s));
        HIPCHECK(hipEventRecord(c->pa, s));
        if(dp->nx2d) {
            hipLaunchKernelGGL((k_tracenx2d<real>), dim3(tblocks), dim3(WAVE), 0, s, P, nx_of<real>(dp), O);
        } else {
#define BHC_TRACE(ST)                                                                                                  \
    if(dp->lds_bytes)                                                                                                  \
        hipLaunchKernelGGL((k_trace2d<real, ST, true>), dim3(tblocks), dim3(WAVE), dp->lds_bytes, s, P, O);            \
    else                                                                                                               \
        hipLaunchKernelGGL((k_trace2d<real, ST, false>), dim3(tblocks), dim3(WAVE), 0, s, P, O);                       \
    break;
            switch(P.ssp_type) {
            case 'C': BHC_TRACE('C')
            case 'S': BHC_TRACE('S')
            case 'P': BHC_TRACE('P')
            case 'N': BHC_TRACE('N')
            case 'Q': BHC_TRACE('Q')
            default: BHC_TRACE('A')
            }
#undef BHC_TRACE
        }
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipEventRecord(c->pb, s));
        uint32_t of = 0, nseg = 0;
        unsigned long long cnt[3] = {0, 0, 0};
        HIPCHECK(hipMemcpyAsync(&of, c->d_overflow, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipMemcpyAsync(&nseg, c->d_seg_count, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipMemcpyAsync(cnt, dp->d_counters, sizeof(cnt), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipStreamSynchronize(s));
        const unsigned long long steps_now = cnt[0];
        nseg = std::min(nseg, O.seg_cap);
        if(phase_add(c, &c->ph_trace_ms)) return -1;
        if(of) {
            if(nj <= 1) return fail("segment buffer too small for a single ray (raise BHC_SEG_BUFFER_MB)");
            int mid = r.first + nj / 2;
            todo.push_back({mid, r.second});
            todo.push_back({r.first, mid});
            // the trace pass wrote only per-ray statistics, the step counter and
            // the error / warning words: the retried halves rewrite the
            // statistics; the counter and the words go back to the completed
            // passes' values, so that the retried rays' warnings count once
            HIPCHECK(hipMemcpyAsync(dp->d_counters, &steps_done, sizeof(unsigned long long), hipMemcpyHostToDevice, s));
            HIPCHECK(hipMemcpyAsync(dp->d_counters + 2, &cand_done, sizeof(unsigned long long), hipMemcpyHostToDevice, s));
            HIPCHECK(hipMemcpyAsync(dp->d_errw, ew_start, sizeof(ew_start), hipMemcpyHostToDevice, s));
            HIPCHECK(hipMemcpyAsync(c->d_prog, &prog_start, sizeof(prog_start), hipMemcpyHostToDevice, s));
            HIPCHECK(hipStreamSynchronize(s));
            continue;
        }
        const bool sparse = (double)(cnt[2] - cand_done) < sparse_items(P.isGaussian != 0) * (double)(steps_now - steps_done);
        steps_done = steps_now;
        cand_done = cnt[2];
        if(first) HIPCHECK(hipEventRecord(c->evm, s));
        HIPCHECK(hipEventRecord(c->pa, s));
        int mode = dp->scatter_mode;
        if(mode == SCATTER_AUTO)
            mode = sparse ? SCATTER_LANES : (RT == RT_TL && c->use_tiles && dp->nbins > 0) ? SCATTER_TILED : SCATTER_WAVE;
        if(mode == SCATTER_TILED && (!(RT == RT_TL && dp->nbins > 0) || own_buffer)) mode = SCATTER_WAVE;
        if(mode == SCATTER_LANES) {
            int sblocks = c->num_cus * 8;
            if(RT == RT_TL && !c->exact_phasor)
                hipLaunchKernelGGL((k_scatter2d_lanes<real, RT, true>), dim3(sblocks), dim3(256), 0, s, P, O);
            else
                hipLaunchKernelGGL((k_scatter2d_lanes<real, RT, false>), dim3(sblocks), dim3(256), 0, s, P, O);
        } else if(mode == SCATTER_TILED) {
            BinCfg B;
            B.nbins = dp->nbins;
            B.nsrc = dp->bin_sources;
            B.total = dp->total_bins;
            B.bin_w = dp->bin_w;
            B.tile_w = dp->tile_w;
            B.tile_lo_off = dp->tile_lo_off;
            // two chunks per CU, of at most dp->chunk segments
            B.chunk = (int)std::min<long long>(dp->chunk, std::max(64ll, (long long)nseg / (2 * c->num_cus) + 1));
            B.counts = dp->d_bins;
            B.offsets = B.counts + dp->total_bins;
            B.cursor = B.offsets + dp->total_bins;
            B.nchunks = B.cursor + dp->total_bins;
            B.chunk_bin = B.nchunks + 1;
            B.chunk_pos = B.chunk_bin + dp->max_chunks;
            B.idx = c->d_bin_idx;
            HIPCHECK(hipMemsetAsync(B.counts, 0, dp->total_bins * sizeof(int32_t), s));
            int gb = c->num_cus * 4;
            size_t hl = (size_t)dp->total_bins * sizeof(int32_t);
            hipLaunchKernelGGL((k_bin_count<real>), dim3(gb), dim3(256), hl, s, P, O, B);
            hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(1024), 0, s, B);
            hipLaunchKernelGGL((k_bin_fill<real>), dim3(gb), dim3(256), hl, s, P, O, B);
            size_t lds = (size_t)dp->tile_w * dp->NRz_per_range * 2 * sizeof(float);
            if(c->exact_phasor)
                hipLaunchKernelGGL((k_scatter_tile<real, false>), dim3(c->num_cus * 4), dim3(TILE_THREADS), lds, s,
                                   P, O, B);
            else
                hipLaunchKernelGGL((k_scatter_tile<real, true>), dim3(c->num_cus * 4), dim3(TILE_THREADS), lds, s,
                                   P, O, B);
        } else {
            int sblocks = c->num_cus * 8;
            if(RT == RT_TL && !c->exact_phasor)
                hipLaunchKernelGGL((k_scatter2d<real, RT, true>), dim3(sblocks), dim3(256), 0, s, P, O);
            else
                hipLaunchKernelGGL((k_scatter2d<real, RT, false>), dim3(sblocks), dim3(256), 0, s, P, O);
        }
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipEventRecord(c->pb, s));
        if(phase_add(c, &c->ph_scatter_ms)) return -1;
        ++c->passes;
        first = false;
    }
    HIPCHECK(hipEventRecord(c->ev1, s));
    return 0;
}
} // namespace

extern "C" int bhc_problem_autotune(bhc_ctx *ctx, bhc_dev_problem *dp, int *mode_out);

namespace {
// Zeros in every output of a problem that reaches the caller: its blocks may
// have served another run, and a launch need not write all of them (arrival
// slots past a receiver's count, rays that an error stopped).
int clear_outputs(bhc_dev_problem *dp, hipStream_t s)
{
    if(dp->d_field) HIPCHECK(hipMemsetAsync(dp->d_field, 0, 2 * dp->nrcv * sizeof(float), s));
    if(dp->d_ncand) HIPCHECK(hipMemsetAsync(dp->d_ncand, 0, dp->nrcv * sizeof(int32_t), s));
    if(dp->d_arr) HIPCHECK(hipMemsetAsync(dp->d_arr, 0, dp->nrcv * dp->max_narr * sizeof(bhc_arrival), s));
    if(dp->d_narr) HIPCHECK(hipMemsetAsync(dp->d_narr, 0, dp->nrcv * sizeof(int32_t), s));
    if(dp->d_neigen) HIPCHECK(hipMemsetAsync(dp->d_neigen, 0, sizeof(int32_t), s));
    if(dp->d_stats) HIPCHECK(hipMemsetAsync(dp->d_stats, 0, 3 * (size_t)dp->njobs * sizeof(int32_t), s));
    if(dp->d_xend) HIPCHECK(hipMemsetAsync(dp->d_xend, 0, (size_t)dp->xend_dim * dp->njobs * sizeof(double), s));
    HIPCHECK(hipMemsetAsync(dp->d_counters, 0, 3 * sizeof(unsigned long long), s));
    HIPCHECK(hipMemsetAsync(dp->d_errw, 0, 4 * sizeof(uint32_t), s));
    dp->cleared = 1;
    return 0;
}

int field_launch(bhc_ctx *ctx, bhc_dev_problem *dp, void *segbuf, size_t segbytes)
{
    HIPCHECK(hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    if(prog_begin(ctx, dp->njobs)) return -1;
    if(clear_outputs(dp, s)) return -1;
    DevOut O = make_out(dp);
    char r0 = dp->run0;
    int rt = (r0 == 'C' || r0 == 'S' || r0 == 'I') ? RT_TL : (r0 == 'E') ? RT_EIG : RT_ARR;
    int rc;
    if(dp->precision == 64) {
        rc = rt == RT_TL ? run_passes<double, RT_TL>(dp, dp->P64, O, segbuf, segbytes)
            : rt == RT_ARR ? run_passes<double, RT_ARR>(dp, dp->P64, O, segbuf, segbytes)
                           : run_passes<double, RT_EIG>(dp, dp->P64, O, segbuf, segbytes);
    } else {
        rc = rt == RT_TL ? run_passes<float, RT_TL>(dp, dp->P32, O, segbuf, segbytes)
            : rt == RT_ARR ? run_passes<float, RT_ARR>(dp, dp->P32, O, segbuf, segbytes)
                           : run_passes<float, RT_EIG>(dp, dp->P32, O, segbuf, segbytes);
    }
    if(rc) return rc;
    if(rt == RT_ARR) {
        int nrcv = (int)dp->nrcv;
        double om = 2.0 * M_PI * dp->freq0;
        hipLaunchKernelGGL(k_arr_merge, dim3((nrcv + 255) / 256), dim3(256), 0, s, dp->d_cand, dp->d_ncand,
                           dp->cand_cap, dp->d_arr, dp->d_narr, dp->max_narr, nrcv, dp->allow_merging,
                           (float)(2.0f * (float)M_PI * (float)dp->freq0), om, dp->precision == 64 ? 1 : 0,
                           dp->d_errw);
        HIPCHECK(hipGetLastError());
    }
    ctx->prog_final = 1;   // every trace pass has completed: all rays have finished
    return 0;
}
} // namespace

extern "C" int bhc_field_launch(bhc_ctx *ctx, bhc_dev_problem *dp)
{
    if(check_idle(ctx, "bhc_field_launch")) return -1;
    if(!dp || dp->ctx != ctx) return fail("bhc_field_launch: problem not uploaded on this context");
    return field_launch(ctx, dp, nullptr, 0);
}

extern "C" int bhc_field_launch_noalloc(bhc_ctx *ctx, bhc_dev_problem *dp)
{
    if(check_idle(ctx, "bhc_field_launch_noalloc")) return -1;
    if(!dp || dp->ctx != ctx) return fail("bhc_field_launch_noalloc: problem not uploaded on this context");
    if(dp->run0 != 'C' && dp->run0 != 'S' && dp->run0 != 'I')
        return fail("bhc_field_launch_noalloc: TL run types (C, S, I) only, not '%c'", dp->run0);
    if(!ctx->scratch) return fail("bhc_field_launch_noalloc: the scratch array is not mapped on device %d", ctx->device);
    // a pass must hold one ray's segments (at most MAXN, plus a partly used
    // slot block at either end); more rays are split over further passes
    const size_t need = ((size_t)MAXN + 2 * (size_t)SEG_BLOCK) * seg_size(dp->precision);
    if(need > NOALLOC_SCRATCH_BYTES)
        return fail("bhc_field_launch_noalloc: one pass needs %zu bytes of scratch, the static scratch holds %zu",
                    need, NOALLOC_SCRATCH_BYTES);
    return field_launch(ctx, dp, ctx->scratch, NOALLOC_SCRATCH_BYTES);
}

extern "C" int bhc_problem_set_scatter(bhc_dev_problem *dp, int mode)
{
    if(!dp || mode < SCATTER_AUTO || mode > SCATTER_LANES) return fail("bhc_problem_set_scatter: bad arguments");
    dp->scatter_mode = mode;
    return 0;
}

// Scatter-mapping search for a resident problem: every available mapping
// (range-binned LDS tiles for TL runs, one wavefront per segment, one lane per
// segment) is launched twice and the fastest kept for later launches.
extern "C" int bhc_problem_autotune(bhc_ctx *ctx, bhc_dev_problem *dp, int *mode_out)
{
    if(check_idle(ctx, "bhc_problem_autotune")) return -1;
    if(!dp || dp->ctx != ctx) return fail("bhc_problem_autotune: problem not uploaded on this context");
    int modes[3] = {SCATTER_TILED, SCATTER_WAVE, SCATTER_LANES};
    int best_mode = SCATTER_AUTO;
    double best = 1e300;
    bool tl = dp->run0 == 'C' || dp->run0 == 'S' || dp->run0 == 'I';
    for(int m : modes) {
        if(m == SCATTER_TILED && !(tl && dp->nbins > 0 && ctx->use_tiles)) continue;
        dp->scatter_mode = m;
        double t = 0.0;
        for(int rep = 0; rep < 2; ++rep) {
            if(bhc_field_launch(ctx, dp)) return -1;
            double ms = 0.0;
            if(bhc_last_kernel_ms(ctx, &ms)) return -1;
            if(rep == 1) t = ms;
        }
        if(t < best) {
            best = t;
            best_mode = m;
        }
    }
    dp->scatter_mode = best_mode;
    if(mode_out) *mode_out = best_mode;
    return 0;
}

extern "C" int bhc_field_download(bhc_ctx *ctx, bhc_dev_problem *dp, bhc_field_out *out)
{
    HIPCHECK(hipSetDevice(ctx->device));
    if(!dp->cleared && clear_outputs(dp, ctx->stream)) return -1;   // not launched yet
    HIPCHECK(hipStreamSynchronize(ctx->stream));
    if(out->field && dp->d_field)
        HIPCHECK(hipMemcpy(out->field, dp->d_field, 2 * dp->nrcv * sizeof(float), hipMemcpyDeviceToHost));
    if(out->arr && dp->d_arr) {
        if(out->max_narr != dp->max_narr) return fail("download: max_narr differs from the upload spec");
        HIPCHECK(hipMemcpy(out->arr, dp->d_arr, dp->nrcv * dp->max_narr * sizeof(bhc_arrival), hipMemcpyDeviceToHost));
        HIPCHECK(hipMemcpy(out->narr, dp->d_narr, dp->nrcv * sizeof(int32_t), hipMemcpyDeviceToHost));
    }
    if(out->hits && dp->d_hits) {
        int n = 0;
        HIPCHECK(hipMemcpy(&n, dp->d_neigen, sizeof(int32_t), hipMemcpyDeviceToHost));
        int m = std::min(n, std::min(out->eigen_memsize, dp->eigen_memsize));
        if(m > 0) HIPCHECK(hipMemcpy(out->hits, dp->d_hits, m * sizeof(bhc_eigen_hit), hipMemcpyDeviceToHost));
        if(out->neigen) *out->neigen = n;
    }
    if(out->ray_nsteps && dp->d_stats) {
        std::vector<int32_t> st(3 * (size_t)dp->njobs);
        HIPCHECK(hipMemcpy(st.data(), dp->d_stats, st.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
        for(int j = 0; j < dp->njobs; ++j) {
            out->ray_nsteps[j] = st[3 * j];
            if(out->ray_ntop) out->ray_ntop[j] = st[3 * j + 1];
            if(out->ray_nbot) out->ray_nbot[j] = st[3 * j + 2];
        }
        if(out->ray_xend)
            HIPCHECK(hipMemcpy(out->ray_xend, dp->d_xend, (size_t)dp->xend_dim * dp->njobs * sizeof(double),
                               hipMemcpyDeviceToHost));
    }
    unsigned long long cnt[2];
    uint32_t ew[4];
    HIPCHECK(hipMemcpy(cnt, dp->d_counters, sizeof(cnt), hipMemcpyDeviceToHost));
    HIPCHECK(hipMemcpy(ew, dp->d_errw, sizeof(ew), hipMemcpyDeviceToHost));
    out->total_steps = (int64_t)cnt[0];
    out->total_contrib = (int64_t)cnt[1];
    out->err = ew[0];
    out->warn = ew[1];
    out->err_count = ew[2];
    out->warn_count = ew[3];
    return 0;
}

extern "C" int bhc_field_run2d(bhc_ctx *ctx, const bhc_problem2d *prob, bhc_field_out *out)
{
    if(check_idle(ctx, "bhc_field_run2d")) return -1;
    bhc_dev_problem *dp = nullptr;
    if(bhc_problem_upload2d(ctx, prob, out, &dp)) return -1;
    int rc = bhc_field_launch(ctx, dp);
    if(!rc) rc = bhc_field_download(ctx, dp, out);
    bhc_problem_release(dp);
    return rc;
}

namespace {
template<typename real> void launch_rays(bhc_dev_problem *dp, const Prob2D<real> &P, const DevOut &O, int blocks)
{
    hipStream_t s = dp->ctx->stream;
#define BHC_RAYS(ST)                                                                                                   \
    if(dp->lds_bytes) hipLaunchKernelGGL((k_ray2d<real, ST, true>), dim3(blocks), dim3(WAVE), dp->lds_bytes, s, P, O); \
    else hipLaunchKernelGGL((k_ray2d<real, ST, false>), dim3(blocks), dim3(WAVE), 0, s, P, O);                         \
    break;
    switch(P.ssp_type) {
    case 'C': BHC_RAYS('C')
    case 'S': BHC_RAYS('S')
    case 'P': BHC_RAYS('P')
    case 'N': BHC_RAYS('N')
    case 'Q': BHC_RAYS('Q')
    default: BHC_RAYS('A')
    }
#undef BHC_RAYS
}
} // namespace

extern "C" int bhc_ray_run2d(bhc_ctx *ctx, const bhc_problem2d *prob, bhc_ray_out *out)
{
    return bhc_ray_run2d_list(ctx, prob, out, nullptr, nullptr, nullptr, -1);
}

extern "C" int bhc_ray_run2d_list(bhc_ctx *ctx, const bhc_problem2d *prob, bhc_ray_out *out, const int32_t *ialpha,
                                  const int32_t *isz, const int32_t *nsteps_in, int32_t nrays)
{
    if(check_idle(ctx, "bhc_ray_run2d")) return -1;
    if(check_problem(prob)) return -1;
    if(out->max_points_per_ray < 3) return fail("max_points_per_ray must be >= 3");
    HIPCHECK(hipSetDevice(ctx->device));
    bhc_field_out spec;
    memset(&spec, 0, sizeof(spec));
    bhc_problem2d p2 = *prob;
    p2.RunType[0] = 'R';
    bhc_dev_problem *dp = nullptr;
    if(bhc_problem_upload2d(ctx, &p2, &spec, &dp)) return -1;
    int njobs = nrays >= 0 ? nrays : dp->njobs;
    if(prog_begin(ctx, njobs)) {
        bhc_problem_release(dp);
        return -1;
    }
    DevOut O = make_out(dp);
    O.job_begin = 0;
    O.job_end = njobs;
    O.max_points = out->max_points_per_ray;
    int32_t *d_ia = nullptr, *d_isz = nullptr, *d_nin = nullptr, *d_nout = nullptr;
    bhc_ray_pt2d *d_pts = nullptr;
    int rc = 0;
    size_t npts = (size_t)njobs * out->max_points_per_ray;
    if(palloc(ctx, &d_pts, npts) || palloc(ctx, &d_nout, njobs)) rc = -1;
    if(!rc && ialpha) {
        if(palloc(ctx, &d_ia, njobs) || palloc(ctx, &d_isz, njobs)) rc = -1;
        else {
            hipMemcpy(d_ia, ialpha, njobs * sizeof(int32_t), hipMemcpyHostToDevice);
            hipMemcpy(d_isz, isz, njobs * sizeof(int32_t), hipMemcpyHostToDevice);
        }
    }
    if(!rc && nsteps_in) {
        if(palloc(ctx, &d_nin, njobs)) rc = -1;
        else hipMemcpy(d_nin, nsteps_in, njobs * sizeof(int32_t), hipMemcpyHostToDevice);
    }
    if(!rc && njobs > 0) {
        O.points = d_pts;
        O.job_alpha = d_ia;
        O.job_sz = d_isz;
        O.nsteps_in = d_nin;
        O.nsteps_out = d_nout;
        hipMemsetAsync(dp->d_errw, 0, 4 * sizeof(uint32_t), ctx->stream);
        hipMemsetAsync(d_pts, 0, npts * sizeof(bhc_ray_pt2d), ctx->stream);
        O.lanes = fan_lanes(njobs, ctx->num_cus, 0);
        const int blocks = std::min((njobs + O.lanes - 1) / O.lanes, ctx->num_cus * 4 * ctx->bpc);
        if(dp->precision == 64) launch_rays(dp, dp->P64, O, blocks);
        else launch_rays(dp, dp->P32, O, blocks);
        if(hipGetLastError() != hipSuccess || hipStreamSynchronize(ctx->stream) != hipSuccess) {
            rc = fail("ray kernel failed");
        } else {
            hipMemcpy(out->points, d_pts, npts * sizeof(bhc_ray_pt2d), hipMemcpyDeviceToHost);
            hipMemcpy(out->nsteps, d_nout, njobs * sizeof(int32_t), hipMemcpyDeviceToHost);
            uint32_t ew[4];
            hipMemcpy(ew, dp->d_errw, sizeof(ew), hipMemcpyDeviceToHost);
            out->err = ew[0];
            out->warn = ew[1];
            out->err_count = ew[2];
            out->warn_count = ew[3];
        }
    }
    void *fr[] = {d_ia, d_isz, d_nin, d_nout, d_pts};
    for(void *p : fr)
        ctx->pool.put(p);
    bhc_problem_release(dp);
    if(!rc) ctx->prog_final = 1;
    return rc;
}

// ===========================================================================
// Nx2D runs (bellhopcxx Nx2D, RunType[5] == '2'): 2D rays on the bearing
// planes of a 3D environment. The receiver side -- field, arrivals, eigen
// hits, range bins, per-ray statistics, the trace / scatter passes and the
// arrivals merge -- is the 2D run's over NSz * NSx * NSy * Ntheta source
// slots (one per bearing plane); only the trace kernel differs.
// ===========================================================================
namespace {
int upload_nx2d(bhc_ctx *ctx, const bhc_problem3d *p, const bhc_field_out *spec, char run0, bhc_dev_problem **out)
{
    *out = nullptr;
    if(!p) return fail("null problem");
    if(p->RunType[5] != '2') return fail("not an Nx2D problem (RunType[5] must be '2')");
    if(p->precision != 64 && p->precision != 32) return fail("precision must be 32 or 64");
    if(p->NSx < 1 || p->NSy < 1 || p->NSz < 1 || p->NRz < 1 || p->NRr < 1 || p->Ntheta < 1 || p->Nalpha < 1
       || p->Nbeta < 1)
        return fail("Nx2D problem: sources, receivers and launch angles must be non-empty");
    if(p->RunType[4] == 'I') return fail("Nx2D problem: irregular receiver grids are not supported");
    if(run0 != 'R' && p->Nbeta != p->Ntheta)
        return fail("Nx2D problem: the beams must lie on the receiver bearings (Nbeta == Ntheta)");
    if(p->iSingle_beta < 0 || p->iSingle_beta > p->Nbeta) return fail("iSingle_beta out of range");
    const long long nsrc = (long long)p->NSz * p->NSx * p->NSy * p->Ntheta;
    const long long nj = (long long)(p->iSingle_alpha >= 1 ? 1 : p->Nalpha) * (p->iSingle_beta >= 1 ? 1 : p->Nbeta)
        * p->NSx * p->NSy * p->NSz;
    if(nsrc * p->Nalpha >= (1ll << 30) || nj >= (1ll << 30)) return fail("Nx2D problem: too many rays");
    // the 2D stand-in that sizes the receiver side: nsrc source slots, the
    // problem's receivers, declinations and beam pattern; its profile and
    // boundaries are placeholders (the trace kernel reads the 3D ones)
    static const double z2[2] = {0.0, 1.0}, c2[4] = {1500.0, 0.0, 1500.0, 0.0}, zero4[4] = {0, 0, 0, 0};
    static const double rho2[2] = {1.0, 1.0};
    bhc_bdry_node2d nodes[2];
    memset(nodes, 0, sizeof(nodes));
    nodes[0].x[0] = -1.0e10;
    nodes[1].x[0] = 1.0e10;
    nodes[0].t[0] = nodes[1].t[0] = 1.0;
    nodes[0].n[1] = nodes[1].n[1] = 1.0;
    std::vector<float> sz((size_t)nsrc, 0.0f);
    for(int i = 0; i < p->NSz; ++i) sz[i] = p->Sz[i];
    bhc_problem2d q;
    memset(&q, 0, sizeof(q));
    q.precision = p->precision;
    memcpy(q.RunType, p->RunType, 7);
    q.RunType[0] = run0;
    q.RunType[5] = ' ';
    memcpy(q.BeamType, p->BeamType, 4);
    q.BeamType[0] = p->RunType[1];
    q.freq0 = p->freq0;
    q.ssp_type = 'C';
    q.ssp_npts = 2;
    q.ssp_z = z2;
    q.ssp_c = c2;
    q.ssp_cz = zero4;
    q.ssp_rho = rho2;
    q.top_hs = p->top_hs;
    q.bot_hs = p->bot_hs;
    q.ati_type[0] = q.bty_type[0] = 'L';
    q.ati_type[1] = q.bty_type[1] = 'S';
    q.ati_npts = q.bty_npts = 2;
    q.ati = nodes;
    q.bty = nodes;
    q.trc_npts = p->trc_npts;
    q.brc_npts = p->brc_npts;
    q.trc = p->trc;
    q.brc = p->brc;
    q.NSz = (int32_t)nsrc;
    q.NRz = p->NRz;
    q.NRr = p->NRr;
    q.NRz_per_range = p->NRz;
    q.Sz = sz.data();
    q.Rz = p->Rz;
    q.Rr = p->Rr;
    q.Delta_r = p->Delta_r;
    q.Nalpha = p->Nalpha;
    q.iSingle_alpha = p->iSingle_alpha;
    q.alpha = p->alpha;
    q.alpha_cos = p->alpha_cos;
    q.alpha_sin = p->alpha_sin;
    q.Dalpha = p->Dalpha;
    q.deltas = p->deltas;
    q.box_r = p->box_x;
    q.box_z = p->box_z;
    q.NSBPPts = p->NSBPPts;
    q.sbp = p->sbp;
    bhc_dev_problem *dp = nullptr;
    if(bhc_problem_upload2d(ctx, &q, spec, &dp)) return -1;
    dp->njobs = (int)nj;
    dp->nx2d = 1;
    dp->xend_dim = 3;
    int rc = 0;
    if(dp->d_xend) {
        ctx->pool.put(dp->d_xend);
        dp->d_xend = nullptr;
        rc = palloc(ctx, &dp->d_xend, 3 * (size_t)nj);
    }
    // the Nx2D blob replaces the stand-in's
    ctx->pool.put(dp->d_blob);
    dp->d_blob = nullptr;
    std::string err;
    if(!rc && p->precision == 64) {
        std::vector<double> blob;
        rc = bhc3d::pack_nx<double>(p, blob, dp->N64, dp->P64, err);
        if(rc) fail("%s", err.c_str());
        if(!rc) rc = palloc(ctx, (double **)&dp->d_blob, blob.size());
        if(!rc && hipMemcpy(dp->d_blob, blob.data(), blob.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
            rc = fail("blob upload failed");
    } else if(!rc) {
        std::vector<float> blob;
        rc = bhc3d::pack_nx<float>(p, blob, dp->N32, dp->P32, err);
        if(rc) fail("%s", err.c_str());
        if(!rc) rc = palloc(ctx, (float **)&dp->d_blob, blob.size());
        if(!rc && hipMemcpy(dp->d_blob, blob.data(), blob.size() * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
            rc = fail("blob upload failed");
    }
    if(rc) {
        bhc_problem_release(dp);
        return -1;
    }
    dp->lds_bytes = 0;
    dp->P64.base = dp->N64.base = dp->N64.s.base = (const double *)dp->d_blob;
    dp->P32.base = dp->N32.base = dp->N32.s.base = (const float *)dp->d_blob;
    dp->P64.Rz = dp->P32.Rz = dp->N64.Rz = dp->N32.Rz = dp->d_Rz;
    dp->P64.Sz = dp->P32.Sz = dp->N64.Sz = dp->N32.Sz = dp->d_Sz;
    dp->P64.field = dp->P32.field = dp->N64.field = dp->N32.field = dp->d_field;
    dp->P64.njobs = dp->P32.njobs = dp->N64.njobs = dp->N32.njobs = (int)nj;
    *out = dp;
    return 0;
}
} // namespace

extern "C" int bhc_field_runnx2d(bhc_ctx *ctx, const bhc_problem3d *prob, bhc_field_out *out)
{
    if(check_idle(ctx, "bhc_field_runnx2d")) return -1;
    HIPCHECK(hipSetDevice(ctx->device));
    const char r0 = prob ? prob->RunType[0] : 0;
    if(r0 != 'C' && r0 != 'S' && r0 != 'I' && r0 != 'A' && r0 != 'a' && r0 != 'E' && r0 != 'V' && r0 != 'v')
        return fail("bhc_field_runnx2d: run type '%c' is not a field run", r0);
    if(!out) return fail("bhc_field_runnx2d: null output");
    const char r1 = prob->RunType[1];
    if((r1 == 'g' || r1 == 'b') && prob->NRr > 1 && !(prob->Delta_r > 0))
        return fail("bhc_field_runnx2d: ray-centred beams need equally spaced receiver ranges");
    bhc_dev_problem *dp = nullptr;
    if(upload_nx2d(ctx, prob, out, r0, &dp)) return -1;
    int rc = field_launch(ctx, dp, nullptr, 0);
    if(!rc) rc = bhc_field_download(ctx, dp, out);
    bhc_problem_release(dp);
    return rc;
}

extern "C" int bhc_ray_runnx2d(bhc_ctx *ctx, const bhc_problem3d *prob, bhc_ray_out *out, double *origin)
{
    if(check_idle(ctx, "bhc_ray_runnx2d")) return -1;
    if(!out || !out->points || !out->nsteps || !origin) return fail("bhc_ray_runnx2d: null output");
    if(out->max_points_per_ray < 3) return fail("max_points_per_ray must be >= 3");
    HIPCHECK(hipSetDevice(ctx->device));
    bhc_field_out spec;
    memset(&spec, 0, sizeof(spec));
    bhc_dev_problem *dp = nullptr;
    if(upload_nx2d(ctx, prob, &spec, 'R', &dp)) return -1;
    const int njobs = dp->njobs;
    if(prog_begin(ctx, njobs)) {
        bhc_problem_release(dp);
        return -1;
    }
    DevOut O = make_out(dp);
    O.job_begin = 0;
    O.job_end = njobs;
    O.max_points = out->max_points_per_ray;
    int32_t *d_nout = nullptr;
    double *d_org = nullptr;
    bhc_ray_pt2d *d_pts = nullptr;
    int rc = 0;
    const size_t npts = (size_t)njobs * out->max_points_per_ray;
    if(palloc(ctx, &d_pts, npts) || palloc(ctx, &d_nout, njobs) || palloc(ctx, &d_org, 4 * (size_t)njobs)) rc = -1;
    if(!rc) {
        O.points = d_pts;
        O.nsteps_out = d_nout;
        hipMemsetAsync(dp->d_errw, 0, 4 * sizeof(uint32_t), ctx->stream);
        hipMemsetAsync(d_pts, 0, npts * sizeof(bhc_ray_pt2d), ctx->stream);
        int blocks = std::max(1, std::min((njobs + 255) / 256, ctx->num_cus * ctx->bpc));
        if(dp->precision == 64)
            hipLaunchKernelGGL(k_raynx2d<double>, dim3(blocks), dim3(256), 0, ctx->stream, dp->P64, dp->N64, O, d_org);
        else
            hipLaunchKernelGGL(k_raynx2d<float>, dim3(blocks), dim3(256), 0, ctx->stream, dp->P32, dp->N32, O, d_org);
        if(hipGetLastError() != hipSuccess || hipStreamSynchronize(ctx->stream) != hipSuccess) {
            rc = fail("Nx2D ray kernel failed");
        } else {
            hipMemcpy(out->points, d_pts, npts * sizeof(bhc_ray_pt2d), hipMemcpyDeviceToHost);
            hipMemcpy(out->nsteps, d_nout, njobs * sizeof(int32_t), hipMemcpyDeviceToHost);
            hipMemcpy(origin, d_org, 4 * (size_t)njobs * sizeof(double), hipMemcpyDeviceToHost);
            uint32_t ew[4];
            hipMemcpy(ew, dp->d_errw, sizeof(ew), hipMemcpyDeviceToHost);
            out->err = ew[0];
            out->warn = ew[1];
            out->err_count = ew[2];
            out->warn_count = ew[3];
        }
    }
    void *fr[] = {d_nout, d_pts, d_org};
    for(void *q : fr)
        ctx->pool.put(q);
    bhc_problem_release(dp);
    if(!rc) ctx->prog_final = 1;
    return rc;
}

// ===========================================================================
// Batched sweeps: many independent 2D TL problems in one persistent launch.
//
// Every wavefront works on one problem at a time (its descriptor is loaded
// with scalar loads and its SSP / boundary tables are staged in the
// workgroup's LDS), its lanes take that problem's rays from a per-problem
// work counter as they free up, and when the problem has no unclaimed rays
// left and the wavefront's rays have all ended, the wavefront moves to the
// first problem that still has rays. Segments carry their problem index and
// one scatter pass serves every problem. When the segment buffer nears its
// end, every wavefront saves its in-flight rays and exits; the host scatters
// what was traced and relaunches, and the saved rays resume where they
// stopped. The SSP type is dispatched at run time.
// ===========================================================================
namespace {

// (p.y and q.y, the second components of p and q, reach no output of a sweep
// and are not kept)
template<typename real> struct RaySave {
    RayPt<real> p0;
    Trace<real> S;
    Infl<real> I;
    int32_t job, is, isz, ia, active, pad;
};

template<typename real> struct BatchDev {
    const Prob2D<real> *probs;
    int32_t nprob;
    int32_t lds_cap;               // reals of LDS per workgroup for staging
    int32_t *ray_next;             // [nprob] next unclaimed ray
    const int32_t *order;          // the launch's problems, those with the longest rays first
    int32_t nlong;                 // of these, the first whose rays are much longer than the rest (long_problems)
    int32_t *pcursor;              // first place in order whose problem may have unclaimed rays
    uint32_t *perr;                // [nprob][4] err, warn, nerr, nwarn
    unsigned long long *psteps;    // [nprob] steps
    const RaySave<real> *save_in;  // [*nsave_in][64]
    const int32_t *save_in_pid;
    const int32_t *nsave_in;       // saved wavefronts of the previous pass
    int32_t *resume_next;
    RaySave<real> *save_out;
    int32_t *save_out_pid;
    int32_t *nsave_out;
    int32_t *more;                 // set when a wavefront stopped taking new problems
    uint32_t suspend_at;           // segment count at which wavefronts suspend
};

// A copy of a structure that is the same for the whole wavefront, word by word
// through the scalar registers: the compiler then keeps its fields there
// instead of in a register of every lane.
template<typename T> __device__ inline T uniform_copy(const T &src)
{
    static_assert(sizeof(T) % 4 == 0, "whole words");
    int w[sizeof(T) / 4];
    __builtin_memcpy(w, &src, sizeof(T));
#pragma unroll
    for(size_t i = 0; i < sizeof(T) / 4; ++i) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    T t;
    __builtin_memcpy(&t, w, sizeof(T));
    return t;
}

// Rays per wavefront of a launch's longest problems: fewer rays meet fewer
// different cases in a step, so each step is shorter.
constexpr int LONG_LANES = 16;

template<typename real> __device__ inline const real *stage_problem(const Prob2D<real> &P, int lds_cap,
                                                                    unsigned char *lds)
{
    if(P.staged_reals <= 0 || P.staged_reals > lds_cap) return P.base;
    real *L = reinterpret_cast<real *>(lds);
    __syncthreads();
    for(int i = threadIdx.x; i < P.staged_reals; i += blockDim.x) L[i] = P.base[i];
    __syncthreads();
    return L;
}

__device__ inline void flush_problem_err(Err &e, uint32_t *perr)
{
    if(e.err) atomicOr(perr + 0, e.err);
    if(e.warn) atomicOr(perr + 1, e.warn);
    if(e.nerr) atomicAdd(perr + 2, e.nerr);
    if(e.nwarn) atomicAdd(perr + 3, e.nwarn);
    e = Err{0, 0, 0, 0};
}

// How a batched trace hands each step to the receivers: as a descriptor in
// the segment buffer for a later scatter pass, or fused (each lane evaluates
// its own step's receivers at once, with the fast or the reference-arithmetic
// phasor), which needs no segment buffer and no second kernel.
enum { TRACE_DESC = 0, TRACE_FUSED_FAST = 1, TRACE_FUSED_EXACT = 2 };

// One wavefront on one problem until the problem has no unclaimed rays and
// the wavefront's rays have ended (returns 0), or until the segment buffer
// nears its end and the rays are saved (returns 1). `resume` restores a saved
// wavefront. The SSP type is a template parameter, as in the single-problem
// kernel, so that each type runs specialised code. STAGE: where the problem's
// staged tables (SSP, boundaries, receiver depths) are read from -- 1, a copy
// in LDS that the compiler knows to be LDS (ds_read, which does not wait for
// the descriptor stores in flight); 2, global memory known to be global; 3, as
// 1, but with a ray-centred problem's receiver depths, which then no longer fit,
// in global memory; 0, either, through a generic pointer (the fused mappings).
template<typename real, char ST, int MODE, int STAGE>
__device__ __attribute__((noinline)) int run_problem(const BatchDev<real> &Bdref, const DevOut &Oref, int pid, int lanes,
                                                     const RaySave<real> *resume, SegBlock &blk_io, unsigned char *lds,
                                                     unsigned long long &all_steps, unsigned long long &all_contrib)
{
    // copies, for the same reason as the problem's below: through the
    // references their fields would be reloaded after every descriptor store;
    // the segment block in registers (through its reference, every append
    // would read it back from memory and wait for the stores in flight)
    const DevOut O = uniform_copy(Oref);
    SegBlock blk = uniform_copy(blk_io);
    const BatchDev<real> Bd = uniform_copy(Bdref);
    pid = __builtin_amdgcn_readfirstlane(pid);
    const int lane = threadIdx.x;
    // a copy: through a reference the problem's fields would be reloaded after
    // every descriptor store (they might alias)
    Prob2D<real> P = uniform_copy(Bd.probs[pid]);
    const real *G = STAGE == 0 ? P.base : as_global(P.base);
    const real *B;
    if constexpr(STAGE == 1 || STAGE == 3) {
        extern __shared__ __align__(16) unsigned char lds_dyn[];
        real *L = reinterpret_cast<real *>(lds_dyn);
        __syncthreads();
        for(int i = threadIdx.x; i < P.staged_reals; i += blockDim.x) L[i] = G[i];
        __syncthreads();
        B = L;
    } else if constexpr(STAGE == 2) {
        B = G;
    } else {
        B = stage_problem(P, Bd.lds_cap, lds);
    }
    if constexpr(STAGE != 0) { // (null stays null)
        P.ray_stats = as_global(P.ray_stats);
        P.ray_xend = as_global(P.ray_xend);
    }
    // the receiver depths: read for every step of a ray-centred beam, and of a
    // Cartesian one by the fused mappings
    const real *RzT;
    if constexpr(STAGE == 1) RzT = B + P.o_rzs;
    else if constexpr(STAGE == 0) RzT = (P.staged_reals > P.o_rzs && P.staged_reals <= Bd.lds_cap ? B : G) + P.o_rzs;
    else RzT = G + P.o_rzs;
    const int nr = P.njobs;
    const bool full = seg_full(P);
    bool pexh = false, active = false, init_fail = false;
    int result = 0;
    Err e = {0, 0, 0, 0};
    RayPt<real> p0;
    Trace<real> S;
    Infl<real> I;
    int job = 0, isz = 0, ia = 0, is = 0;
    unsigned long long steps = 0, contrib = 0;
    if(resume) {
        const RaySave<real> &sv = resume[lane];
        p0 = sv.p0;
        p0.p.y = p0.q.y = (real)0;
        S = sv.S;
        I = sv.I;
        job = sv.job;
        is = sv.is;
        isz = sv.isz;
        ia = sv.ia;
        active = sv.active != 0;
    }
    for(int iter = 0;; ++iter) {
        if(!pexh) {
            const bool want = !active && lane < lanes;
            unsigned long long need = __ballot(want);
            if(need) {
                int cnt = __popcll(need);
                int leader = __ffsll((unsigned long long)need) - 1;
                int base = 0;
                if(lane == leader) base = atomicAdd(Bd.ray_next + pid, cnt);
                base = __shfl(base, leader);
                if(base + cnt >= nr) pexh = true;
                if(want) {
                    int my = base + __popcll(need & ((1ull << lane) - 1ull));
                    if(my < nr) {
                        job = my;
                        JobIndices(job, P, isz, ia);
                        is = 0;
                        active = RayInit<real, ST>(isz, ia, p0, S, I, P, B, G, e);
                        init_fail = !active;
                        if(!active && P.ray_stats) {
                            P.ray_stats[3 * job] = 0;
                            P.ray_stats[3 * job + 1] = 0;
                            P.ray_stats[3 * job + 2] = 0;
                            P.ray_xend[2 * job] = 0.0;
                            P.ray_xend[2 * job + 1] = 0.0;
                        }
                    }
                }
                note_done(O.prog, init_fail);
                init_fail = false;
            }
        }
        if(!__any(active)) break;
        if((iter & 31) == 31) {
            // HasErrored of this problem (its rays stop, other problems go on),
            // and suspension when the segment buffer nears its end
            if(e.err) atomicOr(Bd.perr + 4 * pid, e.err);
            uint32_t ge = __hip_atomic_load(Bd.perr + 4 * pid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t sc = __hip_atomic_load(O.seg_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if(__any(ge != 0u || e.err != 0u)) {
                if(lane == 0) atomicMax(Bd.ray_next + pid, nr);
                break;
            }
            if(__builtin_amdgcn_readfirstlane(sc) >= Bd.suspend_at) {
                int u = 0;
                if(lane == 0) u = atomicAdd(Bd.nsave_out, 1);
                u = __shfl(u, 0);
                if(lane == 0) Bd.save_out_pid[u] = pid;
                RaySave<real> &sv = Bd.save_out[(size_t)u * WAVE + lane];
                RayPt<real> keep = p0;
                keep.p.y = keep.q.y = (real)0;
                sv.p0 = keep;
                sv.S = S;
                sv.I = I;
                sv.job = job;
                sv.is = is;
                sv.isz = isz;
                sv.ia = ia;
                sv.active = active ? 1 : 0;
                result = 1;
                break;
            }
        }
        step_ray<real, MODE != TRACE_DESC>(
            active, p0, I, is, P, RzT, G, isz, ia,
            [&](const RayPt<real> &a, RayPt<real> &b) { return RayStep<real, ST>(a, b, S, P, B, e); },
            [&](const RayPt<real> &a, RayPt<real> &b, bool top) { RayReflect<real, ST>(a, b, top, S, P, B, G, e); },
            [&](bool has) {
                if constexpr(MODE == TRACE_DESC) return reserve_seg<real>(has, lane, O, blk);
                else return 0u;
            },
            [&](SegDesc<real> &d, uint32_t slot) {
                d.prob = pid;
                if constexpr(MODE == TRACE_DESC) {
                    store_seg(d, slot, O, full);
                } else {
                    DevSink<real> sink{&O, &P, 0};
                    seg_items<real, RT_TL, DevSink<real>, MODE == TRACE_FUSED_FAST>(d, P, G, P.Rz, sink);
                    contrib += sink.nc;
                }
            });
        bool fin = false;
        if(active) {
            if(RayTerminate(p0, is, S, MAXN, P, e)) {
                active = false;
                fin = true;
                steps += (unsigned long long)is;
                if(P.ray_stats) {
                    P.ray_stats[3 * job] = is;
                    P.ray_stats[3 * job + 1] = p0.NumTopBnc;
                    P.ray_stats[3 * job + 2] = p0.NumBotBnc;
                    P.ray_xend[2 * job] = (double)p0.x.x;
                    P.ray_xend[2 * job + 1] = (double)p0.x.y;
                }
            }
        }
        note_done(O.prog, fin);
    }
    flush_problem_err(e, Bd.perr + 4 * pid);
    unsigned long long t = steps;
    for(int off = WAVE / 2; off > 0; off >>= 1) t += __shfl_xor(t, off);
    if(lane == 0 && t) atomicAdd(Bd.psteps + pid, t);
    all_steps += steps;
    all_contrib += contrib;
    blk_io = blk;
    return result;
}

template<typename real, int MODE>
__device__ inline int run_problem_any(const BatchDev<real> &Bd, const DevOut &O, int pid, int lanes, const RaySave<real> *resume,
                                      SegBlock &blk, unsigned char *lds, unsigned long long &all_steps,
                                      unsigned long long &all_contrib)
{
    const Prob2D<real> &Pp = Bd.probs[pid];
    const bool lds_fits = Pp.staged_reals > 0 && Pp.staged_reals <= Bd.lds_cap;
#define BHC_RUN(ST)                                                                                                   \
    if constexpr(MODE == TRACE_DESC) {                                                                                \
        if(lds_fits && !(Pp.isRayCen && Pp.staged_reals <= Pp.o_rzs))                                                 \
            return run_problem<real, ST, MODE, 1>(Bd, O, pid, lanes, resume, blk, lds, all_steps, all_contrib);       \
        if(lds_fits) return run_problem<real, ST, MODE, 3>(Bd, O, pid, lanes, resume, blk, lds, all_steps, all_contrib); \
        return run_problem<real, ST, MODE, 2>(Bd, O, pid, lanes, resume, blk, lds, all_steps, all_contrib);                 \
    } else {                                                                                                          \
        return run_problem<real, ST, MODE, 0>(Bd, O, pid, lanes, resume, blk, lds, all_steps, all_contrib);                 \
    }
    switch(Pp.ssp_type) {
    case 'C': BHC_RUN('C')
    case 'P': BHC_RUN('P')
    case 'S': BHC_RUN('S')
    case 'N': BHC_RUN('N')
    case 'Q': BHC_RUN('Q')
    default: BHC_RUN('A')
    }
#undef BHC_RUN
}

// Two wavefronts per SIMD (at most 256 registers): a single one waits for memory
// and for its own dependent FP64 operations in half of its cycles. Each gets half
// of the LDS (sweep_waves). With the launch's structures in scalar registers
// run_problem nearly fits: its 7 to 11 thousand instructions hold 5 to 14 scratch
// reloads (fused in FP64 11 to 37); the kernel around it spills 75 registers
// across its calls, once per problem.
template<typename real, int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) k_trace_batch(BatchDev<real> Bd, DevOut O)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int lane = threadIdx.x;
    SegBlock blk{0u, 0u, 0u};
    unsigned long long all_steps = 0, all_contrib = 0;
    const int nsave_in = __builtin_amdgcn_readfirstlane(*Bd.nsave_in);
    for(;;) {
        // a saved wavefront of the previous pass first
        int u = -1;
        if(nsave_in > 0) {
            if(lane == 0) u = atomicAdd(Bd.resume_next, 1);
            u = __builtin_amdgcn_readfirstlane(__shfl(u, 0));
        }
        if(u >= 0 && u < nsave_in) {
            int pid = __builtin_amdgcn_readfirstlane(Bd.save_in_pid[u]);
            if(run_problem_any<real, MODE>(Bd, O, pid, WAVE, Bd.save_in + (size_t)u * WAVE, blk, lds_raw, all_steps,
                                           all_contrib))
                break;
            continue;
        }
        // no new problems once the segment buffer nears its end: the next
        // pass continues from the work counters
        uint32_t sc = __hip_atomic_load(O.seg_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if(__builtin_amdgcn_readfirstlane(sc) >= Bd.suspend_at) {
            if(lane == 0) atomicOr(Bd.more, 1);
            break;
        }
        int p = 0, lanes = WAVE;
        if(lane == 0) {
            p = __hip_atomic_load(Bd.pcursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while(p < Bd.nprob
                  && __hip_atomic_load(Bd.ray_next + Bd.order[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                      >= Bd.probs[Bd.order[p]].njobs) {
                atomicMax(Bd.pcursor, p + 1);
                ++p;
            }
            if(p < Bd.nlong) lanes = LONG_LANES;
            p = p < Bd.nprob ? Bd.order[p] : -1;
        }
        p = __builtin_amdgcn_readfirstlane(__shfl(p, 0));
        lanes = __builtin_amdgcn_readfirstlane(__shfl(lanes, 0));
        if(p < 0) break;
        // the launch ends with its longest rays: their wavefronts go first
        // where two share a SIMD
        if(lanes < WAVE) __builtin_amdgcn_s_setprio(3);
        else __builtin_amdgcn_s_setprio(0);
        if(run_problem_any<real, MODE>(Bd, O, p, lanes, nullptr, blk, lds_raw, all_steps, all_contrib)) break;
    }
    seal_block<real>(blk, lane, O);
    for(int off = WAVE / 2; off > 0; off >>= 1) {
        all_steps += __shfl_xor(all_steps, off);
        all_contrib += __shfl_xor(all_contrib, off);
    }
    if(lane == 0) atomicAdd(O.counters + 0, all_steps);
    if(lane == 0 && all_contrib) atomicAdd(O.counters + 1, all_contrib);
}

// Scatter of a batched pass: one wavefront per segment, the segment's problem
// descriptor read through a wavefront-uniform pointer.
template<typename real, bool FAST>
__global__ void __launch_bounds__(256) k_scatter_batch(BatchDev<real> Bd, DevOut O)
{
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE));
    const int nwaves = gridDim.x * (blockDim.x / WAVE);
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    unsigned long long nc = 0;
    for(uint32_t s = (uint32_t)wave; s < n; s += (uint32_t)nwaves) {
        SegDesc<real> d;
        load_seg_core(O, s, d);
        if(d.nitems <= 0) continue;
        const Prob2D<real> P = Bd.probs[__builtin_amdgcn_readfirstlane(d.prob)];
        if(seg_full(P)) load_seg_rest(O, s, d);
        DevSink<real> sink{&O, &P, 0};
        scatter_seg<real, RT_TL, FAST>(d, P, sink, lane);
        nc += sink.nc;
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) nc += __shfl_xor(nc, off);
    if(lane == 0 && nc) atomicAdd(O.counters + 1, nc);
}

// Scatter of a batched pass with one lane per segment: a wavefront loads 64
// descriptors at once (one memory round trip for all of them) and every lane
// walks its own segment's receivers. Batched sweeps of hat beams produce a
// segment per step with only a few receivers each, where a wavefront per
// segment would spend its time waiting for the descriptor. Four wavefronts
// per SIMD (128 VGPRs, a few spills in FP64): the lanes wait on descriptor,
// receiver and problem loads, and more wavefronts hide more of it (3% faster
// than three).
template<typename real, bool FAST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) k_scatter_lanes(BatchDev<real> Bd, DevOut O)
{
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    unsigned long long nc = 0;
    const uint32_t stride = gridDim.x * blockDim.x;
    for(uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += stride) {
        SegDesc<real> d;
        load_seg_core(O, s, d);
        const bool act = d.nitems > 0;
        const unsigned long long am = __ballot(act);
        if(!am) continue;
        // The segments of a wavefront mostly belong to one problem (slots are
        // reserved SEG_BLOCK at a time by one tracing wavefront): then its
        // descriptor is read once, with wavefront-uniform (scalar) loads,
        // instead of by every lane.
        const int pu = __builtin_amdgcn_readfirstlane(__shfl(d.prob, __ffsll(am) - 1));
        if(!__any(act && d.prob != pu)) {
            if(!act) continue;
            // a copy: read through a reference, the problem's fields would be
            // reloaded after every field atomic (they might alias)
            const Prob2D<real> P = Bd.probs[pu];
            if(seg_full(P)) load_seg_rest(O, s, d);
            DevSink<real> sink{&O, &P, 0};
            seg_items<real, RT_TL, DevSink<real>, FAST>(d, P, P.base, P.Rz, sink);
            nc += sink.nc;
        } else {
            if(!act) continue;
            const Prob2D<real> P = Bd.probs[d.prob];
            if(seg_full(P)) load_seg_rest(O, s, d);
            DevSink<real> sink{&O, &P, 0};
            seg_items<real, RT_TL, DevSink<real>, FAST>(d, P, P.base, P.Rz, sink);
            nc += sink.nc;
        }
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) nc += __shfl_xor(nc, off);
    if((threadIdx.x & (WAVE - 1)) == 0 && nc) atomicAdd(O.counters + 1, nc);
}

// Scatter of a batched pass with the items of 64 segments flattened over the
// wavefront: the wavefront copies 64 consecutive descriptors to LDS with
// coalesced loads; the segments' range columns are spread over the lanes (a
// prefix sum of the column counts), each column's depth band is computed, and
// the receivers of all bands are spread over the lanes again, so every lane
// evaluates the same number of receivers whatever the segments' sizes.
// Ray-centred segments are walked by their own lane.
template<typename real, bool FAST>
__global__ void __launch_bounds__(128) k_scatter_flat(BatchDev<real> Bd, DevOut O)
{
    constexpr int NW = 2;                                  // wavefronts per workgroup
    constexpr int W16 = (int)(sizeof(Seg<real>) / 16);     // 16-byte words per descriptor
    __shared__ uint4 stage[NW][WAVE * W16];
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = threadIdx.x / WAVE;
    uint32_t n = *O.seg_count;
    if(n > O.seg_cap) n = O.seg_cap;
    const Seg<real> *S = reinterpret_cast<const Seg<real> *>(stage[w]);
    unsigned long long nc = 0;
    const uint32_t gw = blockIdx.x * NW + (uint32_t)w, nw = gridDim.x * NW;
    for(uint32_t base = gw * WAVE; base < n; base += nw * WAVE) {
        const int cnt = (int)min((uint32_t)WAVE, n - base);
        // word k of the descriptors base .. base + cnt - 1 (consecutive lanes,
        // consecutive slots) into the stage's records
        for(int t = lane; t < cnt * O.seg_words; t += WAVE) {
            const int k = t / cnt, i = t - k * cnt;
            stage[w][(size_t)i * W16 + k] = *reinterpret_cast<const uint4 *>(seg_word(O, k, base + i));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int ncol = 0;
        if(lane < cnt && S[lane].d.nitems > 0) {
            const SegDesc<real> &d = S[lane].d;
            const Prob2D<real> &P = Bd.probs[d.prob];
            if(P.isRayCen) {
                DevSink<real> sink{&O, &P, 0};
                seg_items<real, RT_TL, DevSink<real>, FAST>(d, P, P.base, P.Rz, sink);
                nc += sink.nc;
            } else {
                ncol = (d.ir1 - d.ir0) * d.dir + 1;
            }
        }
        int cexcl;
        const int ctot = wave_excl_scan(ncol, lane, cexcl);
        for(int c0 = 0; c0 < ctot; c0 += WAVE) {
            const int ct = c0 + lane;
            const int seg = wave_owner(cexcl, ct);
            const int sexcl = __shfl(cexcl, seg);
            int ir = 0, i0 = 0, i1 = -1;
            if(ct < ctot) {
                const SegDesc<real> &d = S[seg].d;
                const Prob2D<real> &P = Bd.probs[d.prob];
                cart_column(d, ct - sexcl, P, P.base, ir, i0, i1);
            }
            const int icnt = i1 >= i0 ? i1 - i0 + 1 : 0;
            int iexcl;
            const int itot = wave_excl_scan(icnt, lane, iexcl);
            for(int t0 = 0; t0 < itot; t0 += WAVE) {
                const int t = t0 + lane;
                const int own = wave_owner(iexcl, t);
                const int oir = __shfl(ir, own), oi0 = __shfl(i0, own), oex = __shfl(iexcl, own);
                const int oseg = __shfl(seg, own);
                if(t < itot) {
                    const SegDesc<real> &d = S[oseg].d;
                    const Prob2D<real> P = Bd.probs[d.prob];
                    DevSink<real> sink{&O, &P, 0};
                    item_cart_at<real, RT_TL, DevSink<real>, FAST>(d, oir, oi0 + (t - oex), P, P.base, P.Rz, sink);
                    nc += sink.nc;
                }
            }
        }
        // the stage is rewritten by the next group
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    for(int off = WAVE / 2; off > 0; off >>= 1) nc += __shfl_xor(nc, off);
    if(lane == 0 && nc) atomicAdd(O.counters + 1, nc);
}

// Per-pass counters reset by a kernel (the passes are replayed as HIP graphs,
// which take no memset nodes here).
__global__ void k_pass_reset(uint32_t *seg_count, uint32_t *overflow, int32_t *resume, int32_t *nsave_out,
                             int32_t *more)
{
    if(threadIdx.x == 0) {
        *seg_count = 0u;
        *overflow = 0u;
        *resume = 0;
        *nsave_out = 0;
        *more = 0;
    }
}

} // namespace

struct bhc_sweep {
    bhc_ctx *ctx;
    int precision, nprob;
    int with_stats;
    bool any_full;              // some problem's segments need the descriptor's rest
    std::vector<int> njobs, nrz, nrr, nsz;
    std::vector<size_t> field_off, stats_off;   // in floats / rays
    size_t field_floats, total_rays;
    void *d_blobs;
    void *d_probs;
    float *d_rzsz;
    float *d_fields;
    int32_t *d_stats;
    double *d_xend;
    std::vector<double> est;    // steps of a ray, about (the order of the problems)
    int32_t *d_order;           // of the range order_p0, order_p1
    int order_p0, order_p1;
    int nlong;                  // its first problems that LONG_LANES rays per wavefront trace
    int32_t *d_ray_next, *d_pcursor, *d_resume, *d_nsave, *d_more;   // d_nsave: [2], one per parity
    uint32_t *d_perr;
    unsigned long long *d_psteps, *d_counters;
    void *d_save[2];
    int32_t *d_save_pid[2];
    int max_waves;
    int lds_bytes, lds_bytes_max;
    int lds_limit;              // largest budget that can be set
    int passes;
    int scatter_blocks;
    int scatter_lanes;          // 0: one wavefront per segment, 1: one lane per segment, 2: 64 segments' receivers flattened over a wavefront
    double trace_ms, scatter_ms;
    // HIP graphs of one pass (reset, trace, scatter), one per parity of the
    // saved-ray buffers; rebuilt when the launch configuration changes
    bool use_graph;
    hipGraphExec_t graph[2];
    int graph_key[5];
    bool tuned;
};

extern "C" void bhc_sweep_release(bhc_sweep *sw)
{
    if(!sw) return;
    (void)hipSetDevice(sw->ctx->device);
    (void)hipStreamSynchronize(sw->ctx->stream);
    void *ptrs[] = {sw->d_blobs, sw->d_probs, sw->d_rzsz,  sw->d_fields,   sw->d_stats,  sw->d_xend,
                    sw->d_order, sw->d_ray_next, sw->d_pcursor, sw->d_resume, sw->d_nsave, sw->d_more, sw->d_perr, sw->d_psteps,
                    sw->d_counters, sw->d_save[0], sw->d_save[1], sw->d_save_pid[0], sw->d_save_pid[1]};
    for(void *p : ptrs)
        if(p) (void)hipFree(p);
    for(int k = 0; k < 2; ++k)
        if(sw->graph[k]) (void)hipGraphExecDestroy(sw->graph[k]);
    delete sw;
}

namespace {

constexpr int SWEEP_LDS2 = 20480;   // LDS per trace wavefront that leaves room for two per SIMD

// Segments that the sweep's wavefronts may add between two polls: 2 per lane
// per step, 32 steps apart, plus one partly used slot block each.
size_t sweep_margin(int waves) { return (size_t)waves * (2 * 32 * WAVE + 2 * SEG_BLOCK); }

// Wavefronts of a sweep's trace: two per SIMD where the LDS budget and the
// segment buffer (which must hold their margin twice over) allow it, else one.
int sweep_waves(const bhc_sweep *sw, size_t seg_cap)
{
    const bool two = sw->lds_bytes <= SWEEP_LDS2 && 2 * sweep_margin(sw->max_waves) < seg_cap;
    return two ? sw->max_waves : sw->max_waves / 2;
}

template<typename real>
int sweep_upload(bhc_sweep *sw, const bhc_problem2d *const *probs)
{
    bhc_ctx *ctx = sw->ctx;
    int n = sw->nprob;
    std::vector<Prob2D<real>> P(n);
    std::vector<real> blobs;
    std::vector<size_t> boff(n);
    std::vector<float> rzsz;
    std::vector<size_t> rzoff(n), szoff(n);
    size_t max_staged = 0, max_whole = 0;
    sw->field_off.resize(n);
    sw->stats_off.resize(n);
    sw->field_floats = 0;
    sw->total_rays = 0;
    for(int i = 0; i < n; ++i) {
        const bhc_problem2d *p = probs[i];
        std::vector<real> blob;
        std::string err;
        if(pack<real>(p, blob, P[i], err)) return fail("problem %d: %s", i, err.c_str());
        boff[i] = blobs.size();
        blobs.insert(blobs.end(), blob.begin(), blob.end());
        while(blobs.size() % 32) blobs.push_back((real)0);
        sw->any_full = sw->any_full || seg_full(P[i]);
        // the receiver depths are read for every step of a ray-centred beam:
        // staged where they leave room for two wavefronts per SIMD (48 seamount
        // environments of 501 depths, FP32: trace 28.9 ms instead of
        // 30.3). Cartesian beams' descriptors do not need them.
        if(!(P[i].isRayCen && P[i].staged_reals * sizeof(real) <= (size_t)SWEEP_LDS2)) P[i].staged_reals = P[i].o_rzs;
        max_staged = std::max(max_staged, (size_t)P[i].staged_reals);
        // the tables with every column: receiver depths, whole boundary nodes and
        // the sound speeds that splines do not read
        const size_t whole = (size_t)P[i].o_rzs + p->NRz
            + (P[i].node == NODE_LINE ? (size_t)(NODE_SHORT - NODE_LINE) * (p->ati_npts + p->bty_npts) : 0)
            + (p->ssp_type == 'S' || p->ssp_type == 'P' ? 4 * (size_t)p->ssp_npts : 0);
        max_whole = std::max(max_whole, whole);
        rzoff[i] = rzsz.size();
        rzsz.insert(rzsz.end(), p->Rz, p->Rz + p->NRz);
        szoff[i] = rzsz.size();
        rzsz.insert(rzsz.end(), p->Sz, p->Sz + p->NSz);
        // steps of a ray, about: one per step length, boundary node and profile
        // knot passed on a zigzag at 15 degrees
        const double depth = std::max(1e-3, p->bot_hs.depth > 0 ? p->bot_hs.depth : p->box_z);
        sw->est.push_back(p->box_r / p->deltas + p->bty_npts + p->ati_npts + 0.27 * p->box_r / depth * p->ssp_npts);
        sw->njobs.push_back((p->iSingle_alpha >= 1 ? 1 : p->Nalpha) * p->NSz);
        sw->nsz.push_back(p->NSz);
        sw->nrz.push_back(p->NRz_per_range);
        sw->nrr.push_back(p->NRr);
        sw->field_off[i] = sw->field_floats;
        sw->field_floats += 2 * (size_t)p->NSz * p->NRz_per_range * p->NRr;
        sw->field_floats = (sw->field_floats + 63) / 64 * 64;
        sw->stats_off[i] = sw->total_rays;
        sw->total_rays += sw->njobs.back();
    }
    // LDS per workgroup: by default at most 20 KiB, so that eight
    // single-wavefront workgroups (two per SIMD) fit a CU's 160 KiB; up to
    // 40 KiB can be set, which leaves one per SIMD. Larger tables stay in
    // global memory
    size_t cap_reals = std::min<size_t>((size_t)40960, (size_t)ctx->lds_max) / sizeof(real);
    size_t lds_reals = std::min(max_staged, cap_reals);
    sw->lds_bytes_max = (int)(lds_reals * sizeof(real));
    sw->lds_bytes = std::min(sw->lds_bytes_max, SWEEP_LDS2);
    sw->lds_limit = (int)(std::min(max_whole, cap_reals) * sizeof(real));
    if(dalloc((real **)&sw->d_blobs, blobs.size()) || dalloc(&sw->d_rzsz, rzsz.size())
       || dalloc(&sw->d_fields, sw->field_floats) || dalloc((Prob2D<real> **)&sw->d_probs, (size_t)n)
       || dalloc(&sw->d_order, (size_t)n) || dalloc(&sw->d_ray_next, (size_t)n) || dalloc(&sw->d_pcursor, 1) || dalloc(&sw->d_resume, 1)
       || dalloc(&sw->d_nsave, 2) || dalloc(&sw->d_more, 1) || dalloc(&sw->d_perr, 4 * (size_t)n)
       || dalloc(&sw->d_psteps, (size_t)n)
       || dalloc(&sw->d_counters, 2))
        return -1;
    if(sw->with_stats
       && (dalloc(&sw->d_stats, 3 * sw->total_rays) || dalloc(&sw->d_xend, 2 * sw->total_rays)))
        return -1;
    HIPCHECK(hipMemcpy(sw->d_blobs, blobs.data(), blobs.size() * sizeof(real), hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(sw->d_rzsz, rzsz.data(), rzsz.size() * sizeof(float), hipMemcpyHostToDevice));
    for(int i = 0; i < n; ++i) {
        P[i].base = (const real *)sw->d_blobs + boff[i];
        if((size_t)P[i].staged_reals > lds_reals) P[i].staged_reals = 0;
        P[i].Rz = sw->d_rzsz + rzoff[i];
        P[i].Sz = sw->d_rzsz + szoff[i];
        P[i].field = sw->d_fields + sw->field_off[i];
        P[i].njobs = sw->njobs[i];
        if(sw->with_stats) {
            P[i].ray_stats = sw->d_stats + 3 * sw->stats_off[i];
            P[i].ray_xend = sw->d_xend + 2 * sw->stats_off[i];
        }
    }
    HIPCHECK(hipMemcpy(sw->d_probs, P.data(), n * sizeof(Prob2D<real>), hipMemcpyHostToDevice));
    sw->max_waves = ctx->num_cus * 8;   // two per SIMD
    size_t save_units = (size_t)sw->max_waves;
    for(int k = 0; k < 2; ++k)
        if(dalloc((RaySave<real> **)&sw->d_save[k], save_units * WAVE) || dalloc(&sw->d_save_pid[k], save_units))
            return -1;
    sw->scatter_blocks = ctx->num_cus * 8;
    sw->scatter_lanes = 1;
    return 0;
}

// Device view of problems [p0, p1): problem indices inside the launch (work
// counters, saved rays, segment descriptors) are relative to p0.
template<typename real> BatchDev<real> batch_dev(bhc_sweep *sw, int p0, int p1)
{
    BatchDev<real> Bd;
    memset(&Bd, 0, sizeof(Bd));
    Bd.probs = (const Prob2D<real> *)sw->d_probs + p0;
    Bd.nprob = p1 - p0;
    Bd.lds_cap = sw->lds_bytes / (int)sizeof(real);
    Bd.order = sw->d_order;
    Bd.ray_next = sw->d_ray_next + p0;
    Bd.pcursor = sw->d_pcursor;
    Bd.perr = sw->d_perr + 4 * (size_t)p0;
    Bd.psteps = sw->d_psteps + p0;
    Bd.resume_next = sw->d_resume;
    Bd.more = sw->d_more;
    return Bd;
}

template<typename real> DevOut batch_out(bhc_sweep *sw)
{
    bhc_ctx *c = sw->ctx;
    DevOut O;
    memset(&O, 0, sizeof(O));
    O.counters = sw->d_counters;
    O.segs = c->segs;
    O.seg_count = c->d_seg_count;
    O.overflow = c->d_overflow;
    O.seg_cap = seg_slots<real>(c->seg_bytes, sw->any_full);
    O.seg_words = sw->any_full ? SEG_NW<real> : SEG_NC<real>;
    O.prog = prog_of(c);
    return O;
}

// Enqueue one pass of parity `cur` (reads saved rays from buffer cur, saves
// into 1 - cur) on the context's stream.
template<typename real> void enqueue_pass(bhc_sweep *sw, BatchDev<real> Bd, const DevOut &O, int cur, hipEvent_t e_mid)
{
    bhc_ctx *c = sw->ctx;
    hipStream_t s = c->stream;
    Bd.save_in = (const RaySave<real> *)sw->d_save[cur];
    Bd.save_in_pid = sw->d_save_pid[cur];
    Bd.nsave_in = sw->d_nsave + cur;
    Bd.save_out = (RaySave<real> *)sw->d_save[1 - cur];
    Bd.save_out_pid = sw->d_save_pid[1 - cur];
    Bd.nsave_out = sw->d_nsave + (1 - cur);
    const int waves = sweep_waves(sw, O.seg_cap);
    hipLaunchKernelGGL(k_pass_reset, dim3(1), dim3(64), 0, s, c->d_seg_count, c->d_overflow, sw->d_resume,
                       sw->d_nsave + (1 - cur), sw->d_more);
    if(sw->scatter_lanes == 3) {
        // fused: the trace evaluates every step's receivers itself
        if(c->exact_phasor)
            hipLaunchKernelGGL((k_trace_batch<real, TRACE_FUSED_EXACT>), dim3(waves), dim3(WAVE), sw->lds_bytes,
                               s, Bd, O);
        else
            hipLaunchKernelGGL((k_trace_batch<real, TRACE_FUSED_FAST>), dim3(waves), dim3(WAVE), sw->lds_bytes,
                               s, Bd, O);
        if(e_mid) (void)hipEventRecord(e_mid, s);
        return;
    }
    hipLaunchKernelGGL((k_trace_batch<real, TRACE_DESC>), dim3(waves), dim3(WAVE), sw->lds_bytes, s, Bd, O);
    if(e_mid) (void)hipEventRecord(e_mid, s);
    if(sw->scatter_lanes == 2) {
        if(c->exact_phasor)
            hipLaunchKernelGGL((k_scatter_flat<real, false>), dim3(2 * sw->scatter_blocks), dim3(128), 0, s, Bd, O);
        else
            hipLaunchKernelGGL((k_scatter_flat<real, true>), dim3(2 * sw->scatter_blocks), dim3(128), 0, s, Bd, O);
    } else if(sw->scatter_lanes) {
        if(c->exact_phasor)
            hipLaunchKernelGGL((k_scatter_lanes<real, false>), dim3(sw->scatter_blocks), dim3(256), 0, s, Bd, O);
        else
            hipLaunchKernelGGL((k_scatter_lanes<real, true>), dim3(sw->scatter_blocks), dim3(256), 0, s, Bd, O);
    } else {
        if(c->exact_phasor)
            hipLaunchKernelGGL((k_scatter_batch<real, false>), dim3(sw->scatter_blocks), dim3(256), 0, s, Bd, O);
        else
            hipLaunchKernelGGL((k_scatter_batch<real, true>), dim3(sw->scatter_blocks), dim3(256), 0, s, Bd, O);
    }
}

// Trace + scatter problems [p0, p1) in one persistent launch (a sequence of
// passes): zero their fields and counters, then passes until no ray is left.
// Graph mode replays one captured graph per pass; eager mode times the trace
// and scatter kernels of every pass.
template<typename real> int sweep_core(bhc_sweep *sw, int p0, int p1, bool graph)
{
    bhc_ctx *c = sw->ctx;
    hipStream_t s = c->stream;
    if(ensure_segs(c)) return -1;
    BatchDev<real> Bd = batch_dev<real>(sw, p0, p1);
    DevOut O = batch_out<real>(sw);
    size_t margin = sweep_margin(sweep_waves(sw, O.seg_cap));
    if(margin * 2 >= O.seg_cap) return fail("segment buffer too small for a batched sweep (raise BHC_SEG_BUFFER_MB)");
    Bd.suspend_at = (uint32_t)(O.seg_cap - margin);
    const int np = p1 - p0;
    {
        long long rays = 0;
        for(int i = p0; i < p1; ++i) rays += sw->njobs[i];
        if(prog_begin(c, rays)) return -1;
    }
    // The problems with the longest rays go first: a launch ends with its
    // longest ray, and one of 17800 steps among 1700 on average, started last,
    // would run alone at the end.
    if(sw->order_p0 != p0 || sw->order_p1 != p1) {
        std::vector<int32_t> order(np);
        for(int i = 0; i < np; ++i) order[i] = i;
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return sw->est[p0 + a] > sw->est[p0 + b]; });
        // much longer than the mean over the rays, and together on at most a
        // quarter of the wavefronts
        double rays = 0, steps = 0;
        for(int i = p0; i < p1; ++i) {
            rays += sw->njobs[i];
            steps += sw->njobs[i] * sw->est[i];
        }
        long long waves = 0;
        for(sw->nlong = 0; sw->nlong < np; ++sw->nlong) {
            const int q = p0 + order[sw->nlong];
            waves += (sw->njobs[q] + LONG_LANES - 1) / LONG_LANES;
            if(!(sw->est[q] > 1.5 * steps / rays) || waves > sw->max_waves / 4) break;
        }
        HIPCHECK(hipStreamSynchronize(s));
        HIPCHECK(hipMemcpy(sw->d_order, order.data(), np * sizeof(int32_t), hipMemcpyHostToDevice));
        sw->order_p0 = p0;
        sw->order_p1 = p1;
    }
    Bd.nlong = sw->nlong;
    const size_t f0 = sw->field_off[p0], f1 = p1 == sw->nprob ? sw->field_floats : sw->field_off[p1];
    HIPCHECK(hipMemsetAsync(sw->d_fields + f0, 0, (f1 - f0) * sizeof(float), s));
    HIPCHECK(hipMemsetAsync(sw->d_ray_next + p0, 0, np * sizeof(int32_t), s));
    HIPCHECK(hipMemsetAsync(sw->d_pcursor, 0, sizeof(int32_t), s));
    HIPCHECK(hipMemsetAsync(sw->d_nsave, 0, 2 * sizeof(int32_t), s));
    HIPCHECK(hipMemsetAsync(sw->d_perr + 4 * (size_t)p0, 0, 4 * np * sizeof(uint32_t), s));
    HIPCHECK(hipMemsetAsync(sw->d_psteps + p0, 0, np * sizeof(unsigned long long), s));
    HIPCHECK(hipMemsetAsync(sw->d_counters, 0, 2 * sizeof(unsigned long long), s));
    if(sw->with_stats) {
        const size_t r0 = sw->stats_off[p0], r1 = p1 == sw->nprob ? sw->total_rays : sw->stats_off[p1];
        HIPCHECK(hipMemsetAsync(sw->d_stats + 3 * r0, 0, 3 * (r1 - r0) * sizeof(int32_t), s));
        HIPCHECK(hipMemsetAsync(sw->d_xend + 2 * r0, 0, 2 * (r1 - r0) * sizeof(double), s));
    }
    if(graph) {
        int key[5] = {sw->scatter_blocks, sw->lds_bytes, p0, p1, sw->scatter_lanes};
        if(!sw->graph[0] || memcmp(key, sw->graph_key, sizeof(key)) != 0) {
            for(int k = 0; k < 2; ++k) {
                if(sw->graph[k]) (void)hipGraphExecDestroy(sw->graph[k]);
                sw->graph[k] = nullptr;
                hipGraph_t g = nullptr;
                HIPCHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                enqueue_pass<real>(sw, Bd, O, k, nullptr);
                HIPCHECK(hipStreamEndCapture(s, &g));
                hipError_t e = hipGraphInstantiate(&sw->graph[k], g, nullptr, nullptr, 0);
                (void)hipGraphDestroy(g);
                HIPCHECK(e);
            }
            memcpy(sw->graph_key, key, sizeof(key));
        }
    }
    HIPCHECK(hipEventRecord(c->ev0, s));
    int cur = 0;
    sw->passes = 0;
    sw->trace_ms = sw->scatter_ms = 0.0;
    hipEvent_t e0, e1, e2;
    HIPCHECK(hipEventCreate(&e0));
    HIPCHECK(hipEventCreate(&e1));
    HIPCHECK(hipEventCreate(&e2));
    int rc = 0;
    for(;;) {
        (void)hipEventRecord(e0, s);
        if(graph) {
            if(hipGraphLaunch(sw->graph[cur], s) != hipSuccess) {
                rc = fail("sweep: graph launch failed");
                break;
            }
        } else {
            enqueue_pass<real>(sw, Bd, O, cur, e1);
        }
        (void)hipEventRecord(e2, s);
        if(hipGetLastError() != hipSuccess) {
            rc = fail("sweep: kernel launch failed");
            break;
        }
        int32_t ns = 0, more = 0;
        uint32_t of = 0;
        if(hipMemcpyAsync(&ns, sw->d_nsave + (1 - cur), sizeof(int32_t), hipMemcpyDeviceToHost, s) != hipSuccess
           || hipMemcpyAsync(&more, sw->d_more, sizeof(int32_t), hipMemcpyDeviceToHost, s) != hipSuccess
           || hipMemcpyAsync(&of, c->d_overflow, sizeof(uint32_t), hipMemcpyDeviceToHost, s) != hipSuccess
           || hipStreamSynchronize(s) != hipSuccess) {
            rc = fail("sweep: pass failed");
            break;
        }
        float a = 0.f, b = 0.f;
        if(graph) {
            (void)hipEventElapsedTime(&a, e0, e2);
        } else {
            (void)hipEventElapsedTime(&a, e0, e1);
            (void)hipEventElapsedTime(&b, e1, e2);
        }
        sw->trace_ms += a;
        sw->scatter_ms += b;
        ++sw->passes;
        if(of) {
            rc = fail("sweep: segment buffer overflow (suspension margin too small)");
            break;
        }
        if(ns == 0 && !more) break;
        if(sw->passes > 100000) {
            rc = fail("sweep: no progress");
            break;
        }
        cur = 1 - cur;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipEventDestroy(e2);
    HIPCHECK(hipEventRecord(c->ev1, s));
    c->passes = sw->passes;
    if(!rc) c->prog_final = 1;
    return rc;
}

// Launch-configuration search on the sweep's first problems (eager passes,
// kernel times from HIP events): the scatter grid and whether the problems'
// tables are staged in LDS. Keeps the fastest.
template<typename real> int sweep_tune(bhc_sweep *sw)
{
    int nsub = std::min(sw->nprob, 64);
    int cus = sw->ctx->num_cus;
    const int grids[3] = {cus * 4, cus * 8, cus * 16};
    // staging budgets: the default (two wavefronts per SIMD, problems with
    // larger tables unstaged), the largest table's (one wavefront per SIMD where
    // it is over the default) and none
    const int ldss[3] = {std::min(sw->lds_bytes_max, SWEEP_LDS2), sw->lds_bytes_max, 0};
    auto timed = [&](int mode, int blocks, int lds, int n, double &t) -> int {
        sw->scatter_lanes = mode;
        sw->scatter_blocks = blocks;
        sw->lds_bytes = lds;
        for(int rep = 0; rep < 2; ++rep) {
            if(sweep_core<real>(sw, 0, n, false)) return -1;
            if(rep == 1) t = sw->trace_ms + sw->scatter_ms;
        }
        return 0;
    };
    // the staging budget acts on the trace and the mapping / grid on the
    // scatter: choose the scatter's at the default budget, then the budget
    int best_blocks = grids[0], best_lanes = 1, best_lds = ldss[0];
    double best = 1e300, t = 0.0;
    for(int mode = 0; mode < 4; ++mode)
        for(int gi = 0; gi < (mode == 3 ? 1 : 3); ++gi) {   // the fused mode launches no scatter
            if(timed(mode, grids[gi], ldss[0], nsub, t)) return -1;
            if(t < best) {
                best = t;
                best_blocks = grids[gi];
                best_lanes = mode;
            }
        }
    // the budget acts on how well the trace hides its waits, which shows once
    // there is work for every wavefront: 64 problems end with a few long rays on
    // an idle chip, where one wavefront per SIMD is the faster (of 4096 unlike
    // environments, 303 fields/s with the budget that 64 chose, 363 with two
    // wavefronts per SIMD)
    const int nlds = std::min(sw->nprob, 256);
    best = 1e300;
    for(int li = 0; li < 3; ++li) {
        if(li > 0 && ldss[li] == ldss[li - 1]) continue;
        if(timed(best_lanes, best_blocks, ldss[li], nlds, t)) return -1;
        if(t < best) {
            best = t;
            best_lds = ldss[li];
        }
    }
    sw->scatter_blocks = best_blocks;
    sw->lds_bytes = best_lds;
    sw->scatter_lanes = best_lanes;
    sw->tuned = true;
    return 0;
}

} // namespace

extern "C" int bhc_sweep_upload2d(bhc_ctx *ctx, const bhc_problem2d *const *probs, int nprob, int with_stats,
                                  bhc_sweep **out)
{
    *out = nullptr;
    if(!ctx || !probs || nprob < 1) return fail("bhc_sweep_upload2d: no problems");
    int prec = probs[0]->precision;
    for(int i = 0; i < nprob; ++i) {
        if(check_problem(probs[i])) return -1;
        char r0 = probs[i]->RunType[0];
        if(r0 != 'C' && r0 != 'S' && r0 != 'I') return fail("sweep problem %d: only TL run types are batched", i);
        if(probs[i]->precision != prec) return fail("sweep problem %d: all problems must share the precision", i);
    }
    HIPCHECK(hipSetDevice(ctx->device));
    bhc_sweep *sw = new bhc_sweep();
    sw->ctx = ctx;
    sw->precision = prec;
    sw->nprob = nprob;
    sw->with_stats = with_stats;
    sw->use_graph = true;
    if(const char *e = getenv("BHC_SWEEP_GRAPH")) sw->use_graph = atoi(e) != 0;
    int rc = prec == 64 ? sweep_upload<double>(sw, probs) : sweep_upload<float>(sw, probs);
    if(rc) {
        bhc_sweep_release(sw);
        return -1;
    }
    *out = sw;
    return 0;
}

extern "C" int bhc_sweep_launch(bhc_ctx *ctx, bhc_sweep *sw)
{
    if(check_idle(ctx, "bhc_sweep_launch")) return -1;
    if(!ctx || !sw || sw->ctx != ctx) return fail("bhc_sweep_launch: bad arguments");
    HIPCHECK(hipSetDevice(ctx->device));
    return sw->precision == 64 ? sweep_core<double>(sw, 0, sw->nprob, sw->use_graph)
                               : sweep_core<float>(sw, 0, sw->nprob, sw->use_graph);
}

extern "C" int bhc_sweep_launch_range(bhc_ctx *ctx, bhc_sweep *sw, int p0, int p1)
{
    if(check_idle(ctx, "bhc_sweep_launch_range")) return -1;
    if(!ctx || !sw || sw->ctx != ctx) return fail("bhc_sweep_launch_range: bad arguments");
    if(p0 < 0 || p1 > sw->nprob || p0 >= p1)
        return fail("bhc_sweep_launch_range: range [%d, %d) outside the sweep's %d problems", p0, p1, sw->nprob);
    HIPCHECK(hipSetDevice(ctx->device));
    return sw->precision == 64 ? sweep_core<double>(sw, p0, p1, sw->use_graph)
                               : sweep_core<float>(sw, p0, p1, sw->use_graph);
}

extern "C" int bhc_sweep_autotune(bhc_ctx *ctx, bhc_sweep *sw, int *scatter_blocks, int *lds_bytes,
                                  int *scatter_lanes)
{
    if(check_idle(ctx, "bhc_sweep_autotune")) return -1;
    if(!ctx || !sw || sw->ctx != ctx) return fail("bhc_sweep_autotune: bad arguments");
    HIPCHECK(hipSetDevice(ctx->device));
    int rc = sw->precision == 64 ? sweep_tune<double>(sw) : sweep_tune<float>(sw);
    if(scatter_blocks) *scatter_blocks = sw->scatter_blocks;
    if(lds_bytes) *lds_bytes = sw->lds_bytes;
    if(scatter_lanes) *scatter_lanes = sw->scatter_lanes;
    return rc;
}

extern "C" int bhc_sweep_set_launch(bhc_sweep *sw, int scatter_blocks, int lds_bytes)
{
    if(!sw) return fail("bhc_sweep_set_launch: null sweep");
    const int rsz = sw->precision == 64 ? (int)sizeof(double) : (int)sizeof(float);
    if(scatter_blocks < 1 || scatter_blocks > (1 << 20)) return fail("bhc_sweep_set_launch: scatter_blocks out of range");
    if(lds_bytes < 0 || lds_bytes > sw->lds_limit || lds_bytes % rsz)
        return fail("bhc_sweep_set_launch: lds_bytes must be a multiple of %d in [0, %d]", rsz, sw->lds_limit);
    sw->scatter_blocks = scatter_blocks;
    sw->lds_bytes = std::min(lds_bytes, sw->lds_bytes_max);
    sw->tuned = true;
    return 0;
}

extern "C" int bhc_sweep_set_scatter(bhc_sweep *sw, int mapping)
{
    if(!sw || mapping < 0 || mapping > 3) return fail("bhc_sweep_set_scatter: bad arguments");
    sw->scatter_lanes = mapping;
    return 0;
}

extern "C" int bhc_sweep_set_graph(bhc_sweep *sw, int use_graph)
{
    if(!sw) return fail("bhc_sweep_set_graph: null sweep");
    sw->use_graph = use_graph != 0;
    return 0;
}

extern "C" int bhc_sweep_stats(bhc_sweep *sw, double *trace_ms, double *scatter_ms, int *passes, long long *steps,
                               long long *contrib)
{
    if(!sw) return fail("bhc_sweep_stats: null sweep");
    unsigned long long cnt[2] = {0, 0};
    HIPCHECK(hipStreamSynchronize(sw->ctx->stream));
    HIPCHECK(hipMemcpy(cnt, sw->d_counters, sizeof(cnt), hipMemcpyDeviceToHost));
    if(trace_ms) *trace_ms = sw->trace_ms;
    if(scatter_ms) *scatter_ms = sw->scatter_ms;
    if(passes) *passes = sw->passes;
    if(steps) *steps = (long long)cnt[0];
    if(contrib) *contrib = (long long)cnt[1];
    return 0;
}

extern "C" int bhc_sweep_download(bhc_ctx *ctx, bhc_sweep *sw, int iprob, bhc_field_out *out)
{
    if(!ctx || !sw || iprob < 0 || iprob >= sw->nprob || !out) return fail("bhc_sweep_download: bad arguments");
    HIPCHECK(hipSetDevice(ctx->device));
    HIPCHECK(hipStreamSynchronize(ctx->stream));
    size_t nf = 2 * (size_t)sw->nsz[iprob] * sw->nrz[iprob] * sw->nrr[iprob];
    if(out->field)
        HIPCHECK(hipMemcpy(out->field, sw->d_fields + sw->field_off[iprob], nf * sizeof(float),
                           hipMemcpyDeviceToHost));
    uint32_t ew[4];
    HIPCHECK(hipMemcpy(ew, sw->d_perr + 4 * iprob, sizeof(ew), hipMemcpyDeviceToHost));
    out->err = ew[0];
    out->warn = ew[1];
    out->err_count = ew[2];
    out->warn_count = ew[3];
    unsigned long long st = 0;
    HIPCHECK(hipMemcpy(&st, sw->d_psteps + iprob, sizeof(st), hipMemcpyDeviceToHost));
    out->total_steps = (int64_t)st;
    out->total_contrib = 0;
    if(out->ray_nsteps && sw->with_stats) {
        int nj = sw->njobs[iprob];
        std::vector<int32_t> stv(3 * (size_t)nj);
        HIPCHECK(hipMemcpy(stv.data(), sw->d_stats + 3 * sw->stats_off[iprob], stv.size() * sizeof(int32_t),
                           hipMemcpyDeviceToHost));
        for(int j = 0; j < nj; ++j) {
            out->ray_nsteps[j] = stv[3 * j];
            if(out->ray_ntop) out->ray_ntop[j] = stv[3 * j + 1];
            if(out->ray_nbot) out->ray_nbot[j] = stv[3 * j + 2];
        }
        if(out->ray_xend)
            HIPCHECK(hipMemcpy(out->ray_xend, sw->d_xend + 2 * sw->stats_off[iprob], 2 * (size_t)nj * sizeof(double),
                               hipMemcpyDeviceToHost));
    }
    return 0;
}

#include "field3d.h"
