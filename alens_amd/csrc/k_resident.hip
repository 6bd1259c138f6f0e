// k_resident.hip -- BBPGD solves whose operator stays on the chip (gfx950).
//
// The general kernel (k_solve.hip) streams the operator from memory in every iteration and meets at two
// grid barriers; below a few hundred thousand rows its iteration is made of barriers, L2 invalidations and
// dependent round trips, not of bytes.  Here the blocks of one system keep their share of the operator for
// the whole solve - the rods' adjacency slots in LDS, the rows' geometry, rhs and iterate in registers -
// and exchange only (x, g) per row, U per rod and the chunk partials.
//
// Exchanged words carry their own readiness.  Every word is written and read at agent scope (past the
// non-coherent L2s), and a word not yet written in this iteration holds a sentinel that no arithmetic
// produces (a signalling NaN), so a reader polls the data it needs and nothing else: no barrier between
// the phases, no cache write-back or invalidation.
//   gather    every slot of the block polls (x, g) of its row, all slots at once.
//   phase A   v = P(x - alpha g) of every slot; then one lane per rod adds v_j w_j in the slots' order,
//             U = M F, and stores U.
//   phase B   the block polls the velocities of the rods its rows touch into LDS, each rod once; then a lane per
//             row or two: new (x, g), residual and products, stored (x, g); the lanes of a chunk fold its
//             partials in the fixed order and store them.
//   fold      256 lanes poll the partials of the system's chunks and fold them in the fixed order, while the
//             next gather is under way.  When they are all there, every block of the system has finished
//             phase B.
// Buffers rotate so that a fast block never overwrites what a slow one still reads.  The fold of exchange t
// completes only after every block has read all U(t) and finished the gather of (x, g)(t - 1), and has its
// resets of exchange t acknowledged (each block waits for them before it stores its partials).  So in phase A of
// exchange t a block may reset U(t - 1), the partials of t - 2 and (x, g)(t - 2), and write the buffers reset in
// exchange t - 1: U alternates between two buffers, (x, g) and the partials rotate through three.
// Sums, products and their order are those of the general kernel: results are bit-identical.
//
// An iteration is bound by its chain of round trips past the L2 (about 1 us each: velocities, then (x, g) and
// the partials together) and by the lane requests of a CU (about one per ns): waves wait for data or for other blocks
// in 63-67% of their cycles, and for their turn to issue in 12% (FP64, one group) to 22% (FP32, four groups).  So words travel 16 B at a time; velocities are held by slice position (a share's
// are consecutive) and fetched once per block; strides of the LDS are constants; what only the start needs stays
// out of the loop's registers.  Microseconds per iteration, general kernel -> here (slab and box systems in their
// sorted order, FP64 unless noted): 22.8k rows 29 -> 8.1, 107k 29 -> 10.6, 183k in FP32 33 -> 12.6, 472k in FP32
// 31 -> 22.9; 64 systems of 1.37M rows together (each waits only for itself) 10.8 -> 8.1 ms.
//
// Systems do not meet each other at all: a block belongs to one system at a time, takes (system, share)
// pairs from a counter in order, and so the blocks of the first unfinished system are always running.  A batch in
// which too few systems can run at a time is left to the general kernel (turns_ok).
#include <algorithm>
#include <type_traits>

#include "solve_dev.hpp"

namespace alens {

#define LAUNCH_CHECK()                                                                           \
    do {                                                                                         \
        hipError_t e_ = hipGetLastError();                                                       \
        if (e_ != hipSuccess) return HipErr{e_, "kernel launch", __FILE__, __LINE__};             \
    } while (0)

typedef unsigned long long u64;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// sentinel of an exchanged 8-byte word: a signalling NaN (as is its low half as a float)
constexpr u64 kUnset = 0x7FF4A1E57FA1E5C0ull;
constexpr unsigned kUnsetLo = (unsigned)kUnset, kUnsetHi = (unsigned)(kUnset >> 32);

// Agent-scope accesses of the exchange memory, 16 B wide where the data is (the sc1 bit takes a load or store
// past the XCD's L2; a 16-byte access is two 8-byte words, each checked for itself).  One buffer holds every
// region; `at` is a lane's offset, `reg` the region's (a scalar).
constexpr int kAgent = 16;  // sc1
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
struct Exch {
    __amdgpu_buffer_rsrc_t r;
    __device__ inline Exch(void *p, uint32_t bytes) : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00020000)) {}
    __device__ inline u32x4 ld16(uint32_t at, uint32_t reg) const {
        return __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, (int)reg, kAgent);
    }
    __device__ inline u32x2 ld8(uint32_t at, uint32_t reg) const {
        return __builtin_amdgcn_raw_buffer_load_b64(r, (int)at, (int)reg, kAgent);
    }
    __device__ inline void st16(uint32_t at, uint32_t reg, u32x4 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)at, (int)reg, kAgent);
    }
    __device__ inline void st8(uint32_t at, uint32_t reg, u32x2 v) const {
        __builtin_amdgcn_raw_buffer_store_b64(v, r, (int)at, (int)reg, kAgent);
    }
    __device__ inline void unset16(uint32_t at, uint32_t reg) const {
        st16(at, reg, u32x4{kUnsetLo, kUnsetHi, kUnsetLo, kUnsetHi});
    }
};
__device__ inline u32x4 pack16(double a, double b) {
    return u32x4{(unsigned)__double2loint(a), (unsigned)__double2hiint(a), (unsigned)__double2loint(b),
                 (unsigned)__double2hiint(b)};
}
__device__ inline double lo64(u32x4 v) { return __hiloint2double((int)v.y, (int)v.x); }
__device__ inline double hi64(u32x4 v) { return __hiloint2double((int)v.w, (int)v.z); }
__device__ inline uint32_t min3(uint32_t a, uint32_t b, uint32_t c) {
    const uint32_t d = b < c ? b : c;
    return a < d ? a : d;
}
// Folds the words of a load into t, which becomes 0 when one of them is unset: a double is recognised by its high
// half (a signalling NaN whatever the low half is), a pair of floats by the first (a signalling NaN).
__device__ inline uint32_t seen64(uint32_t t, u32x4 v) { return min3(t, v.y ^ kUnsetHi, v.w ^ kUnsetHi); }
__device__ inline uint32_t seen32(uint32_t t, u32x4 v) { return min3(t, v.x ^ kUnsetLo, v.z ^ kUnsetLo); }
// every store of this lane has been acknowledged (the compiler keeps them ahead of it)
__device__ inline void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// block synchronisation for data in LDS: stores to memory stay in flight across it (a __syncthreads waits for
// their acknowledgements, a round trip past the L2 each time)
__device__ inline void lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ inline void reload() { asm volatile("" ::: "memory"); }  // polls read memory again

// Exchanged forms of a (x, g) pair (16 or 8 B) and of a velocity row (48 B, or 32 B with two unused words)
template <typename T>
struct Form;
template <>
struct Form<double> {
    static constexpr int xg = 16, u16 = 3;
    using XG = u32x4;
    static __device__ inline XG get(const Exch &e, uint32_t at, uint32_t reg) { return e.ld16(at, reg); }
    static __device__ inline void put(const Exch &e, uint32_t at, uint32_t reg, double x, double g) {
        e.st16(at, reg, pack16(x, g));
    }
    static __device__ inline void unset(const Exch &e, uint32_t at, uint32_t reg) { e.unset16(at, reg); }
    static __device__ inline uint32_t seen(uint32_t t, XG v) { return seen64(t, v); }
    static __device__ inline uint32_t seen_u(uint32_t t, u32x4 v) { return seen64(t, v); }
    static __device__ inline double x(XG v) { return lo64(v); }
    static __device__ inline double g(XG v) { return hi64(v); }
    static __device__ inline void put_u(const Exch &e, uint32_t at, uint32_t reg, const double (&u)[6]) {
#pragma unroll
        for (int c = 0; c < 3; ++c) e.st16(at + 16u * c, reg, pack16(u[2 * c], u[2 * c + 1]));
    }
    static __device__ inline void get_u(const u32x4 (&w)[3], double (&u)[6]) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            u[2 * c] = lo64(w[c]);
            u[2 * c + 1] = hi64(w[c]);
        }
    }
};
template <>
struct Form<float> {
    static constexpr int xg = 8, u16 = 2;
    using XG = u32x2;
    static __device__ inline XG get(const Exch &e, uint32_t at, uint32_t reg) { return e.ld8(at, reg); }
    static __device__ inline void put(const Exch &e, uint32_t at, uint32_t reg, float x, float g) {
        e.st8(at, reg, u32x2{__float_as_uint(x), __float_as_uint(g)});
    }
    static __device__ inline void unset(const Exch &e, uint32_t at, uint32_t reg) { e.st8(at, reg, u32x2{kUnsetLo, kUnsetHi}); }
    static __device__ inline uint32_t seen(uint32_t t, XG v) {
        const uint32_t d = v.x ^ kUnsetLo;
        return t < d ? t : d;
    }
    static __device__ inline uint32_t seen_u(uint32_t t, u32x4 v) { return seen32(t, v); }
    static __device__ inline float x(XG v) { return __uint_as_float(v.x); }
    static __device__ inline float g(XG v) { return __uint_as_float(v.y); }
    static __device__ inline void put_u(const Exch &e, uint32_t at, uint32_t reg, const float (&u)[6]) {
        e.st16(at, reg, u32x4{__float_as_uint(u[0]), __float_as_uint(u[1]), __float_as_uint(u[2]), __float_as_uint(u[3])});
        e.st16(at + 16u, reg, u32x4{__float_as_uint(u[4]), __float_as_uint(u[5]), 0u, 0u});
    }
    static __device__ inline void get_u(const u32x4 (&w)[2], float (&u)[6]) {
        u[0] = __uint_as_float(w[0].x);
        u[1] = __uint_as_float(w[0].y);
        u[2] = __uint_as_float(w[0].z);
        u[3] = __uint_as_float(w[0].w);
        u[4] = __uint_as_float(w[1].x);
        u[5] = __uint_as_float(w[1].y);
    }
};

// One more poll of a wait; false gives up (this wait was too long, or another block has set the abort word).  need: 0,
// or the ticket count at which every share of the system has a block.  Until then the wait is not counted: a share
// without a block waits for systems before its own, and those end by themselves (tickets are taken in order, so all
// their shares have blocks, whose waits are counted).
__device__ inline bool spin_more(uint32_t &n, uint32_t need, uint32_t *bar) {
    reload();
    if ((++n & 255u) != 0) return true;
    if (__hip_atomic_load(&bar[kBarWords], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return false;
    if (need != 0u && __hip_atomic_load(&bar[kBarTicket * kBarWords], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < need) n = 0;
    if (n < kSpinLimit) return true;
    __hip_atomic_store(&bar[kBarWords], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
}

// Slots before slice position p: whole slices, then p % 64 columns of its slice's depth.
__device__ inline uint32_t slots_before(const uint32_t *sellStart, uint32_t p) {
    const uint32_t sl = p / kSlice, in = p % kSlice, s0 = sellStart[sl];
    return in ? s0 + in * ((sellStart[sl + 1] - s0) / kSlice) : s0;
}
// Positions [p0, p1) of share i of nb of a system with positions [r0, r1): the system's slots cut into equal
// parts, between columns.
__device__ inline uint32_t share_cut(const uint32_t *sellStart, uint32_t r0, uint32_t r1, uint32_t i, uint32_t nb) {
    if (i == 0) return r0;
    if (i >= nb) return r1;
    const uint32_t base = slots_before(sellStart, r0);
    const uint32_t at = base + (uint32_t)((uint64_t)(slots_before(sellStart, r1) - base) * i / nb);
    uint32_t lo = r0 / kSlice, hi = (r1 + kSlice - 1) / kSlice;  // last slice that starts at or before the cut
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sellStart[mid] <= at) lo = mid; else hi = mid;
    }
    const uint32_t depth = (sellStart[lo + 1] - sellStart[lo]) / kSlice;
    const uint32_t in = at > sellStart[lo] && depth ? (at - sellStart[lo] + depth - 1) / depth : 0u;
    const uint32_t p = lo * kSlice + (in < (uint32_t)kSlice ? in : (uint32_t)kSlice);
    return p < r0 ? r0 : (p > r1 ? r1 : p);
}

// How the systems are cut into shares, one per block, for the FP64 and the FP32 solve: a system takes as
// many shares as its chunks need, or its slots at 15/16 of the LDS.  The plan fits when every share does (slots
// in LDS, chunks in the block's lanes), no system has more shares than the launch has blocks and the systems do not
// take too many turns (turns_ok).  In a captured step a wanted plan that does not fit clears the step's rows, and the
// host redoes the step.
//
// Systems whose shares do not all have blocks take turns, and in a turn the blocks that are left over wait; the general
// kernel takes all systems at once.  Whether the turns are shorter depends on how they fill the blocks and on how
// the systems' iterations differ.  Solve times here over those of the general kernel, at three states of a relaxing
// batch each (rods per system; boxes, slabs, or both in turn):
//   FP64  up to 3 turns               3 boxes of 40,000 0.45-0.70, 6 boxes of 40,000 0.71-0.96, 12 slabs of 16,000 0.55-0.62
//         more, 3 systems at a time   64 of 2,000-20,000 0.56-0.86, 100 of 4,000 0.49-0.67, 24 boxes of 16,000 0.70-1.00,
//                                     64 of 2,000-50,000 0.98-1.05
//         more, fewer at a time       8 boxes of 30,000 1.02-1.13, of 34,000 1.15-1.29; 12 boxes of 22,000 0.82-1.07
//   FP32  1 turn                      5 boxes of 26,000 0.50-0.55, 4 slabs of 30,000 0.53-0.65
//         2 turns, 3 at a time        12 boxes of 16,000 0.54-0.85, 8 slabs of 30,000 0.78-0.90, 8 boxes of 30,000 0.85-1.02
//         2 turns, fewer at a time    4 boxes of 60,000 1.03-1.09, 3 slabs of 80,000 0.93-1.13
//         more                        8 boxes of 34,000 1.23-1.52, 24 boxes of 16,000 0.81-1.20, 64 of 2,000-50,000 1.27-1.42
__device__ inline bool turns_ok(int f, int turns, int solving) {
    const bool three = 3 * turns <= solving;
    return f == 0 ? turns <= 3 || three : turns == 1 || (turns == 2 && three);
}

__global__ __launch_bounds__(256) void k_resident_plan(ResidentPlanArgs a) {
    __shared__ uint32_t s_off[kMaxSys + 1];
    __shared__ int s_bad;
    __shared__ uint32_t s_most;
    __shared__ int s_next[kMaxSys], s_solving;
    const int t = threadIdx.x;
    int unfit = 0;
    for (int f = 0; f < 2; ++f) {
        const uint32_t gpb = (uint32_t)a.gpb[f];
        const uint32_t scap = f == 0 ? resident_slots<double>((int)gpb) : resident_slots<float>((int)gpb);
        int32_t *head = a.plan + kPlanHead * f;
        ShareCut *share = reinterpret_cast<ShareCut *>(a.plan + 2 * kPlanHead) + (size_t)f * kPlanShares;
        if (f == 0 && a.alone) {  // one block for the whole solve (one system)
            const uint32_t rows = a.con_off[1] - a.con_off[0], p0 = (uint32_t)a.sys[0].rod_off, p1 = (uint32_t)a.sys[0].rod_end;
            const uint32_t c0 = slots_before(a.sellStart, p0), slots = slots_before(a.sellStart, p1) - c0;
            if (rows <= kAloneRows && alone_bytes(rows, p1 - p0, slots) <= kResidentPool) {
                if (t == 0) {
                    share[0] = ShareCut{0u, 0u, 1u, p0, p1, c0, slots, 0u};
                    head[0] = kPlanAlone;
                    head[1] = 1;
                    head[2] = (int32_t)a.sellStart[a.nslices];
                    head[3] = *a.nchunks;
                    head[4] = head[5] = 1;
                }
                continue;
            }
        }
        uint32_t nb = 0;
        if (t == 0) {
            s_bad = gpb == 0 || (f == 0 && a.alone == kAloneOnly);
            s_most = 1;
            s_solving = 0;
        }
        __syncthreads();
        if (t < a.nsys && gpb > 0 && !s_bad) {
            const uint32_t nch = a.chunk_off[t + 1] - a.chunk_off[t];
            const uint32_t slots = slots_before(a.sellStart, (uint32_t)a.sys[t].rod_end) -
                                   slots_before(a.sellStart, (uint32_t)a.sys[t].rod_off);
            const uint32_t want = scap - scap / 16, by_slots = (slots + want - 1) / want;
            nb = (nch + gpb - 1) / gpb;
            nb = nb > by_slots ? nb : by_slots;
            nb = nb < nch ? nb : nch;  // every share holds a chunk (its partials announce the share's writes)
            nb = nb > 0 ? nb : 1;
            if (nb > a.max_shares[f]) s_bad = 1;
            atomicMax(&s_most, nb);
        }
        s_off[t + 1] = nb;
        if (t == 0) s_off[0] = 0;
        __syncthreads();
        for (int o = 1; o < kMaxSys; o <<= 1) {
            const uint32_t v = t >= o ? s_off[t + 1 - o] : 0u;
            __syncthreads();
            s_off[t + 1] += v;
            __syncthreads();
        }
        const uint32_t total = s_off[a.nsys];
        if (t == 0 && total > (uint32_t)kPlanShares) s_bad = 1;
        if (total > a.max_shares[f]) {
            if (t < a.nsys) {  // the system that starts the turn after the one that system t starts
                int lo = t + 1, hi = a.nsys;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_off[mid] - s_off[t] <= a.max_shares[f]) lo = mid; else hi = mid - 1;
                }
                s_next[t] = lo;
                if (a.chunk_off[t + 1] > a.chunk_off[t]) atomicAdd(&s_solving, 1);
            }
            __syncthreads();
            if (t == 0) {
                int turns = 0;
                for (int q = 0; q < a.nsys; q = s_next[q]) ++turns;
                if (!turns_ok(f, turns, s_solving)) s_bad = 1;
            }
        }
        __syncthreads();
        if (!s_bad) {
            for (uint32_t v = t; v < total; v += 256) {
                int lo = 0, hi = a.nsys;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (s_off[mid] <= v) lo = mid; else hi = mid;
                }
                const uint32_t i = v - s_off[lo], n = s_off[lo + 1] - s_off[lo];
                const uint32_t r0 = (uint32_t)a.sys[lo].rod_off, r1 = (uint32_t)a.sys[lo].rod_end;
                const uint32_t p0 = share_cut(a.sellStart, r0, r1, i, n), p1 = share_cut(a.sellStart, r0, r1, i + 1, n);
                const uint32_t c0 = slots_before(a.sellStart, p0), c1 = slots_before(a.sellStart, p1);
                if (c1 - c0 > scap) s_bad = 1;
                share[v] = ShareCut{(uint32_t)lo, i, n, p0, p1, c0, c1 - c0, 0u};
            }
        }
        __syncthreads();
        const bool bad = s_bad != 0;
        if ((gpb > 0 || (f == 0 && a.alone == kAloneOnly)) && bad) unfit |= 1 << f;
        if (t == 0) {
            head[0] = bad ? kPlanUnfitting : kPlanShared;
            head[1] = (int32_t)total;
            head[2] = f == 0 ? (int32_t)a.sellStart[a.nslices] : unfit;
            head[3] = *a.nchunks;
            head[4] = (int32_t)gpb;
            head[5] = (int32_t)s_most;
        }
        __syncthreads();
    }
    if (a.mv && unfit) {
        // (nor may the other form's solve start: its shares name rows that would never come)
        if (t < 2) a.plan[kPlanHead * t] = kPlanUnfitting;
        for (int q = t; q <= a.nsys; q += 256) a.con_off[q] = a.chunk_off[q] = 0u;
        if (t == 0) {
            *a.mv = 0u;
            *a.nchunks = 0;
        }
    }
}

HipErr launch_resident_plan(hipStream_t st, const ResidentPlanArgs &p) {
    static_assert(kMaxSys == 256, "one thread per system");
    k_resident_plan<<<1, 256, 0, st>>>(p);
    LAUNCH_CHECK();
    return hip_ok();
}

// The exchange memory: three (x, g) buffers of m rows and one spare row, two velocity buffers of n rows, three
// buffers of chunk partials; byte strides.
struct Regions {
    uint32_t x, u, p;
    __host__ __device__ uint32_t X(uint32_t i) const { return i * x; }
    __host__ __device__ uint32_t U(uint32_t e) const { return 3 * x + (e & 1) * u; }
    __host__ __device__ uint32_t P(uint32_t i) const { return 3 * x + 2 * u + i * p; }
    __host__ __device__ uint32_t bytes() const { return 3 * x + 2 * u + 3 * p; }
};
template <typename T>
__host__ __device__ inline Regions regions(uint32_t m, int n, int nchunks) {
    auto al = [](size_t b) { return (uint32_t)((b + 255) & ~(size_t)255); };
    return Regions{al(((size_t)m + 1) * Form<T>::xg), al((size_t)n * Form<T>::u16 * 16), al((size_t)nchunks * 32)};
}
template <typename T>
size_t resident_exchange_bytes(double m, double n, double nchunks) {
    return (size_t)(3 * ((m + 1) * Form<T>::xg + 256) + 2 * (n * Form<T>::u16 * 16 + 256) + 3 * (nchunks * 32 + 256));
}
template size_t resident_exchange_bytes<double>(double, double, double);
template size_t resident_exchange_bytes<float>(double, double, double);

// The exchange memory before a solve: the start point in the third (x, g) buffer, (0, 0) in the spare rows,
// everything else unset; barrier words (the ticket among them) zero.  A plan is for launches with its number of row
// groups and with a block for every share of a system at least: with another one (two groups' chunks on one, a share
// that no block will take) the solve would leave rows out or wait for ever.  Such a plan is refused, with the abort word.
template <typename T>
__global__ void k_resident_reset(unsigned char *__restrict__ ex, Regions g, const typename Vec2<T>::type *__restrict__ xg,
                                 uint32_t m, const uint32_t *__restrict__ md, uint32_t *__restrict__ bar, int keep_abort,
                                 int32_t *__restrict__ head, int gpb, uint32_t grid) {
    using V2 = typename Vec2<T>::type;
    constexpr uint32_t xw = Form<T>::xg / 8;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    u64 *x = reinterpret_cast<u64 *>(ex), *u = reinterpret_cast<u64 *>(ex + g.U(0));
    if (i < (2 * g.u + 3 * g.p) / 8) u[i] = kUnset;
    const uint32_t rows = dcount(m, md);
    if (i < rows * xw) x[i] = x[g.x / 8 + i] = kUnset;
    if (i < rows) {  // (a caller's signalling NaN becomes a quiet one: it must not look unset)
        const V2 v = xg[i];
        reinterpret_cast<V2 *>(ex + g.X(2))[i] = mk2<T>(__builtin_canonicalize(v.x), __builtin_canonicalize(v.y));
    }
    if (i < 3) reinterpret_cast<V2 *>(ex + g.X(i))[m] = mk2<T>(T(0), T(0));
    if (i < (uint32_t)kBarTotalWords && !(keep_abort && i == (uint32_t)kBarWords)) bar[i] = 0u;
    if (i == (uint32_t)kBarWords && head[0] != kPlanUnfitting && (head[0] != kPlanShared || head[4] != gpb || (uint32_t)head[5] > grid)) {
        head[0] = kPlanUnfitting;
        bar[i] = 1u;
    }
}

// Ascending bitonic sort of N keys in LDS by NT threads.
template <int N, int NT>
__device__ inline void sort_keys(uint32_t *key) {
    for (int k = 2; k <= N; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            for (int i = threadIdx.x; i < N / 2; i += NT) {
                const int a = 2 * i - (i & (j - 1)), b = a + j;  // a has bit j clear
                const uint32_t x = key[a], y = key[b];
                if ((x > y) == ((a & k) == 0)) {
                    key[a] = y;
                    key[b] = x;
                }
            }
        }
    }
    __syncthreads();
}

// Four wave results of a group: summed, or their maximum taken, left to right.
__device__ inline double total4(const double *s4, bool sum) {
    if (sum) return ((s4[0] + s4[1]) + s4[2]) + s4[3];
    double t = s4[0];
    t = s4[1] > t ? s4[1] : t;
    t = s4[2] > t ? s4[2] : t;
    return s4[3] > t ? s4[3] : t;
}

// Halving folds (lane l takes lane l + h, h = 32 .. 1) of four quantities of a wave at once, the first two and
// with sum2 the third summed, the others' maximum taken.  Each lane swap halves the lanes in use and packs two
// quantities into one register: a swap of a's upper half with b's lower one leaves a's and b's pairs side by
// side, so one addition serves both; after two levels each quantity has a row of 16 lanes.  Results: lane 0
// v[0], lane 16 v[2], lane 32 v[1], lane 48 v[3], by the order of wave_fold.
__device__ inline void swap_halves32(double &a, double &b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline void swap_rows16(double &a, double &b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double2 fold_passes(const double (&v)[4], bool sum2) {
    double a = v[0], b = v[1], c = v[2], d = v[3];
    swap_halves32(a, b);
    swap_halves32(c, d);
    const double s = c + d, m = d > c ? d : c;
    return make_double2(a + b, sum2 && (threadIdx.x & 63) < 32 ? s : m);
}
__device__ inline double fold_rows(double a, double c, bool sum2) {
    const int l = threadIdx.x & 63;
    swap_rows16(a, c);  // rows: v0, v2, v1, v3
    const bool sum = (l >> 4) == 0 || (l >> 4) == 2 || (sum2 && (l >> 4) == 1);
    auto step = [&](double x, double o) {
        const double s = x + o, m = o > x ? o : x;
        return sum ? s : m;
    };
    double x = step(a, c);
    x = step(x, lanes_up_row<8>(x));
    x = step(x, lanes_up_row<4>(x));
    x = step(x, lanes_up_row<2>(x));
    return step(x, lanes_up_row<1>(x));
}
__device__ inline double wave_fold4(const double (&v)[4], bool sum2) {
    const double2 h = fold_passes(v, sum2);
    return fold_rows(h.x, h.y, sum2);
}
// The same where a wave holds 32 virtual lanes in two passes (fold_passes folds those) and o has the 32 that follow.
__device__ inline double fold_rest(double2 h, double2 o, bool sum2) {
    const double s = h.y + o.y, m = o.y > h.y ? o.y : h.y;
    return fold_rows(h.x + o.x, sum2 && (threadIdx.x & 63) < 32 ? s : m, sum2);
}
// where lane 16 r of wave_fold4 holds its result: quantity 0, 2, 1, 3
__device__ inline int fold4_quantity(int r) { return r == 1 ? 2 : (r == 2 ? 1 : r); }

// A system's report words.
template <typename T>
__device__ inline void report(const SolveArgsT<T> &a, int sy, int iters, int mv, int state, int fb, double res0, double res) {
    double *o = a.out + 8 * (size_t)sy;
    o[0] = (double)iters;
    o[1] = (double)mv;
    o[2] = state == S_CONVERGED ? 1.0 : 0.0;
    o[3] = (double)fb;
    o[4] = state == S_CONVERGED ? 0.0 : (state == S_NONFINITE ? (double)ALENS_E_NONFINITE : (double)ALENS_E_NOCONV);
    o[5] = res0;
    o[6] = res;
    o[7] = (double)(a.con_off[sy + 1] - a.con_off[sy]);  // the system's rows
}

// EXT: the rows include caller rows (lower bounds and compliances other than 0).
template <typename T, int GPB, bool EXT>
__global__ __launch_bounds__(resident_lanes(GPB)) void k_bbpgd_resident(ResidentArgs<T> r) {
    using F = Form<T>;
    constexpr int NT = resident_lanes(GPB), NU = F::u16, W = (int)sizeof(T);
    constexpr int LPC = NT / GPB, RPL = kRedChunk / LPC;  // lanes of a chunk, rows of a lane
    constexpr uint32_t kNone = 0xffffffffu;
    constexpr int NKEY = 1024 * GPB;  // rods named by the block's rows, with repeats
    // LDS: slot weights by component, then a part that holds the slots' values in phase A and the touched rods'
    // velocities in phase B.  Strides are constants, so that a slot's words are immediate offsets of two bases.
    constexpr uint32_t SC = resident_slots<T>(GPB);
    constexpr int GW = (int)((SC + NT - 1) / NT);             // slots of a lane
    constexpr uint32_t oV = 6 * SC * W, B2 = 65536u;          // value part; second base of the immediate offsets
    constexpr uint32_t UC = (resident_pool(GPB) - oV) / (16 * NU);  // velocities it holds
    constexpr int NB = (int)((UC * NU < 1024u * GPB * NU ? UC * NU : 1024u * GPB * NU) + NT - 1) / NT;  // words of a lane
    static_assert(oV + GW * NT * W <= resident_pool(GPB) && oV >= 4 * W * SC && oV < 2 * B2, "LDS layout");
    const SolveArgsT<T> &a = r.s;
    __shared__ __align__(16) unsigned char pool[resident_pool(GPB)];
    __shared__ double shG[GPB * 4 * 4], shF[4 * 4];
    __shared__ double2 shH[RPL == 1 ? GPB * 4 * 64 : 1];  // the odd waves' half-folded partials
    __shared__ uint32_t s_cnt[NT / 64];
    __shared__ int s_abort;
    __shared__ uint32_t s_ticket;
    if (r.head[0] != kPlanShared) return;  // a share does not fit (the host redoes the step), or the plan was refused
    // A chunk's 256 virtual lanes of two passes: with two rows a lane they are the lanes; with one, a wave has 32 of
    // them, pass 0 in its lower half, pass 1 in its upper one.
    const int tid = threadIdx.x, grp = tid / LPC, gl = tid % LPC, lane = tid & 63, wv = gl >> 6;
    const int first_row = RPL == 1 ? 32 * wv + (lane & 31) + (lane >> 5) * kRedThreads : gl;
    const uint32_t total = (uint32_t)r.head[1];
    const Regions rg = regions<T>(a.m, a.n, a.nchunks);
    const Exch ex(r.ex, rg.bytes());
    if (tid == 0) s_abort = 0;
    for (uint32_t turn = 0;; ++turn) {
        if (total <= gridDim.x) {
            if (turn > 0 || blockIdx.x >= total) return;
            if (tid == 0) s_ticket = blockIdx.x;
        } else if (tid == 0) {
            s_ticket = __hip_atomic_fetch_add(&a.bar[kBarTicket * kBarWords], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        const uint32_t share = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_ticket);
        if (share >= total) return;
        const ShareCut cut = r.share[share];
        const int sy = (int)cut.sys;
        const uint32_t nb = cut.of, ib = cut.index, s0 = cut.s0, p0 = cut.p0, p1 = cut.p1;
        const int mono = a.smono[sy];
        const uint32_t ch0 = a.chunk_off[sy], nch = a.chunk_off[sy + 1] - ch0;

        // ---- rows into registers; the rods they touch, each once, by ascending slice position ----
        const uint32_t cb = (uint32_t)((uint64_t)ib * nch / nb), ce = (uint32_t)((uint64_t)(ib + 1) * nch / nb);
        const uint32_t ch = cb + (uint32_t)grp;  // this group's chunk
        const bool act = ch < ce;
        const uint32_t kb = a.con_off[sy] + ch * kRedChunk, kend = a.con_off[sy + 1];
        uint32_t *keys = reinterpret_cast<uint32_t *>(pool), *sP = keys + NKEY;
        uint32_t kk[RPL], pIJ[RPL][2];
        bool ok[RPL];
        T gk[RPL][9], bb[RPL], xo[RPL], go[RPL], lbk[RPL], ivk[RPL];
#pragma unroll
        for (int q = 0; q < RPL; ++q) {
            kk[q] = kb + (uint32_t)(first_row + q * kRedThreads);
            ok[q] = act && kk[q] < kend;
            pIJ[q][0] = pIJ[q][1] = kNone;
            lbk[q] = ivk[q] = T(0);
            if (ok[q]) {
#pragma unroll
                for (int c = 0; c < 9; ++c) gk[q][c] = a.geo[(size_t)c * a.m + kk[q]];
                const uint32_t I = (uint32_t)a.cI[kk[q]], J = (uint32_t)a.cJ[kk[q]];
                pIJ[q][0] = r.spos ? r.spos[I] : I;
                pIJ[q][1] = r.spos ? r.spos[J] : J;
                bb[q] = a.b[kk[q]];
                if (EXT) {
                    lbk[q] = a.lb[kk[q]];
                    ivk[q] = a.invk[kk[q]];
                }
                const typename Vec2<T>::type xg = a.xg[kk[q]];
                xo[q] = xg.x;
                go[q] = xg.y;
            }
            keys[2 * RPL * tid + 2 * q] = pIJ[q][0];
            keys[2 * RPL * tid + 2 * q + 1] = pIJ[q][1];
        }
        sort_keys<NKEY, NT>(keys);
        uint32_t un = 0;  // distinct rods
        {
            constexpr int KPL = 2 * RPL;
            uint32_t v[KPL], cnt = 0;
            bool first[KPL];
#pragma unroll
            for (int q = 0; q < KPL; ++q) {
                const int i = KPL * tid + q;
                v[q] = keys[i];
                first[q] = v[q] != kNone && (i == 0 || keys[i - 1] != v[q]);
                cnt += first[q];
            }
            uint32_t inc = cnt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t t = __shfl_up(inc, o, 64);
                if (lane >= o) inc += t;
            }
            if (lane == 63) s_cnt[tid >> 6] = inc;
            __syncthreads();
            uint32_t at = inc - cnt;
#pragma unroll
            for (int w = 0; w < NT / 64; ++w) {
                if (w < (tid >> 6)) at += s_cnt[w];
                un += s_cnt[w];
            }
#pragma unroll
            for (int q = 0; q < KPL; ++q)
                if (first[q]) sP[at++] = v[q];
            __syncthreads();
        }
        un = (uint32_t)__builtin_amdgcn_readfirstlane((int)un);
        // velocities go through LDS where there is room for them; then a row's rods are LDS addresses, else offsets
        // in the exchange memory.  A lane's words of the block's velocities (past the end: the last word again).
        const bool cached = un <= UC;
        uint32_t uat[NB];
        const uint32_t ulast = un > 0 ? un * NU - 1 : 0u;
#pragma unroll
        for (int z = 0; z < NB; ++z) {
            const uint32_t q = (uint32_t)(tid + z * NT) < ulast ? (uint32_t)(tid + z * NT) : ulast;
            uat[z] = cached && un > 0 ? (sP[q / NU] * NU + q % NU) * 16u : 0u;
        }
#pragma unroll
        for (int q = 0; q < RPL; ++q) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                uint32_t at = ok[q] ? pIJ[q][e] : 0u;
                if (ok[q] && cached) {
                    uint32_t lo = 0, hi = un;  // place of the position in sP
                    while (lo < hi) {
                        const uint32_t mid = (lo + hi) >> 1;
                        if (sP[mid] < at)
                            lo = mid + 1;
                        else
                            hi = mid;
                    }
                    at = lo;
                }
                pIJ[q][e] = at * NU * 16u + (cached ? oV : 0u);
            }
        }
        __syncthreads();
        // ---- slots: weights into LDS, rows (offsets in the exchange memory) into registers ----
        // a rod: degree, LDS address of its first slot's first weight, distance of its slots
        struct Rod {
            uint32_t deg, at, step;
        };
        auto rod_index = [&](uint32_t p) { return a.sord ? (int)a.sord[p] : (int)p; };
        // a slice's columns in this share keep their order, packed: a cut slice is narrower in LDS
        auto rod_at = [&](uint32_t p) {
            const int rod = rod_index(p);
            const uint32_t c0 = p & ~(uint32_t)(kSlice - 1);
            const uint32_t from = c0 > p0 ? c0 : p0, to = c0 + kSlice < p1 ? c0 + kSlice : p1;
            return Rod{a.adjStart[rod + 1] - a.adjStart[rod], (slots_before(a.sellStart, from) - s0 + (p - from)) * W,
                       (to - from) * W};
        };
        uint32_t *sK = reinterpret_cast<uint32_t *>(pool + oV);
        for (uint32_t e = tid; e < (uint32_t)(GW * NT); e += NT) sK[e] = a.m;  // the spare row
        __syncthreads();
        for (uint32_t p = p0 + tid; p < p1; p += NT) {
            const Rod q = rod_at(p);
            const size_t g0 = (size_t)a.sellStart[p / kSlice] + p % kSlice;
            for (uint32_t j = 0; j < q.deg; j += 4) {
                uint32_t K[4];
                T w[4][6];
#pragma unroll
                for (int z = 0; z < 4; ++z) {
                    const size_t ge = g0 + (size_t)(j + z < q.deg ? j + z : j) * kSlice;
                    K[z] = a.sellK[ge] & 0x7fffffffu;
#pragma unroll
                    for (int c = 0; c < 6; ++c) w[z][c] = a.sellW[c * a.epad + ge];
                }
#pragma unroll
                for (int z = 0; z < 4; ++z) {
                    if (j + z >= q.deg) break;
                    const uint32_t at = q.at + (j + z) * q.step;
                    sK[at / W] = K[z];
#pragma unroll
                    for (int c = 0; c < 6; ++c) *reinterpret_cast<T *>(pool + at + c * SC * W) = w[z][c];
                }
            }
        }
        __syncthreads();
        uint32_t kat[GW];
        T lbs[EXT ? GW : 1];
#pragma unroll
        for (int q = 0; q < GW; ++q) {
            const uint32_t K = sK[tid + q * NT];
            kat[q] = K * F::xg;
            if (EXT) lbs[q] = K < a.m ? a.lb[K] : T(0);
        }
        // a lane's first rods stay in registers, with their mobility (as many as leave the loop without spills)
        constexpr int NR = W == 4 && GPB <= 2 ? 2 : 1;
        Rod rods[NR];
        T rmob[NR][6];
#pragma unroll
        for (int z = 0; z < NR; ++z) {
            const uint32_t p = p0 + tid + z * NT;
            rods[z] = p < p1 ? rod_at(p) : Rod{0u, 0u, 0u};
#pragma unroll
            for (int c = 0; c < 6; ++c) rmob[z][c] = rods[z].deg ? a.mob[6 * (size_t)rod_index(p) + c] : T(0);
        }
        __syncthreads();
        __builtin_amdgcn_s_waitcnt(0);  // the share is loaded: nothing in the loop waits for it again

        // where shares wait for blocks, the system's others may start only when earlier systems are done, however
        // long those take; once its first exchange is complete all of them run
        uint32_t need = total > gridDim.x ? share - ib + nb : 0u;
        const T dt = (T)a.dt;
        double alpha = 0.0;
        int odd = 0;              // parity of the iteration
        uint32_t ue = 0, pe = 0;  // velocity exchanges so far; partial buffer in use
        const uint32_t rec = (ch0 + ch) * 32u;

        // The lane index passes through an empty asm where it forms addresses: they are formed there each time
        // instead of being kept live across the loop.
        auto lane_index = [&]() {
            uint32_t t = threadIdx.x;
            asm volatile("" : "+v"(t));
            return t;
        };
        // gather: (x, g) of the rows of this lane's slots (the block's first nq NT slots hold all of its own)
        const int nq_ = __builtin_amdgcn_readfirstlane((int)((cut.slots + NT - 1) / NT));
        const int nz_ = __builtin_amdgcn_readfirstlane(cached ? (int)((un * NU + NT - 1) / NT) : 0);
        typename F::XG wg[GW];
        auto trips = [](int n) {  // a trip count compared anew at each use, not kept as a mask per trip
            asm volatile("" : "+s"(n));
            return n;
        };
        auto gather = [&](uint32_t reg) {
            const int nq = trips(nq_);
#pragma unroll
            for (int q = 0; q < GW; ++q)
                if (q < nq) wg[q] = F::get(ex, kat[q], reg);
        };

        // phase A: velocities of the share's rods from the gathered (x, g) of buffer src.  dst: the (x, g) buffer
        // that this exchange writes (3: none).
        auto phase_A = [&](bool grad, uint32_t src, uint32_t dst) {
            const T al = (T)alpha;
            const uint32_t t = lane_index();
            // the next exchange's velocities, (x, g) and partials are not there yet
            for (uint32_t q = t; q < (p1 - p0) * NU; q += NT) ex.unset16((p0 * NU + q) * 16u, rg.U(ue + 1));
            if (dst < 3) {
#pragma unroll
                for (int q = 0; q < RPL; ++q) {
                    uint32_t kx = kk[q];
                    asm volatile("" : "+v"(kx));
                    if (ok[q]) F::unset(ex, kx * F::xg, rg.X(dst == 2 ? 0 : dst + 1));
                }
            }
            if (act && gl == 0) {
                ex.unset16(rec, rg.P(pe == 2 ? 0 : pe + 1));
                ex.unset16(rec + 16u, rg.P(pe == 2 ? 0 : pe + 1));
            }
            uint32_t spins = 0;
            for (;;) {
                uint32_t seen = 1u;
                const int nq = trips(nq_);
#pragma unroll
                for (int q = 0; q < GW; ++q)
                    if (q < nq) seen = F::seen(seen, wg[q]);
                if (seen != 0u) break;
                if (!spin_more(spins, need, a.bar)) {
                    s_abort = 1;
                    break;
                }
                gather(rg.X(src));
            }
            const int nq = trips(nq_);
#pragma unroll
            for (int q = 0; q < GW; ++q) {
                if (q < nq) {
                    const T v = proj(F::x(wg[q]) - al * F::g(wg[q]), EXT ? lbs[EXT ? q : 0] : T(0));
                    *reinterpret_cast<T *>(pool + oV + (t + q * NT) * W) = grad ? F::g(wg[q]) : v;
                }
            }
            lds_sync();
            // four slots at once: LDS reads, then products in order.  Past the last slot the last one is read
            // again with v = 0, which adds +-0 to a sum that started at +0 and so is never -0.
            auto walk = [&](const Rod &q, uint32_t p, const T (&mb)[6]) {
                if (q.deg == 0) return;  // no row reads it
                T f[6] = {T(0), T(0), T(0), T(0), T(0), T(0)}, u[6];
                const uint32_t last = q.at + (q.deg - 1) * q.step;
                uint32_t at = q.at;
                for (uint32_t j = 0; j < q.deg; j += 4) {
                    T v[4], wt[4][6];
#pragma unroll
                    for (int z = 0; z < 4; ++z) {
                        const uint32_t e = at < last ? at : last, e2 = e + B2;
#pragma unroll
                        for (int c = 0; c < 6; ++c)
                            wt[z][c] = c * SC * W < B2 ? *reinterpret_cast<const T *>(pool + e + c * SC * W)
                                                       : *reinterpret_cast<const T *>(pool + e2 + (c * SC * W - B2));
                        v[z] = oV < B2 ? *reinterpret_cast<const T *>(pool + e + oV)
                                       : *reinterpret_cast<const T *>(pool + e2 + (oV - B2));
                        at += q.step;
                    }
#pragma unroll
                    for (int z = 0; z < 4; ++z) {
                        v[z] = j + z < q.deg ? v[z] : T(0);
#pragma unroll
                        for (int c = 0; c < 6; ++c) f[c] = f[c] + v[z] * wt[z][c];
                    }
                }
                apply_M(mb, f, mono, u);
                F::put_u(ex, p * (16u * NU), rg.U(ue), u);
            };
#pragma unroll
            for (int z = 0; z < NR; ++z) walk(rods[z], p0 + t + z * NT, rmob[z]);
            for (uint32_t p = p0 + t + NR * NT; p < p1; p += NT) {
                const int rod = rod_index(p);
                T mb[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) mb[c] = a.mob[6 * (size_t)rod + c];
                walk(rod_at(p), p, mb);
            }
        };

        // phase B: this lane's rows; (x, g) to buffer dst; the chunk's partials.  false: a wait gave up
        auto phase_B = [&](auto iterate, int mode, uint32_t dst) -> bool {
            constexpr bool ITER = decltype(iterate)::value;
            if (ITER) mode = B_ITER;
            const T al = (T)alpha;
            const uint32_t ur = rg.U(ue);
            if (cached) {
                u32x4 w[NB];
                auto load = [&]() {
                    const int nz = trips(nz_);
#pragma unroll
                    for (int z = 0; z < NB; ++z)
                        if (z < nz) w[z] = ex.ld16(uat[z], ur);
                };
                if (un > 0) {
                    load();
                    uint32_t spins = 0;
                    for (;;) {
                        uint32_t seen = 1u;
                        const int nz = trips(nz_);
#pragma unroll
                        for (int z = 0; z < NB; ++z)
                            if (z < nz) seen = F::seen_u(seen, w[z]);
                        if (seen != 0u) break;
                        if (!spin_more(spins, need, a.bar)) {
                            s_abort = 1;
                            break;
                        }
                        load();
                    }
                }
                lds_sync();  // the slots' values, which share the space, have been read
                const uint32_t t = lane_index();
                const int nz = trips(nz_);
#pragma unroll
                for (int z = 0; z < NB; ++z)
                    if (z < nz && ((z + 1) * NT <= (int)(UC * NU) || t + z * NT < UC * NU))
                        *reinterpret_cast<u32x4 *>(pool + oV + (t + z * NT) * 16u) = w[z];
                lds_sync();
            }
            stores_done();  // the resets of this exchange (their acknowledgement is long back)
            double vs[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, vx[2] = {0.0, 0.0};
#pragma unroll
            for (int q = 0; q < RPL; ++q) {
                if (!ok[q]) continue;
                uint32_t pI = pIJ[q][0], pJ = pIJ[q][1], kx = kk[q];
                T bq = bb[q];
                asm volatile("" : "+v"(pI), "+v"(pJ), "+v"(kx), "+v"(bq));
                u32x4 wI[NU], wJ[NU];
                if (cached) {
#pragma unroll
                    for (int c = 0; c < NU; ++c) {
                        wI[c] = *reinterpret_cast<const u32x4 *>(pool + pI + 16 * c);
                        wJ[c] = *reinterpret_cast<const u32x4 *>(pool + pJ + 16 * c);
                    }
                } else {
                    uint32_t spins = 0;
                    for (;;) {
                        uint32_t seen = 1u;
#pragma unroll
                        for (int c = 0; c < NU; ++c) {
                            wI[c] = ex.ld16(pI + 16u * c, ur);
                            wJ[c] = ex.ld16(pJ + 16u * c, ur);
                        }
#pragma unroll
                        for (int c = 0; c < NU; ++c) seen = F::seen_u(F::seen_u(seen, wI[c]), wJ[c]);
                        if (seen != 0u) break;
                        if (!spin_more(spins, need, a.bar)) {
                            s_abort = 1;
                            break;
                        }
                    }
                }
                T uI[6], uJ[6];
                F::get_u(wI, uI);
                F::get_u(wJ, uJ);
                const T du = dt_row(gk[q], uI, uJ);
                if (mode == B_ALPHA0) {
                    T ag = dt * du;
                    if (EXT && a.invk) ag = ag + ivk[q] * go[q];
                    vs[0] = vs[0] + (double)(go[q] * go[q]);
                    vs[1] = vs[1] + (double)(go[q] * ag);
                } else {
                    const T xn = proj(xo[q] - al * go[q], lbk[q]);
                    T gn = dt * du + bq;
                    if (EXT && a.invk) gn = gn + ivk[q] * xn;
                    const double res = (double)fabs(xn - proj(xn - gn, lbk[q]));
                    if (!isfinite(res))
                        vs[3] = vs[3] + 1.0;
                    else if (res > vx[0])
                        vx[0] = res;
                    if (mode == B_INIT) {
                        if (a.warm) {
                            const double rc = (double)fabs(T(0) - proj(T(0) - bq, lbk[q]));
                            if (!isfinite(rc))
                                vs[4] = vs[4] + 1.0;
                            else if (rc > vx[1])
                                vx[1] = rc;
                        }
                    } else {
                        const T sv = xn - xo[q];
                        const T yv = gn - go[q];
                        vs[0] = vs[0] + (double)(sv * sv);
                        vs[1] = vs[1] + (double)(sv * yv);
                        vs[2] = vs[2] + (double)(yv * yv);
                    }
                    xo[q] = xn;
                    go[q] = gn;
                    F::put(ex, kx * F::xg, rg.X(dst), xn, gn);
                }
            }
            // chunk partials: waves fold by halving, the group's four totals left to right.  The record of this
            // exchange, sums first: start point {non-finite, cold non-finite, residual, cold residual}, first step
            // {g.g, g.Ag, 0, 0}, odd iterations {s.s, s.y, non-finite, residual}, even ones {s.y, y.y, ...}
            double v[4];
            if (ITER) {
                v[0] = odd ? vs[0] : vs[1];
                v[1] = odd ? vs[1] : vs[2];
                v[2] = vs[3];
                v[3] = vx[0];
            } else {
                v[0] = mode == B_INIT ? vs[3] : vs[0];
                v[1] = mode == B_INIT ? vs[4] : vs[1];
                v[2] = mode == B_INIT ? vx[0] : 0.0;
                v[3] = mode == B_INIT ? vx[1] : 0.0;
            }
            double *sg = shG + grp * 4 * 4;
            const bool sum2 = mode != B_INIT;
            if constexpr (RPL == 2) {
                const double x = wave_fold4(v, sum2);
                if ((lane & 15) == 0) sg[fold4_quantity(lane >> 4) * 4 + wv] = x;
            } else {
                // passes, then the other wave's 32 virtual lanes, then within the wave
                double2 h = fold_passes(v, sum2);
                double2 *sh = shH + (grp * 4 + (wv >> 1)) * 64;
                if (wv & 1) sh[lane] = h;
                lds_sync();
                if ((wv & 1) == 0) {
                    const double x = fold_rest(h, sh[lane], sum2);
                    if ((lane & 15) == 0) sg[fold4_quantity(lane >> 4) * 4 + (wv >> 1)] = x;
                }
            }
            lds_sync();
            const bool good = s_abort == 0;
            if (act && gl == 0 && good) {
                double q4[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) q4[q] = total4(sg + q * 4, q < 2 || (q == 2 && mode != B_INIT));
                ex.st16(rec, rg.P(pe), pack16(q4[0], q4[1]));
                ex.st16(rec + 16u, rg.P(pe), pack16(q4[2], q4[3]));
            }
            lds_sync();
            return good;
        };

        // fold: totals of the system's chunk partials of this exchange, NS sums and then maxima
        auto fold = [&](int ns, double (&tot)[4]) -> bool {
            const uint32_t pr = rg.P(pe);
            if (tid < 256) {
                double v[4] = {0.0, 0.0, 0.0, 0.0};
                for (uint32_t c0 = tid; c0 < nch; c0 += 256) {
                    const uint32_t at = (ch0 + c0) * 32u;
                    u32x4 w0 = ex.ld16(at, pr), w1 = ex.ld16(at + 16u, pr);
                    uint32_t spins = 0;
                    while (seen64(seen64(1u, w0), w1) == 0u) {
                        if (!spin_more(spins, need, a.bar)) {
                            s_abort = 1;
                            break;
                        }
                        w0 = ex.ld16(at, pr);
                        w1 = ex.ld16(at + 16u, pr);
                    }
                    const double t[4] = {lo64(w0), hi64(w0), lo64(w1), hi64(w1)};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (q < 2 || (q == 2 && ns == 3))
                            v[q] = v[q] + t[q];
                        else
                            v[q] = t[q] > v[q] ? t[q] : v[q];
                    }
                }
                const double x = wave_fold4(v, ns == 3);
                if ((lane & 15) == 0) shF[fold4_quantity(lane >> 4) * 4 + wv] = x;
            }
            lds_sync();
#pragma unroll
            for (int q = 0; q < 4; ++q) tot[q] = total4(shF + 4 * q, q < 2 || (q == 2 && ns == 3));
            const bool good = s_abort == 0;
            lds_sync();
            return good;
        };

        // exchange it = -1: start point x = P(x0), g = A x + b; 0: first step g^T g / g^T A g; then iterations
        int state = S_ACTIVE, iters = 0, mv = 0, fb = 0;
        double tot[4], res0 = 0.0, res = 0.0;
        uint32_t xs = 2, xe = 0;  // (x, g) buffer in use (at first the start point's) and the next one to write
        gather(rg.X(xs));
        for (int it = -1; it <= a.max_ite; ++it) {
            odd = it & 1;
            const uint32_t dst = it == 0 ? 3u : xe;
            phase_A(it == 0, xs, dst);
            if (!(it > 0 ? phase_B(std::true_type{}, B_ITER, dst) : phase_B(std::false_type{}, it < 0 ? B_INIT : B_ALPHA0, dst))) return;
            if (dst < 3) {
                xs = xe;
                xe = xe == 2 ? 0 : xe + 1;
            }
            gather(rg.X(xs));
            if (!fold(it < 0 ? 2 : 3, tot)) return;
            need = 0u;
            ++ue;
            pe = pe == 2 ? 0 : pe + 1;
            ++mv;
            if (it == 0) {
                alpha = tot[0] / tot[1];
                if (!(alpha > 0.0 && alpha < INFINITY)) alpha = 1.0;
                continue;
            }
            double nf = tot[2], rm = tot[3];
            if (it < 0) {
                nf = tot[0];
                rm = tot[2];
                if (a.warm && (nf > 0.0 || rm > tot[3])) {
                    // the warm start raised the residual: x = 0, g = 0 + b; an exchange of its own publishes it
                    fb = 1;
                    nf = tot[1];
                    rm = tot[3];
                    if (act && gl == 0) {
                        ex.unset16(rec, rg.P(pe == 2 ? 0 : pe + 1));
                        ex.unset16(rec + 16u, rg.P(pe == 2 ? 0 : pe + 1));
                    }
#pragma unroll
                    for (int q = 0; q < RPL; ++q) {
                        if (!ok[q]) continue;
                        xo[q] = T(0);
                        go[q] = T(0) + bb[q];
                        F::unset(ex, kk[q] * F::xg, rg.X(2));
                        F::put(ex, kk[q] * F::xg, rg.X(xe), xo[q], go[q]);
                    }
                    stores_done();
                    lds_sync();
                    if (act && gl == 0) {
                        ex.st16(rec, rg.P(pe), u32x4{0u, 0u, 0u, 0u});
                        ex.st16(rec + 16u, rg.P(pe), u32x4{0u, 0u, 0u, 0u});
                    }
                    if (!fold(2, tot)) return;
                    pe = pe == 2 ? 0 : pe + 1;
                    xs = xe;
                    ++xe;
                    gather(rg.X(xs));
                }
                res0 = rm;
            } else {
                iters = it;
            }
            res = rm;
            if (nf > 0.0) {
                state = S_NONFINITE;
                break;
            }
            if (rm <= a.tol) {
                state = S_CONVERGED;
                break;
            }
            if (it > 0) {
                const double an = tot[0] / tot[1];  // s.s / s.y (odd) or s.y / y.y (even)
                if (an > 0.0 && an < INFINITY) alpha = an;
            }
        }
#pragma unroll
        for (int q = 0; q < RPL; ++q)
            if (ok[q]) a.xg[kk[q]] = mk2<T>(xo[q], go[q]);
        if (ib == 0 && tid == 0) report(a, sy, iters, mv, state, fb, res0, res);
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------------
// A solve that one block holds whole: nothing is exchanged but through LDS.  Groups of 256 lanes hold a chunk each,
// two rows a lane; slot weights, the rows' values and the rods' velocities are in LDS.  An iteration is bound by LDS
// reads (six weights and a value per slot, two velocities per row) and three block synchronisations.  Sums and their
// order are the general kernel's.  Per iteration 2.1 us for 399 rows and 3.4 us for 793, against 7.6 and 9.2 us of the
// shared form, whose one or two blocks spend three round trips past the L2: it is the faster one wherever it fits.
// ------------------------------------------------------------------------------------------------
template <bool EXT>
__global__ __launch_bounds__(512) void k_bbpgd_alone(ResidentArgs<double> r) {
    constexpr int NT = 512;
    static_assert(kAloneRows == 2 * kRedChunk && kRedChunk == 2 * kRedThreads && kRedThreads == 256, "two groups, two rows a lane");
    const SolveArgsT<double> &a = r.s;
    __shared__ __align__(16) unsigned char pool[kResidentPool];
    __shared__ double shG[2][2][4 * 4];
    if (r.head[0] != kPlanAlone) return;  // does not fit: the host redoes the step
    const int tid = threadIdx.x, grp = tid >> 8, gl = tid & 255, lane = tid & 63, wv = (tid >> 6) & 3;
    const ShareCut cut = r.share[0];
    const uint32_t p0 = cut.p0, p1 = cut.p1, S = cut.slots;
    const uint32_t kb = a.con_off[0], R = a.con_off[1] - kb, nch = a.chunk_off[1] - a.chunk_off[0];
    const int mono = a.smono[0];
    const uint32_t oU = 48u * S, oV = oU + 48u * (p1 - p0), oE = oV + 8u * R;  // weights; velocities; values; slots' rows
    // rows
    uint32_t kk[2], pI[2], pJ[2];
    bool ok[2];
    double gk[2][9], bb[2], xo[2], go[2], lbk[2], ivk[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        kk[q] = (uint32_t)(grp * kRedChunk + gl + q * kRedThreads);
        ok[q] = kk[q] < R;
        lbk[q] = ivk[q] = 0.0;
        const uint32_t k = kb + kk[q];
        if (ok[q]) {
#pragma unroll
            for (int c = 0; c < 9; ++c) gk[q][c] = a.geo[(size_t)c * a.m + k];
            const uint32_t I = (uint32_t)a.cI[k], J = (uint32_t)a.cJ[k];
            pI[q] = oU + 48u * ((r.spos ? r.spos[I] : I) - p0);
            pJ[q] = oU + 48u * ((r.spos ? r.spos[J] : J) - p0);
            bb[q] = a.b[k];
            if (EXT) {
                lbk[q] = a.lb[k];
                ivk[q] = a.invk[k];
            }
            const double2 xg = a.xg[k];
            xo[q] = xg.x;
            go[q] = xg.y;
        }
    }
    // slots by component in slice order, a cut last slice packed; a rod: degree, first slot, distance of its slots
    struct Rod {
        uint32_t deg, at, step;
    };
    auto rod_index = [&](uint32_t p) { return a.sord ? (int)a.sord[p] : (int)p; };
    auto rod_at = [&](uint32_t p) {
        const int rod = rod_index(p);
        const uint32_t c0 = p & ~(uint32_t)(kSlice - 1);
        const uint32_t from = c0 > p0 ? c0 : p0, to = c0 + kSlice < p1 ? c0 + kSlice : p1;
        return Rod{a.adjStart[rod + 1] - a.adjStart[rod], slots_before(a.sellStart, from) - cut.s0 + (p - from), to - from};
    };
    double *sW = reinterpret_cast<double *>(pool), *sV = reinterpret_cast<double *>(pool + oV);
    uint16_t *sE = reinterpret_cast<uint16_t *>(pool + oE);
    for (uint32_t p = p0 + tid; p < p1; p += NT) {
        const Rod q = rod_at(p);
        const size_t g0 = (size_t)a.sellStart[p / kSlice] + p % kSlice;
        for (uint32_t j = 0; j < q.deg; j += 4) {
            uint32_t K[4];
            double w[4][6];
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                const size_t ge = g0 + (size_t)(j + z < q.deg ? j + z : j) * kSlice;
                K[z] = a.sellK[ge] & 0x7fffffffu;
#pragma unroll
                for (int c = 0; c < 6; ++c) w[z][c] = a.sellW[c * a.epad + ge];
            }
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                if (j + z >= q.deg) break;
                const uint32_t at = q.at + (j + z) * q.step;
                sE[at] = (uint16_t)(K[z] - kb);
#pragma unroll
                for (int c = 0; c < 6; ++c) sW[c * S + at] = w[z][c];
            }
        }
    }
    constexpr int NR = 2;  // a lane's first rods stay in registers, with their mobility
    Rod rods[NR];
    double rmob[NR][6];
#pragma unroll
    for (int z = 0; z < NR; ++z) {
        const uint32_t p = p0 + tid + z * NT;
        rods[z] = p < p1 ? rod_at(p) : Rod{0u, 0u, 0u};
#pragma unroll
        for (int c = 0; c < 6; ++c) rmob[z][c] = rods[z].deg ? a.mob[6 * (size_t)rod_index(p) + c] : 0.0;
    }
    const double dt = a.dt;
    double alpha = 0.0;
    auto walk = [&](const Rod &q, uint32_t p, const double (&mb)[6]) {
        if (q.deg == 0) return;  // no row reads it
        double f[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, u[6];
        uint32_t at = q.at;
        for (uint32_t j = 0; j < q.deg; ++j, at += q.step) {
            const double v = sV[sE[at]];
#pragma unroll
            for (int c = 0; c < 6; ++c) f[c] = f[c] + v * sW[c * S + at];
        }
        apply_M(mb, f, mono, u);
        double2 *d = reinterpret_cast<double2 *>(pool + oU + 48u * (p - p0));
#pragma unroll
        for (int c = 0; c < 3; ++c) d[c] = make_double2(u[2 * c], u[2 * c + 1]);
    };
    int state = S_ACTIVE, iters = 0, mv = 0, fb = 0;
    double res0 = 0.0, res = 0.0;
    for (int it = -1; it <= a.max_ite; ++it) {
        const bool odd = it & 1;
        // v = P(x - alpha g) of every row (g itself for the first step); then one lane per rod: U = M F
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (ok[q]) sV[kk[q]] = it == 0 ? go[q] : proj(xo[q] - alpha * go[q], lbk[q]);
        lds_sync();
#pragma unroll
        for (int z = 0; z < NR; ++z) walk(rods[z], p0 + tid + z * NT, rmob[z]);
        for (uint32_t p = p0 + tid + NR * NT; p < p1; p += NT) {
            double mb[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) mb[c] = a.mob[6 * (size_t)rod_index(p) + c];
            walk(rod_at(p), p, mb);
        }
        lds_sync();
        // rows: new (x, g), residual and products
        double vs[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, vx[2] = {0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (!ok[q]) continue;
            double uI[6], uJ[6];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double2 wi = reinterpret_cast<const double2 *>(pool + pI[q])[c];
                const double2 wj = reinterpret_cast<const double2 *>(pool + pJ[q])[c];
                uI[2 * c] = wi.x;
                uI[2 * c + 1] = wi.y;
                uJ[2 * c] = wj.x;
                uJ[2 * c + 1] = wj.y;
            }
            const double du = dt_row(gk[q], uI, uJ);
            if (it == 0) {
                double ag = dt * du;
                if (EXT) ag = ag + ivk[q] * go[q];
                vs[0] = vs[0] + go[q] * go[q];
                vs[1] = vs[1] + go[q] * ag;
                continue;
            }
            const double xn = proj(xo[q] - alpha * go[q], lbk[q]);
            double gn = dt * du + bb[q];
            if (EXT) gn = gn + ivk[q] * xn;
            const double e = fabs(xn - proj(xn - gn, lbk[q]));
            if (!isfinite(e))
                vs[3] = vs[3] + 1.0;
            else if (e > vx[0])
                vx[0] = e;
            if (it < 0) {
                if (a.warm) {
                    const double rc = fabs(0.0 - proj(0.0 - bb[q], lbk[q]));
                    if (!isfinite(rc))
                        vs[4] = vs[4] + 1.0;
                    else if (rc > vx[1])
                        vx[1] = rc;
                }
            } else {
                const double sv = xn - xo[q], yv = gn - go[q];
                vs[0] = vs[0] + sv * sv;
                vs[1] = vs[1] + sv * yv;
                vs[2] = vs[2] + yv * yv;
            }
            xo[q] = xn;
            go[q] = gn;
        }
        // chunk partials as in k_bbpgd_resident, then the chunks' totals: sums first
        const bool sum2 = it >= 0;
        double v[4];
        v[0] = it < 0 ? vs[3] : (it == 0 || odd ? vs[0] : vs[1]);
        v[1] = it < 0 ? vs[4] : (it == 0 || odd ? vs[1] : vs[2]);
        v[2] = it < 0 ? vx[0] : vs[3];
        v[3] = it < 0 ? vx[1] : vx[0];
        const double x = wave_fold4(v, sum2);
        double *sg = shG[it & 1][grp];  // two in turn: one is read while the next is written
        if ((lane & 15) == 0) sg[fold4_quantity(lane >> 4) * 4 + wv] = x;
        lds_sync();
        double tot[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool sum = q < 2 || (q == 2 && sum2);
            double c[2] = {0.0, 0.0};
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h)
                if (h < nch) {
                    const double p = total4(shG[it & 1][h] + 4 * q, sum);
                    c[h] = sum ? c[h] + p : (p > c[h] ? p : c[h]);
                }
            tot[q] = sum ? c[0] + c[1] : (c[1] > c[0] ? c[1] : c[0]);
        }
        ++mv;
        if (it == 0) {
            alpha = tot[0] / tot[1];
            if (!(alpha > 0.0 && alpha < INFINITY)) alpha = 1.0;
            continue;
        }
        double nf = tot[2], rm = tot[3];
        if (it < 0) {
            nf = tot[0];
            rm = tot[2];
            if (a.warm && (nf > 0.0 || rm > tot[3])) {  // the warm start raised the residual: x = 0, g = 0 + b
                fb = 1;
                nf = tot[1];
                rm = tot[3];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    xo[q] = 0.0;
                    go[q] = 0.0 + bb[q];
                }
            }
            res0 = rm;
        } else {
            iters = it;
        }
        res = rm;
        if (nf > 0.0) {
            state = S_NONFINITE;
            break;
        }
        if (rm <= a.tol) {
            state = S_CONVERGED;
            break;
        }
        if (it > 0) {
            const double an = tot[0] / tot[1];  // s.s / s.y (odd) or s.y / y.y (even)
            if (an > 0.0 && an < INFINITY) alpha = an;
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (ok[q]) a.xg[kb + kk[q]] = make_double2(xo[q], go[q]);
    if (tid == 0) report(a, 0, iters, mv, state, fb, res0, res);
}

HipErr launch_alone(hipStream_t st, const ResidentArgs<double> &r) {
    if (r.s.lb)
        k_bbpgd_alone<true><<<1, 512, 0, st>>>(r);
    else
        k_bbpgd_alone<false><<<1, 512, 0, st>>>(r);
    LAUNCH_CHECK();
    return hip_ok();
}

template <typename T, int GPB>
static HipErr launch_resident_k(hipStream_t st, ResidentArgs<T> r, int grid) {
    void *args[] = {&r};
    const void *f = r.s.lb ? (const void *)k_bbpgd_resident<T, GPB, true> : (const void *)k_bbpgd_resident<T, GPB, false>;
    ALENS_HIP_TRY(hipLaunchCooperativeKernel(f, dim3(grid), dim3(resident_lanes(GPB)), args, 0, st));
    return hip_ok();
}

template <typename T>
HipErr launch_resident(hipStream_t st, const ResidentArgs<T> &r, int gpb, int grid, bool keep_abort) {
    const Regions g = regions<T>(r.s.m, r.s.n, r.s.nchunks);
    const uint32_t mx = std::max(std::max((2 * g.u + 3 * g.p) / 8, r.s.m * (uint32_t)(Form<T>::xg / 8)), (uint32_t)kBarTotalWords);
    k_resident_reset<T><<<(mx + 255) / 256, 256, 0, st>>>(static_cast<unsigned char *>(r.ex), g, r.s.xg, r.s.m, r.s.m_dev,
                                                          r.s.bar, keep_abort ? 1 : 0, r.head, gpb, (uint32_t)grid);
    LAUNCH_CHECK();
    if constexpr (sizeof(T) == 4)
        if (gpb == 4) return launch_resident_k<T, 4>(st, r, grid);
    return gpb == 2 ? launch_resident_k<T, 2>(st, r, grid) : launch_resident_k<T, 1>(st, r, grid);
}
template HipErr launch_resident<double>(hipStream_t, const ResidentArgs<double> &, int, int, bool);
template HipErr launch_resident<float>(hipStream_t, const ResidentArgs<float> &, int, int, bool);

}  // namespace alens
