// cgpersist.hpp -- the CG iteration of one system as a persistent kernel: the
// Krylov vectors stay in registers and LDS between the iterations, and the
// workgroups exchange nothing but dot-product partials and one vector.
//
// What bounds the kernel-per-phase iteration (cgkernels.hpp) is, on systems that
// fill the chip, bytes: of the 168 bytes per row of an FP64 iteration 96 are
// vector reads and writes that only exist because each phase is a launch of its
// own; on small systems it is the chain of dependent loads and the reduction
// that every launch repeats (4-6 us per kernel).  One kernel for many iterations
// needs neither.  The 256 CUs hold 128 MB of registers and 40 MB of LDS, so the
// vectors of a system of up to 2^21 rows fit on the chip:
//
//  * a workgroup of 1024 threads per CU takes four tiles of 256 threads, the
//    tiles (rows, order, partial sums) of cgkernels.hpp; a thread keeps r and q of
//    its RPT rows in registers, p in LDS, d and g in either;
//  * the matrix rows stay in registers where they fit (RES of the RPT rows: all
//    of them up to 2 FP64 or 4 FP32 rows per thread); the others are read every
//    iteration, 60 bytes per FP64 row, 36 FP32: values, and columns as 16-bit LDS
//    places (k_ghost_plan);
//  * the rows of other tiles that a tile's columns refer to (its ghosts: 800 to 1300
//    for 2048 rows in Z order) have places in its LDS as well.  A tile keeps its
//    ghosts' p itself, by p' = r + beta p, the expression of the row's owner, so all
//    it reads is their r, which every tile publishes for the rows that others refer
//    to (the pattern is symmetric: those with ghost columns) after the update: two
//    grid exchanges per iteration, one read of each ghost, and the product reads
//    nothing but LDS beside the matrix.  Reading r and the old p of a far column
//    where the product meets it, as kc_persist_far does, took 42.8 us an iteration
//    at 128^3 FP64 against 28.0 (its loads, 8 % of the columns, stall the stream);
//    with 32 registers spilled this form took 32.8, and the wait for a row's loads
//    before the next is issued costs less than the spills a second row in flight
//    brings.
//
// Grid reduction without atomics or fences: a workgroup publishes its partial
// sums as 64-bit words, half payload and half sequence number, and the readers
// poll the words themselves.  So the value and its arrival are one word, nothing
// has to be reset, and every workgroup adds the same numbers in the order of
// sum_slots (see GridSum): the bits are those of the kernel-per-phase form.
// Measured with 1024-thread workgroups, a 128-byte line per slot: 1.4 us for 64
// workgroups, 2.3 for 256 (3.1 with the slots 16 bytes apart: writers of one line
// wait for each other); with an agent-scope fence in every wave the same exchange
// took 31-86 us for 256 (each fence is an L2 write-back or invalidate).  The
// published vectors therefore go through agent-scope relaxed stores and loads,
// which pass the per-XCD L2s, and a wave waits for its stores to complete (vmcnt)
// before the workgroup's barrier, behind which its partial sum is published.  (Words
// that carry the iteration's tag, which need no such wait, cost twice the bytes: 5.3
// -> 5.5 us at 32^3 FP64, 9.5 -> 10.7 at 80^3; in FP32 they gained 0.3 us up to 64^3
// and lost 0.9 at 96^3.)
//
// A cooperative launch keeps its workgroups resident together, but costs about 17 us
// more than a plain one, as much as a small solve's whole start.  Launches that do a
// whole solve are therefore plain ones whose workgroups meet first (Meeting): they
// write nothing before all of them have arrived, and if one has not within
// kMeetClocks (other work holds its place), all end and the solve is launched again,
// cooperatively.  Every wait after that is bounded by a clock too: a workgroup that
// waits longer than kSyncSeconds sets `lost` and ends, and so do the others.  A solve
// whose launch is lost, or refused by the device, goes on kernel by kernel from the x
// there is.
//
// Measured per iteration (pressure equation on jittered cubes in Z order,
// kernel-by-kernel form -> this one): FP64 32^3 10.8 -> 5.3 us, 64^3 21.6 -> 7.9, 96^3
// 39.6 -> 12.0, 128^3 65.6 -> 28.0; FP32 32^3 10.9 -> 5.8, 64^3 16.4 -> 7.3, 96^3 27.3
// -> 9.9, 128^3 42.3 -> 14.8.  At 128^3 FP64 12 of the 28 us are the matrix stream
// (126 MB, from the memory-side cache), 16 the rest: two exchanges (2.4 us each on an
// idle chip) with their waits for the slowest workgroup, the ghosts, the LDS reads.
#pragma once

#include "cgkernels.hpp"

#include <algorithm>
#include <vector>

namespace fvhip {
namespace {

constexpr int kPersistThreads = 1024;  // four tiles of kCgBlock threads
constexpr int kPersistSub = kPersistThreads / kCgBlock;
constexpr int kPersistGroups = kCgMaxTiles / kPersistSub;  // workgroups at most
constexpr int kSlotWords = 16;  // up to four doubles as half-payload words; a 128-byte line per slot
constexpr int kCopies = 8;       // of what many workgroups read
constexpr int kSlotBuffer = (kPersistGroups + 8 * kCopies) * kSlotWords;  // workgroups; groups of them
constexpr int kStopApart = 5;  // CgState::stop after a plain launch whose workgroups did not meet
constexpr double kSyncSeconds = 20.0, kFailSeconds = 0.005;
constexpr double kClockHz = 1e8;  // wall_clock64: 100 MHz

// The assembled system, for the persistent forms that scale the matrix and take
// explicit residuals themselves.
struct CsrSystem {
    const int32_t *rowOffs, *diag;
    const double *vals, *rhs;
};

// What PersistSlots::launch says of a launch.
struct PersistLaunch {
    unsigned long long meet;  // Meeting::target
    uint32_t fails;           // exchange of the result's residual, if workgroups 8 to 15 are
                              // to miss it and the waits to end after kFailSeconds (tests)
};

// Arguments by value: the kernel reads them from scalar registers instead of
// chasing the launch description and the system description in memory.
template <typename S>
struct CgPersist {
    int32_t N, tiles, rowsPerTile;
    int32_t iters;        // iterations this launch may run
    uint32_t tag0;        // sequence number of its first exchange
    const int32_t* sellCol;  // slices of one width W: entry k of row i at
    const S* sval;           // (i / 64) * 64 W + 64 k + i % 64
    const S* g;
    S *d, *r, *p;
    S* p2;                   // (kc_persist_far)
    const uint32_t* words;   // the columns, see k_ghost_plan; ghosts of each tile
    const int32_t *ghosts, *count;
    int32_t ghostStride;
    CgState* st;
    unsigned long long* slots;  // 2 * kSlotBuffer
    // WHOLE: the system, its solution, and the solve's limits; fresh: start from x,
    // else go on where a launch ran out of iterations
    CsrSystem m;
    double* x;
    double tol, atol;
    int32_t maxit, fresh;
    CgState* host;            // what the host reads of the state (pinned)
    PersistLaunch launch;
};

template <typename T>
__device__ __forceinline__ void put_shared(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T get_shared(const T* p) {
    return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Keeps x in its register as it is: without this the compiler turns the 32-bit
// offsets, which do not change between iterations, into 64-bit addresses held
// across the loop (two registers each, and the rows no longer fit).
__device__ __forceinline__ void opaque(uint32_t& x) { asm volatile("" : "+v"(x)); }

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ double uniform(double x) {
    const long long b = __double_as_longlong(x);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The byte at base + off, a 32-bit offset: one scalar base and one vector
// register per address.
template <typename T>
__device__ __forceinline__ T* at_byte(T* base, uint32_t off) {
    return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off);
}
template <typename T>
__device__ __forceinline__ const T* at_byte(const T* base, uint32_t off) {
    return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}

// Lane l of the lower half of a group of 2 * OFF lanes: x of lane l + OFF (what
// __shfl_down gives those lanes; the others get something).  Register moves
// between lanes, where __shfl_down goes through the LDS unit (about 130 cycles a
// step, and a reduction is a chain of six).
template <int OFF>
__device__ __forceinline__ uint32_t lane_down(uint32_t x) {
    if constexpr (OFF == 32)
        return __builtin_amdgcn_permlane32_swap(x, x, false, false)[1];
    else if constexpr (OFF == 16)
        return __builtin_amdgcn_permlane16_swap(x, x, false, false)[1];
    else  // row_shl:OFF
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x100 + OFF, 0xf, 0xf, true);
}
template <int OFF>
__device__ __forceinline__ double lane_down(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const uint32_t lo = lane_down<OFF>((uint32_t)b), hi = lane_down<OFF>((uint32_t)(b >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
// Lane 0 of each group of 2 * OFF lanes: the group's sum, in the order of a
// __shfl_down tree (offsets OFF, OFF / 2, ..., 1).
template <int OFF>
__device__ __forceinline__ double lane_sum(double x) {
    x += lane_down<OFF>(x);
    if constexpr (OFF > 1)
        return lane_sum<OFF / 2>(x);
    else
        return x;
}
// x of one lane, in every lane
__device__ __forceinline__ double from_lane(double x, int lane) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const uint32_t lo = __builtin_amdgcn_readlane((int)b, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

struct PersistLds {
    double wave[4][kPersistThreads / 64];  // wave sums of this workgroup's tiles
    double tot[2][4];                      // by parity of the exchange: the grid's sums
    // PersistLaunch's, and how long a wait may last in 65536 clocks (as constants or in
    // scalar registers they cost the loops registers they do not have)
    uint32_t fails, limit;
    int bad, met;
    __device__ void begin(const PersistLaunch& a) {  // one thread, before the first barrier
        fails = a.fails;
        limit = (uint32_t)((a.fails ? kFailSeconds : kSyncSeconds) * kClockHz / 65536);
        bad = 0;
    }
};

// One workgroup's place in the grid exchange.  sum_slots adds the slots of a
// system's tiles as 256 threads: thread t takes t, t + 256, ... and the threads
// are added by a tree per wave of 64 (offsets 32, 16, ..., 1) and then wave by
// wave.  The tiles are dealt to the workgroups so that each of them, and each
// group of them, holds a whole branch of that tree:
//  * more than 256 tiles (256 workgroups): a workgroup holds thread t's tiles;
//    the 32 workgroups of XCD x (hardware workgroup i runs on XCD i % 8) hold the
//    threads of wave x / 2 with parity x % 2, the branch below the last step.
//    The first of them collects its group's sums and publishes theirs, and every
//    workgroup reads the eight group sums: the two hops take as long as polling
//    all 256 slots does on an idle device (2.4 us), with a sixteenth of the
//    polling, which otherwise slows the stores it waits for.  The readers of one
//    line wait for each other, so the group sums are published in kCopies copies
//    for 32 workgroups each (an iteration at 64^3 FP64: all eight in one line 9.9
//    us, one copy 8.6, eight 7.9, 16 or 32 8.0; up to 64 workgroups, copies change
//    nothing).  Polling twice as often costs more than it gains (8.2);
//  * up to 256 tiles (64 workgroups): a workgroup holds tiles l, l + 16, l + 32,
//    l + 48 of a wave, the branch of the first two steps, and every workgroup
//    reads all slots.
struct GridSum {
    unsigned long long* slots;
    uint32_t tag;
    int slot;    // this workgroup's slot
    int nslots;  // workgroups of the grid
    bool large;

    // Takes this workgroup's place in a grid over `tiles` tiles and returns the tile
    // of its part sub.
    __device__ int place(int tiles, int sub) {
        slot = (int)blockIdx.x;
        nslots = (int)gridDim.x;
        large = tiles > kCgBlock;
        if (!large) return 64 * (slot >> 4) + (slot & 15) + 16 * sub;
        const int x = slot & 7;
        return 64 * (x >> 1) + 2 * (slot >> 3) + (x & 1) + kCgBlock * sub;
    }

    __device__ static void publish(unsigned long long* s, double x, uint32_t tag) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(x);
        put_shared(s, b << 32 | tag);
        put_shared(s + 1, (b & 0xffffffff00000000ull) | tag);
    }
    // The values of slot s once they carry the tag; false after kSyncSeconds.
    template <int NV>
    __device__ bool collect(const unsigned long long* s, double (&v)[NV], const PersistLds& L) const {
        unsigned long long w[2 * NV], t0 = 0;
        for (int tries = 0;; ++tries) {
            bool ok = true;
            for (int j = 0; j < 2 * NV; ++j) w[j] = get_shared(s + j);
            for (int j = 0; j < 2 * NV; ++j) ok = ok && (uint32_t)w[j] == tag;
            if (ok) break;
            if ((tries & 63) == 63) {
                const unsigned long long t = wall_clock64();
                if (!t0) t0 = t;
                if ((uint32_t)((t - t0) >> 16) > L.limit) return false;
            }
        }
        for (int j = 0; j < NV; ++j)
            v[j] = __longlong_as_double(
                (long long)(w[2 * j] >> 32 | (w[2 * j + 1] & 0xffffffff00000000ull)));
        return true;
    }

    // The sum over the grid of every thread's v[], in the order of write_slot
    // and sum_slots.  PUBLISHED: this wave's put_shared stores are complete for
    // every workgroup once it returns.  LAST: the launch's last.  False after a timed-out
    // wait.
    template <int NV, bool PUBLISHED, bool LAST = false>
    __device__ bool sum(double (&v)[NV], double (&tot)[NV], PersistLds& L) {
        const int tid = (int)threadIdx.x, lane = tid & 63, wid = tid >> 6;
        for (int j = 0; j < NV; ++j) v[j] = lane_sum<32>(v[j]);
        if (lane == 0)
            for (int j = 0; j < NV; ++j) L.wave[j][wid] = v[j];
        if (PUBLISHED) __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        double* const out = L.tot[tag & 1];
        if (wid == 0) {
            unsigned long long* const buf = slots + (size_t)(tag & 1) * kSlotBuffer;
            // lane k: the partial of tile k, its waves in order (lanes past 3 repeat tile 3)
            double a[NV];
            for (int j = 0; j < NV; ++j) {
                double part = 0.0;
                const int k = min(lane, kPersistSub - 1);
                for (int w = 0; w < kCgBlock / 64; ++w)
                    part += L.wave[j][k * (kCgBlock / 64) + w];
                const double p0 = from_lane(part, 0), p1 = from_lane(part, 1),
                             p2 = from_lane(part, 2), p3 = from_lane(part, 3);
                a[j] = large ? ((p0 + p1) + p2) + p3 : (p0 + p2) + (p1 + p3);
            }
            if (lane == 0 && (!LAST || tag != L.fails || slot >> 3 != 1))
                for (int j = 0; j < NV; ++j)
                    publish(buf + (size_t)slot * kSlotWords + 2 * j, a[j], tag);
            bool ok = true;
            const unsigned long long* from = buf;  // the slots every workgroup reads
            int count = nslots;
            if (large) {
                const int group = slot & 7;  // slots of a group: group + 8 * member
                unsigned long long* const gbuf = buf + (size_t)kPersistGroups * kSlotWords;
                if (slot < 8) {
                    double m[NV];
                    for (int j = 0; j < NV; ++j) m[j] = 0.0;
                    if (lane < kPersistGroups / 8)
                        ok = collect<NV>(buf + (size_t)(group + 8 * lane) * kSlotWords, m, L);
                    for (int j = 0; j < NV; ++j) m[j] = from_lane(lane_sum<16>(m[j]), 0);
                    ok = __all(ok);  // a sum without one of its members is none
                    if (ok && lane < kCopies)
                        for (int j = 0; j < NV; ++j)
                            publish(gbuf + (size_t)(8 * lane + group) * kSlotWords + 2 * j, m[j], tag);
                }
                from = gbuf + (size_t)(8 * (slot & (kCopies - 1))) * kSlotWords;
                count = 8;
            }
            double g[NV];
            for (int j = 0; j < NV; ++j) g[j] = 0.0;
            if (ok && lane < count) ok = collect<NV>(from + (size_t)lane * kSlotWords, g, L);
            for (int j = 0; j < NV; ++j) {
                double r = 0.0;
                if (large) {  // lanes 2 w and 2 w + 1: the last step of wave w's tree
                    g[j] = lane_sum<1>(g[j]);
                    for (int w = 0; w < 4; ++w) r += from_lane(g[j], 2 * w);
                } else {      // lanes 16 w ...: the last four steps
                    g[j] = lane_sum<8>(g[j]);
                    for (int w = 0; w < 4; ++w) r += from_lane(g[j], 16 * w);
                }
                if (lane == 0) out[j] = r;
            }
            if (!ok) L.bad = 1;
        }
        __syncthreads();
        for (int j = 0; j < NV; ++j) tot[j] = uniform(out[j]);
        ++tag;
        return L.bad == 0;
    }
};

// Top bit of a column's byte offset: a row of another tile (an offset into the
// vectors instead of the LDS)
constexpr uint32_t kFar = 0x80000000u;

// b - A x of a tile's rows, their entries in column order, 256 rows at a time: the
// matrix rows are read coalesced into raw ((W + 1) * 256 doubles of LDS) and taken
// from there.  column(u, k): the columns; near(o), far(o), own(u): x at an LDS
// offset, at a vector offset, of this thread's row u; rhs(i): the right-hand side.
// out(u, in, r, b, a, c) gets
// each row's residual and right-hand side (zero past N) and its off-diagonal
// values and columns.  Every thread of the workgroup calls it; barriers before the
// first and after the last use of raw.
template <int RPT, int W, typename Live, typename Col, typename Rhs, typename Near, typename Far,
          typename Own, typename Out>
__device__ __forceinline__ void tile_residual(const CsrSystem& m, int N, int row0, int row1, int iw,
                                              double* raw, Live live, Col column, Rhs rhs,
                                              Near near, Far far, Own own, Out out) {
    const int lane = (int)threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
        __syncthreads();
        const int i0 = row0 + u * kCgBlock, i1 = min(min(i0 + kCgBlock, row1), N);
        int b = 0;
        if (i0 < i1) {
            b = m.rowOffs[i0];
            const int n = m.rowOffs[i1] - b;
            for (int k = (int)threadIdx.x & (kCgBlock - 1); k < n; k += kCgBlock)
                raw[k] = m.vals[b + k];
        }
        __syncthreads();
        if (live(u)) {
            const int i = iw + u * kCgBlock + lane;
            const bool in = i < N;
            const int o = in ? m.rowOffs[i] - b : 0, len = in ? m.rowOffs[i + 1] - b - o : 0;
            const int dg = in ? m.diag[i] : 0;
            const double bi = in ? rhs(i) : 0.0;
            uint32_t c[W];
            double a[W], x[W];
#pragma unroll
            for (int k = 0; k < W; ++k) c[k] = column(u, k);
#pragma unroll
            for (int k = 0; k < W; ++k) x[k] = c[k] & kFar ? far(c[k] & ~kFar) : near(c[k]);
            const double dx = in ? raw[o + dg] * own(u) : 0.0;
            double s = 0.0;
#pragma unroll
            for (int k = 0; k <= W; ++k) {  // the diagonal comes before entry dg
                if (k == dg && in) s += dx;
                if (k < W) {
                    a[k] = k + 1 < len ? raw[o + k + (k >= dg ? 1 : 0)] : 0.0;
                    if (k + 1 < len) s += a[k] * x[k];
                }
            }
            out(u, in, in ? bi - s : 0.0, bi, a, c);
        }
    }
    __syncthreads();
}

// Places of other tiles' rows ("ghosts") a tile's LDS has: as many as its rows can
// refer to where that fits beside the vectors, else what is left of the 160 KB.
template <typename S>
constexpr int ghost_cap(int rpt, int W) {
    if (sizeof(S) == 8) return rpt == 1 ? (W + 1) * kCgBlock : rpt == 2 ? rpt * kCgBlock * W : rpt == 4 ? 3008 : 1760;
    return rpt <= 4 ? rpt * kCgBlock * W : 5632;
}

// The columns of a tile's rows as 16-bit byte offsets in the tile's LDS: its own rows
// first (`own` places), then its ghosts, numbered in the order of rows blocks of 256,
// entries, rows; two columns a word, words as the sliced ELL's values (entry pair j
// of row i at (i / 64) * 32 W + 64 j + i % 64).  ghosts[tile * stride + slot]: the
// rows they are.  Without words only the counts are taken.
__global__ __launch_bounds__(kCgBlock) void k_ghost_plan(int N, int R, int W, int own, int size,
                                                         const int32_t* __restrict__ sellCol,
                                                         uint32_t* __restrict__ words,
                                                         int32_t* __restrict__ ghosts, int stride,
                                                         int32_t* __restrict__ count) {
    __shared__ int waves[kCgBlock / 64];
    const int tid = (int)threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int tile = (int)blockIdx.x, row0 = tile * R, row1 = min(row0 + R, (N + 63) & ~63);
    int base = 0;
    for (int i0 = row0; i0 < row1; i0 += kCgBlock) {
        const int i = i0 + tid;
        const bool in = i < row1;
        uint32_t word = 0;
        for (int k = 0; k < W; ++k) {
            const int c = in ? sellCol[(int64_t)(i >> 6) * 64 * W + 64 * k + lane] : row0;
            const bool far = (uint32_t)(c - row0) >= (uint32_t)R;
            const unsigned long long m = __ballot(far);
            if (lane == 0) waves[wid] = __popcll(m);
            __syncthreads();
            int slot = base + __popcll(m & ((1ull << lane) - 1));
            for (int w = 0; w < kCgBlock / 64; ++w) {
                if (w < wid) slot += waves[w];
                base += waves[w];
            }
            __syncthreads();
            if (!words) continue;
            if (far) ghosts[(int64_t)tile * stride + slot] = c;
            word |= (uint32_t)((far ? own + slot : c - row0) * size) << (k & 1 ? 16 : 0);
            if ((k & 1) && in) {
                words[(int64_t)(i >> 6) * 32 * W + 64 * (k >> 1) + lane] = word;
                word = 0;
            }
        }
    }
    if (tid == 0) count[tile] = base;
}

// The meeting of a plain launch's workgroups: words[0] counts arrivals over all
// launches, `target` is its value after this one's last; words[16] holds the latest
// decision, 2 * tag + 1 (all have arrived) or 2 * tag (one gave up).  The first to
// decide wins, so every workgroup sees the same decision, late ones included.
constexpr int kMeetWords = 32;
// Launches after a missed meeting that do not try one: as many as lose together, at 17 us
// each, what another miss would cost.
constexpr int kApartLaunches = 128;
constexpr unsigned long long kMeetClocks = (unsigned long long)(kClockHz / 500);  // 2 ms
struct Meeting {
    unsigned long long* words;
    unsigned long long target;  // 0: a cooperative launch
    uint32_t tag;

    __device__ unsigned long long decide(bool go) const {
        const unsigned long long mine = 2ull * tag + (go ? 1 : 0);
        unsigned long long seen = get_shared(words + 16);
        while (seen >> 1 != tag && !__hip_atomic_compare_exchange_strong(
                                       words + 16, &seen, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT)) {
        }
        return seen >> 1 != tag ? mine : seen;
    }
    __device__ void arrive() const {
        if (target && threadIdx.x == 0 &&
            __hip_atomic_fetch_add(words, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == target)
            decide(true);
    }
    // Whether all have arrived, in every thread.
    __device__ bool met(PersistLds& L) const {
        if (!target) return true;
        if (threadIdx.x == 0) {
            const unsigned long long t0 = wall_clock64();
            unsigned long long d;
            while ((d = get_shared(words + 16)) >> 1 != tag)
                if (wall_clock64() - t0 > kMeetClocks) {
                    d = decide(false);
                    break;
                }
            L.met = (int)(d & 1);
        }
        __syncthreads();
        return L.met != 0;
    }
};

// The ghosts of a tile, seen by one of its 256 threads: ghost s is thread s % 256's,
// which holds the places in the vectors of its first K (byte offsets, SIZE bytes a
// value).
template <int KG, int SIZE>
struct GhostWalk {
    static constexpr int K = KG;
    const int32_t* list;
    int n, t;
    uint32_t place[K];
    __device__ GhostWalk(const int32_t* ghosts, const int32_t* count, int stride, int tile, int tiles) {
        t = (int)threadIdx.x & (kCgBlock - 1);
        n = tile < tiles ? count[tile] : 0;
        list = ghosts + (int64_t)(tile < tiles ? tile : 0) * stride;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int s = t + j * kCgBlock;
            place[j] = s < n ? (uint32_t)list[s] * (uint32_t)SIZE : 0u;
        }
    }
    // K ghosts at a time: load(j, place) for each, then use(j, s).  The places of the
    // next K are loaded meanwhile.
    template <class Load, class Use>
    __device__ __forceinline__ void each(Load load, Use use) const {
        uint32_t o[K];
#pragma unroll
        for (int j = 0; j < K; ++j) o[j] = place[j];
        for (int s0 = 0; s0 < n; s0 += K * kCgBlock) {
            uint32_t next[K];
            if (s0 + K * kCgBlock < n) {
#pragma unroll
                for (int j = 0; j < K; ++j)
                    next[j] = (uint32_t)list[min(s0 + (K + j) * kCgBlock + t, n - 1)] * (uint32_t)SIZE;
            }
#pragma unroll
            for (int j = 0; j < K; ++j)
                if (s0 + j * kCgBlock + t < n) load(j, o[j]);
#pragma unroll
            for (int j = 0; j < K; ++j)
                if (s0 + j * kCgBlock + t < n) use(j, s0 + j * kCgBlock + t);
#pragma unroll
            for (int j = 0; j < K; ++j) o[j] = next[j];
        }
    }
};

// RPT: rows per thread (the rows a tile gives a thread, rounded up to a power
// of two); W: entries of every slice of the sliced ELL; RES: rows of each thread
// whose values and columns stay in registers; GL: rows whose g is in LDS too, DLDS: d
// (else in registers).  p is in LDS, the tile's own rows' and its ghosts'.  Rows past a
// tile's end take part as zeros; the vectors are allocated to a multiple of 64
// rows, so the rows of the last slice past N are stored too (as zeros).
// WHOLE (FP64): the launch also scales the matrix (from the CSR, also when it goes
// on), takes the initial residual, and after the stop adds the correction to x and
// takes the explicit residual, which goes to CgState::rrep: on small systems the
// nine launches around the iterations cost as much as they do (32^3 heat step of 5
// iterations 144 us with the start and end as kernels in a replayed graph, 103 whole,
// 97 with the ghosts in LDS, 78 with a plain launch, 75 with the state written to
// the host and the start in one exchange; 16^3 Poisson of 125 iterations
// 0.82 -> 0.73 -> 0.56 ms).
template <typename S, int RPT, int W, int RES, int GL, bool DLDS, bool WHOLE>
__global__ __launch_bounds__(kPersistThreads) void kc_persist(CgPersist<S> A) {
    constexpr int kOwn = RPT * kCgBlock, kTile = kOwn + ghost_cap<S>(RPT, W);
    static_assert(kTile * sizeof(S) <= 65536, "16-bit columns");
    __shared__ PersistLds L;
    __shared__ S lp[kPersistSub * kTile], ldAll[DLDS ? kPersistSub * kOwn : 1],
        lgAll[GL ? kPersistSub * GL * kCgBlock : 1];
    // the raw matrix rows of 256 rows of the tile (start and end) share the ghosts' LDS
    static_assert(!WHOLE || (sizeof(S) == 8 && GL == RPT && DLDS && RES == RPT &&
                             ghost_cap<S>(RPT, W) >= (W + 1) * kCgBlock),
                  "whole solves are FP64, with the matrix in registers");
    const int tid = (int)threadIdx.x, lane = tid & 63;
    // a tile is four waves and its rows are dealt in waves of 64, so its bounds
    // are the same in every lane: kept in scalar registers
    const int sub = __builtin_amdgcn_readfirstlane(tid / kCgBlock);
    GridSum gs;
    gs.slots = A.slots;
    gs.tag = A.tag0;
    const int R = A.rowsPerTile;
    const int tile = gs.place(A.tiles, sub);
    CgState* const st = A.st;
    const bool lead = gs.slot == 0 && tid == 0;
    const Meeting meeting{A.slots + 2 * kSlotBuffer, WHOLE ? A.launch.meet : 0, A.tag0};
    meeting.arrive();
    if (!WHOLE || !A.fresh) {
        const int entry = st->stop;
        if (entry || st->lost) {
            if (lead) st->done = entry;  // as the update kernel of a stopped system
            return;
        }
    }
    if (tid == 0) L.begin(A.launch);
    const int row0 = tile * R;
    const int row1 = tile < A.tiles ? min(row0 + R, (A.N + 63) & ~63) : row0;
    // this wave's first row; its row u is iw + 256 u + lane, of slice (iw + 256 u) / 64
    const int iw = row0 + __builtin_amdgcn_readfirstlane(tid & (kCgBlock - 64));
    auto live = [&](int u) { return iw + u * kCgBlock < row1; };
    uint32_t lb = (uint32_t)lane * sizeof(S);
    auto mine = [&](auto* vec, int u) { return at_byte(vec + (iw + u * kCgBlock), lb); };
    S *const tp = lp + sub * kTile, *const ghost = tp + kOwn;
    S *const ld = ldAll + (DLDS ? sub * kOwn : 0), *const lg = lgAll + sub * (GL * kCgBlock);
    auto lds = [&](S* vec, int u) -> S& { return *at_byte(vec + (iw - row0) + u * kCgBlock, lb); };
    auto value = [&](int u, int k) {
        return *at_byte(A.sval + ((int64_t)(iw + u * kCgBlock) * W + 64 * k), lb);
    };
    auto pair = [&](int u, int j) {
        return *at_byte(A.words + ((int64_t)(iw + u * kCgBlock) * (W / 2) + 64 * j), lb / (uint32_t)(sizeof(S) / 4));
    };
    auto col = [](const uint32_t (&c)[W / 2], int k) { return k & 1 ? c[k / 2] >> 16 : c[k / 2] & 0xffffu; };

    // A ghost's p follows p' = r + beta p like its owner's, so all that a tile reads of
    // another's rows is their r.
    const GhostWalk<RPT == 2 || (RPT == 4 && sizeof(S) == 4) ? 6 : 4, sizeof(S)> ghosts(
        A.ghosts, A.count, A.ghostStride, tile, A.tiles);

    // Bit u: row u has a far column.  The pattern is symmetric, so those are the
    // rows that other workgroups read, and only they are published.
    uint32_t shown = 0;

    S rv[RPT], qv[RPT], gr[GL < RPT ? RPT - GL : 1], dr[DLDS ? 1 : RPT];
    S mv[RES ? RES : 1][W];
    uint32_t mc[RES ? RES : 1][W / 2];
    auto d_of = [&](int u) -> S& {
        if constexpr (DLDS)
            return lds(ld, u);
        else
            return dr[u];
    };
    auto g_of = [&](int u) -> S& {
        if (u < GL) return lds(lg, u);
        return gr[GL < RPT ? u - GL : 0];
    };
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
        rv[u] = qv[u] = S(0);
        if (u >= GL) gr[GL < RPT ? u - GL : 0] = S(0);
        if constexpr (!DLDS) dr[u] = S(0);
        uint32_t c[W / 2];
        for (int j = 0; j < W / 2; ++j) c[j] = live(u) ? pair(u, j) : 0u;
        for (int k = 0; k < W; ++k)
            if (col(c, k) >= kOwn * sizeof(S)) shown |= 1u << u;
        if (u < RES) {
            for (int k = 0; k < W; ++k) mv[u][k] = S(0);
            for (int j = 0; j < W / 2; ++j) mc[u][j] = c[j];
        }
    }
    double bnorm, tol, atol, delta, rrep, rho, rhoPrev, alpha, res, res0;
    int maxit, it, stop = 0;
    bool ok = true;
    [[maybe_unused]] auto residual = [&](auto far, auto out) {
        tile_residual<RPT, W>(
            A.m, A.N, row0, row1, iw, reinterpret_cast<double*>(ghost), live,
            [&](int u, int k) {
                const uint32_t c = (uint32_t)*at_byte(
                    A.sellCol + ((int64_t)(iw + u * kCgBlock) * W + 64 * k), (uint32_t)lane * 4u);
                const uint32_t l = c - (uint32_t)row0;
                return l < (uint32_t)R ? l * (uint32_t)sizeof(S) : c * (uint32_t)sizeof(S) | kFar;
            },
            [&](int i) { return A.m.rhs[i]; }, [&](uint32_t o) { return *at_byte(tp, o); }, far,
            [&](int u) { return lds(tp, u); }, out);
    };
    if constexpr (!WHOLE) {
#pragma unroll
        for (int u = 0; u < RPT; ++u)
            if (live(u)) {
                S p0 = S(0), d0 = S(0), g0 = S(0);
                if (u < RES)
                    for (int k = 0; k < W; ++k) mv[u][k] = value(u, k);
                if (iw + u * kCgBlock + lane < A.N) {
                    rv[u] = *mine(A.r, u);
                    p0 = *mine(A.p, u);
                    d0 = *mine(A.d, u);
                    g0 = *mine(A.g, u);
                }
                lds(tp, u) = p0;
                d_of(u) = d0;
                g_of(u) = g0;
            }
    } else {
        // x (in p's place) and g of the own rows, as kc_begin
        const double first = A.m.vals[A.m.rowOffs[0] + A.m.diag[0]];
        auto root = [&](double di) {
            const bool good =
                di != 0.0 && (di > 0.0) == (first > 0.0) && fabs(di) <= 1.7976931348623157e308;
            return good ? copysign(sqrt(fabs(di)), di) : (double)NAN;
        };
#pragma unroll
        for (int u = 0; u < RPT; ++u)
            if (live(u)) {
                const int i = iw + u * kCgBlock + lane;
                const bool in = i < A.N;
                lds(tp, u) = in ? *mine(A.x, u) : 0.0;
                lds(lg, u) = in ? root(A.m.vals[A.m.rowOffs[i] + A.m.diag[i]]) : 0.0;
                lds(ld, u) = !A.fresh && in ? *mine(A.d, u) : 0.0;
            }
        double s2[2] = {0.0, 0.0};
        residual([&](uint32_t o) { return *at_byte(A.x, o); },
                 [&](int u, bool in, double ri, double bi, const double (&a)[W],
                     const uint32_t (&c)[W]) {
                     const double gi = in ? lds(lg, u) : 1.0;
#pragma unroll
                     for (int k = 0; k < W; ++k) {  // as kc_scale
                         double gj;
                         if (c[k] & kFar) {
                             const uint32_t j = (c[k] & ~kFar) / 8u;
                             gj = root(A.m.vals[A.m.rowOffs[j] + A.m.diag[j]]);
                         } else {
                             gj = *at_byte(lg, c[k]);
                         }
                         mv[u][k] = a[k] != 0.0 ? a[k] / (gi * fabs(gj)) : 0.0;
                     }
                     rv[u] = ri;
                     s2[0] += ri * ri;
                     s2[1] += bi * bi;
                 });
        if (!meeting.met(L)) {
            if (lead) st->stop = A.host->stop = kStopApart;
            return;
        }
        if (A.fresh) {
            // ||b||, the relative residual; r = G^-1 r64, p = r, ||G r||^2 and r.r
            double s4[4] = {s2[0], s2[1], 0.0, 0.0}, t4[4];
#pragma unroll
            for (int u = 0; u < RPT; ++u)
                if (live(u)) {
                    const bool in = iw + u * kCgBlock + lane < A.N;
                    const double gi = lds(lg, u);
                    const double ri = in ? rv[u] / gi : 0.0;
                    rv[u] = ri;
                    lds(tp, u) = ri;
                    if (shown >> u & 1) put_shared(mine(A.p, u), ri);
                    const double ur = ri * gi;
                    s4[2] += ur * ur;
                    s4[3] += ri * ri;
                }
            if ((ok = gs.sum<4, true>(s4, t4, L))) {
                bnorm = sqrt(t4[1]);
                if (!(bnorm > 0.0)) bnorm = 1.0;
                res = res0 = sqrt(t4[0]) / bnorm;
                if (lead) A.host->res0 = res0;
                rho = t4[3];
                rhoPrev = alpha = 0.0;
                it = 0;
                // the decision of kc_direction after a start
                const bool conv = res <= A.tol || res * bnorm <= A.atol;
                stop = conv ? 2 : !(res <= 1.7976931348623157e308) ? 3 : A.maxit <= 0 ? 1 : 0;
            }
        } else {
#pragma unroll
            for (int u = 0; u < RPT; ++u)
                if (live(u)) {
                    rv[u] = *mine(A.r, u);
                    lds(tp, u) = *mine(A.p, u);
                }
        }
    }
    if (!WHOLE || !A.fresh) {
        bnorm = uniform(st->bnorm);
        rho = uniform(st->rho);
        rhoPrev = uniform(st->rhoPrev);
        alpha = uniform(st->alpha);
        res = uniform(st->res);
        res0 = uniform(st->res0);
        it = __builtin_amdgcn_readfirstlane(st->it);
    }
    tol = WHOLE ? A.tol : uniform(st->tol);
    atol = WHOLE ? A.atol : uniform(st->atol);
    maxit = WHOLE ? A.maxit : __builtin_amdgcn_readfirstlane(st->maxit);
    delta = WHOLE ? 0.0 : uniform(st->delta);
    rrep = WHOLE ? 0.0 : uniform(st->rrep);
    S beta = S(0);
    {  // the ghosts' p
        S x[ghosts.K];
        ghosts.each([&](int j, uint32_t o) { x[j] = get_shared(at_byte(A.p, o)); },
                    [&](int j, int s) { ghost[s] = x[j]; });
    }
    // streamed rows: loaded when the row before is done (the first one of an iteration
    // at the end of the one before, across its exchanges); the other waves of the SIMD
    // compute meanwhile, and a second set of registers would not fit
    S vn[W];
    uint32_t cn[W / 2];
    auto fetch = [&](int u) {
#pragma unroll
        for (int j = 0; j < W / 2; ++j) cn[j] = pair(u, j);
#pragma unroll
        for (int k = 0; k < W; ++k) vn[k] = value(u, k);
    };
    if (RES < RPT && live(RES)) fetch(RES);
    for (int n = 0; ok && !stop && n < A.iters; ++n) {
        opaque(lb);
        for (int u = 0; u < RES; ++u)
            for (int j = 0; j < W / 2; ++j) opaque(mc[u][j]);
        if (n) {
            S x[ghosts.K];
            ghosts.each([&](int j, uint32_t o) { x[j] = get_shared(at_byte(A.r, o)); },
                        [&](int j, int s) { ghost[s] = x[j] + beta * ghost[s]; });
        }
        __syncthreads();
        // q = As p, p.q
        double v1[1] = {0.0}, t1[1];
        auto row = [&](int u, const S (&v)[W], const uint32_t (&c)[W / 2]) {
            S x[W];
#pragma unroll
            for (int k = 0; k < W; ++k) x[k] = *at_byte(tp, col(c, k));
            const S own = lds(tp, u);
            S sum = own;
#pragma unroll
            for (int k = 0; k < W; ++k) sum += v[k] * x[k];
            qv[u] = sum;
            v1[0] += (double)own * (double)sum;
        };
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            if (!live(u)) break;
            if (u < RES) {
                row(u, mv[u], mc[u]);
            } else {
                row(u, vn, cn);
                if (RPT == 8 && sizeof(S) == 8) __builtin_amdgcn_sched_barrier(0);
                fetch(u + 1 < RPT && live(u + 1) ? u + 1 : RES);
            }
        }
        if (!(ok = gs.sum<1, false>(v1, t1, L))) break;
        // alpha; d += alpha p, r -= alpha q, ||G r||^2 and r.r
        alpha = rho / t1[0];
        ++it;
        rhoPrev = rho;
        const S a = (S)alpha;
        double v2[2] = {0.0, 0.0}, t2[2];
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            if (!live(u)) break;
            const S ri = rv[u] - a * qv[u];
            rv[u] = ri;
            if (shown >> u & 1) put_shared(mine(A.r, u), ri);
            d_of(u) = d_of(u) + a * lds(tp, u);
            const double ur = (double)ri * (double)g_of(u);
            v2[0] += ur * ur;
            v2[1] += (double)ri * (double)ri;
        }
        if (!(ok = gs.sum<2, true>(v2, t2, L))) break;
        // the stop decision (cg_decide) and the next direction
        const double rn = sqrt(t2[0]);
        res = rn / bnorm;
        rho = t2[1];
        if (res <= tol || rn <= atol || it >= maxit || !(res == res) ||
            (delta > 0.0 && rn < delta * rrep)) {
            stop = 1;
            break;
        }
        beta = (S)(rho / rhoPrev);
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            if (!live(u)) break;
            lds(tp, u) = rv[u] + beta * lds(tp, u);
        }
    }
    if constexpr (WHOLE) {
        if (ok && stop) {  // x += |G|^-1 d, the explicit residual of the result
#pragma unroll
            for (int u = 0; u < RPT; ++u)
                if (live(u) && iw + u * kCgBlock + lane < A.N) {
                    const double x = *mine(A.x, u) + lds(ld, u) / fabs(lds(lg, u));
                    lds(tp, u) = x;
                    if (shown >> u & 1)
                        put_shared(mine(A.x, u), x);
                    else
                        *mine(A.x, u) = x;
                }
            double none[1] = {0.0}, all[1], s1[1] = {0.0};
            if ((ok = gs.sum<1, true>(none, all, L))) {
                residual([&](uint32_t o) { return get_shared(at_byte(A.x, o)); },
                         [&](int, bool, double ri, double, const double (&)[W],
                             const uint32_t (&)[W]) { s1[0] += ri * ri; });
                ok = gs.sum<1, false, true>(s1, all, L);
                rrep = sqrt(all[0]) / bnorm;
            }
        }
    }
    if (!ok) {
        if (tid == 0) {
            st->lost = 1;
            if (WHOLE) A.host->lost = 1;
        }
        return;
    }
    if (!WHOLE || !stop) {
#pragma unroll
        for (int u = 0; u < RPT; ++u)
            if (live(u)) {
                *mine(A.r, u) = rv[u];
                *mine(A.p, u) = lds(tp, u);
                *mine(A.d, u) = d_of(u);
            }
    }
    if (lead) {
        st->rho = rho;
        st->rhoPrev = rhoPrev;
        st->alpha = alpha;
        st->res = res;
        st->it = it;
        st->stop = stop;
        st->done = 0;
        st->pbuf = 0;
        if (!WHOLE) st->runs += 1;
        if (WHOLE) {
            st->bnorm = bnorm;
            st->res0 = res0;
            st->rrep = rrep;
            // straight to the host: a copy behind the launch takes 5 us
            A.host->res = res;
            A.host->rrep = rrep;
            A.host->bnorm = bnorm;
            A.host->it = it;
            A.host->stop = stop;
        }
    }
}

// The form for tiles with more ghosts than fit (systems of over 2^20 rows in block
// order, of over 2^19 whose mesh was not renumbered; 128^3 FP64 in block order
// 63 us kernel by kernel, 46 here): a far column's p' is evaluated for each entry, from
// the published r and the published p of the iteration before, and the columns are read
// as 32-bit row numbers.
template <typename S, int RPT, int W, int RES, bool GLDS>
__global__ __launch_bounds__(kPersistThreads) void kc_persist_far(CgPersist<S> A) {
    __shared__ PersistLds L;
    __shared__ S lp[RPT * kPersistThreads], ld[RPT * kPersistThreads],
        lg[GLDS ? RPT * kPersistThreads : 1];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    // a tile is four waves and its rows are dealt in waves of 64, so its bounds
    // are the same in every lane: kept in scalar registers
    const int sub = __builtin_amdgcn_readfirstlane(tid / kCgBlock);
    GridSum gs;
    gs.slots = A.slots;
    gs.tag = A.tag0;
    const int R = A.rowsPerTile;
    const int tile = gs.place(A.tiles, sub);
    // this tile's rows [cbase, cbase + R) have their p in LDS, from lofs on
    const uint32_t cbase = (uint32_t)tile * R, lofs = (uint32_t)sub * (RPT * kCgBlock);
    CgState* const st = A.st;
    const bool lead = gs.slot == 0 && tid == 0;
    const int entry = st->stop;
    if (entry || st->lost) {
        if (lead) st->done = entry;  // as the update kernel of a stopped system
        return;
    }
    if (tid == 0) L.begin(A.launch);
    const int row0 = tile * R;
    const int row1 = tile < A.tiles ? min(row0 + R, (A.N + 63) & ~63) : row0;
    // this wave's first row; its row u is iw + 256 u + lane, of slice (iw + 256 u) / 64
    const int iw = row0 + __builtin_amdgcn_readfirstlane(tid & (kCgBlock - 64));
    auto live = [&](int u) { return iw + u * kCgBlock < row1; };
    uint32_t lb = (uint32_t)lane * sizeof(S);
    auto mine = [&](auto* vec, int u) { return at_byte(vec + (iw + u * kCgBlock), lb); };
    const uint32_t lown = (uint32_t)(iw - (int)cbase) + lofs;  // LDS place of row u: lown + 256 u + lane
    auto lds = [&](S* vec, int u) -> S& { return *at_byte(vec + lown + u * kCgBlock, lb); };
    auto value = [&](int u, int k) {
        return *at_byte(A.sval + ((int64_t)(iw + u * kCgBlock) * W + 64 * k), lb);
    };
    // a column as the byte offset of its p in LDS, or (kFar) of its row in the vectors
    auto column = [&](int u, int k) {
        const uint32_t c = (uint32_t)*at_byte(
            A.sellCol + ((int64_t)(iw + u * kCgBlock) * W + 64 * k), (uint32_t)lane * 4u);
        const uint32_t l = c - cbase;
        return l < (uint32_t)R ? (l + lofs) * (uint32_t)sizeof(S) : c * (uint32_t)sizeof(S) | kFar;
    };

    // Bit u: row u has a far column.  The pattern is symmetric, so those are the
    // rows that other workgroups read, and only they are published.
    uint32_t shown = 0;

    S rv[RPT], qv[RPT], gr[GLDS ? 1 : RPT];
    S mv[RES ? RES : 1][W];
    uint32_t mc[RES ? RES : 1][W];
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
        rv[u] = qv[u] = S(0);
        if (u < RES)
            for (int k = 0; k < W; ++k) {
                mv[u][k] = S(0);
                mc[u][k] = 0;
            }
        if constexpr (!GLDS) gr[u] = S(0);
    }
    double bnorm, tol, atol, delta, rrep, rho, rhoPrev, alpha, res;
    int maxit, it, stop = 0;
    bool ok = true;
    {
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            S p0 = S(0), d0 = S(0), g0 = S(0);
            if (live(u)) {
                if (u < RES) {
#pragma unroll
                    for (int k = 0; k < W; ++k) {
                        mv[u][k] = value(u, k);
                        mc[u][k] = column(u, k);
                        shown |= mc[u][k] >> 31 << u;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < W; ++k) shown |= column(u, k) >> 31 << u;
                }
                if (iw + u * kCgBlock + lane < A.N) {
                    rv[u] = *mine(A.r, u);
                    p0 = *mine(A.p, u);
                    d0 = *mine(A.d, u);
                    g0 = *mine(A.g, u);
                }
                lds(lp, u) = p0;
                lds(ld, u) = d0;
                if constexpr (GLDS) lds(lg, u) = g0;
            }
            if constexpr (!GLDS) gr[u] = g0;
        }
    }
    bnorm = uniform(st->bnorm);
    rho = uniform(st->rho);
    rhoPrev = uniform(st->rhoPrev);
    alpha = uniform(st->alpha);
    res = uniform(st->res);
    it = __builtin_amdgcn_readfirstlane(st->it);
    tol = uniform(st->tol);
    atol = uniform(st->atol);
    maxit = __builtin_amdgcn_readfirstlane(st->maxit);
    delta = uniform(st->delta);
    rrep = uniform(st->rrep);
    S beta = S(0);
    S *pold = A.p, *pnew = A.p2;  // the direction before this iteration's, and the next one's place
    __syncthreads();
    for (int n = 0; ok && !stop && n < A.iters; ++n) {
        opaque(lb);
        for (int u = 0; u < RES; ++u)
            for (int k = 0; k < W; ++k) opaque(mc[u][k]);
        // q = As p, p.q.  A far column's p: as published for the launch's first
        // iteration, afterwards from its published r and old p
        double v1[1] = {0.0}, t1[1];
        auto row = [&](int u, const S (&v)[W], const uint32_t (&c)[W], auto next) {
            S x[W], y[W];
#pragma unroll
            for (int k = 0; k < W; ++k) {
                if (c[k] & kFar) {
                    const uint32_t o = c[k] & ~kFar;
                    y[k] = get_shared(at_byte(pold, o));
                    x[k] = n ? get_shared(at_byte(A.r, o)) : S(0);
                } else {
                    x[k] = *at_byte(lp, c[k]);
                }
            }
            next();
            const S own = lds(lp, u);
            S sum = own;
#pragma unroll
            for (int k = 0; k < W; ++k) {
                if (c[k] & kFar) x[k] = n ? x[k] + beta * y[k] : y[k];
                sum += v[k] * x[k];
            }
            qv[u] = sum;
            v1[0] += (double)own * (double)sum;
        };
        // streamed rows: the next row's columns are in flight during this row, whose
        // values are loaded beside the far columns' vectors
        uint32_t cn[W];
        auto fetch = [&](int u) {
#pragma unroll
            for (int k = 0; k < W; ++k) cn[k] = column(u, k);
        };
        if (RES < RPT && live(RES)) fetch(RES);
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            if (!live(u)) break;
            if (u < RES) {
                row(u, mv[u], mc[u], [] {});
            } else {
                S v[W];
                uint32_t c[W];
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    c[k] = cn[k];
                    v[k] = value(u, k);
                }
                row(u, v, c, [&] {
                    if (u + 1 < RPT && live(u + 1)) fetch(u + 1);
                });
            }
        }
        if (!(ok = gs.sum<1, true>(v1, t1, L))) break;
        // alpha; d += alpha p, r -= alpha q, ||G r||^2 and r.r
        alpha = rho / t1[0];
        ++it;
        rhoPrev = rho;
        const S a = (S)alpha;
        double v2[2] = {0.0, 0.0}, t2[2];
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            if (!live(u)) break;
            const S ri = rv[u] - a * qv[u];
            rv[u] = ri;
            if (shown >> u & 1) put_shared(mine(A.r, u), ri);
            lds(ld, u) = lds(ld, u) + a * lds(lp, u);
            S gi;
            if constexpr (GLDS)
                gi = lds(lg, u);
            else
                gi = gr[u];
            const double ur = (double)ri * (double)gi;
            v2[0] += ur * ur;
            v2[1] += (double)ri * (double)ri;
        }
        if (!(ok = gs.sum<2, true>(v2, t2, L))) break;
        // the stop decision (cg_decide) and the next direction
        const double rn = sqrt(t2[0]);
        res = rn / bnorm;
        rho = t2[1];
        if (res <= tol || rn <= atol || it >= maxit || !(res == res) ||
            (delta > 0.0 && rn < delta * rrep)) {
            stop = 1;
            break;
        }
        beta = (S)(rho / rhoPrev);
        if (n) {
            S* const t = pold;
            pold = pnew;
            pnew = t;
        }
#pragma unroll
        for (int u = 0; u < RPT; ++u) {
            if (!live(u)) break;
            const S pi = rv[u] + beta * lds(lp, u);
            lds(lp, u) = pi;
            if (shown >> u & 1) put_shared(mine(pnew, u), pi);
        }
        __syncthreads();
    }
    if (!ok) {
        if (tid == 0) st->lost = 1;
        return;
    }
#pragma unroll
    for (int u = 0; u < RPT; ++u)
        if (live(u)) {
            *mine(A.r, u) = rv[u];
            *mine(A.p, u) = lds(lp, u);
            *mine(A.d, u) = lds(ld, u);
        }
    if (lead) {
        st->rho = rho;
        st->rhoPrev = rhoPrev;
        st->alpha = alpha;
        st->res = res;
        st->it = it;
        st->stop = stop;
        st->done = 0;
        st->pbuf = 0;
        st->runs += 1;
    }
}

inline const int32_t* uniform_col(const fv_sparsity* sp) {
    return sp->sellUniform ? sp->sellCol.p : sp->uniCol.p;
}

// A buffer of at least n elements; the one there is stays if there is no room for another.
template <typename T>
inline void grow(DBuf<T>& b, fv_ctx* c, size_t n) {
    if (b.n >= n) return;
    DBuf<T> larger;
    larger.alloc(c, n);
    b = std::move(larger);
}

// The ghosts of a pattern's tiles for values of `size` bytes (own: rows a tile has places
// for); null if a tile has more than cap.  The plan stays with the pattern: its systems and
// solvers have the same tiles (cg_tile_rows), so one per value size serves them all.
inline const fv_ghost_plan* ghost_plan(fv_ctx* c, fv_sparsity* sp, int tiles, int R, int W, int own,
                                       int size, int cap) {
    fv_ghost_plan& p = sp->ghostPlan[size == 8 ? 0 : 1];
    uniform_sell(sp);
    auto plan = [&](uint32_t* w, int32_t* g) {
        k_ghost_plan<<<tiles, kCgBlock, 0, c->stream>>>(sp->nRows, R, W, own, size, uniform_col(sp), w, g,
                                                        p.stride, p.count.p);
        FV_LAUNCH_CHECK();
    };
    if (p.stride < 0) {
        p.count.alloc(c, tiles);
        plan(nullptr, nullptr);
        std::vector<int32_t> n(tiles);
        p.count.download(n.data());
        p.stride = *std::max_element(n.begin(), n.end());
    }
    if (p.stride > cap) return nullptr;
    if (!p.words.p) {
        p.ghosts.alloc(c, (size_t)tiles * (p.stride > 0 ? p.stride : 1));
        p.words.alloc(c, ((size_t)sp->nRows + 63) / 64 * 64 * W / 2);
        plan(p.words.p, p.ghosts.p);
    }
    return &p;
}

constexpr size_t kPersistWords = 2 * (size_t)kSlotBuffer + kMeetWords;

// The exchange buffer of a system and its launches.
struct PersistSlots {
    DBuf<unsigned long long> words;
    fv_persist_log* log = nullptr;
    unsigned long long meets = 0;  // arrivals of all plain launches
    int apart = 0;                 // launches that are to be cooperative, after one that did not meet
    bool doubted = false;          // the latest launch's state is to be taken for lost (tests)
    void alloc(fv_ctx* c, fv_persist_log* l) {
        words.alloc(c, kPersistWords);
        log = l;
    }
    void clear(hipStream_t s) {  // no word carries a tag that is still to come
        FV_HIP(hipMemsetAsync(words.p, 0, words.n * sizeof(unsigned long long), s));
        meets = 0;
    }
    // One launch; meeting: as a plain one whose workgroups meet.  False if the device
    // refuses it.
    template <typename Args>
    bool launch(void (*kernel)(Args), int grid, Args& args, bool meeting, hipStream_t s) {
        const int fault = log->take();
        const bool plain = meeting && apart == 0;
        if (meeting && apart > 0) --apart;
        args.launch = PersistLaunch{plain ? meets + grid : 0, 0};
        if (fault == FV_PERSIST_APART && plain) ++args.launch.meet;  // never reached
        doubted = fault == FV_PERSIST_LOST && !log->exchange;
        if (fault == FV_PERSIST_LOST && log->exchange) args.launch.fails = args.tag0 + (uint32_t)log->exchange;
        void* a[] = {&args};
        const void* const k = reinterpret_cast<const void*>(kernel);
        hipError_t e = hipErrorUnknown;
        if (fault != FV_PERSIST_REFUSED)
            e = plain ? hipLaunchKernel(k, dim3(grid), dim3(kPersistThreads), a, 0, s)
                      : hipLaunchCooperativeKernel(k, dim3(grid), dim3(kPersistThreads), a, 0, s);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            ++log->refused;
            return false;
        }
        ++log->launches;
        if (plain) meets += grid;
        return true;
    }
    void did_not_meet() {
        apart = kApartLaunches;
        ++log->apart;
    }
};

// Whether alloc() found room for the buffers of a persistent solver.
template <typename F>
bool persist_room(F&& alloc) {
    try {
        alloc();
        return true;
    } catch (const Error&) {
        (void)hipGetLastError();
        clear_error();
        return false;
    }
}

// Iterations a launch may run, of those that take kPersistMs.  A launch holds up to every CU
// until it ends, and the work of other streams waits; while another thread uses another
// context of the device it is an eighth as long.  Two threads, a Poisson solve at 128^3 beside
// heat steps at 32^3, a second of each: kernel by kernel 35 and 3600, launches of 2 ms 89 and
// 870, of 0.25 ms 72 and 3870, of 0.1 ms 53 and 7210; gradients at 64^3 beside it 24000,
// 1390, 4560, 8430.  Solves beside solves lose by short launches (two at 128^3 45 a second
// each, 38; kernel by kernel 19).
constexpr double kPersistMs = 2.0;
inline int persist_iters(fv_ctx* c, int whole) {
    ctx_touch(c);
    return ctx_beside(c) ? std::max(whole / 8, 1) : whole;
}

// Workgroups of a persistent launch over `tiles` tiles
inline int persist_grid(int tiles) {
    return tiles > kCgBlock ? kPersistGroups : 16 * (tiles / 64) + (tiles % 64 < 16 ? tiles % 64 : 16);
}

// Whether the device keeps the workgroups of such a launch resident together.
inline bool persist_fits(const void* kernel, int device, int grid) {
    int perCu = 0, cus = 0, coop = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, kernel, kPersistThreads, 0) !=
            hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return coop && (int64_t)perCu * cus >= grid;
}

}  // namespace
}  // namespace fvhip
