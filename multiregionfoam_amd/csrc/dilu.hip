// DILU (coupled Cholesky preconditioner) on gfx950: factorisation and the
// forward / backward sweeps of the preconditioner, executed by a schedule of
// chains (one wavefront per workgroup), level groups (a workgroup of up to 16
// per region) and spread levels (the whole device).
//
// Restated arithmetic (per region; interface coefficients are not part of
// the factor, the coupled preconditioner works on each region's lduMatrix):
//   factor    d[u] = diag[u] - sum_{faces f, u(f)=u, face order} upper_f*lower_f / d[l(f)],  rD = 1/d
//   forward   w[u] = rD[u]*r[u] - sum_{lower faces, face order} rD[u]*lower_f*w[l(f)]
//   backward  w[l] -= sum_{upper faces, reverse face order} rD[l]*upper_f*w[u(f)]
//
// General regions only: the sweeps of structured boxes are in dilu_box.hip,
// their factorisation at the end of this file.
//
// Each lane holds one row per step, whose dependencies were computed earlier
// by the same wave (chains) or workgroup (level groups) and are read from LDS,
// or by an earlier launch (spread levels).
// A step of a chain is latency-bound (one LDS round trip plus a short FMA
// chain), so the kernel keeps memory out of the critical path: each row's
// record is a few 16-byte chunks, prefetched kPrefetch steps ahead, every
// prefetch load is unconditional (the compiler then counts outstanding loads
// exactly instead of draining them), and the fast path has no divergent branch.
#include <hip/hip_runtime.h>
#include <type_traits>

#include "sweep.hpp"

namespace mrfg {

namespace {

constexpr int kPrefetch = 8;
constexpr int kWaveRounds = 3;   // prefetch-ring rounds per unrolled group of steps
constexpr int kWaveGroup = kWaveRounds * kPrefetch;
static_assert(kWaveGroup % kRing == 0, "a group of steps spans whole rounds of the LDS ring");
// LDS values of a wave's ring: kRing steps, then zeros up to the largest
// code byte, so that every code byte indexes the ring
constexpr int kRingSlots = 256;
static_assert(kRing * 64 <= kCodeNone, "ring slots lie below the reserved code byte");

}  // namespace

// A chain: one wave whose steps are the region's levels.
// MODE: kDiluFwd / kDiluBwd (T = value type) or kDiluFactor (T = double).
template <typename T, int K, int MODE>
__global__ __launch_bounds__(64) void k_dilu_wave(DiluView<T> V, const SysState *st, const T *in, T *out)
{
    using R = typename RecordOf<T, MODE>::V;
    constexpr int N = RecordOf<T, MODE>::N;
    constexpr int G = packChunks(K + 1, N);      // value chunks per row
    constexpr int NC = packChunks(K, 4);         // ints holding the byte codes
    __shared__ T ring[kRingSlots];
    const int lane = threadIdx.x;
    const int w = MODE == kDiluBwd ? V.order[V.nWaves - 1 - blockIdx.x] : V.order[blockIdx.x];
    const int sys = V.waveSys[w];
    const bool active = MODE == kDiluFactor || st[sys].status == kRunning;
    const int s0 = V.waveSlice[w], nSteps = V.waveSteps[w];
    const int32_t *codes = MODE == kDiluBwd ? V.bCodes : V.fCodes;
    const R *recs = MODE == kDiluFactor ? (const R *)V.prodPack : (const R *)(MODE == kDiluBwd ? V.bPack : V.fPack);
    const unsigned long long tStart = V.trace ? wall_clock64() : 0ull;

    struct Step {
        R v[G];
        int c[NC];
        T a;
    };
    auto sliceOf = [&](int i) {
        i = i < nSteps ? i : nSteps - 1;
        return s0 + (MODE == kDiluBwd ? nSteps - 1 - i : i);
    };
    // the row's record and input, kPrefetch steps ahead.  Every address is
    // computable without another load, and steps past the end re-read the
    // last step, so no load waits for another or is conditional.
    auto load = [&](int i, Step &S) {
        const int s = sliceOf(i);
#pragma unroll
        for (int g = 0; g < G; ++g) S.v[g] = recs[((size_t)s * G + g) * 64 + lane];
#pragma unroll
        for (int h = 0; h < NC; ++h) S.c[h] = codes[((size_t)s * NC + h) * 64 + lane];
        if (MODE != kDiluFactor) S.a = in[s * 64 + lane];
    };

    // FULL groups (below) address a step through per-wave resources: the
    // wave's rows of the records, codes, input and output, a scalar offset of
    // the step's slice in the wave and a per-lane constant
    constexpr bool kCanFull = MODE != kDiluFactor;
    const size_t recBytes = (size_t)nSteps * G * 64 * sizeof(R);
    const bool fullWave = kCanFull && recBytes <= (size_t)INT_MAX;
    const auto rRec = rawBuffer(recs + (size_t)s0 * G * 64, fullWave ? recBytes : 0);
    const auto rCode = rawBuffer(codes + (size_t)s0 * NC * 64, fullWave ? (size_t)nSteps * NC * 64 * sizeof(int) : 0);
    const auto rIn = rawBuffer(kCanFull ? in + (size_t)s0 * 64 : nullptr, fullWave ? (size_t)nSteps * 64 * sizeof(T) : 0);
    const auto rOut = rawBuffer(kCanFull ? out + (size_t)s0 * 64 : nullptr, fullWave ? (size_t)nSteps * 64 * sizeof(T) : 0);
    const unsigned vRec = lane * (unsigned)sizeof(R), vCode = lane * (unsigned)sizeof(int),
                   vRow = lane * (unsigned)sizeof(T);
    auto loadF = [&](int i, Step &S) {
        const unsigned j = (unsigned)(MODE == kDiluBwd ? nSteps - 1 - i : i);
#pragma unroll
        for (int g = 0; g < G; ++g) S.v[g] = bufLoad<R, 0>(rRec, vRec + g * 64 * sizeof(R), j * G * 64 * sizeof(R));
#pragma unroll
        for (int h = 0; h < NC; ++h) S.c[h] = bufLoad<int, 0>(rCode, vCode + h * 64 * sizeof(int), j * NC * 64 * sizeof(int));
        S.a = bufLoad<T, 0>(rIn, vRow, j * 64 * sizeof(T));
    };

    if (active && nSteps > 0) {
        // ring slots above the wave's kRing steps hold zeros: a code without
        // a ring slot (kCodeNone) reads a finite zero there
        for (int q = kRing * 64 + lane; q < kRingSlots; q += 64) ring[q] = T(0);
        __builtin_amdgcn_wave_barrier();
        Step buf[kPrefetch];
        // left to the scheduler, which reorders these loads so the loop's
        // first use waits for all of them; issuing them in consumption order
        // (as the box kernel does) made the waits exact here but the
        // tutorial's solve 1.3 % slower
#pragma unroll
        for (int u = 0; u < kPrefetch; ++u) load(u, buf[u]);
        // ring values of a step's dependencies, read as soon as the previous
        // step has written its slot (a dependency is at most kRing - 1 steps
        // back, and the slot the step overwrites is never among them), so the
        // LDS round trip overlaps the rest of the previous step.  The code
        // byte is the ring slot.
        auto ringSlot = [&](const Step &S, int k) { return (S.c[k / 4] >> (8 * (k % 4))) & 0xFF; };
        T rv[K];
#pragma unroll
        for (int k = 0; k < K; ++k) rv[k] = ring[ringSlot(buf[0], k)];
        // Whole groups of steps: a step past the end reads the clamped last
        // slice and stores nothing (its LDS ring slot is never read), so the
        // group has no early exits and the record waits stay exact within it.
        // A group spans kWaveRounds rounds of the prefetch ring and a whole
        // number of ring rounds, so every step's ring slot is a constant.
        //
        // A group is FULL when its steps and their prefetches all lie inside
        // the wave's steps: there nothing is clamped, the store is
        // unconditional, every address is a scalar offset plus a lane
        // constant, and each dependency term is taken without a select (a
        // missing dependency has a zero coefficient and reads a zero slot, so
        // for rD >= 0 its term is +0 and leaves the value unchanged bit for
        // bit).
        auto runGroup = [&](int i0, auto fullTag) {
            constexpr bool FULL = decltype(fullTag)::value;
#pragma unroll
            for (int uu = 0; uu < kWaveGroup; ++uu) {
                const int u = uu % kPrefetch;
                const int i = i0 + uu;
                const bool inRange = FULL || i < nSteps;
                Step &S = buf[u];
                const T last = (T)elem(S.v[K / N], K % N);   // rD, or diag for the factor
                // branch-free: a missing dependency contributes an exact zero
                T y;
                if (MODE == kDiluFwd) y = S.a * last;
                else if (MODE == kDiluBwd) y = S.a;
                else y = last;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const T c = (T)elem(S.v[k / N], k % N);
                    const bool has = ringSlot(S, k) != kCodeNone;
                    if (MODE == kDiluFactor) y = has ? y - c / rv[k] : y;
                    else if (FULL) y = y - last * c * rv[k];
                    else y = has ? y - last * c * rv[k] : y;
                }
                const int s = FULL ? 0 : sliceOf(i);
                // the ring is private to this wavefront and LDS operations of
                // a wavefront execute in order: no barrier (which would also
                // drain the prefetch loads) is needed between steps
                ring[(uu % kRing) * 64 + lane] = y;
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int k = 0; k < K; ++k) rv[k] = ring[ringSlot(buf[(u + 1) % kPrefetch], k)];
                if (FULL) {
                    bufStore<T, 0>(y, rOut, vRow, (unsigned)(MODE == kDiluBwd ? nSteps - 1 - i : i) * 64 * sizeof(T));
                    loadF(i + kPrefetch, S);
                    continue;
                }
                const int p = s * 64 + lane;
                if (inRange) {
                    if (MODE == kDiluFactor) {
                        const double rd = V.cellOfPos[p] >= 0 ? 1.0 / (double)y : 0.0;
                        V.rDout[p] = rd;
                        constexpr int NP = Pack<double>::N;
                        constexpr int GP = packChunks(K + 1, NP);
                        ((double *)&V.fPack[((size_t)s * GP + K / NP) * 64 + lane])[K % NP] = rd;
                        ((double *)&V.bPack[((size_t)s * GP + K / NP) * 64 + lane])[K % NP] = rd;
                    } else {
                        out[p] = y;
                    }
                }
                load(i + kPrefetch, S);
            }
        };
        for (int i0 = 0; i0 < nSteps; i0 += kWaveGroup) {
            if (kCanFull && fullWave && i0 + kWaveGroup - 1 + kPrefetch < nSteps) runGroup(i0, std::true_type{});
            else runGroup(i0, std::false_type{});
        }
    }
    if (V.trace && lane == 0) {
        unsigned long long *tr = V.trace + 4 * (size_t)blockIdx.x;
        tr[0] = tStart;
        tr[1] = wall_clock64();
        tr[2] = 0;
        tr[3] = (unsigned long long)nSteps;
    }
}

// A level group: one workgroup sweeps a whole region, level by level, up to 16
// slices of a level at a time (one per wave), with a barrier after each level.
// A row's dependencies come from an LDS ring of the region's last kLevelRing
// rows (which spans tens of levels of a mesh of 10^5 cells), or from memory if
// they lie further back.  Rows are loaded kDeep rounds ahead.
//
// The alternative, a wave per 64 rows of a level with every dependency passed
// through memory, costs a memory round trip per level and floods the fabric
// with the polls of waves whose turn is far off: 1257 us a sweep on 78k cells
// renumbered along a front (122 levels of up to 957 rows), against what is
// bound here by one CU's load path (60 bytes a row in FP64, about 64 bytes a
// clock) and the barrier.  Two regions of a system, or the systems of a batch,
// run side by side on CUs of their own.  Regions with wide levels are spread
// over the device instead (layout.cpp, spreadPays).
//
// One CU only has so many cache misses in flight: its rows came at 31 GB/s
// (105 us a sweep of that mesh; 81 us with the helpers below), whatever the
// depth.  So where few groups leave the chip idle, kHelpers more
// workgroups per group, on the same XCD (workgroup b runs on XCD b mod kXcds;
// elsewhere they only do not help), load the rows a little ahead of the sweep
// and drop them: the sweep then hits the XCD's L2.
constexpr int kXcds = 8, kHelpers = 8;
constexpr int kWarmBytes = 3 << 19;   // of the 4 MB of L2

template <int K>
constexpr int kDeepOf = K <= 3 ? 3 : K <= 6 ? 2 : 1;

template <typename T, int K, int MODE>
__global__ __launch_bounds__(1024) void k_dilu_levels(DiluView<T> V, const SysState *st, const T *in, T *out)
{
    using R = typename RecordOf<T, MODE>::V;
    constexpr int N = RecordOf<T, MODE>::N;
    constexpr int G = packChunks(K + 1, N);
    constexpr int kDeep = kDeepOf<K>;
    __shared__ T ring[kLevelRing];
    // helper h of group g is workgroup kXcds + g + kXcds * h (launchGeneralK)
    const bool helper = (int)blockIdx.x >= V.nGroups;
    const int gi = helper ? (int)blockIdx.x % kXcds : (int)blockIdx.x;
    if (helper && ((int)blockIdx.x < kXcds || gi >= V.nGroups)) return;
    const LevelGroup g = V.groups[gi];
    if (MODE != kDiluFactor && st[g.sys].status != kRunning) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned long long tStart = V.trace ? wall_clock64() : 0ull;
    // (constant address space: scalar loads, which no wait for rows includes)
    typedef const __attribute__((address_space(4))) LevelRound ConstRound;
    ConstRound *rounds = (ConstRound *)(V.lvRounds + __builtin_amdgcn_readfirstlane(g.round0));
    const int32_t *deps = MODE == kDiluBwd ? V.bDeps : V.fDeps;
    const R *recs = MODE == kDiluFactor ? (const R *)V.prodPack : (const R *)(MODE == kDiluBwd ? V.bPack : V.fPack);
    // what a later row reads back when it is out of the ring (the factor: d)
    const T *back = MODE == kDiluFactor ? nullptr : out + (size_t)g.slice0 * 64;

    struct Item {
        R v[G];
        int c[K];
        T a;
        int s;       // the wave's slice, -1: none in this round
        int flags;
    };
    auto roundOf = [&](int i) {
        i = min(i, g.nRounds - 1);
        i = __builtin_amdgcn_readfirstlane(MODE == kDiluBwd ? g.nRounds - 1 - i : i);
        return LevelRound{rounds[i].slice, rounds[i].word};
    };
    auto load = [&](int i, LevelRound r, Item &S) {
        const bool has = i < g.nRounds && wave < (r.word >> kRoundBits);
        const int s = r.slice + (has ? wave : 0);   // (a slice to load from in any case: no load is conditional)
#pragma unroll
        for (int q = 0; q < G; ++q) S.v[q] = recs[((size_t)s * G + q) * 64 + lane];
#pragma unroll
        for (int k = 0; k < K; ++k) S.c[k] = deps[((size_t)s * K + k) * 64 + lane];
        if (MODE != kDiluFactor) S.a = in[(size_t)s * 64 + lane];
        S.s = has ? s : -1;
        S.flags = r.word & ((1 << kRoundBits) - 1);
    };
    if (helper) {
        // touch every kHelpers-th round's rows, at most kWarmBytes ahead of
        // the sweep (the counter may still hold the last sweep's value, which
        // only lets the first rounds run further ahead)
        const int window = max(2 * kHelpers, kWarmBytes / (V.lvWaves * 64 * (int)(sizeof(R) * G + sizeof(int) * K + sizeof(T))));
        for (int i = (int)blockIdx.x / kXcds - 1; i < g.nRounds; i += kHelpers) {
            for (int spins = 0; spins < V.waitLimit && i > __hip_atomic_load(&V.lvProgress[gi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + window; ++spins)
                __builtin_amdgcn_s_sleep(8);
            Item S;
            load(i, roundOf(i), S);
#pragma unroll
            for (int q = 0; q < G; ++q) asm volatile("" ::"v"(elem(S.v[q], 0)));
#pragma unroll
            for (int k = 0; k < K; ++k) asm volatile("" ::"v"(S.c[k]));
            if (MODE != kDiluFactor) asm volatile("" ::"v"(S.a));
        }
        return;
    }
    // one slot more than rounds in flight: a round's rows are requested while
    // the ring values of the current one are on their way (the round table's
    // entry, a scalar load, one round earlier still)
    constexpr int kSlots = kDeep + 1;
    Item buf[kSlots];
#pragma unroll
    for (int u = 0; u < kDeep; ++u) load(u, roundOf(u), buf[u]);
    LevelRound next = roundOf(kDeep);
    for (int i0 = 0; i0 < g.nRounds; i0 += kSlots) {
        if (V.lvHelped && threadIdx.x == 0)
            __hip_atomic_store(&V.lvProgress[gi], i0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int u = 0; u < kSlots; ++u) {
            const int i = i0 + u;
            Item &S = buf[u];
            const bool mine = i < g.nRounds && S.s >= 0;
            T v[K];
            if (mine) {
#pragma unroll
                for (int k = 0; k < K; ++k) v[k] = ring[S.c[k] & (kLevelRing - 1)];
            }
            load(i + kDeep, next, buf[(u + kDeep) % kSlots]);
            next = roundOf(i + kDeep + 1);
            if (mine) {
                const T last = (T)elem(S.v[K / N], K % N);   // rD, or diag for the factor
                bool far = false;
#pragma unroll
                for (int k = 0; k < K; ++k) far |= S.c[k] >= kLevelRing;
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(far) != 0, 0)) {
                    // (in memory: a barrier that waits for stores lies
                    // between the row's level and this one, levelRounds.
                    // Such a load waits for the rows in flight as well, which
                    // are counted before it.)
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (S.c[k] >= kLevelRing) v[k] = MODE == kDiluFactor ? (T)V.lvD[(size_t)g.slice0 * 64 + S.c[k] - kLevelRing] : back[S.c[k] - kLevelRing];
                    // (waited for here: after the branch every round would
                    // wait for its rows in flight, also one without such a row)
#pragma unroll
                    for (int k = 0; k < K; ++k) asm volatile("" : "+v"(v[k]));
                }
                T y;
                if (MODE == kDiluFwd) y = S.a * last;
                else if (MODE == kDiluBwd) y = S.a;
                else y = last;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const T c = (T)elem(S.v[k / N], k % N);
                    const bool has = S.c[k] != kNoDep;
                    if (MODE == kDiluFactor) y = has ? y - c / v[k] : y;
                    else y = has ? y - last * c * v[k] : y;
                }
                const size_t p = (size_t)S.s * 64 + lane;
                ring[(p - (size_t)g.slice0 * 64) & (kLevelRing - 1)] = y;
                if (MODE == kDiluFactor) {
                    const double rd = V.cellOfPos[p] >= 0 ? 1.0 / (double)y : 0.0;
                    V.rDout[p] = rd;
                    V.lvD[p] = (double)y;
                    constexpr int NP = Pack<double>::N;
                    constexpr int GP = packChunks(K + 1, NP);
                    ((double *)&V.fPack[((size_t)S.s * GP + K / NP) * 64 + lane])[K % NP] = rd;
                    ((double *)&V.bPack[((size_t)S.s * GP + K / NP) * 64 + lane])[K % NP] = rd;
                } else {
                    out[p] = y;
                }
            }
            if (i < g.nRounds && (S.flags & (MODE == kDiluBwd ? kRoundFirst : kRoundLast))) {
                // the level's values are in the ring before any wave goes on.
                // (Where no row is about to leave the ring only LDS is waited
                // for: waiting for the stores drains the rows in flight.)
                if (S.flags & (MODE == kDiluBwd ? kRoundStoredB : kRoundStoredF)) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
        }
    }
    if (V.trace && threadIdx.x == 0) {
        unsigned long long *tr = V.trace + 4 * ((size_t)V.nWaves + V.nBoxWaves + gi);
        tr[0] = tStart;
        tr[1] = wall_clock64();
        tr[2] = 0;
        tr[3] = (unsigned long long)g.nRounds;
    }
}

// Spread levels: one launch per level, a wave per slice over the whole device,
// every dependency read from memory.  Bound by the launches (3.6 us each in a
// graph) up to some 10^4 rows a level, above by the reads of rows spread over
// memory: 170 us a sweep for 2.0M shuffled cells in 24 levels, where one
// workgroup takes 8300 us and a wave per slice that polls for its dependencies
// took 4500.  No workgroup waits for another.
template <typename T, int K, int MODE>
__global__ __launch_bounds__(256) void k_dilu_spread(DiluView<T> V, const SysState *st, const T *in, T *out, int first,
                                                     int n)
{
    using R = typename RecordOf<T, MODE>::V;
    constexpr int N = RecordOf<T, MODE>::N;
    constexpr int G = packChunks(K + 1, N);
    const int i = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const SpreadSlice q = V.spread[first + i];
    if (MODE != kDiluFactor && st[q.sys].status != kRunning) return;
    const unsigned long long tStart = V.trace ? wall_clock64() : 0ull;
    const int32_t *deps = MODE == kDiluBwd ? V.bDeps : V.fDeps;
    const R *recs = MODE == kDiluFactor ? (const R *)V.prodPack : (const R *)(MODE == kDiluBwd ? V.bPack : V.fPack);
    const size_t s = (size_t)q.slice, p = s * 64 + lane;
    int c[K];
    R v[G];
    T a = T(0), x[K];
#pragma unroll
    for (int k = 0; k < K; ++k) c[k] = deps[(s * K + k) * 64 + lane];
#pragma unroll
    for (int g = 0; g < G; ++g) v[g] = recs[(s * G + g) * 64 + lane];
    if (MODE != kDiluFactor) a = in[p];
    // (stored by an earlier launch)
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const size_t from = c[k] == kNoDep ? p : (size_t)c[k];
        x[k] = MODE == kDiluFactor ? (T)V.lvD[from] : out[from];
    }
    const T last = (T)elem(v[K / N], K % N);   // rD, or diag for the factor
    T y = MODE == kDiluFwd ? a * last : MODE == kDiluBwd ? a : last;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const T f = (T)elem(v[k / N], k % N);
        const T t = MODE == kDiluFactor ? y - f / x[k] : y - last * f * x[k];
        y = c[k] != kNoDep ? t : y;
    }
    if (MODE == kDiluFactor) {
        const double rd = V.cellOfPos[p] >= 0 ? 1.0 / (double)y : 0.0;
        V.rDout[p] = rd;
        V.lvD[p] = (double)y;
        constexpr int NP = Pack<double>::N;
        constexpr int GP = packChunks(K + 1, NP);
        ((double *)&V.fPack[(s * GP + K / NP) * 64 + lane])[K % NP] = rd;
        ((double *)&V.bPack[(s * GP + K / NP) * 64 + lane])[K % NP] = rd;
    } else {
        out[p] = y;
    }
    if (V.trace && q.levels && lane == 0) {
        unsigned long long *tr = V.trace + 4 * ((size_t)V.nWaves + V.nBoxWaves + V.nGroups + q.region);
        if (tr[0] == 0) tr[0] = tStart;
        tr[1] = wall_clock64();
        tr[2] = 0;
        tr[3] = (unsigned long long)q.levels;
    }
}

// ---------------------------------------------------------------------------
// Factorisation of structured-box tiles (the sweeps are in dilu_box.hip).
//
// Lane l = bl + TB*cl of a tile wave owns grid line (bl, cl) of the tile's
// TB x TC lines along the sequential axis; at step t it computes cell
// ia = t - bl - cl of its line.  Each of the cell's three dependencies was
// computed one step earlier: along the line by the lane itself (kept in a
// register), across the line by lane l - 1 and lane l - TB (exchanged through
// 64 LDS values), and across the tile's edge by the neighbouring tile's wave,
// which delivers it to this wave's inbox: (TB + TC) values per step, [cl]
// for the b edge and [TC + bl] for the c edge.  Once per solve and bound by
// three divisions in a row per step, so it keeps one wave per tile.
// ---------------------------------------------------------------------------

constexpr int kFacAhead = 4;     // steps between a record load and its use
constexpr int kFacInAhead = 3;   // steps between an inbox load and its use
constexpr int kFacGroup = 4;     // steps per unrolled group

// KT: the batch's record width K when it is 3 (diag in the last chunk), or 0
// for a wider batch (K read from the view, diag in a chunk of its own).
// LONE: every tile is treated as alone in its region (the tile-local
// factor): no inbox, no deliveries.
// seg, segs: a lone factor of segment seg of segs of the tile's rows (rows
// of the other segments are not this wave's: it neither uses nor writes them)
template <int KT, int AX, bool LONE>
__device__ __forceinline__ void boxFactor(const DiluView<double> &V, const int32_t *m, unsigned long long *inbox,
                                          double *xch, int seg, int segs)
{
    using T = double;
    using U = unsigned long long;
    constexpr U kSent = kHaloSentinel64;
    constexpr bool kExtra = KT == 0;
    constexpr int NL = kExtra ? 3 : 2;
    constexpr int kAxB = AX == 0 ? 1 : 0;
    constexpr int kSlotA = 2 - AX, kSlotB = 2 - kAxB;   // the c neighbour holds the third slot
    const int K = KT ? KT : V.K;
    const int G = packChunks(K + 1, 2);          // chunks per row of the record array
    const int gLast = K / 2, eLast = K % 2;      // chunk / element of diag

    const unsigned lane = threadIdx.x;
    const int TB = m[kBmTB], lg = __builtin_ctz(TB), TC = 64 >> lg, TBC = TB + TC;
    const int nA = m[kBmNA], actB = m[kBmActB], actC = m[kBmActC];
    const int s0 = m[kBmSlice], nSteps = m[kBmSteps];
    const int prevB = LONE ? -1 : m[kBmPrevB], prevC = LONE ? -1 : m[kBmPrevC];
    const int nextB = LONE ? -1 : m[kBmNextB], nextC = LONE ? -1 : m[kBmNextC];
    const int bl = lane & (TB - 1), cl = lane >> lg;
    const bool inTile = bl < actB && cl < actC;
    // this wave's rows [iaLo, iaHi) along the sequential axis and its steps
    int iaLo = 0, iaHi = nA;
    if (LONE && segs > 1) boxSegment(nA, seg, segs, iaLo, iaHi);
    const int tFirst = iaLo, nLocal = iaHi - iaLo + (actB - 1) + (actC - 1);
    if (iaHi <= iaLo) return;   // a segment without rows (nA < segs)
    const bool hasB = bl > 0 || prevB >= 0, hasC = cl > 0 || prevC >= 0;
    const bool useB = bl == 0 && prevB >= 0, useC = cl == 0 && prevC >= 0;
    const unsigned srcB = (lane - 1) & 63, srcC = (lane - TB) & 63;
    // where this lane's values go: the consumer's step is t - (TB - 1)
    // (resp. TC - 1), into the consumer's inbox at [cl] (resp. [TC + bl])
    const bool sendB = bl == TB - 1 && nextB >= 0, sendC = cl == TC - 1 && nextC >= 0;
    const double2 *recs = V.prodPack + (size_t)s0 * G * 64;
    const int rowBytes = G * 64 * (int)sizeof(double2), inRowBytes = TBC * (int)sizeof(U);
    const auto rRec = rawBuffer(recs, (size_t)nSteps * rowBytes);
    const U *myIn = inbox + m[kBmInbox];
    const auto rInbox = rawBuffer(myIn, LONE ? 0 : (size_t)nSteps * inRowBytes);
    auto consumer = [&](int to) {
        if (LONE || to < 0) return rawBuffer(inbox, 0);
        const int32_t *mt = V.boxMeta + (size_t)to * kBoxMeta;
        return rawBuffer(inbox + mt[kBmInbox], (size_t)mt[kBmSteps] * inRowBytes);
    };
    const auto rToB = consumer(nextB), rToC = consumer(nextC);
    const unsigned vRec = lane * (unsigned)sizeof(double2);
    const unsigned vInB = (unsigned)cl * sizeof(U), vInC = (unsigned)(TC + bl) * sizeof(U);
    const unsigned vToB = sendB ? vInB : kNoLane, vToC = sendC ? vInC : kNoLane;

    struct Step {
        double2 v[NL];
        U hb, hc;
    };
    // step i of the wave (clamped: loads past the end re-read the last step)
    auto stepOf = [&](int i) { return tFirst + (i < nLocal ? i : nLocal - 1); };
    auto load = [&](int i, Step &S) {
        const unsigned so = (unsigned)(stepOf(i) * rowBytes);
#pragma unroll
        for (int g = 0; g < 2; ++g) S.v[g] = bufLoad<double2, 0>(rRec, vRec + g * 64 * sizeof(double2), so);
        if (kExtra) S.v[NL - 1] = bufLoad<double2, 0>(rRec, vRec + gLast * 64 * sizeof(double2), so);
    };
    auto loadIn = [&](int i, Step &S) {
        const unsigned so = (unsigned)(stepOf(i) * inRowBytes);
        S.hb = bufLoad<U, kSysCoherent>(rInbox, vInB, so);
        S.hc = bufLoad<U, kSysCoherent>(rInbox, vInC, so);
    };
    xch[lane] = 0.0;
    __builtin_amdgcn_wave_barrier();
    T xbN = xch[srcB], xcN = xch[srcC];
    Step buf[kFacAhead];
#pragma unroll
    for (int u = 0; u < kFacAhead; ++u) buf[u].hb = buf[u].hc = kSent;
#pragma unroll
    for (int u = 0; u < kFacAhead; ++u) {
        if (!LONE && u < kFacInAhead) loadIn(u, buf[u]);
        load(u, buf[u]);
        __builtin_amdgcn_sched_barrier(0);
    }
    T yprev = 0.0;
    for (int i0 = 0; i0 < nLocal; i0 += kFacGroup) {
#pragma unroll
        for (int u = 0; u < kFacGroup; ++u) {
            const int i = i0 + u, t = tFirst + i, ia = t - bl - cl;
            Step &S = buf[u % kFacAhead];
            const bool valid = inTile && (unsigned)(ia - iaLo) < (unsigned)(iaHi - iaLo);
            const bool hasA = ia > iaLo;
            T y, yz;
            for (int pass = 0;; ++pass) {
                y = kExtra ? elem(S.v[NL - 1], eLast) : S.v[1].y;
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const T v = q == kSlotA ? yprev : q == kSlotB ? (useB ? Bits<T>::from(S.hb) : xbN)
                                                                  : (useC ? Bits<T>::from(S.hc) : xcN);
                    const bool has = q == kSlotA ? hasA : q == kSlotB ? hasB : hasC;
                    y = has ? y - elem(S.v[q / 2], q % 2) / v : y;
                }
                yz = valid ? y : 0.0;
                // a sentinel (a NaN) makes the value NaN; a second pass
                // follows the wait for the late values
                if (LONE || pass || __builtin_expect(__builtin_amdgcn_ballot_w64(yz != yz) == 0, 1)) break;
                // poll rounds: each reloads this step's values and those
                // already requested for the next steps, all in flight
                // together; the later ones come with the last round instead
                // of a round trip each (a factor of the 1.4M cell duct takes
                // 145 us, 240 without)
                for (int spins = 0;; ++spins) {
                    U nb[kFacInAhead], nc[kFacInAhead];
#pragma unroll
                    for (int k = 0; k < kFacInAhead; ++k) {
                        nb[k] = haloLoad(myIn + (size_t)stepOf(i + k) * TBC, cl);
                        nc[k] = haloLoad(myIn + (size_t)stepOf(i + k) * TBC, TC + bl);
                    }
#pragma unroll
                    for (int k = 0; k < kFacInAhead; ++k) {
                        Step &F = buf[(u + k) % kFacAhead];
                        F.hb = F.hb == kSent ? nb[k] : F.hb;
                        F.hc = F.hc == kSent ? nc[k] : F.hc;
                    }
                    const bool late = valid && ((useB && S.hb == kSent) || (useC && S.hc == kSent));
                    if (__builtin_amdgcn_ballot_w64(late) == 0) break;
                    // an expired wait ends every later one at once, so a
                    // broken schedule ends the kernel instead of hanging it
                    if (spins >= V.waitLimit || __hip_atomic_load(V.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                        if (lane == 0) atomicOr(V.err, 2);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            // all lanes have read the previous step's values (LDS operations
            // of a wavefront execute in order) before any overwrites them
            xch[lane] = yz;
            __builtin_amdgcn_wave_barrier();
            xbN = xch[srcB];
            xcN = xch[srcC];
            yprev = yz;
            if (i < nLocal) {
                const double rd = valid ? 1.0 / y : 0.0;
                // a segment wave writes its own rows and padding
                const bool mine = !inTile || (unsigned)ia >= (unsigned)nA || valid;
                if (mine) (V.rDout + (size_t)(s0 + t) * 64)[lane] = rd;
                if (V.fPack) {   // (a tile-local factor writes rD only)
                    const size_t e = ((size_t)(s0 + t) * G + gLast) * 64 + lane;
                    ((double *)&V.fPack[e])[eLast] = rd;
                    ((double *)&V.bPack[e])[eLast] = rd;
                }
            }
            if (!LONE) {
                const U yb = Bits<T>::to(y);
                const int tb = t + 1 - TB, tc = t + 1 - TC;
                bufStore<U, kSysCoherent>(yb, rToB, valid ? vToB : kNoLane, (unsigned)((tb > 0 ? tb : 0) * inRowBytes));
                bufStore<U, kSysCoherent>(yb, rToC, valid ? vToC : kNoLane, (unsigned)((tc > 0 ? tc : 0) * inRowBytes));
                loadIn(i + kFacInAhead, buf[(u + kFacInAhead) % kFacAhead]);
            }
            load(i + kFacAhead, S);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

template <int KT, bool LONE>
__global__ __launch_bounds__(64) void k_dilu_box_factor(DiluView<double> V, unsigned long long *inbox)
{
    __shared__ double xch[64];
    const int segs = LONE ? V.boxSegs : 1;
    const int j = (int)blockIdx.x / segs, seg = (int)blockIdx.x - j * segs;
    const int32_t *m = V.boxMeta + (size_t)V.boxOrder[j] * kBoxMeta;
    if (m[kBmSteps] <= 0) return;
    switch (m[kBmAxis]) {
    case 0: boxFactor<KT, 0, LONE>(V, m, inbox, xch, seg, segs); break;
    case 1: boxFactor<KT, 1, LONE>(V, m, inbox, xch, seg, segs); break;
    default: boxFactor<KT, 2, LONE>(V, m, inbox, xch, seg, segs); break;
    }
}

// rD of the FP32 records from the FP64 factor (one thread per row)
template <int K>
__global__ void k_convert_rd(DiluView<float> V, const double *rD64, int nPos)
{
    constexpr int N = Pack<float>::N;
    constexpr int G = packChunks(K + 1, N);
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nPos) return;
    const int s = p / 64, lane = p % 64;
    const float r = (float)rD64[p];
    ((float *)&V.fPack[((size_t)s * G + K / N) * 64 + lane])[K % N] = r;
    ((float *)&V.bPack[((size_t)s * G + K / N) * 64 + lane])[K % N] = r;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

template <typename T, int K, int MODE>
static void launchGeneralK(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s)
{
    if (V.nWaves > 0) k_dilu_wave<T, K, MODE><<<V.nWaves, 64, 0, s>>>(V, st, in, out);
    if (V.nGroups > 0) {
        DiluView<T> L = V;
        L.lvHelped = V.nGroups <= kXcds;
        const int blocks = L.lvHelped ? kXcds * (1 + kHelpers) : V.nGroups;
        k_dilu_levels<T, K, MODE><<<blocks, 64 * V.lvWaves, 0, s>>>(L, st, in, out);
    }
    for (int i = 0; i < V.nSpreadLevels; ++i) {
        const int lv = MODE == kDiluBwd ? V.nSpreadLevels - 1 - i : i;
        const int first = V.spreadLevels[lv], n = V.spreadLevels[lv + 1] - first;
        k_dilu_spread<T, K, MODE><<<(n + 3) / 4, 256, 0, s>>>(V, st, in, out, first, n);
    }
}

template <typename T, int MODE>
static hipError_t launchGeneral(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s)
{
    if (!V.general()) return hipSuccess;
    if (V.lvWaves < 1 || V.lvWaves > 16) return hipErrorInvalidValue;
    switch (V.K) {
    case 3: launchGeneralK<T, 3, MODE>(V, st, in, out, s); break;
    case 6: launchGeneralK<T, 6, MODE>(V, st, in, out, s); break;
    case 12: launchGeneralK<T, 12, MODE>(V, st, in, out, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

static hipError_t launchBoxFactor(const DiluView<double> &V, hipStream_t s)
{
    if (V.nBoxWaves <= 0) return hipSuccess;
    auto *inbox = (unsigned long long *)V.boxInC;
    if (V.boxLone) {
        const int nb = V.nBoxWaves * (V.boxSegs > 1 ? V.boxSegs : 1);
        if (V.K == 3) k_dilu_box_factor<3, true><<<nb, 64, 0, s>>>(V, inbox);
        else k_dilu_box_factor<0, true><<<nb, 64, 0, s>>>(V, inbox);
        return hipGetLastError();
    }
    if (V.boxSegs > 1) return hipErrorInvalidValue;   // segments only where tiles are lone
    if (V.K == 3) k_dilu_box_factor<3, false><<<V.nBoxWaves, 64, 0, s>>>(V, inbox);
    else k_dilu_box_factor<0, false><<<V.nBoxWaves, 64, 0, s>>>(V, inbox);
    return hipGetLastError();
}

// The general sweep on s and the box sweep on V.side when both exist and a
// side stream is set (the box sweep forked after the work already on s and
// joined before the next), else both on s.
template <typename T, typename GenF, typename BoxF>
static hipError_t bothSweeps(const DiluView<T> &V, hipStream_t s, GenF &&gen, BoxF &&box)
{
    const bool fork = V.side && V.fork && V.join && V.general() && V.nBoxWaves > 0;
    if (!fork) {
        hipError_t e = gen(s);
        return e != hipSuccess ? e : box(s);
    }
    hipError_t e = hipEventRecord(V.fork, s);
    if (e == hipSuccess) e = hipStreamWaitEvent(V.side, V.fork, 0);
    if (e == hipSuccess) e = box(V.side);
    if (e == hipSuccess) e = hipEventRecord(V.join, V.side);
    if (e == hipSuccess) e = gen(s);
    if (e == hipSuccess) e = hipStreamWaitEvent(s, V.join, 0);
    return e;
}

template <typename T>
hipError_t diluForward(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s)
{
    return bothSweeps(
        V, s, [&](hipStream_t q) { return launchGeneral<T, kDiluFwd>(V, st, in, out, q); },
        [&](hipStream_t q) { return boxForward<T>(V, st, in, out, q); });
}

template <typename T>
hipError_t diluBackward(const DiluView<T> &V, const SysState *st, T *inout, hipStream_t s)
{
    return bothSweeps(
        V, s, [&](hipStream_t q) { return launchGeneral<T, kDiluBwd>(V, st, inout, inout, q); },
        [&](hipStream_t q) { return boxBackward<T>(V, st, inout, q); });
}

__global__ void k_fill_u64(unsigned long long *a, int n, unsigned long long v)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = v;
}

__global__ void k_fill_u32(unsigned int *a, int n, unsigned int v)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = v;
}

hipError_t diluFactor(const DiluView<double> &V, hipStream_t s)
{
    // box tiles publish d through an inbox buffer of their own, reset first
    if (V.nBoxIn > 0) k_fill_u64<<<256, 256, 0, s>>>((unsigned long long *)V.boxInC, V.nBoxIn, kHaloSentinel64);
    hipError_t e = launchGeneral<double, kDiluFactor>(V, nullptr, nullptr, nullptr, s);
    return e != hipSuccess ? e : launchBoxFactor(V, s);
}

hipError_t diluFactorTileLocal(const DiluView<double> &V, double *rD, int segs, hipStream_t s)
{
    if (V.nBoxWaves <= 0) return hipSuccess;
    if (segs < 1) return hipErrorInvalidValue;
    DiluView<double> L = V;
    L.rDout = rD;
    L.fPack = nullptr;
    L.bPack = nullptr;
    L.boxLone = true;
    L.boxSegs = segs;
    L.trace = nullptr;
    return launchBoxFactor(L, s);
}

hipError_t diluConvertRD(const DiluView<float> &V32, const double *rD64, int nSlices, hipStream_t s)
{
    const int nPos = nSlices * 64, blocks = (nPos + 255) / 256;
    switch (V32.K) {
    case 3: k_convert_rd<3><<<blocks, 256, 0, s>>>(V32, rD64, nPos); break;
    case 6: k_convert_rd<6><<<blocks, 256, 0, s>>>(V32, rD64, nPos); break;
    case 12: k_convert_rd<12><<<blocks, 256, 0, s>>>(V32, rD64, nPos); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t fillHalo64(void *h, int n, hipStream_t s)
{
    k_fill_u64<<<256, 256, 0, s>>>((unsigned long long *)h, n, kHaloSentinel64);
    return hipGetLastError();
}

hipError_t fillHalo32(void *h, int n, hipStream_t s)
{
    k_fill_u32<<<256, 256, 0, s>>>((unsigned int *)h, n, kHaloSentinel32);
    return hipGetLastError();
}

template hipError_t diluForward<double>(const DiluView<double> &, const SysState *, const double *, double *,
                                        hipStream_t);
template hipError_t diluForward<float>(const DiluView<float> &, const SysState *, const float *, float *,
                                       hipStream_t);
template hipError_t diluBackward<double>(const DiluView<double> &, const SysState *, double *, hipStream_t);
template hipError_t diluBackward<float>(const DiluView<float> &, const SysState *, float *, hipStream_t);

}  // namespace mrfg
