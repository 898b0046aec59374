// Forward and backward DILU sweeps of structured-box tiles on gfx950.
//
//   forward   w[u] = rD[u]*r[u] - sum_{lower faces, face order} rD[u]*lower_f*w[l(f)]
//   backward  w[l] -= sum_{upper faces, reverse face order} rD[l]*upper_f*w[u(f)]
//
// A tile holds TB x TC = 64 grid lines along the region's longest axis; lane
// l = bl + TB*cl of its compute wave owns line (bl, cl).  At step T it
// computes cell ia = T - bl - cl of the line (T runs up in the forward and
// down in the backward sweep), so a cell's three neighbours are
//   along the line  the lane's own value of the previous step (a register),
//   along b, c      the previous step's values of lanes l -/+ 1, l -/+ TB,
//                   through a (TB + 1) x (TC + 1) LDS plane of the step,
// and on the tile's edge the neighbouring tile's value, which that tile's
// compute wave stores to this tile's inbox (agent-scope relaxed atomics, a
// sentinel marks values that have not arrived) and which is put into the
// spare row and column of the plane.
//
// A sweep is bound by the chain of steps along the region's diagonal
// (nA + nB + nC of them) and the hops between tiles, not by bandwidth: the
// box of 160x80x80 cells keeps fewer than 60 of its 100 tiles busy at a
// time.  So the work of a tile is split by what waits for what, one
// wavefront each (on SIMDs of their own):
//   stream   loads records and input kAhead steps ahead, forms every product
//            that needs no neighbour (and BiCGStab's p / s update where it is
//            fused) and writes the row to an LDS ring;
//   feed     polls the inbox, several batches of loads in flight, and puts
//            what has arrived into the planes;
//   compute  runs the recurrence on the ring and the planes: it never waits
//            on a global load, and its stores drain on their own.
// One wave that did all of it waited in every step for loads and stores issued
// a few steps before (vmcnt counts both, in order).  Measured on that box with
// its 200x100x19 neighbour (1.4M cells, FP64, inside the solve): 93 us a sweep
// and 165 ns a step before, 65 us and 81 ns now; a hop takes 2.2 us, of which
// 0.65 us are the 8 steps to the producer's edge, 0.25 us the hand-over in
// groups of kSub and the rest memory (store, poll, store to LDS).
#include <type_traits>

#include "sweep.hpp"

namespace mrfg {

namespace {

constexpr int kG = 8;          // steps per unrolled group of the compute wave
constexpr int kSub = 4;        // steps between its looks at the other waves' progress
constexpr int kRec = 16;       // record ring (steps)
constexpr int kIn = 16;        // ring of planes (steps)
constexpr int kChunk = 4;      // steps the stream wave hands over at a time
constexpr int kAhead = 8;      // steps of global loads the stream wave has in flight
constexpr int kLook = 2;       // steps the compute wave reads rows ahead
constexpr int kAll = 1 << 30;  // progress of a wave that has nothing (more) to do
constexpr int kPlane = 136;    // values per plane: (TB + 1) * (TC + 1) <= 130
// (the rings leave the other waves several steps of slack beyond what the
// compute wave needs next: with none, each hand-over waits for the other)
static_assert(kRec >= kSub + kLook + 2 * kChunk && kIn >= kSub + kG, "look-ahead and slack fit the rings");
static_assert(kAhead % kChunk == 0 && kRec % kAhead == 0 && kRec % kG == 0 && kIn % kG == 0 && kG % kSub == 0,
              "rings hold whole groups");

// Row values handed from the stream to the compute wave, in 16-byte chunks:
// the three products rD*c in slot order and the row's first term (rD*r
// forward, w backward).
template <typename T>
struct RowV {
    static constexpr int kChunks = 4 / Pack<T>::N;
    typename Pack<T>::V v[kChunks];
    __device__ T operator[](int i) const { return elem(v[i / Pack<T>::N], i % Pack<T>::N); }
};
template <typename T>
using RowSlot = typename Pack<T>::V[RowV<T>::kChunks][64];
template <typename T>
__device__ inline RowV<T> getRow(const RowSlot<T> &s, int lane)
{
    RowV<T> r;
#pragma unroll
    for (int k = 0; k < RowV<T>::kChunks; ++k) r.v[k] = s[k][lane];
    return r;
}
__device__ inline void putRow(RowSlot<double> &s, int lane, const double (&c)[3], double y0)
{
    s[0][lane] = double2{c[0], c[1]};
    s[1][lane] = double2{c[2], y0};
}
__device__ inline void putRow(RowSlot<float> &s, int lane, const float (&c)[3], float y0)
{
    s[0][lane] = float4{c[0], c[1], c[2], y0};
}

template <typename T>
struct Shared {
    RowSlot<T> rec[kRec];
    // plane of step i: the values of step i, and in its spare row and column
    // the edge values that step i + 1 needs
    T plane[kIn][kPlane];
    T spare[64];       // the feed wave's writes that are not due
    // steps whose rows (less the look-ahead) and whose edge values are there
    struct alignas(8) Ready {
        int rows, edges;
    } ready;
    int consumed;      // steps the compute wave has finished
};

// (LDS operations of a wavefront execute in order, so a counter written
// after the data it covers is seen after it; these only keep the compiler
// from moving the accesses)
__device__ inline void compilerFence() { asm volatile("" ::: "memory"); }
// (relaxed atomics: a volatile access would stay in the generic address
// space and wait for every global access in flight)
__device__ inline int look(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ inline int peek(const int *p)
{
    compilerFence();
    const int v = __builtin_amdgcn_readfirstlane(look(p));
    compilerFence();
    return v;
}
__device__ inline void post(int *p, int v)
{
    compilerFence();
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    compilerFence();
}

// The tile, from its descriptor (wave-uniform)
struct Tile {
    int TB, lg, TC, nA, axis, actB, actC, s0, nSteps, inbox;
    __device__ explicit Tile(const int32_t *m)
        : TB(m[kBtTB]), lg(__builtin_ctz(m[kBtTB])), TC(64 >> lg), nA(m[kBtNA]), axis(m[kBtAxis]), actB(m[kBtActB]),
          actC(m[kBtActC]), s0(m[kBtSlice]), nSteps(m[kBtSteps]), inbox(m[kBtInbox])
    {
    }
    // plane cells of lane (b, c) and of the edge values it may need
    template <bool FWD>
    __device__ int cell(int b, int c) const { return FWD ? (c + 1) * (TB + 1) + b + 1 : c * (TB + 1) + b; }
};

// the value of lane l - 1 (forward) / l + 1 (backward), zero past the wave's end
template <typename T, bool FWD>
__device__ inline T laneBefore(T v)
{
    auto move = [](unsigned u) {   // wave_shr:1 / wave_shl:1
        return (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, FWD ? 0x138 : 0x130, 0xf, 0xf, true);
    };
    if constexpr (sizeof(T) == 8) {
        const unsigned long long u = Bits<T>::to(v);
        return Bits<T>::from(((unsigned long long)move((unsigned)(u >> 32)) << 32) | move((unsigned)u));
    } else {
        return Bits<T>::from(move(Bits<T>::to(v)));
    }
}

// The rows [lo, hi) of the sequential axis that a workgroup sweeps
struct Span {
    int lo, hi;
};

// ---------------------------------------------------------------------------
// compute wave
// ---------------------------------------------------------------------------

// FLAT: the tile has no neighbour along c at all (one line of cells across,
// as in 2-D): the c term is left out, and a LONE tile needs no plane, since
// the one exchange left is a DPP move.
template <typename T, int MODE, int AX, bool LONE, bool FLAT>
__device__ __forceinline__ void boxCompute(const DiluView<T> &V, const int32_t *m, const Tile &t, Span sp, T *out,
                                           typename Bits<T>::U *inbox, Shared<T> &sh, unsigned &nSlow)
{
    using U = typename Bits<T>::U;
    constexpr bool kFwd = MODE != kDiluBwd;
    // record slot (2 - axis of the neighbour) of the line, b and c neighbour:
    // the slot order is the reference's face order
    constexpr int kAxB = AX == 0 ? 1 : 0;
    constexpr int kSlotA = 2 - AX, kSlotB = 2 - kAxB, kSlotC = 3 - kSlotA - kSlotB;

    const unsigned lane = threadIdx.x & 63;
    const int TB = t.TB, TC = t.TC, bl = lane & (TB - 1), cl = lane >> t.lg;
    const bool inTile = bl < t.actB && cl < t.actC;
    const int tLo = (t.actB - 1) + (t.actC - 1);   // rows valid from step lo + tLo on for every lane
    const int nL = sp.hi - sp.lo + tLo;
    // the consumers: the next tiles' inboxes (rows of E values for the b
    // edge, then as many for the c edge).  A value's row in the consumer's
    // inbox is the consumer's step that needs it
    const int E = max(TB, TC);
    const int toB = LONE ? -1 : m[kFwd ? kBtInNextB : kBtInPrevB], toC = LONE ? -1 : m[kFwd ? kBtInNextC : kBtInPrevC];
    const int lB = m[kFwd ? kBtLNextB : kBtLPrevB], lC = m[kFwd ? kBtLNextC : kBtLPrevC];   // their steps
    const bool sendB = toB >= 0 && inTile && (kFwd ? bl == TB - 1 : bl == 0);
    const bool sendC = toC >= 0 && inTile && (kFwd ? cl == TC - 1 : cl == 0);
    const int dB = kFwd ? 1 - TB : TB - 1, dC = kFwd ? 1 - TC : TC - 1;
    const int mOff = min(min(toB >= 0 ? dB : 0, toC >= 0 ? dC : 0), 0);
    const auto rToB = rawBuffer(inbox + (toB >= 0 ? toB : 0), toB >= 0 ? (size_t)lB * E * sizeof(U) : 0);
    const auto rToC = rawBuffer(inbox + (toC >= 0 ? toC + lC * E : 0), toC >= 0 ? (size_t)lC * E * sizeof(U) : 0);
    const unsigned vToB = sendB ? (unsigned)cl * sizeof(U) : kNoLane;
    const unsigned vToC = sendC ? (unsigned)bl * sizeof(U) : kNoLane;
    const auto rOut = rawBuffer(out + (size_t)t.s0 * 64, (size_t)t.nSteps * 64 * sizeof(T));
    const unsigned vOut = inTile ? lane * (unsigned)sizeof(T) : kNoLane;

    const int own = t.cell<kFwd>(bl, cl), nbB = own + (kFwd ? -1 : 1), nbC = own + (kFwd ? -(TB + 1) : TB + 1);

    // The progress of the other waves is read kSub steps before it is needed,
    // so that a step only waits for it when one of them is behind.
    unsigned long long seen = 0;
    const unsigned long long *ready = reinterpret_cast<const unsigned long long *>(&sh.ready);
    auto lookReady = [&]() {
        compilerFence();
        seen = __hip_atomic_load(ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        compilerFence();
    };
    auto isReady = [&](int need) {
        int r = __builtin_amdgcn_readfirstlane((int)(unsigned)seen);
        if (!LONE) r = min(r, __builtin_amdgcn_readfirstlane((int)(unsigned)(seen >> 32)));
        return r >= need;
    };
    auto waitReady = [&](int need) {
        if (__builtin_expect(!isReady(need), 0)) {
            ++nSlow;
            for (int spins = 0;; ++spins) {
                lookReady();
                if (isReady(need)) break;
                // an expired wait ends every later one after 1024 looks, so
                // a broken schedule ends the kernel instead of hanging it
                if ((spins & 1023) == 1023 && (spins > (kWaitLimit << 3) || __hip_atomic_load(V.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                    if (lane == 0) atomicOr(V.err, 2);
                    break;
                }
            }
        }
    };
    lookReady();
    waitReady(1);
    RowV<T> row[kLook];
#pragma unroll
    for (int u = 0; u < kLook; ++u) row[u] = getRow<T>(sh.rec[u], lane);
    T xb = sh.plane[kIn - 1][nbB], xc = T(0), yprev = T(0);
    if (!FLAT) xc = sh.plane[kIn - 1][nbC];
    auto runGroup = [&](int g, auto fullTag) {
        constexpr bool FULL = decltype(fullTag)::value;
        // time of the group's first step, and the scalar offsets of its lowest
        const int T0 = kFwd ? sp.lo + g : sp.hi - 1 + tLo - g;
        const int Tlow = kFwd ? T0 : T0 - (kG - 1);
        const RowSlot<T> *recG = &sh.rec[g & (kRec - 1)], *recN = &sh.rec[(g + kG) & (kRec - 1)];
        T(*plane)[kPlane] = &sh.plane[g & (kIn - 1)];
#pragma unroll
        for (int u = 0; u < kG; ++u) {
            const int Tu = kFwd ? T0 + u : T0 - u;
            const int ia = Tu - bl - cl;
            const bool valid = FULL ? inTile : inTile && (unsigned)(ia - sp.lo) < (unsigned)(sp.hi - sp.lo);
            const RowV<T> r = row[u % kLook];
            T p[3];
            p[kSlotA] = r[kSlotA] * yprev;
            p[kSlotB] = r[kSlotB] * xb;
            if (!FLAT) p[kSlotC] = r[kSlotC] * xc;
            T y = r[3];
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (!(FLAT && q == kSlotC)) y = y - p[q];
            if (!FULL) y = valid ? y : T(0);
            constexpr bool kMove = LONE && FLAT;
            if (!kMove) plane[u][own] = y;
            // (other lanes' values are read back: not to be reordered, which
            // a lane's own addresses would allow)
            compilerFence();
            // the exchange comes first: its round trip is the step's chain,
            // and the stores below overlap it
            if (kMove) {
                xb = laneBefore<T, kFwd>(y);
            } else if (u % kSub != kSub - 1) {
                xb = plane[u][nbB];
                if (!FLAT) xc = plane[u][nbC];
            }
            __builtin_amdgcn_sched_barrier(0);
            yprev = y;
            const U yb = Bits<T>::to(y);
            if (!LONE) {
                if (FULL) {   // one scalar offset for both
                    const unsigned so = (unsigned)((Tu + mOff) * E) * sizeof(U);
                    bufStore<U, kSysCoherent>(yb, rToB, vToB + (unsigned)((dB - mOff) * E) * sizeof(U), so);
                    bufStore<U, kSysCoherent>(yb, rToC, vToC + (unsigned)((dC - mOff) * E) * sizeof(U), so);
                } else {
                    // (a valid row's consumer step is valid too; an invalid
                    // row's is only kept non-negative)
                    bufStore<U, kSysCoherent>(yb, rToB, valid ? vToB : kNoLane, (unsigned)(max(Tu + dB, 0) * E) * sizeof(U));
                    bufStore<U, kSysCoherent>(yb, rToC, valid ? vToC : kNoLane, (unsigned)(max(Tu + dC, 0) * E) * sizeof(U));
                }
            }
            if (FULL) bufStore<T, 0>(y, rOut, vOut + (unsigned)(Tu - Tlow) * 64 * sizeof(T), (unsigned)Tlow * 64 * sizeof(T));
            else bufStore<T, 0>(y, rOut, valid ? vOut : kNoLane, (unsigned)(Tu > 0 ? Tu : 0) * 64 * sizeof(T));
            if (u % kSub == kSub - 1) {
                // the steps so far are done; the edge values and rows of the
                // next ones have to be there
                post(&sh.consumed, g + u + 1);
                waitReady(g + u + 1 + kSub);
                lookReady();
                if (!kMove) xb = plane[u][nbB];
                if (!FLAT) xc = plane[u][nbC];
            }
            row[u % kLook] = getRow<T>(u + kLook < kG ? recG[u + kLook] : recN[u + kLook - kG], lane);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    waitReady(kSub);
    lookReady();
    for (int g = 0; g < nL; g += kG) {
        // FULL: every in-tile row of the group's steps is one of the span's
        const int tMin = kFwd ? sp.lo + g : sp.hi - 1 + tLo - (g + kG - 1), tMax = tMin + kG - 1;
        if (tMin >= sp.lo + tLo && tMax <= sp.hi - 1) runGroup(g, std::true_type{});
        else runGroup(g, std::false_type{});
    }
}

// ---------------------------------------------------------------------------
// stream wave
// ---------------------------------------------------------------------------

// KT: the batch's record width K when it is 3 (two FP64 chunks or one FP32
// chunk per row, rD in the last), or 0 for a wider batch (K read from the
// view, rD in a chunk of its own).
template <typename T, int KT, int MODE, int INP>
__device__ __forceinline__ void boxStream(const DiluView<T> &V, const Tile &t, Span sp, const T *in, Shared<T> &sh,
                                          const SweepInput<T> &inp)
{
    using R = typename RecordOf<T, MODE>::V;
    constexpr int N = RecordOf<T, MODE>::N;
    constexpr bool kFwd = MODE != kDiluBwd;
    constexpr int G2 = 2 / N + 1;                // chunks holding slots 0..2
    constexpr bool kExtra = KT == 0;             // rD in a chunk of its own
    constexpr int NL = G2 + (kExtra ? 1 : 0);
    const int K = KT ? KT : V.K;
    const int G = packChunks(K + 1, N), gLast = K / N, eLast = K % N;
    const unsigned lane = threadIdx.x & 63;
    const int bl = lane & (t.TB - 1), cl = lane >> t.lg;
    const bool inTile = bl < t.actB && cl < t.actC;
    const int tLo = (t.actB - 1) + (t.actC - 1), nL = sp.hi - sp.lo + tLo;
    const unsigned rowBytes = (unsigned)G * 64 * sizeof(R);
    const R *recs = (const R *)(MODE == kDiluBwd ? V.bPack : V.fPack);
    const auto rRec = rawBuffer(recs + (size_t)t.s0 * G * 64, (size_t)t.nSteps * rowBytes);
    const size_t rowsBytes = (size_t)t.nSteps * 64 * sizeof(T);
    const auto rIn = rawBuffer((INP ? inp.r : in) + (size_t)t.s0 * 64, rowsBytes);
    // the fused input's other operands: the vector it is stored to (p, read
    // first for its old value; s) and v
    const auto rDst = INP ? rawBuffer(inp.dst + (size_t)t.s0 * 64, rowsBytes) : rawBuffer(in, 0);
    const auto rV = INP ? rawBuffer(inp.v + (size_t)t.s0 * 64, rowsBytes) : rawBuffer(in, 0);
    const unsigned vRec = lane * (unsigned)sizeof(R), vRow = lane * (unsigned)sizeof(T);

    struct Step {
        R v[NL];
        T a, pOld, vv;
    };
    // step i's slice (loads past the end re-read the last step's)
    auto timeOf = [&](int i) {
        i = i < nL ? i : nL - 1;
        return kFwd ? sp.lo + i : sp.hi - 1 + tLo - i;
    };
    auto load = [&](int i, Step &S) {
        const unsigned j = (unsigned)timeOf(i);
        const unsigned so = j * rowBytes, sv = j * (unsigned)(64 * sizeof(T));
#pragma unroll
        for (int g = 0; g < G2; ++g) S.v[g] = bufLoad<R, 0>(rRec, vRec + g * 64 * sizeof(R), so);
        if (kExtra) S.v[NL - 1] = bufLoad<R, 0>(rRec, vRec + gLast * 64 * sizeof(R), so);
        S.a = bufLoad<T, 0>(rIn, vRow, sv);
        if (INP == kInpP) S.pOld = bufLoad<T, 0>(rDst, vRow, sv);
        if (INP) S.vv = bufLoad<T, 0>(rV, vRow, sv);
    };
    Step buf[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
        load(u, buf[u]);
        __builtin_amdgcn_sched_barrier(0);
    }
    int consumed = 0;
    for (int g = 0; g < nL; g += kAhead) {
        RowSlot<T> *recG = &sh.rec[g & (kRec - 1)];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int i = g + u;
            if (u % kChunk == 0) {
                // room for the next chunk in the ring (bounded: the compute
                // wave ends even if its waits expire)
                for (int spins = 0; consumed + kRec < i + kChunk && spins < (kWaitLimit << 4); ++spins) {
                    consumed = peek(&sh.consumed);
                    if (consumed + kRec < i + kChunk) __builtin_amdgcn_s_sleep(1);
                }
            }
            const Step &S = buf[u];
            T last;
            if (kExtra) last = (T)elem(S.v[NL - 1], eLast);
            else last = (T)elem(S.v[3 / N], 3 % N);
            // the row's input: BiCGStab's p or s update where fused (the
            // expressions of k_bicg_p / k_bicg_s), else the loaded value
            T ain = S.a;
            if (INP == kInpP) ain = S.a + inp.c1 * S.pOld - inp.c2 * S.vv;
            else if (INP == kInpS) ain = S.a - inp.c1 * S.vv;
            T c[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) c[q] = last * (T)elem(S.v[q / N], q % N);
            putRow(recG[u], lane, c, kFwd ? ain * last : ain);
            if (u % kChunk == kChunk - 1) post(&sh.ready.rows, i + 1 - kLook);
            if (INP) {
                // (only the span's rows: a segment's wave shares slices with
                // the others', and a step past the end re-reads the last)
                const int Ti = timeOf(i), ia = Ti - bl - cl;
                const bool valid = inTile & ((unsigned)(ia - sp.lo) < (unsigned)(sp.hi - sp.lo)) & (i < nL);
                bufStore<T, 0>(ain, rDst, valid ? vRow : kNoLane, (unsigned)Ti * (unsigned)(64 * sizeof(T)));
            }
            load(i + kAhead, buf[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    post(&sh.ready.rows, kAll);
}

// ---------------------------------------------------------------------------
// feed wave
// ---------------------------------------------------------------------------

// Rows of the inbox arrive in order, one per step of the producer.  Lane l
// follows b value l % TC in every TB-th row and c value l % TB in every
// TC-th; a batch of loads covers at least the next 8 rows of both, and
// kBatches batches are in flight, so a value is seen a fraction of a memory
// round trip after it could be.  (A load of a row that another batch has
// already delivered is ignored.)  What a hop costs is this wave's instructions
// as much as memory: with 16 rows and four batches, a batch took 170
// instructions and was looked at 1.4 us after its issue.
template <typename T, int MODE, int LG>
__device__ __forceinline__ void boxFeed(const DiluView<T> &V, const int32_t *m, const Tile &t,
                                        const typename Bits<T>::U *inbox, Shared<T> &sh)
{
    using U = typename Bits<T>::U;
    constexpr U kSent = Bits<T>::kSent;
    constexpr bool kFwd = MODE != kDiluBwd;
    constexpr int TB = 1 << LG, TC = 64 >> LG, E = TB > TC ? TB : TC;
    constexpr int kRB = TB >= 8 ? 1 : 8 / TB, kRC = TC >= 8 ? 1 : 8 / TC;   // loads per batch
    constexpr int kBatches = 2;
    constexpr int kRow = E * (int)sizeof(U);
    const int lane = threadIdx.x & 63;
    const bool prevB = m[kFwd ? kBtInPrevB : kBtInNextB] >= 0, prevC = m[kFwd ? kBtInPrevC : kBtInNextC] >= 0;
    const int nL = t.nSteps;
    // first and one-past-last step of the lane's values, and its next row
    const int cv = lane & (TC - 1), bv = lane & (TB - 1);
    const int offB = (kFwd ? 0 : TB - 1) + cv, offC = bv + (kFwd ? 0 : TC - 1);
    const int firstB = kFwd ? offB : nL - offB - t.nA, firstC = kFwd ? offC : nL - offC - t.nA;
    const int endB = prevB && cv < t.actC ? firstB + t.nA : INT_MIN, endC = prevC && bv < t.actB ? firstC + t.nA : INT_MIN;
    int nb = firstB + (lane >> (6 - LG)), nc = firstC + (lane >> LG);
    // inbox rows by step: step i is row T = i (forward) / nL - 1 - i.  (A
    // row outside the inbox is not loaded, the hardware returns zero, and it
    // is never taken.  Nor is any row of a side without a neighbour, which a
    // flat tile would ask for eight full rows of in each batch: a fed tile of
    // 1000x66 cells went at 145 ns a step.)
    const auto rB = rawBuffer(inbox + t.inbox, prevB ? (size_t)nL * kRow : 0);
    const auto rC = rawBuffer(inbox + t.inbox + (size_t)nL * E, prevC ? (size_t)nL * kRow : 0);
    auto offsetOf = [&](int i, int v) { return (unsigned)((kFwd ? i : nL - 1 - i) * kRow + v * (int)sizeof(U)); };
    // where they go: the plane of the step before
    U *toB = (U *)&sh.plane[0][t.cell<kFwd>(kFwd ? -1 : TB, cv)], *toC = (U *)&sh.plane[0][t.cell<kFwd>(bv, kFwd ? -1 : TC)];
    U *spare = (U *)&sh.spare[lane];
    struct Batch {
        U b[kRB], c[kRC];
        int nb, nc;
    } ring[kBatches];
    auto issue = [&](Batch &q) {
        q.nb = nb;
        q.nc = nc;
#pragma unroll
        for (int k = 0; k < kRB; ++k) q.b[k] = bufLoad<U, kSysCoherent>(rB, offsetOf(nb + k * TB, cv), 0);
#pragma unroll
        for (int k = 0; k < kRC; ++k) q.c[k] = bufLoad<U, kSysCoherent>(rC, offsetOf(nc + k * TC, bv), 0);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int k = 0; k < kBatches; ++k) issue(ring[k]);
    // (bounded: `idle` rounds in a row without a step, not the rounds of a
    // long sweep, and none once another wait has expired.  The loop has one
    // exit, after whole rounds of batches: an exit in between made the
    // compiler drain every load at the start of a round.)
    int done = 0;
    for (int idle = 0; idle < V.waitLimit && done != kAll; ++idle) {
        if (__builtin_expect((idle & 1023) == 1023, 0) && __hip_atomic_load(V.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            idle = V.waitLimit - 1;
#pragma unroll
        for (int s = 0; s < kBatches; ++s) {
            Batch &q = ring[s];
            const int room = look(&sh.consumed) + kIn;
            const int limB = min(endB, room), limC = min(endC, room);
#pragma unroll
            for (int k = 0; k < kRB; ++k) {
                const int i = q.nb + k * TB;
                const bool take = (i == nb) & (i < limB) & (q.b[k] != kSent);
                U *to = take ? toB + ((i - 1) & (kIn - 1)) * kPlane : spare;
                *to = q.b[k];
                nb = take ? nb + TB : nb;
            }
#pragma unroll
            for (int k = 0; k < kRC; ++k) {
                const int i = q.nc + k * TC;
                const bool take = (i == nc) & (i < limC) & (q.c[k] != kSent);
                U *to = take ? toC + ((i - 1) & (kIn - 1)) * kPlane : spare;
                *to = q.c[k];
                nc = take ? nc + TC : nc;
            }
            compilerFence();
            issue(q);
            // the steps before the first one that lacks a value, in the
            // compute wave's units of kSub
            const int lacks = min(nb < endB ? nb : kAll, nc < endC ? nc : kAll);
            if (__builtin_amdgcn_ballot_w64(lacks < done + kSub) == 0) {
                do done += kSub;
                while (done < nL && __builtin_amdgcn_ballot_w64(lacks < done + kSub) == 0);
                done = done < nL ? done : kAll;
                idle = -1;
                post(&sh.ready.edges, done);
            }
        }
    }
    if (done != kAll && lane == 0) atomicOr(V.err, 2);
}

template <typename T>
__device__ inline SweepInput<T> sweepInputOf(int inpKind, SweepInput<T> in, const SysState &S)
{
    if (inpKind == kInpP) {
        in.c1 = (T)S.beta;
        in.c2 = (T)(S.beta * S.omega);
    } else {
        in.c1 = (T)S.alpha;
    }
    return in;
}

template <typename T, int MODE, bool LONE>
__device__ __forceinline__ void computeAll(const DiluView<T> &V, const int32_t *m, const Tile &t, Span sp, T *out,
                                           typename Bits<T>::U *inbox, Shared<T> &sh, unsigned &nSlow)
{
    const bool flat = t.TC == 1 && (LONE || (m[kBtInPrevC] < 0 && m[kBtInNextC] < 0));
    const int sel = t.axis * 2 + (flat ? 1 : 0);
    switch (sel) {
    case 0: boxCompute<T, MODE, 0, LONE, false>(V, m, t, sp, out, inbox, sh, nSlow); break;
    case 1: boxCompute<T, MODE, 0, LONE, true>(V, m, t, sp, out, inbox, sh, nSlow); break;
    case 2: boxCompute<T, MODE, 1, LONE, false>(V, m, t, sp, out, inbox, sh, nSlow); break;
    case 3: boxCompute<T, MODE, 1, LONE, true>(V, m, t, sp, out, inbox, sh, nSlow); break;
    case 4: boxCompute<T, MODE, 2, LONE, false>(V, m, t, sp, out, inbox, sh, nSlow); break;
    default: boxCompute<T, MODE, 2, LONE, true>(V, m, t, sp, out, inbox, sh, nSlow); break;
    }
}

template <typename T>
__device__ inline void initShared(Shared<T> &sh, bool fed)
{
    // (missing neighbours' values are finite: their coefficients are zero)
    for (int q = threadIdx.x; q < kIn * kPlane; q += blockDim.x) sh.plane[q / kPlane][q % kPlane] = T(0);
    if (threadIdx.x == 0) {
        sh.ready.rows = 0;
        sh.ready.edges = fed ? 0 : kAll;
        sh.consumed = 0;
    }
}

}  // namespace

// One workgroup per tile (a LONE launch: per tile segment).  Workgroups are
// dispatched in the order of their tiles' dependencies, so a tile only waits
// for tiles that are resident or done (sweep_gate.hpp: also beside other
// batches' sweeps).
template <typename T, int KT, int MODE, bool LONE, int INP = kInpPlain>
__global__ __launch_bounds__(LONE ? 128 : 192) void k_dilu_box(DiluView<T> V, const SysState *st, const T *in, T *out,
                                                               typename Bits<T>::U *inbox,
                                                               typename Bits<T>::U *inboxClear,
                                                               SweepInput<T> inpBase = SweepInput<T>{})
{
    __shared__ Shared<T> sh;
    const int segs = LONE ? V.boxSegs : 1;
    const int j = (int)blockIdx.x / segs, seg = (int)blockIdx.x - j * segs;
    const int32_t *m = V.boxTile + (size_t)(MODE == kDiluBwd ? V.nBoxWaves - 1 - j : j) * kBoxTile;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool active = st[m[kBtSys]].status == kRunning;
    const Tile t(m);
    const unsigned long long tStart = V.trace ? wall_clock64() : 0ull;
    unsigned nSlow = 0;
    // the tile's entries of the opposite sweep's inbox, which nobody reads
    // during this one: those that a neighbour delivers to, once the feed wave
    // has nothing left to wait for.  (Clearing whole rows beforehand held the
    // first edge values up by 2 * 64 values a step and tile in flat boxes: a
    // sweep of 3000x66 cells took 611 us, 441 us now.)
    auto clearInbox = [&]() {
        constexpr bool kFwd = MODE != kDiluBwd;
        const int E = max(t.TB, t.TC), lgC = 6 - t.lg;
        typename Bits<T>::U *ofB = inboxClear + t.inbox, *ofC = ofB + (size_t)t.nSteps * E;
        const int nB = m[kFwd ? kBtInNextB : kBtInPrevB] >= 0 ? t.nSteps * t.TC : 0;
        const int nC = m[kFwd ? kBtInNextC : kBtInPrevC] >= 0 ? t.nSteps * t.TB : 0;
        const int lane = threadIdx.x & 63;
        for (int q = lane; q < nB; q += 64) ofB[(size_t)(q >> lgC) * E + (q & (t.TC - 1))] = Bits<T>::kSent;
        for (int q = lane; q < nC; q += 64) ofC[(size_t)(q >> t.lg) * E + (q & (t.TB - 1))] = Bits<T>::kSent;
    };
    if (active && t.nSteps > 0) {
        constexpr bool kFwd = MODE != kDiluBwd;
        const bool fed = !LONE && (m[kFwd ? kBtInPrevB : kBtInNextB] >= 0 || m[kFwd ? kBtInPrevC : kBtInNextC] >= 0);
        initShared(sh, fed);
        __syncthreads();
        Span sp{0, t.nA};
        if (LONE && segs > 1) boxSegment(t.nA, seg, segs, sp.lo, sp.hi);
        if (sp.hi > sp.lo) {
            if (wave == 0) {
                computeAll<T, MODE, LONE>(V, m, t, sp, out, inbox, sh, nSlow);
            } else if (wave == 1) {
                const SweepInput<T> inp = INP ? sweepInputOf(INP, inpBase, st[m[kBtSys]]) : inpBase;
                boxStream<T, KT, MODE, INP>(V, t, sp, in, sh, inp);
            } else if constexpr (!LONE) {
                switch (fed ? t.lg : 7) {
                case 0: boxFeed<T, MODE, 0>(V, m, t, inbox, sh); break;
                case 1: boxFeed<T, MODE, 1>(V, m, t, inbox, sh); break;
                case 2: boxFeed<T, MODE, 2>(V, m, t, inbox, sh); break;
                case 3: boxFeed<T, MODE, 3>(V, m, t, inbox, sh); break;
                case 4: boxFeed<T, MODE, 4>(V, m, t, inbox, sh); break;
                case 5: boxFeed<T, MODE, 5>(V, m, t, inbox, sh); break;
                case 6: boxFeed<T, MODE, 6>(V, m, t, inbox, sh); break;
                default: break;   // no neighbour to wait for
                }
                clearInbox();
            }
        }
    } else if (!LONE && wave == 2) {
        clearInbox();
    }
    if (V.trace && threadIdx.x == 0 && segs == 1) {
        unsigned long long *tr = V.trace + 4 * ((size_t)V.nWaves + blockIdx.x);
        tr[0] = tStart;
        tr[1] = wall_clock64();
        tr[2] = nSlow;
        tr[3] = (unsigned long long)t.nSteps;
    }
}

// Both sweeps of lone tiles in one launch: a workgroup sweeps its tile (or
// tile segment) forward and then backward, since its backward rows depend
// only on its own forward rows.
template <typename T, int INP = kInpPlain>
__global__ __launch_bounds__(128) void k_dilu_box_pair(DiluView<T> V, const SysState *st, const T *in, T *out,
                                                       SweepInput<T> inpBase = SweepInput<T>{})
{
    using U = typename Bits<T>::U;
    __shared__ Shared<T> sh;
    const int segs = V.boxSegs;
    const int j = (int)blockIdx.x / segs, seg = (int)blockIdx.x - j * segs;
    const int32_t *m = V.boxTile + (size_t)j * kBoxTile;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Tile t(m);
    if (st[m[kBtSys]].status != kRunning || t.nSteps <= 0) return;
    Span sp{0, t.nA};
    if (segs > 1) boxSegment(t.nA, seg, segs, sp.lo, sp.hi);
    if (sp.hi <= sp.lo) return;
    unsigned nSlow = 0;
    initShared(sh, false);
    __syncthreads();
    if (wave == 0) computeAll<T, kDiluFwd, true>(V, m, t, sp, out, (U *)nullptr, sh, nSlow);
    else boxStream<T, 3, kDiluFwd, INP>(V, t, sp, in, sh, INP ? sweepInputOf(INP, inpBase, st[m[kBtSys]]) : inpBase);
    // the forward rows of the compute wave are read back by the stream wave
    // (of the same workgroup)
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    initShared(sh, false);
    __syncthreads();
    if (wave == 0) computeAll<T, kDiluBwd, true>(V, m, t, sp, out, (U *)nullptr, sh, nSlow);
    else boxStream<T, 3, kDiluBwd, kInpPlain>(V, t, sp, out, sh, SweepInput<T>{});
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

template <typename T, int MODE>
static hipError_t launchSweep(const DiluView<T> &V, const SysState *st, const T *in, T *out, void *use, void *clr,
                              hipStream_t s)
{
    using U = typename Bits<T>::U;
    if (V.nBoxWaves <= 0) return hipSuccess;
    if (!V.boxTile) return hipErrorInvalidValue;
    const int n = V.nBoxWaves;
    if (V.boxLone) {
        const int nb = n * (V.boxSegs > 1 ? V.boxSegs : 1);
        if (V.K == 3) k_dilu_box<T, 3, MODE, true><<<nb, 128, 0, s>>>(V, st, in, out, (U *)use, (U *)clr);
        else k_dilu_box<T, 0, MODE, true><<<nb, 128, 0, s>>>(V, st, in, out, (U *)use, (U *)clr);
        return hipGetLastError();
    }
    if (V.boxSegs > 1) return hipErrorInvalidValue;   // segments only in lone sweeps
    if (V.K == 3) k_dilu_box<T, 3, MODE, false><<<n, 192, 0, s>>>(V, st, in, out, (U *)use, (U *)clr);
    else k_dilu_box<T, 0, MODE, false><<<n, 192, 0, s>>>(V, st, in, out, (U *)use, (U *)clr);
    return hipGetLastError();
}

template <typename T>
hipError_t boxForward(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s)
{
    return launchSweep<T, kDiluFwd>(V, st, in, out, V.boxInF, V.boxInB, s);
}

template <typename T>
hipError_t boxBackward(const DiluView<T> &V, const SysState *st, T *inout, hipStream_t s)
{
    return launchSweep<T, kDiluBwd>(V, st, inout, inout, V.boxInB, V.boxInF, s);
}

template <typename T>
hipError_t diluApplyLone(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s)
{
    // (records are wider than a box's three slots only beside other regions)
    if (V.nBoxWaves <= 0 || V.general() || V.K != 3 || !V.boxLone || !V.boxTile) return hipErrorInvalidValue;
    const int nb = V.nBoxWaves * (V.boxSegs > 1 ? V.boxSegs : 1);
    k_dilu_box_pair<T><<<nb, 128, 0, s>>>(V, st, in, out);
    return hipGetLastError();
}

template <typename T>
hipError_t diluApplyFused(const DiluView<T> &V, const SysState *st, int inp, const T *r, T *dst, const T *v, T *out,
                          hipStream_t s)
{
    if (!diluCanFuse(V) || (inp != kInpP && inp != kInpS) || !V.boxTile) return hipErrorInvalidValue;
    SweepInput<T> in;
    in.r = r;
    in.dst = dst;
    in.v = v;
    if (V.boxLone) {
        const int nb = V.nBoxWaves * (V.boxSegs > 1 ? V.boxSegs : 1);
        if (inp == kInpP) k_dilu_box_pair<T, kInpP><<<nb, 128, 0, s>>>(V, st, dst, out, in);
        else k_dilu_box_pair<T, kInpS><<<nb, 128, 0, s>>>(V, st, dst, out, in);
        return hipGetLastError();
    }
    using U = typename Bits<T>::U;
    const int n = V.nBoxWaves;
    U *use = (U *)V.boxInF, *clr = (U *)V.boxInB;
    if (inp == kInpP) k_dilu_box<T, 3, kDiluFwd, false, kInpP><<<n, 192, 0, s>>>(V, st, dst, out, use, clr, in);
    else k_dilu_box<T, 3, kDiluFwd, false, kInpS><<<n, 192, 0, s>>>(V, st, dst, out, use, clr, in);
    hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : boxBackward<T>(V, st, out, s);
}

hipError_t boxTilesPerCU(int *tiles)
{
    const void *kernels[] = {(const void *)k_dilu_box<double, 3, kDiluBwd, false>, (const void *)k_dilu_box<double, 3, kDiluFwd, false, kInpP>,
                             (const void *)k_dilu_box<double, 0, kDiluFwd, false>};
    *tiles = INT_MAX;
    for (const void *k : kernels) {
        int n = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, 192, 0);
        if (e != hipSuccess) return e;
        if (n < 1) return hipErrorInvalidValue;
        *tiles = n < *tiles ? n : *tiles;
    }
    return hipSuccess;
}

#define MRFG_BOX_INSTANTIATE(T)                                                                                      \
    template hipError_t boxForward<T>(const DiluView<T> &, const SysState *, const T *, T *, hipStream_t);            \
    template hipError_t boxBackward<T>(const DiluView<T> &, const SysState *, T *, hipStream_t);                      \
    template hipError_t diluApplyLone<T>(const DiluView<T> &, const SysState *, const T *, T *, hipStream_t);         \
    template hipError_t diluApplyFused<T>(const DiluView<T> &, const SysState *, int, const T *, T *, const T *, T *, \
                                          hipStream_t);
MRFG_BOX_INSTANTIATE(double)
MRFG_BOX_INSTANTIATE(float)

}  // namespace mrfg
