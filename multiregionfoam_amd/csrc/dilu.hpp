// DILU (coupled Cholesky preconditioner) executed by a wave schedule
// (dilu.hip).  See layout.hpp for how the schedule and dependency codes are
// built.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"
#include "layout.hpp"

namespace mrfg {

enum { kDiluFwd = 0, kDiluBwd = 1, kDiluFactor = 2 };

// Inbox entries of box tiles hold the raw bits of a value; one equal to the sentinel has
// not been published yet in the current sweep (signalling-NaN payloads that
// arithmetic never produces).
constexpr unsigned long long kHaloSentinel64 = 0xFFF4A5A5A5A5A5A5ull;
constexpr unsigned int kHaloSentinel32 = 0xFFA5A5A5u;

// Per-row DILU records, packed in 16-byte chunks so that a step of a wave
// costs few vector-memory instructions.  Chunk g of lane l of slice s sits
// at (s*G + g)*64 + l.
//   values  [c_0..c_{K-1}, rD]: forward = lower coefficients, backward =
//           upper coefficients, factor = upper*lower products with the
//           diagonal in place of rD;
// Rows of general waves also have codes that say where each dependency is:
//   chains        one byte each (kCodeNone or an LDS ring slot), four per
//                 int, int j of lane l of slice s at (s*NC + j)*64 + l;
//   level groups  one int each, that of slot k at (s*K + k)*64 + l: kNoDep,
//                 an LDS ring slot (< kLevelRing), or kLevelRing + the row's
//                 place in the group; spread levels: the row's position.
template <typename T>
struct Pack;
template <>
struct Pack<double> {
    using V = double2;
    static constexpr int N = 2;
};
template <>
struct Pack<float> {
    using V = float4;
    static constexpr int N = 4;
};
constexpr int packChunks(int n, int per) { return (n + per - 1) / per; }
constexpr int kCodeNone = 0xFF;

// One workgroup's sweep of a level group: rounds of up to lvWaves slices
// (layout.hpp, LevelRound)
struct LevelGroup {
    int slice0, round0, nRounds, sys;
};

constexpr int kWaitLimit = 1 << 20;   // polls of one wait before it raises the error flag (about a second)

// A slice of a region whose levels are spread over the device
struct SpreadSlice {
    int slice, sys;
    int region;      // among the spread regions
    int levels;      // of the region, in the first slice of a level; else 0
};

template <typename T>
struct DiluView {
    // chain waves in dispatch order
    const int32_t *order = nullptr;
    const int32_t *waveSlice = nullptr, *waveSteps = nullptr, *waveSys = nullptr;
    int nWaves = 0, K = 3;
    const int32_t *fCodes = nullptr, *bCodes = nullptr;
    // level groups
    const LevelGroup *groups = nullptr;
    const LevelRound *lvRounds = nullptr;
    const int32_t *fDeps = nullptr, *bDeps = nullptr;
    int nGroups = 0, lvWaves = 1;
    int *lvProgress = nullptr;           // per group: the round its sweep has reached
    bool lvHelped = false;               // set by the launcher: helper workgroups read lvProgress
    double *lvD = nullptr;               // factor: d per row of the level groups and spread levels
    // spread levels: the slices of all regions' first level, of their second
    // and so on; level l has those from spreadLevels[l] on (on the host)
    const SpreadSlice *spread = nullptr;
    const int *spreadLevels = nullptr;
    int nSpreadLevels = 0;
    typename Pack<T>::V *fPack = nullptr, *bPack = nullptr;
    const double2 *prodPack = nullptr;   // factor records (FP64)
    double *rDout = nullptr;             // factor: plain rD per row
    const int32_t *cellOfPos = nullptr;  // factor: padding rows get rD = 0
    bool general() const { return nWaves > 0 || nGroups > 0 || nSpreadLevels > 0; }   // regions that are no boxes
    int *err = nullptr;                  // bit 2: a halo wait expired
    int waitLimit = kWaitLimit;
    // structured-box tiles (dilu_box.hip; the factor in dilu.hip): their own
    // dispatch order, kBoxMeta ints of tile geometry per wave, and compact
    // inboxes of 2 max(TB, TC) values per step per tile, one per direction
    const int32_t *boxOrder = nullptr;
    int nBoxWaves = 0;
    bool boxLone = false;                // every box tile is alone in its region
    // lone sweeps only (the tile-local preconditioner): each tile's rows are
    // cut along the sequential axis into boxSegs segments of nA / boxSegs
    // rows, each swept by a wave of its own with the coupling across the cut
    // left out
    int boxSegs = 1;
    const int32_t *boxMeta = nullptr;
    const int32_t *boxTile = nullptr;    // kBoxTile ints per box tile, in dispatch order
    void *boxInF = nullptr, *boxInB = nullptr, *boxInC = nullptr;
    int nBoxIn = 0;
    // optional trace: per wave start / end realtime clock ticks, slow-path
    // hits and steps (4 entries each); chain waves by dispatch index, then box
    // tiles, then level groups, then spread regions
    unsigned long long *trace = nullptr;
    // host side: when both kinds of waves exist, the box sweep runs on `side`
    // concurrently with the general sweep (regions never depend on each
    // other), forked and joined with the two events
    hipStream_t side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};

// A forward sweep of box tiles may compute its input itself, BiCGStab's
// update of the vector it preconditions, and store that vector (the
// expressions of k_bicg_p / k_bicg_s, so the results are the same):
//   kInpP: in = r + c1*dst - c2*v (c1 = beta, c2 = beta*omega), stored to dst (p);
//   kInpS: in = r - c1*v (c1 = alpha), stored to dst (s).
enum { kInpPlain = 0, kInpP = 1, kInpS = 2 };
template <typename T>
struct SweepInput {
    const T *r = nullptr;
    T *dst = nullptr;
    const T *v = nullptr;
    T c1 = T(0), c2 = T(0);
};

// Forward sweep out = (D+L)^-1 in (with the D^-1 scaling of DILU) and the
// backward sweep in place; systems whose status is not running are skipped.
// the box tiles alone (dilu_box.hip)
template <typename T>
hipError_t boxForward(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s);
template <typename T>
hipError_t boxBackward(const DiluView<T> &V, const SysState *st, T *inout, hipStream_t s);
template <typename T>
hipError_t diluForward(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s);
template <typename T>
hipError_t diluBackward(const DiluView<T> &V, const SysState *st, T *inout, hipStream_t s);
// Both sweeps in one launch when every wave is a lone box tile (no general
// waves): out = M^-1 in, each wave forward then backward over its own rows.
template <typename T>
hipError_t diluApplyLone(const DiluView<T> &V, const SysState *st, const T *in, T *out, hipStream_t s);
// The preconditioner applied to BiCGStab's p (inp = kInpP: p = r + beta*p -
// beta*omega*v) or s (kInpS: s = r - alpha*v) of every system, with the
// update computed and stored by the forward sweeps (batches of K = 3 box
// tiles only, no general waves): out = M^-1 dst.  The scalars come from each
// system's state.
template <typename T>
hipError_t diluApplyFused(const DiluView<T> &V, const SysState *st, int inp, const T *r, T *dst, const T *v, T *out,
                          hipStream_t s);
template <typename T>
bool diluCanFuse(const DiluView<T> &V)
{
    return !V.general() && V.nBoxWaves > 0 && V.K == 3;
}
// Factorisation: rD = 1/d for every row of the batch (FP64), written to
// rDout and into the forward and backward records.
hipError_t diluFactor(const DiluView<double> &V, hipStream_t s);
// The tile-local factor: rD of every box tile's rows with the couplings across
// tile edges (and across the cuts between its segs segments) left out, each
// tile segment factorised alone, written to rD only (rows of general waves
// are left as they are).  FP64, from the FP64 product records.
hipError_t diluFactorTileLocal(const DiluView<double> &V, double *rD, int segs, hipStream_t s);
// Segment s of segs of a box tile's nA rows along its sequential axis: rows
// [lo, hi) (shared by the host's record derivation and the device sweeps)
__host__ __device__ inline void boxSegment(int nA, int s, int segs, int &lo, int &hi)
{
    lo = (int)((long long)s * nA / segs);
    hi = (int)((long long)(s + 1) * nA / segs);
}
// Workgroups of the box sweeps (FP64, with inboxes) that a CU of the current
// device holds at once
hipError_t boxTilesPerCU(int *tiles);
// XCDs of a device with `cus` CUs
constexpr int kCusPerXcd = 32;
inline int xcdsOf(int cus) { return cus > kCusPerXcd ? cus / kCusPerXcd : 1; }

// Values of a box tile's inbox: per step one row for the b and one for the c edge
__host__ __device__ inline int boxInboxValues(int nSteps, int TB) { return nSteps * 2 * (TB > 64 / TB ? TB : 64 / TB); }

// A box tile as its sweeps see it: one descriptor per tile in forward
// dispatch order (the backward sweep takes them in reverse), with the inbox
// of every neighbouring tile (-1: none) and the steps of the next ones, so a
// workgroup starts after two dependent loads
enum {
    kBtTB = 0, kBtNA, kBtAxis, kBtActB, kBtActC, kBtSlice, kBtSteps, kBtSys, kBtInbox,
    kBtInPrevB, kBtInPrevC, kBtInNextB, kBtInNextC, kBtLPrevB, kBtLPrevC, kBtLNextB, kBtLNextC,
    kBoxTile = 20
};
// rD of the FP32 records from the FP64 factor
hipError_t diluConvertRD(const DiluView<float> &V32, const double *rD64, int nSlices, hipStream_t s);
hipError_t fillHalo64(void *h, int n, hipStream_t s);
hipError_t fillHalo32(void *h, int n, hipStream_t s);

}  // namespace mrfg
