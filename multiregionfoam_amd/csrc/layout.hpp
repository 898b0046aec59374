// Device layout of coupled block systems.
//
// Rows ("positions") of a system are grouped into 64-row slices; a slice is
// one step of one DILU wave.  A wave is a sequence of steps executed by one
// wavefront, lane l of step t holding one row (or nothing).  The waves of a
// system form its DILU schedule:
//
//   * structured hex regions (detected from the LDU addressing: faces to
//     c+1, c+nx, c+nx*ny in upper-triangular order) are cut into tiles of 64
//     grid lines along the longest axis; lane (b,c) of a tile walks its line
//     with a skew of b+c steps, so each of a cell's three lower neighbours
//     was computed one step earlier by the same or an adjacent lane;
//   * any other region is scheduled by levels (a cell's level is one more
//     than its lower neighbours' largest): a chain, one wave whose steps are
//     the levels, where every level fits 64 rows and reaches at most
//     kRing - 1 levels back (2-D and multi-block meshes, whose levels are
//     anti-diagonals), else a level group, swept by one workgroup that meets
//     at a barrier after each level, or spread levels, each swept by the whole
//     device, where they are wide.
//
// Either way the schedule is a topological order of the factor's dependency
// graph, so the Cholesky/DILU factor and sweeps computed in it are the
// reference preconditioner itself.  A chain's wave reads its dependencies
// from an LDS ring of its last kRing steps, a level group from an LDS ring of
// the region's last kLevelRing rows, or from memory where they lie further
// back, spread levels from memory.
//
// Per slice of 64 rows:
//   SpMV   sliced ELL, column-major inside the slice: entry k of lane l at
//          (ellOff[s] + k) * 64 + l; diagonal kept apart; row entries in the
//          LDU face-loop order (lower ascending, then upper ascending).
//   GGI    rows with interface faces are flagged in a 64-bit mask; their
//          faces hold the boundary coefficient and the weighted gather pairs
//          (position, weight) of the other region's cells.
//   DILU   K dependency slots per row at (s*K + k)*64 + l: forward = lower
//          neighbours in face order with lower coefficients and upper*lower
//          products, backward = upper neighbours in reverse face order with
//          upper coefficients; codes: kNoDep, in a chain the ring slot, in a
//          level group the ring slot or kLevelRing + the row's place in the
//          region's slices, in spread levels that place.
#pragma once

#include "coupled_system.hpp"

#include <climits>
#include <cstdint>
#include <string>
#include <vector>

namespace mrfg {

constexpr int kSlice = 64;          // rows per slice = wavefront size
constexpr int kSlicesPerBlock = 4;  // 256-thread blocks for SpMV / vector ops
constexpr int kRing = 3;            // LDS ring depth (steps) of a DILU wave (slots < 192)
constexpr int32_t kNoDep = -1;
constexpr int kLevelRing = 16384;   // rows of a level group's LDS ring (128 KB in FP64); a power of two

// A round of a level group's workgroup: the slices of one level that it takes
// side by side, one per wave.
struct LevelRound {
    int32_t slice;   // the first
    int32_t word;    // their number << kRoundBits | flags
};
enum {
    kRoundLast = 1,      // ends its level: a barrier follows (forward)
    kRoundFirst = 2,     // starts its level: a barrier follows (backward)
    kRoundStoredF = 4,   // at that barrier the rows stored so far have to be
    kRoundStoredB = 8,   // in memory (forward / backward)
    kRoundBits = 4
};

// Per-wave metadata of a structured-box tile wave (kBoxMeta ints each).
enum {
    kBmTB = 0,      // lanes along the tile's first tangential axis (TC = 64/TB)
    kBmNA,          // cells along the sequential axis
    kBmPrevB,       // wave of the tile before / after along each tangential axis (-1: none)
    kBmPrevC,
    kBmNextB,
    kBmNextC,
    kBmAxis,        // sequential axis (0 x, 1 y, 2 z); b, c are the other two, ascending
    kBmActB,        // active lanes along b / c in this tile
    kBmActC,
    kBmSlice,       // first slice (filled by the batch)
    kBmSteps,
    kBmInbox,       // first inbox value of this wave (filled by the batch)
    kBmSys,
    kBoxMeta = 16
};

// Per-slice geometry: the sequential axis (-1: not a 3-D box tile, the columns
// are listed); log2 of TB, actB << 8 and actC << 16; for the rows on the tile's
// edges the distance to the neighbour's position across it (0: none); the
// slice's step of the tile; nA.
enum { kSgAxis = 0, kSgTile, kSgPrevB, kSgNextB, kSgPrevC, kSgNextC, kSgStep, kSgNA, kSliceGeom = 8 };

struct RegionSchedule {
    std::string kind;                // "box", "chain", "levels" or "spread"
    int n[3] = {0, 0, 0};            // box dimensions
    int seqAxis = -1, tileB = 0, tileC = 0;
    int nWaves = 0, maxSteps = 0;
};

struct SystemLayout {
    long long nCells = 0, nFaces = 0, nPairs = 0;
    int nPos = 0, nSlices = 0, nWaves = 0, K = 0;
    std::vector<RegionSchedule> schedules;
    std::vector<int32_t> regionOffset;       // first global cell of each region
    std::vector<int32_t> cellOfPos;          // global cell or -1 (padding)
    std::vector<int32_t> posOfCell;
    // waves, in dispatch order
    std::vector<int32_t> waveSlice, waveSteps, waveKey;
    // SpMV
    std::vector<int32_t> ellOff;             // nSlices + 1, in 64-entry columns
    std::vector<int32_t> ellCol;
    std::vector<double> ellVal;
    // per slice, kSliceGeom ints: where the neighbours of a 3-D box tile's
    // rows are.  Such a slice has six entries per row in the order of the
    // axes (z, y, x lower, then x, y, z upper; zero where there is none), so
    // their columns follow from the tile
    std::vector<int32_t> sliceGeom;
    std::vector<double> diag, source, sumA, psi0;
    // GGI interface rows
    std::vector<uint64_t> ifMask;            // per slice
    std::vector<int32_t> ifBase;             // per slice, first interface row
    std::vector<int32_t> ifRowFace;          // interface rows + 1
    std::vector<double> ifCoeff;             // per interface face
    std::vector<int32_t> ifPairOff;          // faces + 1
    std::vector<int32_t> ifPairCol;
    std::vector<double> ifPairW;
    // DILU
    std::vector<int32_t> fCode, bCode;       // nSlices * K * 64
    std::vector<double> fVal, fProd, bVal;
    // per wave: the slices of each level of a level group or of spread levels
    // (empty for others)
    std::vector<std::vector<int32_t>> waveLevels;
    std::vector<uint8_t> waveFar;            // per wave: 1 if a dependency lies beyond the LDS ring
    std::vector<uint8_t> waveSpread;         // per wave: 1 if its levels are spread over the device
    // structured-box tile waves: their rows keep the DILU values in fixed
    // slots (slot = 2 - axis of the neighbour: z, y, x, which is both the
    // face order of the lower neighbours and the reverse face order of the
    // upper ones; zero where a neighbour is missing) and have no codes: the
    // dependencies follow from the tile geometry in boxMeta
    std::vector<uint8_t> waveBox;            // per wave: 1 if a box tile
    std::vector<int32_t> boxMeta;            // kBoxMeta per wave
    // where each value came from, so re-assembled coefficients can be put in
    // place on the device: face values are numbered 2*(faceOffset[r] + f)
    // (+0 the lower coefficient, +1 the upper; a symmetric region's lower
    // entries name its upper), interface-side faces in interface order, side
    // a then side b
    std::vector<int32_t> faceOffset;         // per region
    std::vector<int32_t> ellSrc;             // per ELL entry, -1 for padding
    std::vector<int32_t> fSrc, bSrc;         // per DILU slot (as fVal / bVal), -1 for none
    std::vector<int32_t> ifSrc;              // per interface-row face (as ifCoeff)
};

// Build the layout.  `preferLevels` forces the level schedule for every
// region (used to test the general path on structured meshes).
SystemLayout buildLayout(const CoupledSystem &sys, bool preferLevels = false);

// Append the rounds of a level group of `levels` (slices per level) from
// slice0 on, for workgroups of `waves` waves; `far`: with dependencies beyond
// the LDS ring, whose rows the marked barriers put into memory in time.
void levelRounds(const std::vector<int32_t> &levels, int slice0, int waves, bool far, std::vector<LevelRound> &out);

// Detect a lexicographically numbered structured hex box from LDU
// addressing; returns false if the region is not one.
bool detectBox(const LduRegion &R, int n[3]);

}  // namespace mrfg
