#include "layout.hpp"

#include <algorithm>
#include <numeric>
#include <stdexcept>

namespace mrfg {

namespace {

struct RowDeps {
    // CSR of lower / upper neighbours per global cell, in face order
    std::vector<int32_t> lo_off, lo_nb, lo_face;
    std::vector<int32_t> up_off, up_nb, up_face;
};

// One DILU wave under construction: cells[step * 64 + lane] (global cell or -1)
struct WaveBuild {
    int key = 0;       // dispatch key: tiles on one anti-diagonal / one level share it
    int region = 0;
    int steps = 0;
    std::vector<int32_t> cells;
    // structured-box tile (box = false for level waves)
    bool box = false;
    int tb = 0, tc = 0, TB = 0, nA = 0, seqAxis = 0, actB = 0, actC = 0;
    std::vector<int32_t> levels;   // level group or spread levels: slices per level
    bool spread = false;
};

void tangential(int a, int &b, int &c)
{
    if (a == 0) { b = 1; c = 2; }
    else if (a == 1) { b = 0; c = 2; }
    else { b = 0; c = 1; }
}

// Model of one sweep's time (us) for a tiling: the dependency chain of a
// tile (its steps plus one cross-tile hop per tile boundary crossed) against
// the bandwidth time of all slots.
double tileCost(const int n[3], int a, int TB, int TC)
{
    int b, c;
    tangential(a, b, c);
    int nTB = (n[b] + TB - 1) / TB, nTC = (n[c] + TC - 1) / TC;
    int steps = n[a] + std::min(TB, n[b]) - 1 + std::min(TC, n[c]) - 1;
    double slots = (double)nTB * nTC * steps * 64.0;
    double chain = steps * 0.06 + (nTB + nTC - 2) * 2.0;
    double bw = slots * 56.0 / 4.0e6;
    return std::max(chain, bw) + 0.05 * bw;
}

void boxWaves(const int n[3], int regionIdx, int cellOffset, RegionSchedule &rs, std::vector<WaveBuild> &out)
{
    int a = 0;
    for (int q = 1; q < 3; ++q)
        if (n[q] > n[a]) a = q;
    int b, c;
    tangential(a, b, c);
    int bestTB = 64;
    double best = 1e300;
    for (int TB = 1; TB <= 64; TB *= 2) {
        int TC = 64 / TB;
        if (TB > 1 && TB / 2 >= n[b]) continue;
        if (TC > 1 && TC / 2 >= n[c]) continue;
        double cst = tileCost(n, a, TB, TC);
        if (cst < best) {
            best = cst;
            bestTB = TB;
        }
    }
    const int TB = bestTB, TC = 64 / TB;
    rs.kind = "box";
    for (int q = 0; q < 3; ++q) rs.n[q] = n[q];
    rs.seqAxis = a;
    rs.tileB = TB;
    rs.tileC = TC;
    const int nTB = (n[b] + TB - 1) / TB, nTC = (n[c] + TC - 1) / TC;
    for (int tc = 0; tc < nTC; ++tc)
        for (int tb = 0; tb < nTB; ++tb) {
            WaveBuild w;
            w.key = tb + tc;
            w.region = regionIdx;
            int maxBl = std::min(TB, n[b] - tb * TB) - 1, maxCl = std::min(TC, n[c] - tc * TC) - 1;
            w.box = true;
            w.tb = tb;
            w.tc = tc;
            w.TB = TB;
            w.nA = n[a];
            w.seqAxis = a;
            w.actB = maxBl + 1;
            w.actC = maxCl + 1;
            w.steps = n[a] + maxBl + maxCl;
            w.cells.assign((size_t)w.steps * kSlice, -1);
            for (int cl = 0; cl <= maxCl; ++cl)
                for (int bl = 0; bl <= maxBl; ++bl) {
                    int lane = bl + TB * cl;
                    int idx[3];
                    idx[b] = tb * TB + bl;
                    idx[c] = tc * TC + cl;
                    for (int ia = 0; ia < n[a]; ++ia) {
                        idx[a] = ia;
                        int cell = idx[0] + n[0] * (idx[1] + n[1] * idx[2]);
                        w.cells[(size_t)(ia + bl + cl) * kSlice + lane] = cellOffset + cell;
                    }
                }
            rs.maxSteps = std::max(rs.maxSteps, w.steps);
            out.push_back(std::move(w));
            rs.nWaves++;
        }
}

// Whether a region's levels are swept by the whole device, one launch per
// level, rather than by one workgroup (a level group).  What a sweep takes
// (FP64, launches replayed from a graph):
//   spread   3.6 us a level (1340 us for 382 levels of 2.0M cells numbered
//            along a front, 170 us for 20 levels of 2.0M shuffled cells)
//   group    0.8 ns a row (389 us for 0.5M cells along a front, 241 levels),
//            and 1.1 ns for each line of 128 bytes that a slice reads back
//            from beyond the LDS ring (2030 us for the 2.0M along a front,
//            1960 us for 0.5M shuffled, 8300 us for 2.0M shuffled)
// so a level is worth 4500 rows and such a line 1.5.  The other choice: spread
// 870 us for the 0.5M along a front, 1180 (against 967) for 1.3M in 328
// levels; a group 143 us (against 61) for 59k shuffled cells in 17 levels.
bool spreadPays(int c0, int c1, const RowDeps &D, const std::vector<std::vector<int32_t>> &byLevel)
{
    constexpr long long kRowsPerLevel = 4500;
    constexpr int kLine = 128 / sizeof(double);
    const long long rows = c1 - c0, need = kRowsPerLevel * (long long)byLevel.size();
    if (rows >= need) return true;
    std::vector<int32_t> place(c1 - c0);   // in the group's slices
    int32_t at = 0;
    long long lines = 0;
    std::vector<int32_t> back;             // lines of a slice
    for (const std::vector<int32_t> &cells : byLevel) {
        const int32_t end = at + (int32_t)((cells.size() + kSlice - 1) / kSlice) * kSlice;
        for (size_t i = 0; i < cells.size(); ++i) place[cells[i] - c0] = at + (int32_t)i;
        for (size_t i = 0; i < cells.size(); i += kSlice) {
            back.clear();
            for (size_t l = i; l < std::min(i + kSlice, cells.size()); ++l)
                for (int q = D.lo_off[cells[l]]; q < D.lo_off[cells[l] + 1]; ++q) {
                    const int32_t from = place[D.lo_nb[q] - c0];
                    if (end - from > kLevelRing) back.push_back(from / kLine);
                }
            std::sort(back.begin(), back.end());
            lines += std::unique(back.begin(), back.end()) - back.begin();
        }
        at = end;
    }
    return 2 * rows + 3 * lines >= 2 * need;
}

void levelWaves(int regionIdx, int c0, int c1, const RowDeps &D, RegionSchedule &rs, std::vector<WaveBuild> &out)
{
    std::vector<int32_t> level(c1 - c0, 0);
    int maxLevel = 0;
    for (int c = c0; c < c1; ++c) {
        int lv = 0;
        for (int q = D.lo_off[c]; q < D.lo_off[c + 1]; ++q) lv = std::max(lv, level[D.lo_nb[q] - c0] + 1);
        level[c - c0] = lv;
        maxLevel = std::max(maxLevel, lv);
    }
    std::vector<std::vector<int32_t>> byLevel(maxLevel + 1);
    for (int c = c0; c < c1; ++c) byLevel[level[c - c0]].push_back(c);
    size_t maxWidth = 0;
    for (const auto &b : byLevel) maxWidth = std::max(maxWidth, b.size());
    int reach = 1;   // levels between a cell and its furthest neighbour
    for (int c = c0; c < c1; ++c)
        for (int q = D.lo_off[c]; q < D.lo_off[c + 1]; ++q) reach = std::max(reach, level[c - c0] - level[D.lo_nb[q] - c0]);
    WaveBuild w;
    w.key = 0;
    w.region = regionIdx;
    // one wave walks narrow levels as its steps: every dependency comes from
    // its own LDS ring and no step waits for another wave.  Wider levels (or
    // levels that reach further back) go to a workgroup with a barrier per
    // level, or are spread over the device where they are wide enough.
    const bool chain = maxWidth <= (size_t)kSlice && reach <= kRing - 1;
    for (int lv = 0; lv <= maxLevel; ++lv) {
        const int n = (int)((byLevel[lv].size() + kSlice - 1) / kSlice);
        const size_t at = w.cells.size();
        w.cells.resize(at + (size_t)n * kSlice, -1);
        std::copy(byLevel[lv].begin(), byLevel[lv].end(), w.cells.begin() + at);
        if (!chain) w.levels.push_back(n);
        w.steps += n;
    }
    w.spread = !chain && spreadPays(c0, c1, D, byLevel);
    rs.kind = chain ? "chain" : w.spread ? "spread" : "levels";
    rs.nWaves = 1;
    rs.maxSteps = w.steps;
    out.push_back(std::move(w));
}

}  // namespace

bool detectBox(const LduRegion &R, int n[3])
{
    const int N = R.nCells;
    if (N < 2 || R.nFaces < 1) return false;
    int d1 = 0, d2 = 0, d3 = 0;   // smallest distinct offsets
    for (int f = 0; f < R.nFaces; ++f) {
        int d = R.uAddr[f] - R.lAddr[f];
        if (d == d1 || d == d2 || d == d3) continue;
        if (!d1 || d < d1) { d3 = d2; d2 = d1; d1 = d; }
        else if (!d2 || d < d2) { d3 = d2; d2 = d; }
        else if (!d3 || d < d3) d3 = d;
    }
    int nx, ny, nz;
    if (d1 != 1) return false;
    if (!d2) { nx = N; ny = 1; nz = 1; }
    else if (!d3) { nx = d2; ny = N / d2; nz = 1; }
    else { nx = d2; if (d3 % d2) return false; ny = d3 / d2; nz = N / d3; }
    if ((long long)nx * ny * nz != N || nx < 1 || ny < 1 || nz < 1) return false;
    // verify the face list is exactly the lexicographic box pattern
    int f = 0;
    for (int c = 0; c < N; ++c) {
        int i = c % nx, j = (c / nx) % ny, k = c / (nx * ny);
        int nb[3] = {i + 1 < nx ? c + 1 : -1, j + 1 < ny ? c + nx : -1, k + 1 < nz ? c + nx * ny : -1};
        for (int q = 0; q < 3; ++q) {
            if (nb[q] < 0) continue;
            if (f >= R.nFaces || R.lAddr[f] != c || R.uAddr[f] != nb[q]) return false;
            ++f;
        }
    }
    if (f != R.nFaces) return false;
    n[0] = nx;
    n[1] = ny;
    n[2] = nz;
    return true;
}

// A row beyond the ring is read back from memory, so a barrier that waits for
// stores has to lie between its level and the reader's.  One such barrier at
// each level end where the rows since the last one and the next level's would
// exceed the ring is enough: if a forward row of level A had none before its
// reader's level L, all rows from A's first to L's last would fit the ring, and
// the row would be read from there (backward alike).
void levelRounds(const std::vector<int32_t> &levels, int slice0, int waves, bool far, std::vector<LevelRound> &out)
{
    const int nL = (int)levels.size();
    std::vector<int> stored(nL, 0);
    constexpr int kMost = kLevelRing / kSlice;
    long long sum = 0;
    for (int lv = 0; far && lv + 1 < nL; ++lv) {
        sum += levels[lv];
        if (sum + levels[lv + 1] > kMost) stored[lv] |= kRoundStoredF, sum = 0;
    }
    sum = 0;
    for (int lv = nL - 1; far && lv > 0; --lv) {
        sum += levels[lv];
        if (sum + levels[lv - 1] > kMost) stored[lv] |= kRoundStoredB, sum = 0;
    }
    int s = slice0;
    for (int lv = 0; lv < nL; ++lv)
        for (int k = 0; k < levels[lv]; k += waves) {
            const int cnt = std::min(waves, levels[lv] - k);
            int flags = 0;
            if (k + cnt == levels[lv]) flags |= kRoundLast | (stored[lv] & kRoundStoredF);
            if (k == 0) flags |= kRoundFirst | (stored[lv] & kRoundStoredB);
            out.push_back({s, cnt << kRoundBits | flags});
            s += cnt;
        }
}

SystemLayout buildLayout(const CoupledSystem &sys, bool preferLevels)
{
    sys.check();
    SystemLayout L;
    const int nR = (int)sys.regions.size();
    L.regionOffset.resize(nR + 1, 0);
    for (int r = 0; r < nR; ++r) L.regionOffset[r + 1] = L.regionOffset[r] + sys.regions[r].nCells;
    const int N = L.regionOffset[nR];
    L.nCells = N;
    L.nFaces = sys.nFaces();
    L.nPairs = sys.nPairs();

    // ---- lower/upper neighbour lists per cell (face order) ----
    std::vector<int32_t> nLo(N, 0), nUp(N, 0);
    for (int r = 0; r < nR; ++r) {
        const LduRegion &R = sys.regions[r];
        int o = L.regionOffset[r];
        for (int f = 0; f < R.nFaces; ++f) {
            nLo[o + R.uAddr[f]]++;
            nUp[o + R.lAddr[f]]++;
        }
    }
    RowDeps D;
    D.lo_off.assign(N + 1, 0);
    D.up_off.assign(N + 1, 0);
    for (int c = 0; c < N; ++c) {
        D.lo_off[c + 1] = D.lo_off[c] + nLo[c];
        D.up_off[c + 1] = D.up_off[c] + nUp[c];
    }
    D.lo_nb.resize(D.lo_off[N]);
    D.lo_face.resize(D.lo_off[N]);
    D.up_nb.resize(D.up_off[N]);
    D.up_face.resize(D.up_off[N]);
    {
        std::vector<int32_t> fl(D.lo_off.begin(), D.lo_off.end() - 1), fu(D.up_off.begin(), D.up_off.end() - 1);
        for (int r = 0; r < nR; ++r) {
            const LduRegion &R = sys.regions[r];
            int o = L.regionOffset[r];
            for (int f = 0; f < R.nFaces; ++f) {
                int l = o + R.lAddr[f], u = o + R.uAddr[f];
                D.lo_nb[fl[u]] = l;
                D.lo_face[fl[u]++] = f;
                D.up_nb[fu[l]] = u;
                D.up_face[fu[l]++] = f;
            }
        }
    }
    int K = 3;
    for (int c = 0; c < N; ++c) K = std::max(K, std::max(nLo[c], nUp[c]));
    L.K = K;

    // ---- DILU schedule: waves of every region, ordered by dispatch key ----
    std::vector<WaveBuild> waves;
    L.schedules.resize(nR);
    for (int r = 0; r < nR; ++r) {
        int n[3];
        if (!preferLevels && detectBox(sys.regions[r], n))
            boxWaves(n, r, L.regionOffset[r], L.schedules[r], waves);
        else
            levelWaves(r, L.regionOffset[r], L.regionOffset[r + 1], D, L.schedules[r], waves);
    }
    std::vector<int> ord(waves.size());
    std::iota(ord.begin(), ord.end(), 0);
    std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return waves[x].key < waves[y].key; });
    L.nWaves = (int)waves.size();
    L.waveSlice.resize(L.nWaves);
    L.waveSteps.resize(L.nWaves);
    L.waveKey.resize(L.nWaves);
    L.waveLevels.resize(L.nWaves);
    L.waveFar.assign(L.nWaves, 0);
    L.waveSpread.assign(L.nWaves, 0);
    int slice = 0;
    for (int wi = 0; wi < L.nWaves; ++wi) {
        const WaveBuild &w = waves[ord[wi]];
        L.waveSlice[wi] = slice;
        L.waveSteps[wi] = w.steps;
        L.waveKey[wi] = w.key;
        L.waveLevels[wi] = w.levels;
        L.waveSpread[wi] = w.spread ? 1 : 0;
        slice += w.steps;
    }
    L.nSlices = slice;
    L.nPos = slice * kSlice;
    L.cellOfPos.assign(L.nPos, -1);
    L.posOfCell.assign(N, -1);
    std::vector<int32_t> waveOfSlice(L.nSlices);
    for (int wi = 0; wi < L.nWaves; ++wi) {
        const WaveBuild &w = waves[ord[wi]];
        for (int t = 0; t < w.steps; ++t) {
            waveOfSlice[L.waveSlice[wi] + t] = wi;
            for (int l = 0; l < kSlice; ++l) {
                int c = w.cells[(size_t)t * kSlice + l];
                if (c < 0) continue;
                int p = (L.waveSlice[wi] + t) * kSlice + l;
                L.cellOfPos[p] = c;
                L.posOfCell[c] = p;
            }
        }
    }
    for (int c = 0; c < N; ++c)
        if (L.posOfCell[c] < 0) throw std::runtime_error("DILU schedule does not cover every cell");

    // level groups: first and one-past-last slice (of the wave) of each slice's level
    std::vector<int32_t> lvBegin(L.nSlices, -1), lvEnd(L.nSlices, -1);
    for (int wi = 0; wi < L.nWaves; ++wi) {
        int t = 0;
        for (int n : L.waveLevels[wi]) {
            for (int k = 0; k < n; ++k) {
                lvBegin[L.waveSlice[wi] + t + k] = t;
                lvEnd[L.waveSlice[wi] + t + k] = t + n;
            }
            t += n;
        }
    }

    // structured-box waves: tile neighbours and fixed-slot records (slot =
    // 2 - axis: z, y, x, the face order of a cell's lower neighbours and the
    // reverse face order of its upper neighbours)
    L.waveBox.assign(L.nWaves, 0);
    L.boxMeta.assign((size_t)L.nWaves * kBoxMeta, -1);
    {
        std::vector<std::vector<int>> tileWave(nR);
        std::vector<int> tileNB(nR, 0);
        for (int wi = 0; wi < L.nWaves; ++wi) {
            const WaveBuild &w = waves[ord[wi]];
            if (!w.box) continue;
            const RegionSchedule &rs = L.schedules[w.region];
            int b, cc;
            tangential(rs.seqAxis, b, cc);
            int nTB = (rs.n[b] + rs.tileB - 1) / rs.tileB, nTC = (rs.n[cc] + rs.tileC - 1) / rs.tileC;
            if (tileWave[w.region].empty()) tileWave[w.region].assign((size_t)nTB * nTC, -1);
            tileNB[w.region] = nTB;
            tileWave[w.region][(size_t)w.tc * nTB + w.tb] = wi;
        }
        for (int wi = 0; wi < L.nWaves; ++wi) {
            const WaveBuild &w = waves[ord[wi]];
            if (!w.box) continue;
            L.waveBox[wi] = 1;
            const RegionSchedule &rs = L.schedules[w.region];
            int b, cc;
            tangential(rs.seqAxis, b, cc);
            const int nTB = tileNB[w.region], nTC = (rs.n[cc] + rs.tileC - 1) / rs.tileC;
            auto tw = [&](int tb, int tc) {
                return tb < 0 || tc < 0 || tb >= nTB || tc >= nTC ? -1 : tileWave[w.region][(size_t)tc * nTB + tb];
            };
            int32_t *m = &L.boxMeta[(size_t)wi * kBoxMeta];
            m[kBmTB] = w.TB;
            m[kBmNA] = w.nA;
            m[kBmPrevB] = tw(w.tb - 1, w.tc);
            m[kBmPrevC] = tw(w.tb, w.tc - 1);
            m[kBmNextB] = tw(w.tb + 1, w.tc);
            m[kBmNextC] = tw(w.tb, w.tc + 1);
            m[kBmAxis] = rs.seqAxis;
            m[kBmActB] = w.actB;
            m[kBmActC] = w.actC;
        }
    }

    auto regionOf = [&](int c) {
        return int(std::upper_bound(L.regionOffset.begin(), L.regionOffset.end(), c) - L.regionOffset.begin()) - 1;
    };

    L.diag.assign(L.nPos, 0.0);
    L.source.assign(L.nPos, 0.0);
    L.psi0.assign(L.nPos, 0.0);
    L.sumA.assign(L.nPos, 0.0);
    for (int r = 0; r < nR; ++r) {
        const LduRegion &R = sys.regions[r];
        int o = L.regionOffset[r];
        for (int c = 0; c < R.nCells; ++c) {
            int p = L.posOfCell[o + c];
            L.diag[p] = R.diag[c];
            L.source[p] = R.source[c];
            L.psi0[p] = R.psi[c];
        }
    }
    // sumA: diag, then the face loop, then minus interface coefficients
    // (lduMatrix::sumA restated on the coupled system)
    {
        std::vector<double> s(N);
        for (int r = 0; r < nR; ++r) {
            const LduRegion &R = sys.regions[r];
            int o = L.regionOffset[r];
            for (int c = 0; c < R.nCells; ++c) s[o + c] = R.diag[c];
            for (int f = 0; f < R.nFaces; ++f) {
                s[o + R.uAddr[f]] += R.lower[f];
                s[o + R.lAddr[f]] += R.upper[f];
            }
        }
        for (const auto &I : sys.interfaces) {
            const InterfaceSide *sides[2] = {&I.a, &I.b};
            for (int q = 0; q < 2; ++q) {
                const InterfaceSide &S = *sides[q];
                int o = L.regionOffset[S.region];
                for (int f = 0; f < S.nFaces(); ++f) s[o + S.fc[f]] -= S.coeff[f];
            }
        }
        for (int c = 0; c < N; ++c) L.sumA[L.posOfCell[c]] = s[c];
    }

    // ---- interface faces per row (interface order, then face order) ----
    std::vector<std::vector<std::pair<int, int>>> rowFaces(N);
    for (size_t i = 0; i < sys.interfaces.size(); ++i) {
        const CoupledInterface &I = sys.interfaces[i];
        const InterfaceSide *sides[2] = {&I.a, &I.b};
        for (int q = 0; q < 2; ++q) {
            const InterfaceSide &S = *sides[q];
            int o = L.regionOffset[S.region];
            for (int f = 0; f < S.nFaces(); ++f) rowFaces[o + S.fc[f]].push_back({(int)i * 2 + q, f});
        }
    }

    // ---- geometry of the 3-D box slices (the columns of their SpMV entries) ----
    L.sliceGeom.assign((size_t)L.nSlices * kSliceGeom, 0);
    for (int s = 0; s < L.nSlices; ++s) L.sliceGeom[(size_t)s * kSliceGeom + kSgAxis] = -1;
    for (int wi = 0; wi < L.nWaves; ++wi) {
        if (!L.waveBox[wi]) continue;
        const RegionSchedule &rs = L.schedules[waves[ord[wi]].region];
        if (rs.n[0] < 2 || rs.n[1] < 2 || rs.n[2] < 2) continue;
        const int32_t *m = &L.boxMeta[(size_t)wi * kBoxMeta];
        const int TB = m[kBmTB], TC = kSlice / TB;
        // lane l's row of step t is cell ia = t - bl - cl of its line, in the
        // tile and in its neighbours alike
        auto across = [&](int to, int dStep, int dLane) {
            return m[to] < 0 ? 0 : (L.waveSlice[m[to]] - L.waveSlice[wi] + dStep) * kSlice + dLane;
        };
        int g[kSliceGeom] = {m[kBmAxis],
                             __builtin_ctz(TB) | m[kBmActB] << 8 | m[kBmActC] << 16,
                             across(kBmPrevB, TB - 1, TB - 1),
                             across(kBmNextB, 1 - TB, 1 - TB),
                             across(kBmPrevC, TC - 1, TB * (TC - 1)),
                             across(kBmNextC, 1 - TC, -TB * (TC - 1)),
                             0,
                             m[kBmNA]};
        for (int t = 0; t < L.waveSteps[wi]; ++t) {
            g[kSgStep] = t;
            std::copy(g, g + kSliceGeom, &L.sliceGeom[(size_t)(L.waveSlice[wi] + t) * kSliceGeom]);
        }
    }

    // ---- per-slice ELL (SpMV) ----
    L.ellOff.assign(L.nSlices + 1, 0);
    L.ifMask.assign(L.nSlices, 0);
    L.ifBase.assign(L.nSlices, 0);
    L.ifRowFace.assign(1, 0);
    L.ifPairOff.assign(1, 0);
    for (int s = 0; s < L.nSlices; ++s) {
        int wE = 0;
        for (int l = 0; l < kSlice; ++l) {
            int c = L.cellOfPos[s * kSlice + l];
            if (c < 0) continue;
            wE = std::max(wE, (D.lo_off[c + 1] - D.lo_off[c]) + (D.up_off[c + 1] - D.up_off[c]));
        }
        if (L.sliceGeom[(size_t)s * kSliceGeom + kSgAxis] >= 0) wE = 6;
        L.ellOff[s + 1] = L.ellOff[s] + wE;
    }
    L.ellCol.assign((size_t)L.ellOff[L.nSlices] * kSlice, 0);
    L.ellVal.assign((size_t)L.ellOff[L.nSlices] * kSlice, 0.0);
    L.ellSrc.assign((size_t)L.ellOff[L.nSlices] * kSlice, -1);
    L.faceOffset.assign(nR, 0);
    for (int r = 1; r < nR; ++r) L.faceOffset[r] = L.faceOffset[r - 1] + sys.regions[r - 1].nFaces;
    std::vector<int32_t> sideOffset(2 * sys.interfaces.size() + 1, 0);
    for (size_t i = 0; i < sys.interfaces.size(); ++i) {
        sideOffset[2 * i + 1] = sideOffset[2 * i] + sys.interfaces[i].a.nFaces();
        sideOffset[2 * i + 2] = sideOffset[2 * i + 1] + sys.interfaces[i].b.nFaces();
    }
    const size_t nDep = (size_t)L.nSlices * K * kSlice;
    L.fCode.assign(nDep, kNoDep);
    L.bCode.assign(nDep, kNoDep);
    L.fVal.assign(nDep, 0.0);
    L.fProd.assign(nDep, 0.0);
    L.bVal.assign(nDep, 0.0);
    L.fSrc.assign(nDep, -1);
    L.bSrc.assign(nDep, -1);

    auto waveStep = [&](int p, int &w, int &t, int &lane) {
        int s = p / kSlice;
        lane = p % kSlice;
        w = waveOfSlice[s];
        t = s - L.waveSlice[w];
    };

    for (int s = 0; s < L.nSlices; ++s) {
        L.ifBase[s] = (int32_t)L.ifRowFace.size() - 1;
        const int wE = L.ellOff[s + 1] - L.ellOff[s];
        for (int l = 0; l < kSlice; ++l) {
            int p = s * kSlice + l;
            int c = L.cellOfPos[p];
            // padding entries of the SpMV point at the row itself with value 0
            for (int k = 0; k < wE; ++k) L.ellCol[(size_t)(L.ellOff[s] + k) * kSlice + l] = p;
            if (c < 0) continue;
            int r = regionOf(c);
            const LduRegion &R = sys.regions[r];
            const std::vector<double> &lo = R.symmetric ? R.upper : R.lower;
            auto loSrc = [&](int f) { return 2 * (L.faceOffset[r] + f) + (R.symmetric ? 1 : 0); };
            auto upSrc = [&](int f) { return 2 * (L.faceOffset[r] + f) + 1; };
            int k = 0;
            // the entry of a 3-D box row is that of the neighbour's axis
            const bool byAxis = L.sliceGeom[(size_t)s * kSliceGeom + kSgAxis] >= 0;
            auto axisOf = [&](int d) {
                const RegionSchedule &rs = L.schedules[r];
                return d == 1 ? 0 : d == rs.n[0] ? 1 : 2;
            };
            for (int q = D.lo_off[c]; q < D.lo_off[c + 1]; ++q, ++k) {
                if (byAxis) k = 2 - axisOf(c - D.lo_nb[q]);
                size_t e = (size_t)(L.ellOff[s] + k) * kSlice + l;
                L.ellCol[e] = L.posOfCell[D.lo_nb[q]];
                L.ellVal[e] = lo[D.lo_face[q]];
                L.ellSrc[e] = loSrc(D.lo_face[q]);
            }
            for (int q = D.up_off[c]; q < D.up_off[c + 1]; ++q, ++k) {
                if (byAxis) k = 3 + axisOf(D.up_nb[q] - c);
                size_t e = (size_t)(L.ellOff[s] + k) * kSlice + l;
                L.ellCol[e] = L.posOfCell[D.up_nb[q]];
                L.ellVal[e] = R.upper[D.up_face[q]];
                L.ellSrc[e] = upSrc(D.up_face[q]);
            }

            int w, t, lane;
            waveStep(p, w, t, lane);
            const int T = L.waveSteps[w];
            if (L.waveBox[w]) {
                // box tile rows: fixed slots by the axis of the neighbour
                // (slot 2 - axis), zero where there is none; the dependencies
                // themselves follow from the tile geometry
                const RegionSchedule &rs = L.schedules[r];
                const int sxy = rs.n[0] * rs.n[1];
                auto slotOf = [&](int d) { return d == 1 ? 2 : d == rs.n[0] ? 1 : d == sxy ? 0 : -1; };
                for (int q = D.lo_off[c]; q < D.lo_off[c + 1]; ++q) {
                    int sl = slotOf(c - D.lo_nb[q]);
                    if (sl < 0) throw std::runtime_error("box region with an unexpected lower neighbour");
                    int f = D.lo_face[q];
                    size_t e = ((size_t)s * K + sl) * kSlice + l;
                    L.fVal[e] = lo[f];
                    L.fProd[e] = R.upper[f] * lo[f];
                    L.fSrc[e] = loSrc(f);
                }
                for (int q = D.up_off[c]; q < D.up_off[c + 1]; ++q) {
                    int sl = slotOf(D.up_nb[q] - c);
                    if (sl < 0) throw std::runtime_error("box region with an unexpected upper neighbour");
                    L.bVal[((size_t)s * K + sl) * kSlice + l] = R.upper[D.up_face[q]];
                    L.bSrc[((size_t)s * K + sl) * kSlice + l] = upSrc(D.up_face[q]);
                }
            } else {
                // forward sweep: lower neighbours, ascending face order
                k = 0;
                for (int q = D.lo_off[c]; q < D.lo_off[c + 1]; ++q, ++k) {
                    int f = D.lo_face[q];
                    int pd = L.posOfCell[D.lo_nb[q]];
                    int wd, td, ld;
                    waveStep(pd, wd, td, ld);
                    size_t e = ((size_t)s * K + k) * kSlice + l;
                    L.fVal[e] = lo[f];
                    L.fProd[e] = R.upper[f] * lo[f];
                    L.fSrc[e] = loSrc(f);
                    if (wd != w) throw std::runtime_error("DILU dependency crosses waves");
                    if (lvEnd[s] >= 0) {
                        if (lvEnd[pd / kSlice] > lvBegin[s]) throw std::runtime_error("DILU schedule violates a forward dependency");
                        // in the ring until the rows kLevelRing further on are written
                        const int at = td * kSlice + ld;
                        const bool far = !L.waveSpread[w] && lvEnd[s] * kSlice - at > kLevelRing;
                        L.fCode[e] = L.waveSpread[w] ? at : far ? kLevelRing + at : at & (kLevelRing - 1);
                        if (far) L.waveFar[w] = 1;
                    } else {
                        if (t - td < 1 || t - td > kRing - 1) throw std::runtime_error("DILU schedule violates a forward dependency");
                        L.fCode[e] = (td % kRing) * kSlice + ld;
                    }
                }
                // backward sweep: upper neighbours, reverse face order; processing
                // index i = T-1-t, so the ring slot of a dependency uses its own i
                k = 0;
                for (int q = D.up_off[c + 1] - 1; q >= D.up_off[c]; --q, ++k) {
                    int pd = L.posOfCell[D.up_nb[q]];
                    int wd, td, ld;
                    waveStep(pd, wd, td, ld);
                    size_t e = ((size_t)s * K + k) * kSlice + l;
                    L.bVal[e] = R.upper[D.up_face[q]];
                    L.bSrc[e] = upSrc(D.up_face[q]);
                    if (wd != w) throw std::runtime_error("DILU dependency crosses waves");
                    if (lvEnd[s] >= 0) {
                        if (lvBegin[pd / kSlice] < lvEnd[s]) throw std::runtime_error("DILU schedule violates a backward dependency");
                        const int at = td * kSlice + ld;
                        const bool far = !L.waveSpread[w] && at - lvBegin[s] * kSlice >= kLevelRing;
                        L.bCode[e] = L.waveSpread[w] ? at : far ? kLevelRing + at : at & (kLevelRing - 1);
                        if (far) L.waveFar[w] = 1;
                    } else {
                        if (td - t < 1 || td - t > kRing - 1) throw std::runtime_error("DILU schedule violates a backward dependency");
                        L.bCode[e] = ((T - 1 - td) % kRing) * kSlice + ld;
                    }
                }
            }
            // interface faces of this row
            if (!rowFaces[c].empty()) {
                L.ifMask[s] |= 1ULL << l;
                for (auto &pf : rowFaces[c]) {
                    const CoupledInterface &I = sys.interfaces[pf.first / 2];
                    const InterfaceSide &S = (pf.first % 2) ? I.b : I.a;
                    const InterfaceSide &O = (pf.first % 2) ? I.a : I.b;
                    int oN = L.regionOffset[O.region];
                    int f = pf.second;
                    L.ifCoeff.push_back(S.coeff[f]);
                    L.ifSrc.push_back(sideOffset[pf.first] + f);
                    for (int q = S.off[f]; q < S.off[f + 1]; ++q) {
                        L.ifPairCol.push_back(L.posOfCell[oN + O.fc[S.idx[q]]]);
                        L.ifPairW.push_back(S.w[q]);
                    }
                    L.ifPairOff.push_back((int32_t)L.ifPairW.size());
                }
                L.ifRowFace.push_back((int32_t)L.ifCoeff.size());
            }
        }
    }
    return L;
}

}  // namespace mrfg
