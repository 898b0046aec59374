// Host replay of a level group's schedule (csrc/layout.cpp), built and called
// by test_level_schedule.py.  The rows of a level run in any order; a row
// written in it is in the LDS ring after the barrier that ends the level, and
// in memory after the next barrier that waits for stores.  Every dependency
// must be where its code says, before its reader's level starts.
#include "../multiregionfoam_amd/csrc/layout.hpp"

#include <cstdio>
#include <cstring>
#include <stdexcept>

using namespace mrfg;

// noWaits: the schedule without barriers that wait for stores;
// out: ring reads, far reads, barriers, barriers that wait for stores, reads of
// spread levels
extern "C" int replay(int nCells, int nFaces, const int32_t *lower, const int32_t *upper, int waves, int noWaits,
                      long long *out, char *why, int nWhy)
try {
    CoupledSystem sys;
    sys.regions.resize(1);
    LduRegion &R = sys.regions[0];
    R.nCells = nCells;
    R.nFaces = nFaces;
    R.lAddr.assign(lower, lower + nFaces);
    R.uAddr.assign(upper, upper + nFaces);
    R.lower.assign(nFaces, -1.0);
    R.upper = R.lower;
    R.diag = R.source = R.psi = std::vector<double>(nCells, 1.0);
    const SystemLayout L = buildLayout(sys);
    const bool spread = L.schedules[0].kind == "spread";
    if (!spread && L.schedules[0].kind != "levels") throw std::runtime_error("no levels: " + L.schedules[0].kind);
    std::vector<LevelRound> rounds;
    levelRounds(L.waveLevels[0], 0, waves, L.waveFar[0] != 0 && !noWaits, rounds);
    // neighbours in the order of the dependency slots
    std::vector<std::vector<int>> lo(nCells), up(nCells);
    for (int f = 0; f < nFaces; ++f) {
        lo[R.uAddr[f]].push_back(R.lAddr[f]);
        up[R.lAddr[f]].insert(up[R.lAddr[f]].begin(), R.uAddr[f]);
    }
    auto fail = [&](const char *what, int cell) {
        std::snprintf(why, nWhy, "%s at cell %d", what, cell);
        return 1;
    };
    std::memset(out, 0, 5 * sizeof(long long));
    if (spread != (L.waveSpread[0] != 0)) return fail("wrong kind of wave", -1);
    if (spread) {
        std::vector<int> levelOf(L.nSlices);
        int s = 0;
        for (size_t lv = 0; lv < L.waveLevels[0].size(); ++lv)
            for (int k = 0; k < L.waveLevels[0][lv]; ++k) levelOf[s++] = (int)lv;
        if (s != L.nSlices) return fail("slice left out", -1);
        for (int c = 0; c < nCells; ++c)
            for (bool fwd : {true, false})
                for (int k = 0; k < L.K; ++k) {
                    const std::vector<int> &nb = fwd ? lo[c] : up[c];
                    const int p = L.posOfCell[c], q = (fwd ? L.fCode : L.bCode)[((size_t)(p / kSlice) * L.K + k) * kSlice + p % kSlice];
                    if ((q == kNoDep) != (k >= (int)nb.size())) return fail("wrong number of dependencies", c);
                    if (q == kNoDep) continue;
                    ++out[4];
                    if (q != L.posOfCell[nb[k]]) return fail("wrong row", c);
                    const int from = levelOf[q / kSlice], to = levelOf[p / kSlice];
                    if (fwd ? from >= to : from <= to) return fail("row of a level launched later", c);
                }
        return 0;
    }
    for (bool fwd : {true, false}) {
        enum { kNone, kWritten, kInMemory };
        std::vector<int> ring(kLevelRing, -1), state(L.nPos, kNone), seen(L.nSlices, 0), level;
        const std::vector<int32_t> &code = fwd ? L.fCode : L.bCode;
        const int nR = (int)rounds.size();
        for (int i = 0; i < nR; ++i) {
            const LevelRound &r = rounds[fwd ? i : nR - 1 - i];
            const int cnt = r.word >> kRoundBits;
            if (cnt < 1 || cnt > waves) return fail("round of a wrong size", -1);
            for (int k = 0; k < cnt; ++k) {
                const int s = r.slice + k;
                if (s < 0 || s >= L.nSlices || seen[s]++) return fail("slice outside or twice", -1);
                level.push_back(s);
            }
            if (!(r.word & (fwd ? kRoundLast : kRoundFirst))) continue;
            // the level's reads, against what the levels before it left
            std::vector<char> written(kLevelRing, 0);
            for (int s : level)
                for (int l = 0; l < kSlice; ++l) written[(s * kSlice + l) & (kLevelRing - 1)] = 1;
            for (int s : level)
                for (int l = 0; l < kSlice; ++l) {
                    const int c = L.cellOfPos[s * kSlice + l];
                    if (c < 0) continue;
                    const std::vector<int> &nb = fwd ? lo[c] : up[c];
                    for (int k = 0; k < L.K; ++k) {
                        const int q = code[((size_t)s * L.K + k) * kSlice + l];
                        if ((q == kNoDep) != (k >= (int)nb.size())) return fail("wrong number of dependencies", c);
                        if (q == kNoDep) continue;
                        const int want = L.posOfCell[nb[k]];
                        if (q >= kLevelRing) {
                            ++out[1];
                            if (q - kLevelRing != want) return fail("wrong far row", c);
                            if (state[want] != kInMemory) return fail("far row not in memory yet", c);
                        } else {
                            ++out[0];
                            if (ring[q] != want) return fail("row not in the ring", c);
                            if (written[q]) return fail("ring slot overwritten by the reader's level", c);
                        }
                    }
                }
            ++out[2];
            for (int s : level)
                for (int l = 0; l < kSlice; ++l) {
                    const int p = s * kSlice + l;
                    ring[p & (kLevelRing - 1)] = p;
                    state[p] = kWritten;
                }
            level.clear();
            if (r.word & (fwd ? kRoundStoredF : kRoundStoredB)) {
                ++out[3];
                for (int &x : state)
                    if (x == kWritten) x = kInMemory;
            }
        }
        for (int x : seen)
            if (!x) return fail("slice left out", -1);
    }
    return 0;
} catch (const std::exception &e) {
    std::snprintf(why, nWhy, "%s", e.what());
    return 2;
}
