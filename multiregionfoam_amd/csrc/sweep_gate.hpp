// Which batches' box sweeps may be in flight on a device together.
//
// A tile's workgroup waits for other tiles of its kernel, so the earliest
// unfinished tile has to be running.  An XCD starts its share of a kernel's
// workgroups in order but on its own, so with one kernel that always holds:
// where the earliest unfinished tile has not started, its XCD holds none of
// the kernel's tiles and has room.  Tiles of other kernels can take that room
// while they wait in turn for tiles that the first kernel keeps from starting.
// They cannot if, per XCD, the tiles of all kernels but the largest leave a
// slot free: the largest then always runs its earliest tile and ends, and so
// does the next largest after it.
//
// A box tile takes 51 KB of LDS in FP64, so 3 fit a CU and 96 an XCD: two
// batches of up to 760 tiles run together, of 300 tiles three.  (Other
// processes on the device are not seen; there a wait that expires fails the
// call.)
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <vector>

namespace mrfg {

class SweepGate {
public:
    // slots: tiles that an XCD holds at once
    explicit SweepGate(int slots) : slots_(slots) {}

    // Hold `tiles` tiles per XCD; waits, first come first served, until they
    // may be in flight with those held already.
    void acquire(int tiles)
    {
        if (tiles <= 0) return;
        std::unique_lock<std::mutex> lk(m_);
        const uint64_t me = next_++;
        cv_.wait(lk, [&] { return me == turn_ && fits(tiles); });
        held_.push_back(tiles);
        ++turn_;
        cv_.notify_all();
    }
    void release(int tiles)
    {
        if (tiles <= 0) return;
        std::lock_guard<std::mutex> lk(m_);
        held_.erase(std::find(held_.begin(), held_.end(), tiles));
        cv_.notify_all();
    }

private:
    bool fits(int tiles) const
    {
        int sum = tiles, most = tiles;
        for (int t : held_) {
            sum += t;
            most = std::max(most, t);
        }
        return sum - most < slots_;
    }
    std::mutex m_;
    std::condition_variable cv_;
    std::vector<int> held_;
    uint64_t next_ = 0, turn_ = 0;
    int slots_;
};

// Holds a gate's tiles for a scope.
class SweepHold {
public:
    SweepHold(SweepGate &gate, int tiles) : gate_(gate), tiles_(tiles) { gate_.acquire(tiles_); }
    ~SweepHold() { gate_.release(tiles_); }
    SweepHold(const SweepHold &) = delete;
    SweepHold &operator=(const SweepHold &) = delete;

private:
    SweepGate &gate_;
    int tiles_;
};

}  // namespace mrfg
