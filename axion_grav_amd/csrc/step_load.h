// The step data under way on each device, host side only.
#pragma once
#include <stdint.h>

#include <atomic>

namespace axg {

// What the passes of one step touch, for a lattice of n3 sites with elem bytes a complex value and resid bytes of residual a
// field: three fields, and with GW sourcing the six transformed sources twice and the four accumulators,
// half a field each.
constexpr int64_t step_bytes(int64_t n3, int64_t elem, int64_t resid, bool gw)
{
    return n3 * ((gw ? 11 : 3) * elem + 3 * resid);
}

// Of the 256 MiB last-level cache, what a step's data may take and still be there in the next pass.
constexpr int64_t STEP_CACHE = (int64_t)240 << 20;

// Counts a lattice's step data for as long as its steps are queued or running.  Where the lattices stepped at once
// (one handle a thread) do not fit the cache together, none of them has it to itself and ordinary accesses cost
// instead of gain.  Microseconds per lattice step, streamed and cached: 128^3 FP32C one lattice 94 and 74, two at
// once 82 and 92; FP32 one 86 and 68, two 75 and 83; 96^3 FP32C (84 MiB) one 54 and 47, two 40.9 and 34.6, three
// 38.7 and 40.6.  The sum is asked at each step, so a run that begins alone streams from when another
// joins it.  Other processes on the device are not seen.  The results do not depend on it.
class StepLoad {
public:
    static constexpr int DEVICES = 16;  // devices beyond share a count: their lattices may stream without need
    StepLoad(int device, int64_t bytes) : sum_(under_way(device)), bytes_(bytes) { sum_ += bytes_; }
    ~StepLoad() { sum_ -= bytes_; }
    StepLoad(const StepLoad&) = delete;
    StepLoad& operator=(const StepLoad&) = delete;
    // Do all the lattices under way fit the cache together?
    bool fits() const { return sum_.load(std::memory_order_relaxed) <= STEP_CACHE; }

private:
    static std::atomic<int64_t>& under_way(int device)
    {
        static std::atomic<int64_t> sums[DEVICES] = {};
        return sums[(unsigned)device % DEVICES];
    }
    std::atomic<int64_t>& sum_;
    const int64_t bytes_;
};

}  // namespace axg
