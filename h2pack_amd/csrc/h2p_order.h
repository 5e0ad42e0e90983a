// Order of the block tasks of a launch (host).
#pragma once
#include <algorithm>
#include <iterator>
#include <vector>

namespace h2p {

// A part's tasks: [off, off + big) on whole workgroups, then n - big as wave
// units, each range in descending order of work.
struct PartRange {
    int off, big, n;
};

// The tasks of several parts as one list in the same order: the workgroup
// tasks of all parts, then their wave tasks, each range merged by `before`
// (a strict weak order, more work first; equal tasks in the order of the
// parts).  Linear in the tasks: sorting the list anew took 3.5 ms of the
// upload at 20,000 blocks.  big: its workgroup tasks.
template <class T, class Before>
std::vector<T> merge_parts(const std::vector<T> &tasks, const std::vector<PartRange> &parts, Before before, int *big) {
    std::vector<T> out, half;
    *big = 0;
    for (int wave = 0; wave < 2; wave++) {
        std::vector<T> run;
        for (const PartRange &p : parts) {
            const auto b = tasks.begin() + p.off + (wave ? p.big : 0), e = tasks.begin() + p.off + (wave ? p.n : p.big);
            half.clear();
            half.reserve(run.size() + (e - b));
            std::merge(run.begin(), run.end(), b, e, std::back_inserter(half), before);
            run.swap(half);
        }
        if (!wave) *big = (int)run.size();
        out.insert(out.end(), run.begin(), run.end());
    }
    return out;
}

}  // namespace h2p
