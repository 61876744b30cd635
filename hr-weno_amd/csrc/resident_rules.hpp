// resident_rules.hpp -- host rules of the launches whose blocks wait for each other
// (kernels_resident.hpp).  Plain C++.
#pragma once
#include <algorithm>
#include <climits>
#include <cstdint>
#include <cstdlib>

namespace hrw {

// Whether a launch of nsteps steps may write its result over its input.  A block loads some of its
// neighbours' initial cells, so none may store its result before its neighbours have loaded.  With
// alpha = max|u| every block waits for all maxima in the first stage; otherwise a block first waits
// for its neighbours at the start of the second step, and a launch of a single step has no wait.
constexpr bool resident_in_place(bool several_blocks, bool alphamax, int64_t nsteps)
{
    return !several_blocks || alphamax || nsteps >= 2;
}

// Steps of a line in one launch at most: some ms (3 to 15 us a step), so that other streams and threads
// get their turn in a long call, and what is done again after a wait in vain is little.
constexpr int64_t kResLaunchSteps = 1024;
// The same of a batch, whose steps take up to some 100 us.
constexpr int64_t kBatchLaunchSteps = 64;

// Steps of the next launch of a call with `left` steps to go, `most` (3 or more) in one launch: no
// launch of a single step but for a call of one.
constexpr int64_t launch_steps(int64_t left, int64_t most)
{
    const int64_t n = std::min(left, most);
    return left - n == 1 ? n - 1 : n;
}

// The polls of a wait: what `text` (the environment variable HRW_RESIDENT_POLLS, or null) says in whole
// decimal digits, else `usual`.
inline int resident_polls(const char *text, int usual)
{
    if (!text || *text < '0' || *text > '9') return usual;
    char *end = nullptr;
    const long v = std::strtol(text, &end, 10);
    return *end == '\0' && v <= INT_MAX ? (int)v : usual;
}

// After a launch whose blocks waited in vain (a fifth of a second lost), an object's next calls take the
// launches per stage at once: 1, then 2, 4 .. 256 of them between tries that end so, until one does not.
struct BackOff {
    int left = 0, next = 1;
    bool skip()
    {
        if (left == 0) return false;
        --left;
        return true;
    }
    void in_vain()
    {
        left = next;
        next = std::min(2 * next, 256);
    }
    void went() { left = 0, next = 1; }
};

// Blocks of one line of a batch at most.  They wait for each other, so all must come to be on the
// device at once: at most one per CU (two fit on one, which leaves room beside them), and no more than
// a wavefront gathers the maxima of.
constexpr int kBatchResGroup = 64;
constexpr int batch_line_blocks(int cus) { return std::min(kBatchResGroup, cus); }

// The numbers of an object's exchanges.  They go on from launch to launch without a gap: a maximum
// carries one bit of its number, which tells it from the word's last one only if every number in
// between was published.  So a launch takes its numbers when it has gone through, not when it is
// tried, and after one whose blocks waited in vain the words are cleared and the numbers start anew.
constexpr unsigned kResFirstTag = 4;   // the number after which cleared words read as not arrived
struct ExchangeNumbers {
    unsigned next = kResFirstTag;
    bool clear = false;                // the words are clear, or hold the numbers before `next`
    // Whether the words have to be cleared before a launch of `used` exchanges.
    bool need_clear(unsigned used) const { return !clear || next > 0xffffffffu - used; }
    void cleared()
    {
        next = kResFirstTag;
        clear = true;
    }
    void launched(unsigned used) { next += used; }
    void lost() { clear = false; }
};

}  // namespace hrw
