// launch_split.hpp -- splitting a batch over launches (host code, no HIP).
//
// A HIP launch takes fewer than 2^32 work-items in one grid dimension --
// work-items, not workgroups, so the limit on workgroups falls with the
// threads of each: 2^26 of 64 threads, 2^23 of 512.  A larger grid is not
// always refused: its size can wrap around, and all but the workgroups beyond
// the limit are then skipped without an error.  So kernels that number
// (system, group of its work) pairs along grid x are launched through
// launch_split, which keeps every part below it.
#pragma once

#include <cstdint>

namespace rsa
{

constexpr int64_t LAUNCH_ITEMS = (int64_t(1) << 32) - 1;

// Calls launch(s0, ns, g0, ng) for parts that cover `systems` x `groups`:
// systems [s0, s0 + ns), groups [g0, g0 + ng) of each.  A part takes at most
// ceil(ns / unit) * unit * ng workgroups of `threads` threads, fewer than 2^32
// work-items, and s0 is a multiple of `unit` (at most 64).  The groups are
// split only where one unit of systems exceeds a launch.  Stops at the first
// status other than 0 and returns it.
template <typename F>
auto launch_split(int64_t systems, int64_t groups, int threads, int unit, F&& launch)
    -> decltype(launch(int64_t(0), int64_t(0), int64_t(0), int64_t(0)))
{
    using status = decltype(launch(int64_t(0), int64_t(0), int64_t(0), int64_t(0)));
    const int64_t cap = LAUNCH_ITEMS / threads;
    const int64_t ng = groups < cap / unit ? groups : cap / unit;
    if(systems <= 0 || ng <= 0)
        return status(0);
    const int64_t ns = cap / ng / unit * unit;
    for(int64_t s0 = 0; s0 < systems; s0 += ns)
        for(int64_t g0 = 0; g0 < groups; g0 += ng)
        {
            const status st = launch(s0, systems - s0 < ns ? systems - s0 : ns, g0,
                                     groups - g0 < ng ? groups - g0 : ng);
            if(st != status(0))
                return st;
        }
    return status(0);
}

} // namespace rsa
