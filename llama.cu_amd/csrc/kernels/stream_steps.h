// A wave's way through its steps of K with the loads of several steps always on their way.
#pragma once
#include "common.h"

// Steps 0 .. n - 1 with AHEAD steps' loads on their way: fetch(u, i) asks for step i into place u, use(u, i) multiplies it.  No way leads out of the loop, and
// nothing in it is asked for under a condition: the compiler, which counts the loads that it may leave on their way, otherwise waits for all of them once in
// AHEAD steps, and a wave takes a trip to memory for each AHEAD steps.
template <int AHEAD, class Fetch, class Use>
__device__ __forceinline__ void stream_steps(int n, Fetch fetch, Use use) {
    if (n < AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD - 1; ++u)
            if (u < n) fetch(u, u);
#pragma unroll
        for (int u = 0; u < AHEAD - 1; ++u)
            if (u < n) use(u, u);
        return;
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
        fetch(u, u);
        __builtin_amdgcn_sched_barrier(0);           // (out of order, the first places' loads would count as the youngest)
    }
    int i = 0;
    for (; i + 2 * AHEAD <= n; i += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            use(u, i + u);
            fetch(u, i + u + AHEAD);
            __builtin_amdgcn_sched_barrier(0);       // (together, the loads would come behind the last place's use)
        }
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
        use(u, i + u);
        if (i + u + AHEAD < n) fetch(u, i + u + AHEAD);
    }
#pragma unroll
    for (int u = 0; u < AHEAD - 1; ++u)
        if (i + u + AHEAD < n) use(u, i + u + AHEAD);
}
