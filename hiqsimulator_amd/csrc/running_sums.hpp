// Running sums of block probabilities, as a workgroup forms them: every thread
// has a run of consecutive blocks, a tree scan over the threads' sums gives where
// its run ends.  The scan rounds in another order than the sums inside a run, so
// the two ends of neighbouring runs can be ulps apart, in either direction.  A
// search for the first running sum above u must not find a block of probability
// zero there, so:
//   * the end of a run is the largest scan value up to it of a run that holds
//     anything (an empty run ends where the one before it does);
//   * a run's sums stop at its end, and its last block that holds anything takes
//     what is left.
// Then running sums never fall and are equal over empty blocks.  NaN stays NaN.
#pragma once

#include <hip/hip_runtime.h>

namespace hq {

// One thread's run, over its blocks in order.
struct BlockRun {
     double sum = 0.0;
     int last = -1;  // its last block that holds anything
     __host__ __device__ void add(double p, int i)
     {
          sum += p;
          if (!(p <= 0.0)) last = i;
     }
     // Where the run ends by itself; `scan`: the tree's sum up to and with it.
     __host__ __device__ double end(double scan) const { return last < 0 ? 0.0 : scan; }
};

// The larger one; NaN if either is.
__host__ __device__ inline double larger(double a, double b) { return a > b || a != a ? a : b; }

// What is stored for block i of a run: `run`, the sum up to and with it from the
// previous run's end, limited by this run's `end`.
__host__ __device__ inline double running_sum(double run, int i, int last, double end)
{
     return i < last && !(run > end) ? run : end;
}

}  // namespace hq
