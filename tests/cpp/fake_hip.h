// A HIP runtime and kernels of the host, for checks of the runtime's own logic
// (csrc/mlp_runtime.cpp) without a GPU: device memory is host memory, a launch
// runs at once or is recorded by an open capture, and the kernels do only what
// the host logic looks at (a slot's rounds, its active flag, what the last
// round left out).  Counts what was launched and how.
#ifndef FAKE_HIP_H_
#define FAKE_HIP_H_

#include <cstddef>
#include <functional>
#include <vector>

struct Counts {
  int evals = 0;         // launches of k_sweep in a round
  int pruned = 0;        // ... of k_psweep
  int fills = 0;         // ... of k_sweep completing rows
  int eager = 0;         // of these, launched outside a graph
  int instantiated = 0;  // graphs
  int replayed = 0;
  int fused_grid = 0;    // workgroups of the last launch of a fused round, LDS of each
  size_t fused_lds = 0;
  int narrow = 0, wide = 0;  // merges by MLP_MERGE_WIDE
  int worked = 0;        // evaluations of a neighborhood of a slot that did not return at once
};
extern Counts counts;
// rounds after which a slot of N positions finds nothing more
extern std::function<int(int)> rounds_of_slot;
// The stream synchronisation with this number (from 1) fails; 0: none.
extern int fail_sync;
// Whether the slot's last round left rows out and nothing completed them since.
bool left_out(int slot);

#endif  // FAKE_HIP_H_
