// steps.hip -- the kernels of the forms that a run has on request only, compiled
// from solver.hip as a code object of their own: the persistent form's (k_steps)
// and the paired flux kernels whose workgroups walk several tiles.  The runtime
// loads a code object whole when the first of its kernels is used, and these 74
// are 2.4 of the 4.5 MB of device code: in one object with the others every
// process paid for them on its first launch (a process' first initialize, step
// and read, 2k cells: 10.5 ms before the paired kernels came, 21 with all in one
// object, 13 as it is).
#define MA_STEPS_UNIT
#pragma clang diagnostic ignored "-Wunused-function"  // the other unit's kernels
#include "solver.hip"
