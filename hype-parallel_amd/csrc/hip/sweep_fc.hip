// sweep_fc.hip -- the stage kernel again, compiled with FMA contraction
// (-ffp-contract=on) into its own namespace.  Selected per problem with
// HYPE_OPT_FMA: a*b+c is fused within an expression of the source, which is
// faster and no less accurate, but no longer bitwise equal to the uncontracted
// reference arithmetic (see include/hype2d.h).  The front end decides what is
// fused, from the expression alone, so the kernels of all tile layouts round
// alike.  (-ffp-contract=fast, fusing across expressions wherever instruction
// selection meets the operands in one block, rounded Euler's split tiles unlike
// its one-wave tiles: a small grid's results alone were not those of a batch.
// It is 1 % faster, on the primitive path of Baer-Nunziato 3 %.)  This unit
// holds Euler and Kapila; sweep_fc_bn.hip holds Baer-Nunziato.
#define HYPE_KNS hype_fc
#define HYPE_CONTRACTED_BUILD 1
#include "sweep.hip"
