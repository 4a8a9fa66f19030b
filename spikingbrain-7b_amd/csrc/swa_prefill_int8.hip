// The prompt attention's kernels over INT8 caches, compiled by themselves: their loops start on a cache line (-falign-loops=64). It is where
// the loops happen to lie that takes up to 8 % of the builds for three or seven query heads per kv head (us, as they fell -> aligned: 28 : 4
// heads, 4 x 2048 tokens behind 8000 with 30 decodes 466 -> 446, 1 x 3000 behind 3000 279 -> 269; 12 : 4 140 -> 129; 30 : 10 275 -> 254; the other
// head counts within 2 % either way, 72 calls of nine head counts 0.985 on average). The kernels over elements lose 0.4 to 0.9 % by the same
// alignment, those over fp8 0.1, and go without.
#define SB_PREFILL_INT8
#include "swa_prefill_mfma.hip"
