// The row tiles that may have up to 288 rows (row_tiles_kernel<.., EITHER = true>), a unit of their own: their loops begin at the first byte of
// a line of 64 (build.py).  Where the first instruction of a step lies depends else on all the code in front of it, and the step on that: 4096 rows
// in 8 groups, 4096 x 14336, us, with the same loop 32, 4, 24, 28 and 48 bytes into a line 253.0, 254.3, 255.9, 256.2 and 259.0; in another run 247.0
// with 32, 248.8 with 4, 250.4 with 28, and 247.8 at its beginning in two builds whose code in front differs.  The tiles of 256 rows do not gain by it
// (a training step of 8191 tokens to 4 of 60 experts 1693 -> 1697).
#define AAMD_ROW_TILES_HIGHER
#include "gemm_rows.hip"
