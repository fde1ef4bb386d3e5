// Mixed-radix pass kernel, the passes of a real four-step that meet the real
// array: twiddled columns of real words, and rows stored as real words.  (The
// columns of half-spectrum bins stay on the generic kernel: two bins and a
// two-level root per point spill here, whatever the grouping.)
//
// Against the generic LDS kernel on the same passes (MI355X): r2c of 64 x 48,000 60 -> 37 us, of 16 x
// 1,000,000 325 -> 224; c2r of 64 x 48,000 76 -> 54, of 16 x 1,000,000 421 -> 308, bound by the columns
// left on that kernel; r2c by one or two rounds of workgroups a pass.
#include "engine.h"
#include "mix_kernel.h"

namespace ifft {

hipError_t launch_mix_four(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    if (P.store_mode == ST_C2R_HALF) return launch_mix<LD_C2C, ST_C2R_HALF>(P, grid, block, lds, s);
    if (P.store_mode == ST_C2R_PAIR) return launch_mix<LD_C2C, ST_C2R_PAIR>(P, grid, block, lds, s);
    if (P.load_mode == LD_REAL_HALF) return launch_mix<LD_REAL_HALF, ST_TWIDDLE>(P, grid, block, lds, s);
    return launch_mix<LD_R2C_PAIR, ST_TWIDDLE>(P, grid, block, lds, s);
}

}  // namespace ifft
