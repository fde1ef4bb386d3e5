// Mixed-radix pass kernel, complex transforms, and the choice of instance.
#include "engine.h"
#include "mix_kernel.h"

namespace ifft {

// Measured choice (MI355X).  With three waves per SIMD (168 registers) nothing spills; with four
// the largest radices spill a few.  Workgroups of up to 256 threads run faster with three (float
// r2c rows of 1920 over 16 x 1080: 0.113 ms with four, 0.098 ms with three; 375-point columns 57 ->
// 54 us): several share a CU either way.  Larger ones fit a CU twice only with four (1080-point
// columns 0.186 -> 0.171 ms, odd pairs of 4095 0.105 -> 0.094 ms), unless the grid gives each CU
// one at most (256 rows of 4095: 15.8 us with four, 14.2 us with three).
int mix_wpe(unsigned grid, unsigned block) { return block <= 256 || grid <= 256 ? 3 : 4; }

hipError_t launch_mix_r2c(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s);
hipError_t launch_mix_c2r(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s);

hipError_t launch_fft_mix(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    if (P.load_mode == LD_C2C && P.store_mode == ST_C2C) return launch_mix<LD_C2C, ST_C2C>(P, grid, block, lds, s);
    if (P.load_mode == LD_C2C && P.store_mode == ST_TWIDDLE)
        return launch_mix<LD_C2C, ST_TWIDDLE>(P, grid, block, lds, s);
    if (P.load_mode == LD_C2C || P.store_mode == ST_TWIDDLE) return launch_mix_four(P, grid, block, lds, s);
    if (P.store_mode == ST_R2C_HALF || P.store_mode == ST_R2C_PAIR) return launch_mix_r2c(P, grid, block, lds, s);
    return launch_mix_c2r(P, grid, block, lds, s);
}

}  // namespace ifft
