// Mixed-radix pass kernel, half spectra to real.
#include "engine.h"
#include "mix_kernel.h"

namespace ifft {

hipError_t launch_mix_c2r(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    if (P.load_mode == LD_C2R_HALF) return launch_mix<LD_C2R_HALF, ST_C2R_HALF>(P, grid, block, lds, s);
    return launch_mix<LD_C2R_PAIR, ST_C2R_PAIR>(P, grid, block, lds, s);
}

}  // namespace ifft
