// Mixed-radix pass kernel, real to half spectra.
#include "engine.h"
#include "mix_kernel.h"

namespace ifft {

hipError_t launch_mix_r2c(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    if (P.load_mode == LD_REAL_HALF) return launch_mix<LD_REAL_HALF, ST_R2C_HALF>(P, grid, block, lds, s);
    return launch_mix<LD_R2C_PAIR, ST_R2C_PAIR>(P, grid, block, lds, s);
}

}  // namespace ifft
