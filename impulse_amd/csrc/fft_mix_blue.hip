// Mixed-radix Bluestein pass (one LDS pass per chirp-z transform).
#include "engine.h"
#include "mix_kernel.h"

namespace ifft {

hipError_t launch_fft_mix_blue(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    switch (P.load_mode) {
        case LD_C2C: return launch_mix_blue<LD_C2C, ST_C2C>(P, grid, block, lds, s);
        case LD_REAL_HALF: return launch_mix_blue<LD_REAL_HALF, ST_R2C_HALF>(P, grid, block, lds, s);
        case LD_R2C_PAIR: return launch_mix_blue<LD_R2C_PAIR, ST_R2C_PAIR>(P, grid, block, lds, s);
        case LD_C2R_HALF: return launch_mix_blue<LD_C2R_HALF, ST_C2R_HALF>(P, grid, block, lds, s);
        default: return launch_mix_blue<LD_C2R_PAIR, ST_C2R_PAIR>(P, grid, block, lds, s);
    }
}

}  // namespace ifft
