// Launches the small workgroups of the power-of-two kernel on the stand-in HIP runtime, on grids that no
// plan asks for, and prints what each launch was: the modes that the per-point path lacks are either
// their own instance or refused.
#include <cstdio>
#include <cstring>

#include "fft_params.h"

namespace ifft {
hipError_t launch_fft_pow2(const FftParams &P, int map, unsigned grid, unsigned block, size_t lds, hipStream_t s);
}
extern "C" const char *standin_launches();

int main()
{
    const int maps[] = {0, 1, 2};   // rows, columns, rows loaded and columns stored
    for (int store : {(int)ifft::ST_CONV_TWIDDLE, (int)ifft::ST_R2C_ROWPAIR})
        for (int map : maps)
            for (unsigned grid : {8u, 1000000u}) {
                ifft::FftParams P;
                std::memset(&P, 0, sizeof(P));
                P.N = 512;
                P.NT = 32;
                P.TB = map == 0 ? 2 : 4;   // a wavefront; four transforms where the lanes walk across them
                P.load_mode = ifft::LD_C2C;
                P.store_mode = store;
                const hipError_t e = ifft::launch_fft_pow2(P, map, grid, (unsigned)(P.TB * P.NT), 8192, nullptr);
                const char *l = standin_launches();
                std::printf("%d %d %u %d %s", store == ifft::ST_CONV_TWIDDLE, map, grid, (int)e, *l ? l : "-\n");
            }
    return 0;
}
