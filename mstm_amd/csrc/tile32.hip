// tile32.hip -- FP32 direct tiles (tile.hpp)
#include "kernels.hpp"
#include "tile.hpp"

template <>
hipError_t launch_direct_tiles<float>(const float *tab, const int2 *tiles, int ntiles, int L, const float *xin,
                                    float *partial, int npad, int nr, int G, int nq, hipStream_t st,
                                    const int *gate)
{
    return tile_dispatch<float>(tab, tiles, ntiles, L, xin, partial, npad, nr, G, nq, st, gate);
}
