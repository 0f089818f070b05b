// tile64.hip -- FP64 direct tiles (tile.hpp)
#include "kernels.hpp"
#include "tile.hpp"

template <>
hipError_t launch_direct_tiles<double>(const double *tab, const int2 *tiles, int ntiles, int L, const double *xin,
                                    double *partial, int npad, int nr, int G, int nq, hipStream_t st,
                                    const int *gate)
{
    return tile_dispatch<double>(tab, tiles, ntiles, L, xin, partial, npad, nr, G, nq, st, gate);
}
