// the LU panels' choice of route (kernels.hpp) on the host
#include "../../mstm_amd/csrc/kernels.hpp"

extern "C" int lu_route_host(int rows, int capacity) { return lu_panel_exchanges(rows, capacity); }
