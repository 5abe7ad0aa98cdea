#include "mg_strip_impl.hpp"

template int fvx::launch_strip<double, fvx::kDirichlet>(int, int, bool, TileArgs<double>, hipStream_t);
