#include "mg_strip_impl.hpp"

template int fvx::launch_strip<float, fvx::kNoflux>(int, int, bool, TileArgs<float>, hipStream_t);
