// Tiles of up to 128 rows of experts in mask mode or with a base window code other than 0.
#include "nq_pf_tile.hpp"

namespace nq { template int launch_tiles<true>(const PfGemm&, int, int, hipStream_t); }
