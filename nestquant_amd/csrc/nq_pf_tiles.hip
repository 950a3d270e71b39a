// Tiles of up to 128 rows of plain experts (every chunk refined, base window code 0).
#include "nq_pf_tile.hpp"

namespace nq { template int launch_tiles<false>(const PfGemm&, int, int, hipStream_t); }
