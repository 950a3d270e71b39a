// Tiles of up to 256 rows of either kind.
#include "nq_pf_tile.hpp"

namespace nq
{
template int launch_gemm_tg<16, false>(const PfGemm&, int, int, hipStream_t);
template int launch_gemm_tg<16, true>(const PfGemm&, int, int, hipStream_t);
}
