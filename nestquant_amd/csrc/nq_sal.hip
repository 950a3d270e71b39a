// Decode salience export as a launch of its own (reference sm120/nqsal.cu:19-78, called at sm120/serve/nq_vllm.py:558,572): at most 8
// tokens of 8 picks per call, no host synchronisation, static pointers, so the call can sit in a captured decode step. A layer
// call can carry it in its routing launch instead (NqMoeArgs.with_salience), where it costs nothing: this launch is 5 us of
// latency (9.4 us with one wavefront per token and the picks' sums as a chain of lane exchanges).
#include "nq_sal.hpp"
#include "nq_host.hpp"

namespace nq {

__global__ void __launch_bounds__(512) nq_sal_k(SalArgs a)
{
    __shared__ SalShared S;
    salience<8>(a, &S);
}

int launch_sal(const void* x, int x_dtype, int64_t sx, const void* w, int w_dtype, const void* ids, int ids_dtype, int T, int H, int K,
               int E, float rsf, double* acc, double* host, hipStream_t st)
{
    SalArgs a{x, sx, w, ids, T, H, K, E, x_dtype, w_dtype, ids_dtype, rsf, acc, host};
    nq_sal_k<<<1, 512, 0, st>>>(a);
    NQ_LAUNCH_CHECK("nq_sal");
    return 0;
}

}  // namespace nq
