// fp32 SGD at k = 128, a file of its own so that the launchers compile in parallel.
#include "hogwild_launch.h"
#include "rules_fp32.h"

namespace mf {

int launch_sgd_k128(const char* who, const Call& c, float* p, float* q, float lrate, float lambda, void* stream)
{
    return launch_coh<128, SgdRule>(who, c, [&](auto a) { a.p = p; a.q = q; a.lrate = lrate; a.lambda = lambda; return a; }, 0, stream, whole_epoch(c));
}
float inflight_sgd_k128(uint32_t num_workers, uint32_t cap) { return inflight_of<SgdRule<128, true>>(num_workers, 0, cap); }

}  // namespace mf
