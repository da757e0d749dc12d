// fp32 SGD at k = 128, a file of its own so that the launchers compile in parallel.
#include "hogwild_launch.h"
#include "rules_fp32.h"

namespace mf {

// Six workgroups per compute unit: the kernel's registers would let a seventh in, which buys no time and leaves a sixth more
// updates in flight (single elements of an epoch of 100M ratings then lie 0.66 of the model's root mean square from where
// six leave them).  Six of 24 KB fit in the 160 KB of LDS, seven do not.
constexpr size_t kSixWorkgroups = 24u << 10;

int launch_sgd_k128(const char* who, const Call& c, float* p, float* q, float lrate, float lambda, void* stream)
{
    return launch_coh<128, SgdRule>(who, c, [&](auto a) { a.p = p; a.q = q; a.lrate = lrate; a.lambda = lambda; return a; }, kSixWorkgroups, stream, whole_epoch(c));
}
float inflight_sgd_k128(uint32_t num_workers, uint32_t cap) { return inflight_of<SgdRule<128, true>>(num_workers, kSixWorkgroups, cap); }

}  // namespace mf
