// MASCOT kernels without the sampled-statistics code (launches in which no rating is sampled).
#include "launch_mascot.h"
#include "rule_mascot.h"

namespace mf {

int launch_mascot_plain(const MascotCall& c, Range r)
{
    // Five workgroups per compute unit at k = 128: the kernel's 80 registers would let six in, and then an epoch of 100M
    // ratings with some groups binary32 takes 14.88 ms instead of 14.75.  Five of 28 KB fit in the 160 KB of LDS, six do not.
    constexpr size_t kFiveWorkgroups = 28u << 10;
    const size_t lds = c.k == 128 && c.lds < kFiveWorkgroups ? kFiveWorkgroups : c.lds;
    return launch_k_coh<MascotPlainRule>(c.who, c.k, c.c, [&](auto a) { return c.fill(a); }, lds, c.stream, r);
}
size_t mascot_table_lds_bytes(uint32_t user_groups, uint32_t item_groups) { return MascotRule<128, true>::lds_bytes(user_groups, item_groups); }

}  // namespace mf
