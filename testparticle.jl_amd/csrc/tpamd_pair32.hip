// tpamd_pair32.hip -- the FP32C kernels of two gathers a step (see
// tpamd_gridpair.h), float storage, cells or nodes.
#include "tpamd_gridpair.h"

namespace {

template <int MODE, bool UXB>
void go(const LaunchReq& r, bool per, bool cells)
{
    if (cells) per ? launch_pair<S32P<MODE, UXB, true, true>>(r) : launch_pair<S32P<MODE, UXB, false, true>>(r);
    else per ? launch_pair<S32P<MODE, UXB, true, false>>(r) : launch_pair<S32P<MODE, UXB, false, false>>(r);
}

}  // namespace

namespace tpamd {

void launch_pair32(const LaunchReq& r, bool time, bool uxb, bool per, bool cells)
{
    if (!time) go<kPairEB, false>(r, per, cells);
    else if (uxb) go<kPairTime, true>(r, per, cells);
    else go<kPairTime, false>(r, per, cells);
}

}  // namespace tpamd
