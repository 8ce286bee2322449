// tpamd_pair64.hip -- the FP64 kernels of two gathers a step (see
// tpamd_gridpair.h), double or float storage, cells or nodes.
#include "tpamd_gridpair.h"

namespace {

template <int MODE, bool UXB, typename T>
void go(const LaunchReq& r, bool per, bool cells)
{
    if (cells) per ? launch_pair<S64P<MODE, UXB, true, T, true>>(r) : launch_pair<S64P<MODE, UXB, false, T, true>>(r);
    else per ? launch_pair<S64P<MODE, UXB, true, T, false>>(r) : launch_pair<S64P<MODE, UXB, false, T, false>>(r);
}

}  // namespace

namespace tpamd {

void launch_pair64(const LaunchReq& r, bool time, bool uxb, bool per, bool f32, bool cells)
{
    if (!time) f32 ? go<kPairEB, false, float>(r, per, cells) : go<kPairEB, false, double>(r, per, cells);
    else if (uxb) f32 ? go<kPairTime, true, float>(r, per, cells) : go<kPairTime, true, double>(r, per, cells);
    else f32 ? go<kPairTime, false, float>(r, per, cells) : go<kPairTime, false, double>(r, per, cells);
}

}  // namespace tpamd
