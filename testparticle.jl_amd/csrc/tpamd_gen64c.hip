// tpamd_gen64c.hip -- the generic FP64 kernels of tpamd_gen64.hip, with every
// grid read from its cell-replicated copy.  Kernels of their own: a test of the
// layout in the gather cost solves on nodes up to a tenth (adaptive, FP64).
#include "tpamd_pusher.h"

namespace tpamd {

void launch_generic64_cells(const LaunchReq& r, int alg)
{
    with_launcher(r, [&](const auto& l) {
        if (alg == 0) l.template go<S64C, 0>();
        else l.template go<S64C, 1>();
    });
}

}  // namespace tpamd
