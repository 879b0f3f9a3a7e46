// egs_scatter_fused.h for f16 operands
#include "egs_fused_launch.h"

namespace egs {
namespace host {

int launch_fused_f16(const ScatterFusedParams &p, bool w_nmajor, int R, size_t lds, int blocks, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    return w_nmajor ? launch_scatter_fused_ks<ElemF16, true>(p, R, lds, blocks, dw, dwt, s) : launch_scatter_fused_ks<ElemF16, false>(p, R, lds, blocks, dw, dwt, s);
}

}  // namespace host
}  // namespace egs
