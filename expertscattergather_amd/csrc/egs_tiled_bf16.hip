// egs_tiled.h for bf16 operands
#include "egs_tiled_launch.h"

namespace egs {
namespace host {

int tiled_rows_bf16(TiledRowsParams &p, bool w_trans, hipStream_t s)
{
    return w_trans ? launch_tiled<ElemBF16, ElemBF16::ES, true>(p, s) : launch_tiled<ElemBF16, ElemBF16::ES, false>(p, s);
}
int tiled_dw_bf16(TiledDwParams &p, hipStream_t s) { return launch_tiled_dw<ElemBF16>(p, s); }

}  // namespace host
}  // namespace egs
