// egs_tiled.h for f16 operands
#include "egs_tiled_launch.h"

namespace egs {
namespace host {

int tiled_rows_f16(TiledRowsParams &p, bool w_trans, hipStream_t s)
{
    return w_trans ? launch_tiled<ElemF16, ElemF16::ES, true>(p, s) : launch_tiled<ElemF16, ElemF16::ES, false>(p, s);
}
int tiled_dw_f16(TiledDwParams &p, hipStream_t s) { return launch_tiled_dw<ElemF16>(p, s); }

}  // namespace host
}  // namespace egs
