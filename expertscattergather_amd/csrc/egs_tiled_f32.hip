// egs_tiled.h for f32 operands
#include "egs_tiled_launch.h"

namespace egs {
namespace host {

int tiled_rows_f32(TiledRowsParams &p, bool w_trans, hipStream_t s)
{
    return w_trans ? launch_tiled<ElemF32, ElemF32::ES, true>(p, s) : launch_tiled<ElemF32, ElemF32::ES, false>(p, s);
}
int tiled_dw_f32(TiledDwParams &p, hipStream_t s) { return launch_tiled_dw<ElemF32>(p, s); }

}  // namespace host
}  // namespace egs
