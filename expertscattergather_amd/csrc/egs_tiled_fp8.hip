// egs_tiled.h for bf16 rows and fp8 (e4m3) weights
#include "egs_tiled_launch.h"

namespace egs {
namespace host {

int tiled_rows_fp8w(TiledRowsParams &p, bool w_trans, hipStream_t s)
{
    return w_trans ? launch_tiled<ElemBF16, 1, true>(p, s) : launch_tiled<ElemBF16, 1, false>(p, s);
}

}  // namespace host
}  // namespace egs
