// rows_small_kernel for bf16 operands
#include "egs_small_launch.h"

namespace egs {
namespace host {

int launch_rows_small_bf16(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s) { return launch_rows_small_tt<ElemBF16>(j, dw, dwt, s); }

}  // namespace host
}  // namespace egs
