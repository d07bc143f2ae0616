// instantiations of the single pass, one element type per file so that they compile side by side
#include "fused_rows.hpp"

namespace nrl {
void launch_fused_bf16(const FusedLaunch& l) { fused_launch<NRL_BF16>(l); }
}  // namespace nrl
