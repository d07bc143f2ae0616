// instantiations of the single pass, one element type per file so that they compile side by side
#include "fused_rows.hpp"

namespace nrl {
void launch_fused_f32(const FusedLaunch& l) { fused_launch<NRL_F32>(l); }
}  // namespace nrl
