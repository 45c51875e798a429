// Phase kernels for f32 inputs (a translation unit per type: they compile side by side).
#include "phase_kernels.h"

namespace hot {
template int phase_launch_impl<float>(int, ColSel, const PhaseArgs&, size_t, hipStream_t);
}
