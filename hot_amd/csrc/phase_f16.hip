// Phase kernels for f16 inputs (a translation unit per type: they compile side by side).
#include "phase_kernels.h"

namespace hot {
template int phase_launch_impl<f16_t>(int, ColSel, const PhaseArgs&, size_t, hipStream_t);
}
