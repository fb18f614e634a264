// gefenx_step_f32.hip -- the step kernels for fp32 parameters.
#include "gefenx_step_kernels.h"

template struct gx::StepKernels<gx::F32>;
