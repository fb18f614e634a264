// gefenx_step_f16.hip -- the step kernels for fp16 parameters.
#include "gefenx_step_kernels.h"

template struct gx::StepKernels<gx::F16>;
