// gefenx_step_bf16.hip -- the step kernels for bf16 parameters.
#include "gefenx_step_kernels.h"

template struct gx::StepKernels<gx::BF16>;
