// The persistent decode step of step.hip for BF16 weights.
#define ITTS_STEP_BF16
#include "step.hip"
