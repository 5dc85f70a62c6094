// hbem_solve_f32.hip -- the thin solves of hbem_solve.hip for FP32 factors, a
// translation unit of their own so that the two sets of kernels compile side by side.
#define HBEM_SOLVE_F32
#include "hbem_solve.hip"
