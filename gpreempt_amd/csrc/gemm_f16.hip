#include "gemm_launch.hpp"

template int gp::launch_typed<_Float16>(const gp::MatPlan &, const gp_preempt_ctx *, gp_stream, gp_launch_info *);
template int gp::launch_group_typed<_Float16>(const gp::MatPlan *, int, const gp_preempt_ctx *, gp_stream, gp_launch_info *);
