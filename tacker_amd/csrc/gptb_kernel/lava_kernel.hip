// Generated by fusion/code/gen_run.py -- do not edit.
// GPTB form of lava (src/gptb_kernel/lava_kernel.cu:3-140): block positions [ptb_start_block_pos,
// ptb_end_block_pos) served by the ptb_iter_block_step workgroups of the launch.
extern "C" __global__ __launch_bounds__(256, 4) void general_ptb_lava(
    par_str d_par_gpu,
    dim_str d_dim_gpu,
    box_str* d_box_gpu,
    FOUR_VECTOR* d_rv_gpu,
    float* d_qv_gpu,
    FOUR_VECTOR* d_fv_gpu,
    int grid_dimension_x,
    int grid_dimension_y,
    int grid_dimension_z,
    int block_dimension_x,
    int block_dimension_y,
    int block_dimension_z,
    int ptb_start_block_pos,
    int ptb_iter_block_step,
    int ptb_end_block_pos,
    int thread_base)
{
    (void)grid_dimension_y;
    (void)grid_dimension_z;
    (void)block_dimension_x;
    (void)block_dimension_y;
    (void)block_dimension_z;
    tk::lava_role<4>(d_par_gpu, d_dim_gpu, d_box_gpu, d_rv_gpu, d_qv_gpu, d_fv_gpu, grid_dimension_x, (int)blockIdx.x, ptb_iter_block_step, ptb_start_block_pos, ptb_end_block_pos, (int)threadIdx.x - thread_base, (int)blockDim.x);
}
