// Generated by fusion/code/gen_run.py -- do not edit.
// GPTB form of cutcp (src/gptb_kernel/cutcp_kernel.cu:12-183): block positions [ptb_start_block_pos,
// ptb_end_block_pos) served by the ptb_iter_block_step workgroups of the launch.
extern "C" __global__ void general_ptb_cutcp(
    int binDim_x,
    int binDim_y,
    float* binZeroAddr,
    float h,
    float cutoff2,
    float inv_cutoff2,
    float* regionZeroAddr,
    int zRegionIndex_t,
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
    (void)zRegionIndex_t;
    (void)block_dimension_x;
    (void)block_dimension_y;
    (void)block_dimension_z;
    tk::cutcp_role<4>(binDim_x, binDim_y, binZeroAddr, h, cutoff2, inv_cutoff2, regionZeroAddr, grid_dimension_x, grid_dimension_y, grid_dimension_z, (int)blockIdx.x, ptb_iter_block_step, ptb_start_block_pos, ptb_end_block_pos, (int)threadIdx.x - thread_base, (int)blockDim.x);
}
