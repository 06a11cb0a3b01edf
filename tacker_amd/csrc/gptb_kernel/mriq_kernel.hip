// Generated by fusion/code/gen_run.py -- do not edit.
// GPTB form of mriq (src/gptb_kernel/mriq_kernel.cu:3-70): block positions [ptb_start_block_pos,
// ptb_end_block_pos) served by the ptb_iter_block_step workgroups of the launch.
extern "C" __global__ void g_general_ptb_mriq(
    int numK,
    int kGlobalIndex,
    float* x,
    float* y,
    float* z,
    float* Qr,
    float* Qi,
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
    (void)kGlobalIndex;
    (void)grid_dimension_z;
    (void)block_dimension_x;
    (void)block_dimension_y;
    (void)block_dimension_z;
    tk::mriq_role<16>(numK, x, y, z, Qr, Qi, grid_dimension_x, grid_dimension_y, (int)blockIdx.x, ptb_iter_block_step, ptb_start_block_pos, ptb_end_block_pos, (int)threadIdx.x - thread_base, (int)blockDim.x);
}
