// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of lava with path; parameter order = lava's GPTB list, then path's.

// lava-path  workgroup split  1 lava : 1 path workgroups per group
extern "C" __global__ __launch_bounds__(256) void lava_path_mix_wg_1_1(
    par_str lava0_d_par_gpu,
    dim_str lava0_d_dim_gpu,
    box_str* lava0_d_box_gpu,
    FOUR_VECTOR* lava0_d_rv_gpu,
    float* lava0_d_qv_gpu,
    FOUR_VECTOR* lava0_d_fv_gpu,
    int lava0_grid_dimension_x,
    int lava0_grid_dimension_y,
    int lava0_grid_dimension_z,
    int lava0_block_dimension_x,
    int lava0_block_dimension_y,
    int lava0_block_dimension_z,
    int lava0_ptb_start_block_pos,
    int lava0_ptb_iter_block_step,
    int lava0_ptb_end_block_pos,
    int path1_iteration,
    int* path1_gpuWall,
    int* path1_gpuSrc,
    int* path1_gpuResults,
    int path1_cols,
    int path1_rows,
    int path1_startStep,
    int path1_border,
    int path1_grid_dimension_x,
    int path1_grid_dimension_y,
    int path1_grid_dimension_z,
    int path1_block_dimension_x,
    int path1_block_dimension_y,
    int path1_block_dimension_z,
    int path1_ptb_start_block_pos,
    int path1_ptb_iter_block_step,
    int path1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)path1_rows;
    (void)path1_grid_dimension_x;
    (void)path1_grid_dimension_y;
    (void)path1_grid_dimension_z;
    (void)path1_block_dimension_x;
    (void)path1_block_dimension_y;
    (void)path1_block_dimension_z;
    (void)path1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, sp.role_block, sp.role_blocks, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::path_role(path1_iteration, path1_gpuWall, path1_gpuSrc, path1_gpuResults, path1_cols, path1_startStep, path1_border, sp.role_block, sp.role_blocks, path1_ptb_start_block_pos, path1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lava-path  workgroup split  1 lava : 2 path workgroups per group
extern "C" __global__ __launch_bounds__(256) void lava_path_mix_wg_1_2(
    par_str lava0_d_par_gpu,
    dim_str lava0_d_dim_gpu,
    box_str* lava0_d_box_gpu,
    FOUR_VECTOR* lava0_d_rv_gpu,
    float* lava0_d_qv_gpu,
    FOUR_VECTOR* lava0_d_fv_gpu,
    int lava0_grid_dimension_x,
    int lava0_grid_dimension_y,
    int lava0_grid_dimension_z,
    int lava0_block_dimension_x,
    int lava0_block_dimension_y,
    int lava0_block_dimension_z,
    int lava0_ptb_start_block_pos,
    int lava0_ptb_iter_block_step,
    int lava0_ptb_end_block_pos,
    int path1_iteration,
    int* path1_gpuWall,
    int* path1_gpuSrc,
    int* path1_gpuResults,
    int path1_cols,
    int path1_rows,
    int path1_startStep,
    int path1_border,
    int path1_grid_dimension_x,
    int path1_grid_dimension_y,
    int path1_grid_dimension_z,
    int path1_block_dimension_x,
    int path1_block_dimension_y,
    int path1_block_dimension_z,
    int path1_ptb_start_block_pos,
    int path1_ptb_iter_block_step,
    int path1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)path1_rows;
    (void)path1_grid_dimension_x;
    (void)path1_grid_dimension_y;
    (void)path1_grid_dimension_z;
    (void)path1_block_dimension_x;
    (void)path1_block_dimension_y;
    (void)path1_block_dimension_z;
    (void)path1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, sp.role_block, sp.role_blocks, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::path_role(path1_iteration, path1_gpuWall, path1_gpuSrc, path1_gpuResults, path1_cols, path1_startStep, path1_border, sp.role_block, sp.role_blocks, path1_ptb_start_block_pos, path1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lava-path  workgroup split  2 lava : 1 path workgroups per group
extern "C" __global__ __launch_bounds__(256) void lava_path_mix_wg_2_1(
    par_str lava0_d_par_gpu,
    dim_str lava0_d_dim_gpu,
    box_str* lava0_d_box_gpu,
    FOUR_VECTOR* lava0_d_rv_gpu,
    float* lava0_d_qv_gpu,
    FOUR_VECTOR* lava0_d_fv_gpu,
    int lava0_grid_dimension_x,
    int lava0_grid_dimension_y,
    int lava0_grid_dimension_z,
    int lava0_block_dimension_x,
    int lava0_block_dimension_y,
    int lava0_block_dimension_z,
    int lava0_ptb_start_block_pos,
    int lava0_ptb_iter_block_step,
    int lava0_ptb_end_block_pos,
    int path1_iteration,
    int* path1_gpuWall,
    int* path1_gpuSrc,
    int* path1_gpuResults,
    int path1_cols,
    int path1_rows,
    int path1_startStep,
    int path1_border,
    int path1_grid_dimension_x,
    int path1_grid_dimension_y,
    int path1_grid_dimension_z,
    int path1_block_dimension_x,
    int path1_block_dimension_y,
    int path1_block_dimension_z,
    int path1_ptb_start_block_pos,
    int path1_ptb_iter_block_step,
    int path1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)path1_rows;
    (void)path1_grid_dimension_x;
    (void)path1_grid_dimension_y;
    (void)path1_grid_dimension_z;
    (void)path1_block_dimension_x;
    (void)path1_block_dimension_y;
    (void)path1_block_dimension_z;
    (void)path1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, sp.role_block, sp.role_blocks, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::path_role(path1_iteration, path1_gpuWall, path1_gpuSrc, path1_gpuResults, path1_cols, path1_startStep, path1_border, sp.role_block, sp.role_blocks, path1_ptb_start_block_pos, path1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lava-path  order split  1 of 2 workgroups start with lava, the others with path
extern "C" __global__ __launch_bounds__(256) void lava_path_mix_ord_1_1(
    par_str lava0_d_par_gpu,
    dim_str lava0_d_dim_gpu,
    box_str* lava0_d_box_gpu,
    FOUR_VECTOR* lava0_d_rv_gpu,
    float* lava0_d_qv_gpu,
    FOUR_VECTOR* lava0_d_fv_gpu,
    int lava0_grid_dimension_x,
    int lava0_grid_dimension_y,
    int lava0_grid_dimension_z,
    int lava0_block_dimension_x,
    int lava0_block_dimension_y,
    int lava0_block_dimension_z,
    int lava0_ptb_start_block_pos,
    int lava0_ptb_iter_block_step,
    int lava0_ptb_end_block_pos,
    int path1_iteration,
    int* path1_gpuWall,
    int* path1_gpuSrc,
    int* path1_gpuResults,
    int path1_cols,
    int path1_rows,
    int path1_startStep,
    int path1_border,
    int path1_grid_dimension_x,
    int path1_grid_dimension_y,
    int path1_grid_dimension_z,
    int path1_block_dimension_x,
    int path1_block_dimension_y,
    int path1_block_dimension_z,
    int path1_ptb_start_block_pos,
    int path1_ptb_iter_block_step,
    int path1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)path1_rows;
    (void)path1_grid_dimension_x;
    (void)path1_grid_dimension_y;
    (void)path1_grid_dimension_z;
    (void)path1_block_dimension_x;
    (void)path1_block_dimension_y;
    (void)path1_block_dimension_z;
    (void)path1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::path_role(path1_iteration, path1_gpuWall, path1_gpuSrc, path1_gpuResults, path1_cols, path1_startStep, path1_border, (int)blockIdx.x, (int)gridDim.x, path1_ptb_start_block_pos, path1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// lava-path  order split  1 of 3 workgroups start with lava, the others with path
extern "C" __global__ __launch_bounds__(256) void lava_path_mix_ord_1_2(
    par_str lava0_d_par_gpu,
    dim_str lava0_d_dim_gpu,
    box_str* lava0_d_box_gpu,
    FOUR_VECTOR* lava0_d_rv_gpu,
    float* lava0_d_qv_gpu,
    FOUR_VECTOR* lava0_d_fv_gpu,
    int lava0_grid_dimension_x,
    int lava0_grid_dimension_y,
    int lava0_grid_dimension_z,
    int lava0_block_dimension_x,
    int lava0_block_dimension_y,
    int lava0_block_dimension_z,
    int lava0_ptb_start_block_pos,
    int lava0_ptb_iter_block_step,
    int lava0_ptb_end_block_pos,
    int path1_iteration,
    int* path1_gpuWall,
    int* path1_gpuSrc,
    int* path1_gpuResults,
    int path1_cols,
    int path1_rows,
    int path1_startStep,
    int path1_border,
    int path1_grid_dimension_x,
    int path1_grid_dimension_y,
    int path1_grid_dimension_z,
    int path1_block_dimension_x,
    int path1_block_dimension_y,
    int path1_block_dimension_z,
    int path1_ptb_start_block_pos,
    int path1_ptb_iter_block_step,
    int path1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)path1_rows;
    (void)path1_grid_dimension_x;
    (void)path1_grid_dimension_y;
    (void)path1_grid_dimension_z;
    (void)path1_block_dimension_x;
    (void)path1_block_dimension_y;
    (void)path1_block_dimension_z;
    (void)path1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::path_role(path1_iteration, path1_gpuWall, path1_gpuSrc, path1_gpuResults, path1_cols, path1_startStep, path1_border, (int)blockIdx.x, (int)gridDim.x, path1_ptb_start_block_pos, path1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// lava-path  order split  2 of 3 workgroups start with lava, the others with path
extern "C" __global__ __launch_bounds__(256) void lava_path_mix_ord_2_1(
    par_str lava0_d_par_gpu,
    dim_str lava0_d_dim_gpu,
    box_str* lava0_d_box_gpu,
    FOUR_VECTOR* lava0_d_rv_gpu,
    float* lava0_d_qv_gpu,
    FOUR_VECTOR* lava0_d_fv_gpu,
    int lava0_grid_dimension_x,
    int lava0_grid_dimension_y,
    int lava0_grid_dimension_z,
    int lava0_block_dimension_x,
    int lava0_block_dimension_y,
    int lava0_block_dimension_z,
    int lava0_ptb_start_block_pos,
    int lava0_ptb_iter_block_step,
    int lava0_ptb_end_block_pos,
    int path1_iteration,
    int* path1_gpuWall,
    int* path1_gpuSrc,
    int* path1_gpuResults,
    int path1_cols,
    int path1_rows,
    int path1_startStep,
    int path1_border,
    int path1_grid_dimension_x,
    int path1_grid_dimension_y,
    int path1_grid_dimension_z,
    int path1_block_dimension_x,
    int path1_block_dimension_y,
    int path1_block_dimension_z,
    int path1_ptb_start_block_pos,
    int path1_ptb_iter_block_step,
    int path1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)path1_rows;
    (void)path1_grid_dimension_x;
    (void)path1_grid_dimension_y;
    (void)path1_grid_dimension_z;
    (void)path1_block_dimension_x;
    (void)path1_block_dimension_y;
    (void)path1_block_dimension_z;
    (void)path1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::path_role(path1_iteration, path1_gpuWall, path1_gpuSrc, path1_gpuResults, path1_cols, path1_startStep, path1_border, (int)blockIdx.x, (int)gridDim.x, path1_ptb_start_block_pos, path1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
