// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of lava with nn; parameter order = lava's GPTB list, then nn's.

// lava-nn  workgroup split  1 lava : 1 nn workgroups per group
extern "C" __global__ __launch_bounds__(256) void lava_nn_mix_wg_1_1(
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
    LatLong* nn1_d_locations,
    float* nn1_d_distances,
    int nn1_numRecords,
    float nn1_lat,
    float nn1_lng,
    int nn1_grid_dimension_x,
    int nn1_grid_dimension_y,
    int nn1_grid_dimension_z,
    int nn1_block_dimension_x,
    int nn1_block_dimension_y,
    int nn1_block_dimension_z,
    int nn1_ptb_start_block_pos,
    int nn1_ptb_iter_block_step,
    int nn1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)nn1_grid_dimension_z;
    (void)nn1_block_dimension_y;
    (void)nn1_block_dimension_z;
    (void)nn1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, sp.role_block, sp.role_blocks, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::nn_role(nn1_d_locations, nn1_d_distances, nn1_numRecords, nn1_lat, nn1_lng, nn1_grid_dimension_x, nn1_grid_dimension_y, nn1_block_dimension_x, sp.role_block, sp.role_blocks, nn1_ptb_start_block_pos, nn1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lava-nn  workgroup split  1 lava : 2 nn workgroups per group
extern "C" __global__ __launch_bounds__(256) void lava_nn_mix_wg_1_2(
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
    LatLong* nn1_d_locations,
    float* nn1_d_distances,
    int nn1_numRecords,
    float nn1_lat,
    float nn1_lng,
    int nn1_grid_dimension_x,
    int nn1_grid_dimension_y,
    int nn1_grid_dimension_z,
    int nn1_block_dimension_x,
    int nn1_block_dimension_y,
    int nn1_block_dimension_z,
    int nn1_ptb_start_block_pos,
    int nn1_ptb_iter_block_step,
    int nn1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)nn1_grid_dimension_z;
    (void)nn1_block_dimension_y;
    (void)nn1_block_dimension_z;
    (void)nn1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, sp.role_block, sp.role_blocks, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::nn_role(nn1_d_locations, nn1_d_distances, nn1_numRecords, nn1_lat, nn1_lng, nn1_grid_dimension_x, nn1_grid_dimension_y, nn1_block_dimension_x, sp.role_block, sp.role_blocks, nn1_ptb_start_block_pos, nn1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lava-nn  workgroup split  2 lava : 1 nn workgroups per group
extern "C" __global__ __launch_bounds__(256) void lava_nn_mix_wg_2_1(
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
    LatLong* nn1_d_locations,
    float* nn1_d_distances,
    int nn1_numRecords,
    float nn1_lat,
    float nn1_lng,
    int nn1_grid_dimension_x,
    int nn1_grid_dimension_y,
    int nn1_grid_dimension_z,
    int nn1_block_dimension_x,
    int nn1_block_dimension_y,
    int nn1_block_dimension_z,
    int nn1_ptb_start_block_pos,
    int nn1_ptb_iter_block_step,
    int nn1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)nn1_grid_dimension_z;
    (void)nn1_block_dimension_y;
    (void)nn1_block_dimension_z;
    (void)nn1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, sp.role_block, sp.role_blocks, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::nn_role(nn1_d_locations, nn1_d_distances, nn1_numRecords, nn1_lat, nn1_lng, nn1_grid_dimension_x, nn1_grid_dimension_y, nn1_block_dimension_x, sp.role_block, sp.role_blocks, nn1_ptb_start_block_pos, nn1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lava-nn  order split  1 of 2 workgroups start with lava, the others with nn
extern "C" __global__ __launch_bounds__(256) void lava_nn_mix_ord_1_1(
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
    LatLong* nn1_d_locations,
    float* nn1_d_distances,
    int nn1_numRecords,
    float nn1_lat,
    float nn1_lng,
    int nn1_grid_dimension_x,
    int nn1_grid_dimension_y,
    int nn1_grid_dimension_z,
    int nn1_block_dimension_x,
    int nn1_block_dimension_y,
    int nn1_block_dimension_z,
    int nn1_ptb_start_block_pos,
    int nn1_ptb_iter_block_step,
    int nn1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)nn1_grid_dimension_z;
    (void)nn1_block_dimension_y;
    (void)nn1_block_dimension_z;
    (void)nn1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::nn_role(nn1_d_locations, nn1_d_distances, nn1_numRecords, nn1_lat, nn1_lng, nn1_grid_dimension_x, nn1_grid_dimension_y, nn1_block_dimension_x, (int)blockIdx.x, (int)gridDim.x, nn1_ptb_start_block_pos, nn1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// lava-nn  order split  1 of 3 workgroups start with lava, the others with nn
extern "C" __global__ __launch_bounds__(256) void lava_nn_mix_ord_1_2(
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
    LatLong* nn1_d_locations,
    float* nn1_d_distances,
    int nn1_numRecords,
    float nn1_lat,
    float nn1_lng,
    int nn1_grid_dimension_x,
    int nn1_grid_dimension_y,
    int nn1_grid_dimension_z,
    int nn1_block_dimension_x,
    int nn1_block_dimension_y,
    int nn1_block_dimension_z,
    int nn1_ptb_start_block_pos,
    int nn1_ptb_iter_block_step,
    int nn1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)nn1_grid_dimension_z;
    (void)nn1_block_dimension_y;
    (void)nn1_block_dimension_z;
    (void)nn1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::nn_role(nn1_d_locations, nn1_d_distances, nn1_numRecords, nn1_lat, nn1_lng, nn1_grid_dimension_x, nn1_grid_dimension_y, nn1_block_dimension_x, (int)blockIdx.x, (int)gridDim.x, nn1_ptb_start_block_pos, nn1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// lava-nn  order split  2 of 3 workgroups start with lava, the others with nn
extern "C" __global__ __launch_bounds__(256) void lava_nn_mix_ord_2_1(
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
    LatLong* nn1_d_locations,
    float* nn1_d_distances,
    int nn1_numRecords,
    float nn1_lat,
    float nn1_lng,
    int nn1_grid_dimension_x,
    int nn1_grid_dimension_y,
    int nn1_grid_dimension_z,
    int nn1_block_dimension_x,
    int nn1_block_dimension_y,
    int nn1_block_dimension_z,
    int nn1_ptb_start_block_pos,
    int nn1_ptb_iter_block_step,
    int nn1_ptb_end_block_pos)
{
    (void)lava0_grid_dimension_y;
    (void)lava0_grid_dimension_z;
    (void)lava0_block_dimension_x;
    (void)lava0_block_dimension_y;
    (void)lava0_block_dimension_z;
    (void)lava0_ptb_iter_block_step;
    (void)nn1_grid_dimension_z;
    (void)nn1_block_dimension_y;
    (void)nn1_block_dimension_z;
    (void)nn1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lava_role<4>(lava0_d_par_gpu, lava0_d_dim_gpu, lava0_d_box_gpu, lava0_d_rv_gpu, lava0_d_qv_gpu, lava0_d_fv_gpu, lava0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava0_ptb_start_block_pos, lava0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::nn_role(nn1_d_locations, nn1_d_distances, nn1_numRecords, nn1_lat, nn1_lng, nn1_grid_dimension_x, nn1_grid_dimension_y, nn1_block_dimension_x, (int)blockIdx.x, (int)gridDim.x, nn1_ptb_start_block_pos, nn1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
