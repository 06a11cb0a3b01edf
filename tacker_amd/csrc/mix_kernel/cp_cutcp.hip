// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of cp with cutcp; parameter order = cp's GPTB list, then cutcp's.

// cp-cutcp  workgroup split  1 cp : 1 cutcp workgroups per group
extern "C" __global__ __launch_bounds__(256) void cp_cutcp_mix_wg_1_1(
    int cp0_numatoms,
    float cp0_gridspacing,
    float* cp0_energygrid,
    int cp0_grid_dimension_x,
    int cp0_grid_dimension_y,
    int cp0_grid_dimension_z,
    int cp0_block_dimension_x,
    int cp0_block_dimension_y,
    int cp0_block_dimension_z,
    int cp0_ptb_start_block_pos,
    int cp0_ptb_iter_block_step,
    int cp0_ptb_end_block_pos,
    int cutcp1_binDim_x,
    int cutcp1_binDim_y,
    float* cutcp1_binZeroAddr,
    float cutcp1_h,
    float cutcp1_cutoff2,
    float cutcp1_inv_cutoff2,
    float* cutcp1_regionZeroAddr,
    int cutcp1_zRegionIndex_t,
    int cutcp1_grid_dimension_x,
    int cutcp1_grid_dimension_y,
    int cutcp1_grid_dimension_z,
    int cutcp1_block_dimension_x,
    int cutcp1_block_dimension_y,
    int cutcp1_block_dimension_z,
    int cutcp1_ptb_start_block_pos,
    int cutcp1_ptb_iter_block_step,
    int cutcp1_ptb_end_block_pos)
{
    (void)cp0_block_dimension_x;
    (void)cp0_block_dimension_y;
    (void)cp0_block_dimension_z;
    (void)cp0_ptb_iter_block_step;
    (void)cutcp1_zRegionIndex_t;
    (void)cutcp1_block_dimension_x;
    (void)cutcp1_block_dimension_y;
    (void)cutcp1_block_dimension_z;
    (void)cutcp1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::cp_role(cp0_numatoms, cp0_gridspacing, cp0_energygrid, cp0_grid_dimension_x, cp0_grid_dimension_y, cp0_grid_dimension_z, sp.role_block, sp.role_blocks, cp0_ptb_start_block_pos, cp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::cutcp_role<4>(cutcp1_binDim_x, cutcp1_binDim_y, cutcp1_binZeroAddr, cutcp1_h, cutcp1_cutoff2, cutcp1_inv_cutoff2, cutcp1_regionZeroAddr, cutcp1_grid_dimension_x, cutcp1_grid_dimension_y, cutcp1_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp1_ptb_start_block_pos, cutcp1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cp-cutcp  workgroup split  1 cp : 2 cutcp workgroups per group
extern "C" __global__ __launch_bounds__(256) void cp_cutcp_mix_wg_1_2(
    int cp0_numatoms,
    float cp0_gridspacing,
    float* cp0_energygrid,
    int cp0_grid_dimension_x,
    int cp0_grid_dimension_y,
    int cp0_grid_dimension_z,
    int cp0_block_dimension_x,
    int cp0_block_dimension_y,
    int cp0_block_dimension_z,
    int cp0_ptb_start_block_pos,
    int cp0_ptb_iter_block_step,
    int cp0_ptb_end_block_pos,
    int cutcp1_binDim_x,
    int cutcp1_binDim_y,
    float* cutcp1_binZeroAddr,
    float cutcp1_h,
    float cutcp1_cutoff2,
    float cutcp1_inv_cutoff2,
    float* cutcp1_regionZeroAddr,
    int cutcp1_zRegionIndex_t,
    int cutcp1_grid_dimension_x,
    int cutcp1_grid_dimension_y,
    int cutcp1_grid_dimension_z,
    int cutcp1_block_dimension_x,
    int cutcp1_block_dimension_y,
    int cutcp1_block_dimension_z,
    int cutcp1_ptb_start_block_pos,
    int cutcp1_ptb_iter_block_step,
    int cutcp1_ptb_end_block_pos)
{
    (void)cp0_block_dimension_x;
    (void)cp0_block_dimension_y;
    (void)cp0_block_dimension_z;
    (void)cp0_ptb_iter_block_step;
    (void)cutcp1_zRegionIndex_t;
    (void)cutcp1_block_dimension_x;
    (void)cutcp1_block_dimension_y;
    (void)cutcp1_block_dimension_z;
    (void)cutcp1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::cp_role(cp0_numatoms, cp0_gridspacing, cp0_energygrid, cp0_grid_dimension_x, cp0_grid_dimension_y, cp0_grid_dimension_z, sp.role_block, sp.role_blocks, cp0_ptb_start_block_pos, cp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::cutcp_role<4>(cutcp1_binDim_x, cutcp1_binDim_y, cutcp1_binZeroAddr, cutcp1_h, cutcp1_cutoff2, cutcp1_inv_cutoff2, cutcp1_regionZeroAddr, cutcp1_grid_dimension_x, cutcp1_grid_dimension_y, cutcp1_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp1_ptb_start_block_pos, cutcp1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cp-cutcp  workgroup split  2 cp : 1 cutcp workgroups per group
extern "C" __global__ __launch_bounds__(256) void cp_cutcp_mix_wg_2_1(
    int cp0_numatoms,
    float cp0_gridspacing,
    float* cp0_energygrid,
    int cp0_grid_dimension_x,
    int cp0_grid_dimension_y,
    int cp0_grid_dimension_z,
    int cp0_block_dimension_x,
    int cp0_block_dimension_y,
    int cp0_block_dimension_z,
    int cp0_ptb_start_block_pos,
    int cp0_ptb_iter_block_step,
    int cp0_ptb_end_block_pos,
    int cutcp1_binDim_x,
    int cutcp1_binDim_y,
    float* cutcp1_binZeroAddr,
    float cutcp1_h,
    float cutcp1_cutoff2,
    float cutcp1_inv_cutoff2,
    float* cutcp1_regionZeroAddr,
    int cutcp1_zRegionIndex_t,
    int cutcp1_grid_dimension_x,
    int cutcp1_grid_dimension_y,
    int cutcp1_grid_dimension_z,
    int cutcp1_block_dimension_x,
    int cutcp1_block_dimension_y,
    int cutcp1_block_dimension_z,
    int cutcp1_ptb_start_block_pos,
    int cutcp1_ptb_iter_block_step,
    int cutcp1_ptb_end_block_pos)
{
    (void)cp0_block_dimension_x;
    (void)cp0_block_dimension_y;
    (void)cp0_block_dimension_z;
    (void)cp0_ptb_iter_block_step;
    (void)cutcp1_zRegionIndex_t;
    (void)cutcp1_block_dimension_x;
    (void)cutcp1_block_dimension_y;
    (void)cutcp1_block_dimension_z;
    (void)cutcp1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::cp_role(cp0_numatoms, cp0_gridspacing, cp0_energygrid, cp0_grid_dimension_x, cp0_grid_dimension_y, cp0_grid_dimension_z, sp.role_block, sp.role_blocks, cp0_ptb_start_block_pos, cp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::cutcp_role<4>(cutcp1_binDim_x, cutcp1_binDim_y, cutcp1_binZeroAddr, cutcp1_h, cutcp1_cutoff2, cutcp1_inv_cutoff2, cutcp1_regionZeroAddr, cutcp1_grid_dimension_x, cutcp1_grid_dimension_y, cutcp1_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp1_ptb_start_block_pos, cutcp1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cp-cutcp  order split  1 of 2 workgroups start with cp, the others with cutcp
extern "C" __global__ __launch_bounds__(256) void cp_cutcp_mix_ord_1_1(
    int cp0_numatoms,
    float cp0_gridspacing,
    float* cp0_energygrid,
    int cp0_grid_dimension_x,
    int cp0_grid_dimension_y,
    int cp0_grid_dimension_z,
    int cp0_block_dimension_x,
    int cp0_block_dimension_y,
    int cp0_block_dimension_z,
    int cp0_ptb_start_block_pos,
    int cp0_ptb_iter_block_step,
    int cp0_ptb_end_block_pos,
    int cutcp1_binDim_x,
    int cutcp1_binDim_y,
    float* cutcp1_binZeroAddr,
    float cutcp1_h,
    float cutcp1_cutoff2,
    float cutcp1_inv_cutoff2,
    float* cutcp1_regionZeroAddr,
    int cutcp1_zRegionIndex_t,
    int cutcp1_grid_dimension_x,
    int cutcp1_grid_dimension_y,
    int cutcp1_grid_dimension_z,
    int cutcp1_block_dimension_x,
    int cutcp1_block_dimension_y,
    int cutcp1_block_dimension_z,
    int cutcp1_ptb_start_block_pos,
    int cutcp1_ptb_iter_block_step,
    int cutcp1_ptb_end_block_pos)
{
    (void)cp0_block_dimension_x;
    (void)cp0_block_dimension_y;
    (void)cp0_block_dimension_z;
    (void)cp0_ptb_iter_block_step;
    (void)cutcp1_zRegionIndex_t;
    (void)cutcp1_block_dimension_x;
    (void)cutcp1_block_dimension_y;
    (void)cutcp1_block_dimension_z;
    (void)cutcp1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::cp_role(cp0_numatoms, cp0_gridspacing, cp0_energygrid, cp0_grid_dimension_x, cp0_grid_dimension_y, cp0_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cp0_ptb_start_block_pos, cp0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::cutcp_role<4>(cutcp1_binDim_x, cutcp1_binDim_y, cutcp1_binZeroAddr, cutcp1_h, cutcp1_cutoff2, cutcp1_inv_cutoff2, cutcp1_regionZeroAddr, cutcp1_grid_dimension_x, cutcp1_grid_dimension_y, cutcp1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cutcp1_ptb_start_block_pos, cutcp1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// cp-cutcp  order split  1 of 3 workgroups start with cp, the others with cutcp
extern "C" __global__ __launch_bounds__(256) void cp_cutcp_mix_ord_1_2(
    int cp0_numatoms,
    float cp0_gridspacing,
    float* cp0_energygrid,
    int cp0_grid_dimension_x,
    int cp0_grid_dimension_y,
    int cp0_grid_dimension_z,
    int cp0_block_dimension_x,
    int cp0_block_dimension_y,
    int cp0_block_dimension_z,
    int cp0_ptb_start_block_pos,
    int cp0_ptb_iter_block_step,
    int cp0_ptb_end_block_pos,
    int cutcp1_binDim_x,
    int cutcp1_binDim_y,
    float* cutcp1_binZeroAddr,
    float cutcp1_h,
    float cutcp1_cutoff2,
    float cutcp1_inv_cutoff2,
    float* cutcp1_regionZeroAddr,
    int cutcp1_zRegionIndex_t,
    int cutcp1_grid_dimension_x,
    int cutcp1_grid_dimension_y,
    int cutcp1_grid_dimension_z,
    int cutcp1_block_dimension_x,
    int cutcp1_block_dimension_y,
    int cutcp1_block_dimension_z,
    int cutcp1_ptb_start_block_pos,
    int cutcp1_ptb_iter_block_step,
    int cutcp1_ptb_end_block_pos)
{
    (void)cp0_block_dimension_x;
    (void)cp0_block_dimension_y;
    (void)cp0_block_dimension_z;
    (void)cp0_ptb_iter_block_step;
    (void)cutcp1_zRegionIndex_t;
    (void)cutcp1_block_dimension_x;
    (void)cutcp1_block_dimension_y;
    (void)cutcp1_block_dimension_z;
    (void)cutcp1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::cp_role(cp0_numatoms, cp0_gridspacing, cp0_energygrid, cp0_grid_dimension_x, cp0_grid_dimension_y, cp0_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cp0_ptb_start_block_pos, cp0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::cutcp_role<4>(cutcp1_binDim_x, cutcp1_binDim_y, cutcp1_binZeroAddr, cutcp1_h, cutcp1_cutoff2, cutcp1_inv_cutoff2, cutcp1_regionZeroAddr, cutcp1_grid_dimension_x, cutcp1_grid_dimension_y, cutcp1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cutcp1_ptb_start_block_pos, cutcp1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// cp-cutcp  order split  2 of 3 workgroups start with cp, the others with cutcp
extern "C" __global__ __launch_bounds__(256) void cp_cutcp_mix_ord_2_1(
    int cp0_numatoms,
    float cp0_gridspacing,
    float* cp0_energygrid,
    int cp0_grid_dimension_x,
    int cp0_grid_dimension_y,
    int cp0_grid_dimension_z,
    int cp0_block_dimension_x,
    int cp0_block_dimension_y,
    int cp0_block_dimension_z,
    int cp0_ptb_start_block_pos,
    int cp0_ptb_iter_block_step,
    int cp0_ptb_end_block_pos,
    int cutcp1_binDim_x,
    int cutcp1_binDim_y,
    float* cutcp1_binZeroAddr,
    float cutcp1_h,
    float cutcp1_cutoff2,
    float cutcp1_inv_cutoff2,
    float* cutcp1_regionZeroAddr,
    int cutcp1_zRegionIndex_t,
    int cutcp1_grid_dimension_x,
    int cutcp1_grid_dimension_y,
    int cutcp1_grid_dimension_z,
    int cutcp1_block_dimension_x,
    int cutcp1_block_dimension_y,
    int cutcp1_block_dimension_z,
    int cutcp1_ptb_start_block_pos,
    int cutcp1_ptb_iter_block_step,
    int cutcp1_ptb_end_block_pos)
{
    (void)cp0_block_dimension_x;
    (void)cp0_block_dimension_y;
    (void)cp0_block_dimension_z;
    (void)cp0_ptb_iter_block_step;
    (void)cutcp1_zRegionIndex_t;
    (void)cutcp1_block_dimension_x;
    (void)cutcp1_block_dimension_y;
    (void)cutcp1_block_dimension_z;
    (void)cutcp1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::cp_role(cp0_numatoms, cp0_gridspacing, cp0_energygrid, cp0_grid_dimension_x, cp0_grid_dimension_y, cp0_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cp0_ptb_start_block_pos, cp0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::cutcp_role<4>(cutcp1_binDim_x, cutcp1_binDim_y, cutcp1_binZeroAddr, cutcp1_h, cutcp1_cutoff2, cutcp1_inv_cutoff2, cutcp1_regionZeroAddr, cutcp1_grid_dimension_x, cutcp1_grid_dimension_y, cutcp1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cutcp1_ptb_start_block_pos, cutcp1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
