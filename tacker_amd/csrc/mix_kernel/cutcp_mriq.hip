// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of cutcp with mriq; parameter order = cutcp's GPTB list, then mriq's.

// cutcp-mriq  workgroup split  1 cutcp : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void cutcp_mriq_mix_wg_1_1(
    int cutcp0_binDim_x,
    int cutcp0_binDim_y,
    float* cutcp0_binZeroAddr,
    float cutcp0_h,
    float cutcp0_cutoff2,
    float cutcp0_inv_cutoff2,
    float* cutcp0_regionZeroAddr,
    int cutcp0_zRegionIndex_t,
    int cutcp0_grid_dimension_x,
    int cutcp0_grid_dimension_y,
    int cutcp0_grid_dimension_z,
    int cutcp0_block_dimension_x,
    int cutcp0_block_dimension_y,
    int cutcp0_block_dimension_z,
    int cutcp0_ptb_start_block_pos,
    int cutcp0_ptb_iter_block_step,
    int cutcp0_ptb_end_block_pos,
    int mriq1_numK,
    int mriq1_kGlobalIndex,
    float* mriq1_x,
    float* mriq1_y,
    float* mriq1_z,
    float* mriq1_Qr,
    float* mriq1_Qi,
    int mriq1_grid_dimension_x,
    int mriq1_grid_dimension_y,
    int mriq1_grid_dimension_z,
    int mriq1_block_dimension_x,
    int mriq1_block_dimension_y,
    int mriq1_block_dimension_z,
    int mriq1_ptb_start_block_pos,
    int mriq1_ptb_iter_block_step,
    int mriq1_ptb_end_block_pos)
{
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cutcp-mriq  workgroup split  1 cutcp : 2 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void cutcp_mriq_mix_wg_1_2(
    int cutcp0_binDim_x,
    int cutcp0_binDim_y,
    float* cutcp0_binZeroAddr,
    float cutcp0_h,
    float cutcp0_cutoff2,
    float cutcp0_inv_cutoff2,
    float* cutcp0_regionZeroAddr,
    int cutcp0_zRegionIndex_t,
    int cutcp0_grid_dimension_x,
    int cutcp0_grid_dimension_y,
    int cutcp0_grid_dimension_z,
    int cutcp0_block_dimension_x,
    int cutcp0_block_dimension_y,
    int cutcp0_block_dimension_z,
    int cutcp0_ptb_start_block_pos,
    int cutcp0_ptb_iter_block_step,
    int cutcp0_ptb_end_block_pos,
    int mriq1_numK,
    int mriq1_kGlobalIndex,
    float* mriq1_x,
    float* mriq1_y,
    float* mriq1_z,
    float* mriq1_Qr,
    float* mriq1_Qi,
    int mriq1_grid_dimension_x,
    int mriq1_grid_dimension_y,
    int mriq1_grid_dimension_z,
    int mriq1_block_dimension_x,
    int mriq1_block_dimension_y,
    int mriq1_block_dimension_z,
    int mriq1_ptb_start_block_pos,
    int mriq1_ptb_iter_block_step,
    int mriq1_ptb_end_block_pos)
{
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cutcp-mriq  workgroup split  2 cutcp : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void cutcp_mriq_mix_wg_2_1(
    int cutcp0_binDim_x,
    int cutcp0_binDim_y,
    float* cutcp0_binZeroAddr,
    float cutcp0_h,
    float cutcp0_cutoff2,
    float cutcp0_inv_cutoff2,
    float* cutcp0_regionZeroAddr,
    int cutcp0_zRegionIndex_t,
    int cutcp0_grid_dimension_x,
    int cutcp0_grid_dimension_y,
    int cutcp0_grid_dimension_z,
    int cutcp0_block_dimension_x,
    int cutcp0_block_dimension_y,
    int cutcp0_block_dimension_z,
    int cutcp0_ptb_start_block_pos,
    int cutcp0_ptb_iter_block_step,
    int cutcp0_ptb_end_block_pos,
    int mriq1_numK,
    int mriq1_kGlobalIndex,
    float* mriq1_x,
    float* mriq1_y,
    float* mriq1_z,
    float* mriq1_Qr,
    float* mriq1_Qi,
    int mriq1_grid_dimension_x,
    int mriq1_grid_dimension_y,
    int mriq1_grid_dimension_z,
    int mriq1_block_dimension_x,
    int mriq1_block_dimension_y,
    int mriq1_block_dimension_z,
    int mriq1_ptb_start_block_pos,
    int mriq1_ptb_iter_block_step,
    int mriq1_ptb_end_block_pos)
{
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cutcp-mriq  order split  1 of 2 workgroups start with cutcp, the others with mriq
extern "C" __global__ __launch_bounds__(256) void cutcp_mriq_mix_ord_1_1(
    int cutcp0_binDim_x,
    int cutcp0_binDim_y,
    float* cutcp0_binZeroAddr,
    float cutcp0_h,
    float cutcp0_cutoff2,
    float cutcp0_inv_cutoff2,
    float* cutcp0_regionZeroAddr,
    int cutcp0_zRegionIndex_t,
    int cutcp0_grid_dimension_x,
    int cutcp0_grid_dimension_y,
    int cutcp0_grid_dimension_z,
    int cutcp0_block_dimension_x,
    int cutcp0_block_dimension_y,
    int cutcp0_block_dimension_z,
    int cutcp0_ptb_start_block_pos,
    int cutcp0_ptb_iter_block_step,
    int cutcp0_ptb_end_block_pos,
    int mriq1_numK,
    int mriq1_kGlobalIndex,
    float* mriq1_x,
    float* mriq1_y,
    float* mriq1_z,
    float* mriq1_Qr,
    float* mriq1_Qi,
    int mriq1_grid_dimension_x,
    int mriq1_grid_dimension_y,
    int mriq1_grid_dimension_z,
    int mriq1_block_dimension_x,
    int mriq1_block_dimension_y,
    int mriq1_block_dimension_z,
    int mriq1_ptb_start_block_pos,
    int mriq1_ptb_iter_block_step,
    int mriq1_ptb_end_block_pos)
{
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// cutcp-mriq  order split  1 of 3 workgroups start with cutcp, the others with mriq
extern "C" __global__ __launch_bounds__(256) void cutcp_mriq_mix_ord_1_2(
    int cutcp0_binDim_x,
    int cutcp0_binDim_y,
    float* cutcp0_binZeroAddr,
    float cutcp0_h,
    float cutcp0_cutoff2,
    float cutcp0_inv_cutoff2,
    float* cutcp0_regionZeroAddr,
    int cutcp0_zRegionIndex_t,
    int cutcp0_grid_dimension_x,
    int cutcp0_grid_dimension_y,
    int cutcp0_grid_dimension_z,
    int cutcp0_block_dimension_x,
    int cutcp0_block_dimension_y,
    int cutcp0_block_dimension_z,
    int cutcp0_ptb_start_block_pos,
    int cutcp0_ptb_iter_block_step,
    int cutcp0_ptb_end_block_pos,
    int mriq1_numK,
    int mriq1_kGlobalIndex,
    float* mriq1_x,
    float* mriq1_y,
    float* mriq1_z,
    float* mriq1_Qr,
    float* mriq1_Qi,
    int mriq1_grid_dimension_x,
    int mriq1_grid_dimension_y,
    int mriq1_grid_dimension_z,
    int mriq1_block_dimension_x,
    int mriq1_block_dimension_y,
    int mriq1_block_dimension_z,
    int mriq1_ptb_start_block_pos,
    int mriq1_ptb_iter_block_step,
    int mriq1_ptb_end_block_pos)
{
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// cutcp-mriq  order split  2 of 3 workgroups start with cutcp, the others with mriq
extern "C" __global__ __launch_bounds__(256) void cutcp_mriq_mix_ord_2_1(
    int cutcp0_binDim_x,
    int cutcp0_binDim_y,
    float* cutcp0_binZeroAddr,
    float cutcp0_h,
    float cutcp0_cutoff2,
    float cutcp0_inv_cutoff2,
    float* cutcp0_regionZeroAddr,
    int cutcp0_zRegionIndex_t,
    int cutcp0_grid_dimension_x,
    int cutcp0_grid_dimension_y,
    int cutcp0_grid_dimension_z,
    int cutcp0_block_dimension_x,
    int cutcp0_block_dimension_y,
    int cutcp0_block_dimension_z,
    int cutcp0_ptb_start_block_pos,
    int cutcp0_ptb_iter_block_step,
    int cutcp0_ptb_end_block_pos,
    int mriq1_numK,
    int mriq1_kGlobalIndex,
    float* mriq1_x,
    float* mriq1_y,
    float* mriq1_z,
    float* mriq1_Qr,
    float* mriq1_Qi,
    int mriq1_grid_dimension_x,
    int mriq1_grid_dimension_y,
    int mriq1_grid_dimension_z,
    int mriq1_block_dimension_x,
    int mriq1_block_dimension_y,
    int mriq1_block_dimension_z,
    int mriq1_ptb_start_block_pos,
    int mriq1_ptb_iter_block_step,
    int mriq1_ptb_end_block_pos)
{
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
