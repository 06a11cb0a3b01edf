// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of lbm with mrif; parameter order = lbm's GPTB list, then mrif's.

// lbm-mrif  workgroup split  1 lbm : 1 mrif workgroups per group
extern "C" __global__ __launch_bounds__(256) void lbm_mrif_mix_wg_1_1(
    float* lbm0_srcGrid,
    float* lbm0_dstGrid,
    int lbm0_grid_dimension_x,
    int lbm0_grid_dimension_y,
    int lbm0_grid_dimension_z,
    int lbm0_block_dimension_x,
    int lbm0_block_dimension_y,
    int lbm0_block_dimension_z,
    int lbm0_ptb_start_block_pos,
    int lbm0_ptb_iter_block_step,
    int lbm0_ptb_end_block_pos,
    int mrif1_numK,
    int mrif1_kGlobalIndex,
    float* mrif1_x,
    float* mrif1_y,
    float* mrif1_z,
    float* mrif1_outR,
    float* mrif1_outI,
    int mrif1_grid_dimension_x,
    int mrif1_grid_dimension_y,
    int mrif1_grid_dimension_z,
    int mrif1_block_dimension_x,
    int mrif1_block_dimension_y,
    int mrif1_block_dimension_z,
    int mrif1_ptb_start_block_pos,
    int mrif1_ptb_iter_block_step,
    int mrif1_ptb_end_block_pos)
{
    (void)lbm0_grid_dimension_z;
    (void)lbm0_block_dimension_y;
    (void)lbm0_block_dimension_z;
    (void)lbm0_ptb_iter_block_step;
    (void)mrif1_kGlobalIndex;
    (void)mrif1_grid_dimension_z;
    (void)mrif1_block_dimension_x;
    (void)mrif1_block_dimension_y;
    (void)mrif1_block_dimension_z;
    (void)mrif1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::lbm_role(lbm0_srcGrid, lbm0_dstGrid, lbm0_grid_dimension_x, lbm0_grid_dimension_y, lbm0_block_dimension_x, sp.role_block, sp.role_blocks, lbm0_ptb_start_block_pos, lbm0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mrif_role<4>(mrif1_numK, mrif1_x, mrif1_y, mrif1_z, mrif1_outR, mrif1_outI, mrif1_grid_dimension_x, mrif1_grid_dimension_y, sp.role_block, sp.role_blocks, mrif1_ptb_start_block_pos, mrif1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lbm-mrif  workgroup split  1 lbm : 2 mrif workgroups per group
extern "C" __global__ __launch_bounds__(256) void lbm_mrif_mix_wg_1_2(
    float* lbm0_srcGrid,
    float* lbm0_dstGrid,
    int lbm0_grid_dimension_x,
    int lbm0_grid_dimension_y,
    int lbm0_grid_dimension_z,
    int lbm0_block_dimension_x,
    int lbm0_block_dimension_y,
    int lbm0_block_dimension_z,
    int lbm0_ptb_start_block_pos,
    int lbm0_ptb_iter_block_step,
    int lbm0_ptb_end_block_pos,
    int mrif1_numK,
    int mrif1_kGlobalIndex,
    float* mrif1_x,
    float* mrif1_y,
    float* mrif1_z,
    float* mrif1_outR,
    float* mrif1_outI,
    int mrif1_grid_dimension_x,
    int mrif1_grid_dimension_y,
    int mrif1_grid_dimension_z,
    int mrif1_block_dimension_x,
    int mrif1_block_dimension_y,
    int mrif1_block_dimension_z,
    int mrif1_ptb_start_block_pos,
    int mrif1_ptb_iter_block_step,
    int mrif1_ptb_end_block_pos)
{
    (void)lbm0_grid_dimension_z;
    (void)lbm0_block_dimension_y;
    (void)lbm0_block_dimension_z;
    (void)lbm0_ptb_iter_block_step;
    (void)mrif1_kGlobalIndex;
    (void)mrif1_grid_dimension_z;
    (void)mrif1_block_dimension_x;
    (void)mrif1_block_dimension_y;
    (void)mrif1_block_dimension_z;
    (void)mrif1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::lbm_role(lbm0_srcGrid, lbm0_dstGrid, lbm0_grid_dimension_x, lbm0_grid_dimension_y, lbm0_block_dimension_x, sp.role_block, sp.role_blocks, lbm0_ptb_start_block_pos, lbm0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mrif_role<4>(mrif1_numK, mrif1_x, mrif1_y, mrif1_z, mrif1_outR, mrif1_outI, mrif1_grid_dimension_x, mrif1_grid_dimension_y, sp.role_block, sp.role_blocks, mrif1_ptb_start_block_pos, mrif1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lbm-mrif  workgroup split  2 lbm : 1 mrif workgroups per group
extern "C" __global__ __launch_bounds__(256) void lbm_mrif_mix_wg_2_1(
    float* lbm0_srcGrid,
    float* lbm0_dstGrid,
    int lbm0_grid_dimension_x,
    int lbm0_grid_dimension_y,
    int lbm0_grid_dimension_z,
    int lbm0_block_dimension_x,
    int lbm0_block_dimension_y,
    int lbm0_block_dimension_z,
    int lbm0_ptb_start_block_pos,
    int lbm0_ptb_iter_block_step,
    int lbm0_ptb_end_block_pos,
    int mrif1_numK,
    int mrif1_kGlobalIndex,
    float* mrif1_x,
    float* mrif1_y,
    float* mrif1_z,
    float* mrif1_outR,
    float* mrif1_outI,
    int mrif1_grid_dimension_x,
    int mrif1_grid_dimension_y,
    int mrif1_grid_dimension_z,
    int mrif1_block_dimension_x,
    int mrif1_block_dimension_y,
    int mrif1_block_dimension_z,
    int mrif1_ptb_start_block_pos,
    int mrif1_ptb_iter_block_step,
    int mrif1_ptb_end_block_pos)
{
    (void)lbm0_grid_dimension_z;
    (void)lbm0_block_dimension_y;
    (void)lbm0_block_dimension_z;
    (void)lbm0_ptb_iter_block_step;
    (void)mrif1_kGlobalIndex;
    (void)mrif1_grid_dimension_z;
    (void)mrif1_block_dimension_x;
    (void)mrif1_block_dimension_y;
    (void)mrif1_block_dimension_z;
    (void)mrif1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::lbm_role(lbm0_srcGrid, lbm0_dstGrid, lbm0_grid_dimension_x, lbm0_grid_dimension_y, lbm0_block_dimension_x, sp.role_block, sp.role_blocks, lbm0_ptb_start_block_pos, lbm0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mrif_role<4>(mrif1_numK, mrif1_x, mrif1_y, mrif1_z, mrif1_outR, mrif1_outI, mrif1_grid_dimension_x, mrif1_grid_dimension_y, sp.role_block, sp.role_blocks, mrif1_ptb_start_block_pos, mrif1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// lbm-mrif  order split  1 of 2 workgroups start with lbm, the others with mrif
extern "C" __global__ __launch_bounds__(256) void lbm_mrif_mix_ord_1_1(
    float* lbm0_srcGrid,
    float* lbm0_dstGrid,
    int lbm0_grid_dimension_x,
    int lbm0_grid_dimension_y,
    int lbm0_grid_dimension_z,
    int lbm0_block_dimension_x,
    int lbm0_block_dimension_y,
    int lbm0_block_dimension_z,
    int lbm0_ptb_start_block_pos,
    int lbm0_ptb_iter_block_step,
    int lbm0_ptb_end_block_pos,
    int mrif1_numK,
    int mrif1_kGlobalIndex,
    float* mrif1_x,
    float* mrif1_y,
    float* mrif1_z,
    float* mrif1_outR,
    float* mrif1_outI,
    int mrif1_grid_dimension_x,
    int mrif1_grid_dimension_y,
    int mrif1_grid_dimension_z,
    int mrif1_block_dimension_x,
    int mrif1_block_dimension_y,
    int mrif1_block_dimension_z,
    int mrif1_ptb_start_block_pos,
    int mrif1_ptb_iter_block_step,
    int mrif1_ptb_end_block_pos)
{
    (void)lbm0_grid_dimension_z;
    (void)lbm0_block_dimension_y;
    (void)lbm0_block_dimension_z;
    (void)lbm0_ptb_iter_block_step;
    (void)mrif1_kGlobalIndex;
    (void)mrif1_grid_dimension_z;
    (void)mrif1_block_dimension_x;
    (void)mrif1_block_dimension_y;
    (void)mrif1_block_dimension_z;
    (void)mrif1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lbm_role(lbm0_srcGrid, lbm0_dstGrid, lbm0_grid_dimension_x, lbm0_grid_dimension_y, lbm0_block_dimension_x, (int)blockIdx.x, (int)gridDim.x, lbm0_ptb_start_block_pos, lbm0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mrif_role<4>(mrif1_numK, mrif1_x, mrif1_y, mrif1_z, mrif1_outR, mrif1_outI, mrif1_grid_dimension_x, mrif1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif1_ptb_start_block_pos, mrif1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// lbm-mrif  order split  1 of 3 workgroups start with lbm, the others with mrif
extern "C" __global__ __launch_bounds__(256) void lbm_mrif_mix_ord_1_2(
    float* lbm0_srcGrid,
    float* lbm0_dstGrid,
    int lbm0_grid_dimension_x,
    int lbm0_grid_dimension_y,
    int lbm0_grid_dimension_z,
    int lbm0_block_dimension_x,
    int lbm0_block_dimension_y,
    int lbm0_block_dimension_z,
    int lbm0_ptb_start_block_pos,
    int lbm0_ptb_iter_block_step,
    int lbm0_ptb_end_block_pos,
    int mrif1_numK,
    int mrif1_kGlobalIndex,
    float* mrif1_x,
    float* mrif1_y,
    float* mrif1_z,
    float* mrif1_outR,
    float* mrif1_outI,
    int mrif1_grid_dimension_x,
    int mrif1_grid_dimension_y,
    int mrif1_grid_dimension_z,
    int mrif1_block_dimension_x,
    int mrif1_block_dimension_y,
    int mrif1_block_dimension_z,
    int mrif1_ptb_start_block_pos,
    int mrif1_ptb_iter_block_step,
    int mrif1_ptb_end_block_pos)
{
    (void)lbm0_grid_dimension_z;
    (void)lbm0_block_dimension_y;
    (void)lbm0_block_dimension_z;
    (void)lbm0_ptb_iter_block_step;
    (void)mrif1_kGlobalIndex;
    (void)mrif1_grid_dimension_z;
    (void)mrif1_block_dimension_x;
    (void)mrif1_block_dimension_y;
    (void)mrif1_block_dimension_z;
    (void)mrif1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lbm_role(lbm0_srcGrid, lbm0_dstGrid, lbm0_grid_dimension_x, lbm0_grid_dimension_y, lbm0_block_dimension_x, (int)blockIdx.x, (int)gridDim.x, lbm0_ptb_start_block_pos, lbm0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mrif_role<4>(mrif1_numK, mrif1_x, mrif1_y, mrif1_z, mrif1_outR, mrif1_outI, mrif1_grid_dimension_x, mrif1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif1_ptb_start_block_pos, mrif1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// lbm-mrif  order split  2 of 3 workgroups start with lbm, the others with mrif
extern "C" __global__ __launch_bounds__(256) void lbm_mrif_mix_ord_2_1(
    float* lbm0_srcGrid,
    float* lbm0_dstGrid,
    int lbm0_grid_dimension_x,
    int lbm0_grid_dimension_y,
    int lbm0_grid_dimension_z,
    int lbm0_block_dimension_x,
    int lbm0_block_dimension_y,
    int lbm0_block_dimension_z,
    int lbm0_ptb_start_block_pos,
    int lbm0_ptb_iter_block_step,
    int lbm0_ptb_end_block_pos,
    int mrif1_numK,
    int mrif1_kGlobalIndex,
    float* mrif1_x,
    float* mrif1_y,
    float* mrif1_z,
    float* mrif1_outR,
    float* mrif1_outI,
    int mrif1_grid_dimension_x,
    int mrif1_grid_dimension_y,
    int mrif1_grid_dimension_z,
    int mrif1_block_dimension_x,
    int mrif1_block_dimension_y,
    int mrif1_block_dimension_z,
    int mrif1_ptb_start_block_pos,
    int mrif1_ptb_iter_block_step,
    int mrif1_ptb_end_block_pos)
{
    (void)lbm0_grid_dimension_z;
    (void)lbm0_block_dimension_y;
    (void)lbm0_block_dimension_z;
    (void)lbm0_ptb_iter_block_step;
    (void)mrif1_kGlobalIndex;
    (void)mrif1_grid_dimension_z;
    (void)mrif1_block_dimension_x;
    (void)mrif1_block_dimension_y;
    (void)mrif1_block_dimension_z;
    (void)mrif1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::lbm_role(lbm0_srcGrid, lbm0_dstGrid, lbm0_grid_dimension_x, lbm0_grid_dimension_y, lbm0_block_dimension_x, (int)blockIdx.x, (int)gridDim.x, lbm0_ptb_start_block_pos, lbm0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mrif_role<4>(mrif1_numK, mrif1_x, mrif1_y, mrif1_z, mrif1_outR, mrif1_outI, mrif1_grid_dimension_x, mrif1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif1_ptb_start_block_pos, mrif1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
