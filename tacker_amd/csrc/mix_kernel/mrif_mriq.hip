// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of mrif with mriq; parameter order = mrif's GPTB list, then mriq's.

// mrif-mriq  workgroup split  1 mrif : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_mriq_mix_wg_1_1(
    int mrif0_numK,
    int mrif0_kGlobalIndex,
    float* mrif0_x,
    float* mrif0_y,
    float* mrif0_z,
    float* mrif0_outR,
    float* mrif0_outI,
    int mrif0_grid_dimension_x,
    int mrif0_grid_dimension_y,
    int mrif0_grid_dimension_z,
    int mrif0_block_dimension_x,
    int mrif0_block_dimension_y,
    int mrif0_block_dimension_z,
    int mrif0_ptb_start_block_pos,
    int mrif0_ptb_iter_block_step,
    int mrif0_ptb_end_block_pos,
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-mriq  workgroup split  1 mrif : 2 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_mriq_mix_wg_1_2(
    int mrif0_numK,
    int mrif0_kGlobalIndex,
    float* mrif0_x,
    float* mrif0_y,
    float* mrif0_z,
    float* mrif0_outR,
    float* mrif0_outI,
    int mrif0_grid_dimension_x,
    int mrif0_grid_dimension_y,
    int mrif0_grid_dimension_z,
    int mrif0_block_dimension_x,
    int mrif0_block_dimension_y,
    int mrif0_block_dimension_z,
    int mrif0_ptb_start_block_pos,
    int mrif0_ptb_iter_block_step,
    int mrif0_ptb_end_block_pos,
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-mriq  workgroup split  2 mrif : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_mriq_mix_wg_2_1(
    int mrif0_numK,
    int mrif0_kGlobalIndex,
    float* mrif0_x,
    float* mrif0_y,
    float* mrif0_z,
    float* mrif0_outR,
    float* mrif0_outI,
    int mrif0_grid_dimension_x,
    int mrif0_grid_dimension_y,
    int mrif0_grid_dimension_z,
    int mrif0_block_dimension_x,
    int mrif0_block_dimension_y,
    int mrif0_block_dimension_z,
    int mrif0_ptb_start_block_pos,
    int mrif0_ptb_iter_block_step,
    int mrif0_ptb_end_block_pos,
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-mriq  order split  1 of 2 workgroups start with mrif, the others with mriq
extern "C" __global__ __launch_bounds__(256) void mrif_mriq_mix_ord_1_1(
    int mrif0_numK,
    int mrif0_kGlobalIndex,
    float* mrif0_x,
    float* mrif0_y,
    float* mrif0_z,
    float* mrif0_outR,
    float* mrif0_outI,
    int mrif0_grid_dimension_x,
    int mrif0_grid_dimension_y,
    int mrif0_grid_dimension_z,
    int mrif0_block_dimension_x,
    int mrif0_block_dimension_y,
    int mrif0_block_dimension_z,
    int mrif0_ptb_start_block_pos,
    int mrif0_ptb_iter_block_step,
    int mrif0_ptb_end_block_pos,
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mrif-mriq  order split  1 of 3 workgroups start with mrif, the others with mriq
extern "C" __global__ __launch_bounds__(256) void mrif_mriq_mix_ord_1_2(
    int mrif0_numK,
    int mrif0_kGlobalIndex,
    float* mrif0_x,
    float* mrif0_y,
    float* mrif0_z,
    float* mrif0_outR,
    float* mrif0_outI,
    int mrif0_grid_dimension_x,
    int mrif0_grid_dimension_y,
    int mrif0_grid_dimension_z,
    int mrif0_block_dimension_x,
    int mrif0_block_dimension_y,
    int mrif0_block_dimension_z,
    int mrif0_ptb_start_block_pos,
    int mrif0_ptb_iter_block_step,
    int mrif0_ptb_end_block_pos,
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mrif-mriq  order split  2 of 3 workgroups start with mrif, the others with mriq
extern "C" __global__ __launch_bounds__(256) void mrif_mriq_mix_ord_2_1(
    int mrif0_numK,
    int mrif0_kGlobalIndex,
    float* mrif0_x,
    float* mrif0_y,
    float* mrif0_z,
    float* mrif0_outR,
    float* mrif0_outI,
    int mrif0_grid_dimension_x,
    int mrif0_grid_dimension_y,
    int mrif0_grid_dimension_z,
    int mrif0_block_dimension_x,
    int mrif0_block_dimension_y,
    int mrif0_block_dimension_z,
    int mrif0_ptb_start_block_pos,
    int mrif0_ptb_iter_block_step,
    int mrif0_ptb_end_block_pos,
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
