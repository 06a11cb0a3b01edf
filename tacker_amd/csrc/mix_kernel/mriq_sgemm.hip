// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of mriq with sgemm; parameter order = mriq's GPTB list, then sgemm's.

// mriq-sgemm  workgroup split  1 mriq : 1 sgemm workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_sgemm_mix_wg_1_1(
    int mriq0_numK,
    int mriq0_kGlobalIndex,
    float* mriq0_x,
    float* mriq0_y,
    float* mriq0_z,
    float* mriq0_Qr,
    float* mriq0_Qi,
    int mriq0_grid_dimension_x,
    int mriq0_grid_dimension_y,
    int mriq0_grid_dimension_z,
    int mriq0_block_dimension_x,
    int mriq0_block_dimension_y,
    int mriq0_block_dimension_z,
    int mriq0_ptb_start_block_pos,
    int mriq0_ptb_iter_block_step,
    int mriq0_ptb_end_block_pos,
    float* sgemm1_A,
    float* sgemm1_B,
    float* sgemm1_C,
    int sgemm1_NORMAL_M,
    int sgemm1_NORMAL_N,
    int sgemm1_NORMAL_K,
    int sgemm1_grid_dimension_x,
    int sgemm1_grid_dimension_y,
    int sgemm1_grid_dimension_z,
    int sgemm1_block_dimension_x,
    int sgemm1_block_dimension_y,
    int sgemm1_block_dimension_z,
    int sgemm1_ptb_start_block_pos,
    int sgemm1_ptb_iter_block_step,
    int sgemm1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)sgemm1_block_dimension_x;
    (void)sgemm1_block_dimension_y;
    (void)sgemm1_block_dimension_z;
    (void)sgemm1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::sgemm_role(sgemm1_A, sgemm1_B, sgemm1_C, sgemm1_NORMAL_M, sgemm1_NORMAL_N, sgemm1_NORMAL_K, sgemm1_grid_dimension_x, sgemm1_grid_dimension_y, sgemm1_grid_dimension_z, sp.role_block, sp.role_blocks, sgemm1_ptb_start_block_pos, sgemm1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-sgemm  workgroup split  1 mriq : 2 sgemm workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_sgemm_mix_wg_1_2(
    int mriq0_numK,
    int mriq0_kGlobalIndex,
    float* mriq0_x,
    float* mriq0_y,
    float* mriq0_z,
    float* mriq0_Qr,
    float* mriq0_Qi,
    int mriq0_grid_dimension_x,
    int mriq0_grid_dimension_y,
    int mriq0_grid_dimension_z,
    int mriq0_block_dimension_x,
    int mriq0_block_dimension_y,
    int mriq0_block_dimension_z,
    int mriq0_ptb_start_block_pos,
    int mriq0_ptb_iter_block_step,
    int mriq0_ptb_end_block_pos,
    float* sgemm1_A,
    float* sgemm1_B,
    float* sgemm1_C,
    int sgemm1_NORMAL_M,
    int sgemm1_NORMAL_N,
    int sgemm1_NORMAL_K,
    int sgemm1_grid_dimension_x,
    int sgemm1_grid_dimension_y,
    int sgemm1_grid_dimension_z,
    int sgemm1_block_dimension_x,
    int sgemm1_block_dimension_y,
    int sgemm1_block_dimension_z,
    int sgemm1_ptb_start_block_pos,
    int sgemm1_ptb_iter_block_step,
    int sgemm1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)sgemm1_block_dimension_x;
    (void)sgemm1_block_dimension_y;
    (void)sgemm1_block_dimension_z;
    (void)sgemm1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::sgemm_role(sgemm1_A, sgemm1_B, sgemm1_C, sgemm1_NORMAL_M, sgemm1_NORMAL_N, sgemm1_NORMAL_K, sgemm1_grid_dimension_x, sgemm1_grid_dimension_y, sgemm1_grid_dimension_z, sp.role_block, sp.role_blocks, sgemm1_ptb_start_block_pos, sgemm1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-sgemm  workgroup split  2 mriq : 1 sgemm workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_sgemm_mix_wg_2_1(
    int mriq0_numK,
    int mriq0_kGlobalIndex,
    float* mriq0_x,
    float* mriq0_y,
    float* mriq0_z,
    float* mriq0_Qr,
    float* mriq0_Qi,
    int mriq0_grid_dimension_x,
    int mriq0_grid_dimension_y,
    int mriq0_grid_dimension_z,
    int mriq0_block_dimension_x,
    int mriq0_block_dimension_y,
    int mriq0_block_dimension_z,
    int mriq0_ptb_start_block_pos,
    int mriq0_ptb_iter_block_step,
    int mriq0_ptb_end_block_pos,
    float* sgemm1_A,
    float* sgemm1_B,
    float* sgemm1_C,
    int sgemm1_NORMAL_M,
    int sgemm1_NORMAL_N,
    int sgemm1_NORMAL_K,
    int sgemm1_grid_dimension_x,
    int sgemm1_grid_dimension_y,
    int sgemm1_grid_dimension_z,
    int sgemm1_block_dimension_x,
    int sgemm1_block_dimension_y,
    int sgemm1_block_dimension_z,
    int sgemm1_ptb_start_block_pos,
    int sgemm1_ptb_iter_block_step,
    int sgemm1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)sgemm1_block_dimension_x;
    (void)sgemm1_block_dimension_y;
    (void)sgemm1_block_dimension_z;
    (void)sgemm1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::sgemm_role(sgemm1_A, sgemm1_B, sgemm1_C, sgemm1_NORMAL_M, sgemm1_NORMAL_N, sgemm1_NORMAL_K, sgemm1_grid_dimension_x, sgemm1_grid_dimension_y, sgemm1_grid_dimension_z, sp.role_block, sp.role_blocks, sgemm1_ptb_start_block_pos, sgemm1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-sgemm  order split  1 of 2 workgroups start with mriq, the others with sgemm
extern "C" __global__ __launch_bounds__(256) void mriq_sgemm_mix_ord_1_1(
    int mriq0_numK,
    int mriq0_kGlobalIndex,
    float* mriq0_x,
    float* mriq0_y,
    float* mriq0_z,
    float* mriq0_Qr,
    float* mriq0_Qi,
    int mriq0_grid_dimension_x,
    int mriq0_grid_dimension_y,
    int mriq0_grid_dimension_z,
    int mriq0_block_dimension_x,
    int mriq0_block_dimension_y,
    int mriq0_block_dimension_z,
    int mriq0_ptb_start_block_pos,
    int mriq0_ptb_iter_block_step,
    int mriq0_ptb_end_block_pos,
    float* sgemm1_A,
    float* sgemm1_B,
    float* sgemm1_C,
    int sgemm1_NORMAL_M,
    int sgemm1_NORMAL_N,
    int sgemm1_NORMAL_K,
    int sgemm1_grid_dimension_x,
    int sgemm1_grid_dimension_y,
    int sgemm1_grid_dimension_z,
    int sgemm1_block_dimension_x,
    int sgemm1_block_dimension_y,
    int sgemm1_block_dimension_z,
    int sgemm1_ptb_start_block_pos,
    int sgemm1_ptb_iter_block_step,
    int sgemm1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)sgemm1_block_dimension_x;
    (void)sgemm1_block_dimension_y;
    (void)sgemm1_block_dimension_z;
    (void)sgemm1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::sgemm_role(sgemm1_A, sgemm1_B, sgemm1_C, sgemm1_NORMAL_M, sgemm1_NORMAL_N, sgemm1_NORMAL_K, sgemm1_grid_dimension_x, sgemm1_grid_dimension_y, sgemm1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, sgemm1_ptb_start_block_pos, sgemm1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mriq-sgemm  order split  1 of 3 workgroups start with mriq, the others with sgemm
extern "C" __global__ __launch_bounds__(256) void mriq_sgemm_mix_ord_1_2(
    int mriq0_numK,
    int mriq0_kGlobalIndex,
    float* mriq0_x,
    float* mriq0_y,
    float* mriq0_z,
    float* mriq0_Qr,
    float* mriq0_Qi,
    int mriq0_grid_dimension_x,
    int mriq0_grid_dimension_y,
    int mriq0_grid_dimension_z,
    int mriq0_block_dimension_x,
    int mriq0_block_dimension_y,
    int mriq0_block_dimension_z,
    int mriq0_ptb_start_block_pos,
    int mriq0_ptb_iter_block_step,
    int mriq0_ptb_end_block_pos,
    float* sgemm1_A,
    float* sgemm1_B,
    float* sgemm1_C,
    int sgemm1_NORMAL_M,
    int sgemm1_NORMAL_N,
    int sgemm1_NORMAL_K,
    int sgemm1_grid_dimension_x,
    int sgemm1_grid_dimension_y,
    int sgemm1_grid_dimension_z,
    int sgemm1_block_dimension_x,
    int sgemm1_block_dimension_y,
    int sgemm1_block_dimension_z,
    int sgemm1_ptb_start_block_pos,
    int sgemm1_ptb_iter_block_step,
    int sgemm1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)sgemm1_block_dimension_x;
    (void)sgemm1_block_dimension_y;
    (void)sgemm1_block_dimension_z;
    (void)sgemm1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::sgemm_role(sgemm1_A, sgemm1_B, sgemm1_C, sgemm1_NORMAL_M, sgemm1_NORMAL_N, sgemm1_NORMAL_K, sgemm1_grid_dimension_x, sgemm1_grid_dimension_y, sgemm1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, sgemm1_ptb_start_block_pos, sgemm1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mriq-sgemm  order split  2 of 3 workgroups start with mriq, the others with sgemm
extern "C" __global__ __launch_bounds__(256) void mriq_sgemm_mix_ord_2_1(
    int mriq0_numK,
    int mriq0_kGlobalIndex,
    float* mriq0_x,
    float* mriq0_y,
    float* mriq0_z,
    float* mriq0_Qr,
    float* mriq0_Qi,
    int mriq0_grid_dimension_x,
    int mriq0_grid_dimension_y,
    int mriq0_grid_dimension_z,
    int mriq0_block_dimension_x,
    int mriq0_block_dimension_y,
    int mriq0_block_dimension_z,
    int mriq0_ptb_start_block_pos,
    int mriq0_ptb_iter_block_step,
    int mriq0_ptb_end_block_pos,
    float* sgemm1_A,
    float* sgemm1_B,
    float* sgemm1_C,
    int sgemm1_NORMAL_M,
    int sgemm1_NORMAL_N,
    int sgemm1_NORMAL_K,
    int sgemm1_grid_dimension_x,
    int sgemm1_grid_dimension_y,
    int sgemm1_grid_dimension_z,
    int sgemm1_block_dimension_x,
    int sgemm1_block_dimension_y,
    int sgemm1_block_dimension_z,
    int sgemm1_ptb_start_block_pos,
    int sgemm1_ptb_iter_block_step,
    int sgemm1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)sgemm1_block_dimension_x;
    (void)sgemm1_block_dimension_y;
    (void)sgemm1_block_dimension_z;
    (void)sgemm1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::sgemm_role(sgemm1_A, sgemm1_B, sgemm1_C, sgemm1_NORMAL_M, sgemm1_NORMAL_N, sgemm1_NORMAL_K, sgemm1_grid_dimension_x, sgemm1_grid_dimension_y, sgemm1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, sgemm1_ptb_start_block_pos, sgemm1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
