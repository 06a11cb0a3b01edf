// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of fft with mriq; parameter order = fft's GPTB list, then mriq's.

// fft-mriq  workgroup split  1 fft : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void fft_mriq_mix_wg_1_1(
    float* fft0_data,
    int fft0_grid_dimension_x,
    int fft0_grid_dimension_y,
    int fft0_grid_dimension_z,
    int fft0_block_dimension_x,
    int fft0_block_dimension_y,
    int fft0_block_dimension_z,
    int fft0_ptb_start_block_pos,
    int fft0_ptb_iter_block_step,
    int fft0_ptb_end_block_pos,
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
    (void)fft0_grid_dimension_y;
    (void)fft0_grid_dimension_z;
    (void)fft0_block_dimension_x;
    (void)fft0_block_dimension_y;
    (void)fft0_block_dimension_z;
    (void)fft0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::fft_role<4>(fft0_data, fft0_grid_dimension_x, sp.role_block, sp.role_blocks, fft0_ptb_start_block_pos, fft0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// fft-mriq  workgroup split  1 fft : 2 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void fft_mriq_mix_wg_1_2(
    float* fft0_data,
    int fft0_grid_dimension_x,
    int fft0_grid_dimension_y,
    int fft0_grid_dimension_z,
    int fft0_block_dimension_x,
    int fft0_block_dimension_y,
    int fft0_block_dimension_z,
    int fft0_ptb_start_block_pos,
    int fft0_ptb_iter_block_step,
    int fft0_ptb_end_block_pos,
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
    (void)fft0_grid_dimension_y;
    (void)fft0_grid_dimension_z;
    (void)fft0_block_dimension_x;
    (void)fft0_block_dimension_y;
    (void)fft0_block_dimension_z;
    (void)fft0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::fft_role<4>(fft0_data, fft0_grid_dimension_x, sp.role_block, sp.role_blocks, fft0_ptb_start_block_pos, fft0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// fft-mriq  workgroup split  2 fft : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void fft_mriq_mix_wg_2_1(
    float* fft0_data,
    int fft0_grid_dimension_x,
    int fft0_grid_dimension_y,
    int fft0_grid_dimension_z,
    int fft0_block_dimension_x,
    int fft0_block_dimension_y,
    int fft0_block_dimension_z,
    int fft0_ptb_start_block_pos,
    int fft0_ptb_iter_block_step,
    int fft0_ptb_end_block_pos,
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
    (void)fft0_grid_dimension_y;
    (void)fft0_grid_dimension_z;
    (void)fft0_block_dimension_x;
    (void)fft0_block_dimension_y;
    (void)fft0_block_dimension_z;
    (void)fft0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::fft_role<4>(fft0_data, fft0_grid_dimension_x, sp.role_block, sp.role_blocks, fft0_ptb_start_block_pos, fft0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, sp.role_block, sp.role_blocks, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// fft-mriq  order split  1 of 2 workgroups start with fft, the others with mriq
extern "C" __global__ __launch_bounds__(256) void fft_mriq_mix_ord_1_1(
    float* fft0_data,
    int fft0_grid_dimension_x,
    int fft0_grid_dimension_y,
    int fft0_grid_dimension_z,
    int fft0_block_dimension_x,
    int fft0_block_dimension_y,
    int fft0_block_dimension_z,
    int fft0_ptb_start_block_pos,
    int fft0_ptb_iter_block_step,
    int fft0_ptb_end_block_pos,
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
    (void)fft0_grid_dimension_y;
    (void)fft0_grid_dimension_z;
    (void)fft0_block_dimension_x;
    (void)fft0_block_dimension_y;
    (void)fft0_block_dimension_z;
    (void)fft0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::fft_role<4>(fft0_data, fft0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, fft0_ptb_start_block_pos, fft0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// fft-mriq  order split  1 of 3 workgroups start with fft, the others with mriq
extern "C" __global__ __launch_bounds__(256) void fft_mriq_mix_ord_1_2(
    float* fft0_data,
    int fft0_grid_dimension_x,
    int fft0_grid_dimension_y,
    int fft0_grid_dimension_z,
    int fft0_block_dimension_x,
    int fft0_block_dimension_y,
    int fft0_block_dimension_z,
    int fft0_ptb_start_block_pos,
    int fft0_ptb_iter_block_step,
    int fft0_ptb_end_block_pos,
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
    (void)fft0_grid_dimension_y;
    (void)fft0_grid_dimension_z;
    (void)fft0_block_dimension_x;
    (void)fft0_block_dimension_y;
    (void)fft0_block_dimension_z;
    (void)fft0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::fft_role<4>(fft0_data, fft0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, fft0_ptb_start_block_pos, fft0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// fft-mriq  order split  2 of 3 workgroups start with fft, the others with mriq
extern "C" __global__ __launch_bounds__(256) void fft_mriq_mix_ord_2_1(
    float* fft0_data,
    int fft0_grid_dimension_x,
    int fft0_grid_dimension_y,
    int fft0_grid_dimension_z,
    int fft0_block_dimension_x,
    int fft0_block_dimension_y,
    int fft0_block_dimension_z,
    int fft0_ptb_start_block_pos,
    int fft0_ptb_iter_block_step,
    int fft0_ptb_end_block_pos,
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
    (void)fft0_grid_dimension_y;
    (void)fft0_grid_dimension_z;
    (void)fft0_block_dimension_x;
    (void)fft0_block_dimension_y;
    (void)fft0_block_dimension_z;
    (void)fft0_ptb_iter_block_step;
    (void)mriq1_kGlobalIndex;
    (void)mriq1_grid_dimension_z;
    (void)mriq1_block_dimension_x;
    (void)mriq1_block_dimension_y;
    (void)mriq1_block_dimension_z;
    (void)mriq1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::fft_role<4>(fft0_data, fft0_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, fft0_ptb_start_block_pos, fft0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::mriq_role<4>(mriq1_numK, mriq1_x, mriq1_y, mriq1_z, mriq1_Qr, mriq1_Qi, mriq1_grid_dimension_x, mriq1_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq1_ptb_start_block_pos, mriq1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
