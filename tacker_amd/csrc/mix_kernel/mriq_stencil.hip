// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of mriq with stencil; parameter order = mriq's GPTB list, then stencil's.

// mriq-stencil  workgroup split  1 mriq : 1 stencil workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_stencil_mix_wg_1_1(
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
    float stencil1_c0,
    float stencil1_c1,
    float* stencil1_A0,
    float* stencil1_Anext,
    int stencil1_nx,
    int stencil1_ny,
    int stencil1_nz,
    int stencil1_grid_dimension_x,
    int stencil1_grid_dimension_y,
    int stencil1_grid_dimension_z,
    int stencil1_block_dimension_x,
    int stencil1_block_dimension_y,
    int stencil1_block_dimension_z,
    int stencil1_ptb_start_block_pos,
    int stencil1_ptb_iter_block_step,
    int stencil1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, sp.role_block, sp.role_blocks, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-stencil  workgroup split  1 mriq : 2 stencil workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_stencil_mix_wg_1_2(
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
    float stencil1_c0,
    float stencil1_c1,
    float* stencil1_A0,
    float* stencil1_Anext,
    int stencil1_nx,
    int stencil1_ny,
    int stencil1_nz,
    int stencil1_grid_dimension_x,
    int stencil1_grid_dimension_y,
    int stencil1_grid_dimension_z,
    int stencil1_block_dimension_x,
    int stencil1_block_dimension_y,
    int stencil1_block_dimension_z,
    int stencil1_ptb_start_block_pos,
    int stencil1_ptb_iter_block_step,
    int stencil1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, sp.role_block, sp.role_blocks, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-stencil  workgroup split  2 mriq : 1 stencil workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_stencil_mix_wg_2_1(
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
    float stencil1_c0,
    float stencil1_c1,
    float* stencil1_A0,
    float* stencil1_Anext,
    int stencil1_nx,
    int stencil1_ny,
    int stencil1_nz,
    int stencil1_grid_dimension_x,
    int stencil1_grid_dimension_y,
    int stencil1_grid_dimension_z,
    int stencil1_block_dimension_x,
    int stencil1_block_dimension_y,
    int stencil1_block_dimension_z,
    int stencil1_ptb_start_block_pos,
    int stencil1_ptb_iter_block_step,
    int stencil1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, sp.role_block, sp.role_blocks, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-stencil  order split  1 of 2 workgroups start with mriq, the others with stencil
extern "C" __global__ __launch_bounds__(256) void mriq_stencil_mix_ord_1_1(
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
    float stencil1_c0,
    float stencil1_c1,
    float* stencil1_A0,
    float* stencil1_Anext,
    int stencil1_nx,
    int stencil1_ny,
    int stencil1_nz,
    int stencil1_grid_dimension_x,
    int stencil1_grid_dimension_y,
    int stencil1_grid_dimension_z,
    int stencil1_block_dimension_x,
    int stencil1_block_dimension_y,
    int stencil1_block_dimension_z,
    int stencil1_ptb_start_block_pos,
    int stencil1_ptb_iter_block_step,
    int stencil1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mriq-stencil  order split  1 of 3 workgroups start with mriq, the others with stencil
extern "C" __global__ __launch_bounds__(256) void mriq_stencil_mix_ord_1_2(
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
    float stencil1_c0,
    float stencil1_c1,
    float* stencil1_A0,
    float* stencil1_Anext,
    int stencil1_nx,
    int stencil1_ny,
    int stencil1_nz,
    int stencil1_grid_dimension_x,
    int stencil1_grid_dimension_y,
    int stencil1_grid_dimension_z,
    int stencil1_block_dimension_x,
    int stencil1_block_dimension_y,
    int stencil1_block_dimension_z,
    int stencil1_ptb_start_block_pos,
    int stencil1_ptb_iter_block_step,
    int stencil1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mriq-stencil  order split  2 of 3 workgroups start with mriq, the others with stencil
extern "C" __global__ __launch_bounds__(256) void mriq_stencil_mix_ord_2_1(
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
    float stencil1_c0,
    float stencil1_c1,
    float* stencil1_A0,
    float* stencil1_Anext,
    int stencil1_nx,
    int stencil1_ny,
    int stencil1_nz,
    int stencil1_grid_dimension_x,
    int stencil1_grid_dimension_y,
    int stencil1_grid_dimension_z,
    int stencil1_block_dimension_x,
    int stencil1_block_dimension_y,
    int stencil1_block_dimension_z,
    int stencil1_ptb_start_block_pos,
    int stencil1_ptb_iter_block_step,
    int stencil1_ptb_end_block_pos)
{
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
