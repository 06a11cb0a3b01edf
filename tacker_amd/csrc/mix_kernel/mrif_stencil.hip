// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of mrif with stencil; parameter order = mrif's GPTB list, then stencil's.

// mrif-stencil  workgroup split  1 mrif : 1 stencil workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_stencil_mix_wg_1_1(
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, sp.role_block, sp.role_blocks, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-stencil  workgroup split  1 mrif : 2 stencil workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_stencil_mix_wg_1_2(
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, sp.role_block, sp.role_blocks, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-stencil  workgroup split  2 mrif : 1 stencil workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_stencil_mix_wg_2_1(
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, sp.role_block, sp.role_blocks, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-stencil  order split  1 of 2 workgroups start with mrif, the others with stencil
extern "C" __global__ __launch_bounds__(256) void mrif_stencil_mix_ord_1_1(
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mrif-stencil  order split  1 of 3 workgroups start with mrif, the others with stencil
extern "C" __global__ __launch_bounds__(256) void mrif_stencil_mix_ord_1_2(
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// mrif-stencil  order split  2 of 3 workgroups start with mrif, the others with stencil
extern "C" __global__ __launch_bounds__(256) void mrif_stencil_mix_ord_2_1(
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
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)stencil1_block_dimension_x;
    (void)stencil1_block_dimension_y;
    (void)stencil1_block_dimension_z;
    (void)stencil1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, (int)blockIdx.x, (int)gridDim.x, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::stencil_role(stencil1_c0, stencil1_c1, stencil1_A0, stencil1_Anext, stencil1_nx, stencil1_ny, stencil1_nz, stencil1_grid_dimension_x, stencil1_grid_dimension_y, stencil1_grid_dimension_z, (int)blockIdx.x, (int)gridDim.x, stencil1_ptb_start_block_pos, stencil1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
