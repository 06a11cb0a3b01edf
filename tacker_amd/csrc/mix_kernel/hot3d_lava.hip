// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of hot3d with lava; parameter order = hot3d's GPTB list, then lava's.

// hot3d-lava  workgroup split  1 hot3d : 1 lava workgroups per group
extern "C" __global__ __launch_bounds__(256) void hot3d_lava_mix_wg_1_1(
    float* hot3d0_p,
    float* hot3d0_tIn,
    float* hot3d0_tOut,
    float hot3d0_sdc,
    int hot3d0_nx,
    int hot3d0_ny,
    int hot3d0_nz,
    float hot3d0_ce,
    float hot3d0_cw,
    float hot3d0_cn,
    float hot3d0_cs,
    float hot3d0_ct,
    float hot3d0_cb,
    float hot3d0_cc,
    int hot3d0_grid_dimension_x,
    int hot3d0_grid_dimension_y,
    int hot3d0_grid_dimension_z,
    int hot3d0_block_dimension_x,
    int hot3d0_block_dimension_y,
    int hot3d0_block_dimension_z,
    int hot3d0_ptb_start_block_pos,
    int hot3d0_ptb_iter_block_step,
    int hot3d0_ptb_end_block_pos,
    par_str lava1_d_par_gpu,
    dim_str lava1_d_dim_gpu,
    box_str* lava1_d_box_gpu,
    FOUR_VECTOR* lava1_d_rv_gpu,
    float* lava1_d_qv_gpu,
    FOUR_VECTOR* lava1_d_fv_gpu,
    int lava1_grid_dimension_x,
    int lava1_grid_dimension_y,
    int lava1_grid_dimension_z,
    int lava1_block_dimension_x,
    int lava1_block_dimension_y,
    int lava1_block_dimension_z,
    int lava1_ptb_start_block_pos,
    int lava1_ptb_iter_block_step,
    int lava1_ptb_end_block_pos)
{
    (void)hot3d0_grid_dimension_z;
    (void)hot3d0_block_dimension_z;
    (void)hot3d0_ptb_iter_block_step;
    (void)lava1_grid_dimension_y;
    (void)lava1_grid_dimension_z;
    (void)lava1_block_dimension_x;
    (void)lava1_block_dimension_y;
    (void)lava1_block_dimension_z;
    (void)lava1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::hot3d_role(hot3d0_p, hot3d0_tIn, hot3d0_tOut, hot3d0_sdc, hot3d0_nx, hot3d0_ny, hot3d0_nz, hot3d0_ce, hot3d0_cw, hot3d0_cn, hot3d0_cs, hot3d0_ct, hot3d0_cb, hot3d0_cc, hot3d0_grid_dimension_x, hot3d0_grid_dimension_y, hot3d0_block_dimension_x, hot3d0_block_dimension_y, sp.role_block, sp.role_blocks, hot3d0_ptb_start_block_pos, hot3d0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::lava_role<4>(lava1_d_par_gpu, lava1_d_dim_gpu, lava1_d_box_gpu, lava1_d_rv_gpu, lava1_d_qv_gpu, lava1_d_fv_gpu, lava1_grid_dimension_x, sp.role_block, sp.role_blocks, lava1_ptb_start_block_pos, lava1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// hot3d-lava  workgroup split  1 hot3d : 2 lava workgroups per group
extern "C" __global__ __launch_bounds__(256) void hot3d_lava_mix_wg_1_2(
    float* hot3d0_p,
    float* hot3d0_tIn,
    float* hot3d0_tOut,
    float hot3d0_sdc,
    int hot3d0_nx,
    int hot3d0_ny,
    int hot3d0_nz,
    float hot3d0_ce,
    float hot3d0_cw,
    float hot3d0_cn,
    float hot3d0_cs,
    float hot3d0_ct,
    float hot3d0_cb,
    float hot3d0_cc,
    int hot3d0_grid_dimension_x,
    int hot3d0_grid_dimension_y,
    int hot3d0_grid_dimension_z,
    int hot3d0_block_dimension_x,
    int hot3d0_block_dimension_y,
    int hot3d0_block_dimension_z,
    int hot3d0_ptb_start_block_pos,
    int hot3d0_ptb_iter_block_step,
    int hot3d0_ptb_end_block_pos,
    par_str lava1_d_par_gpu,
    dim_str lava1_d_dim_gpu,
    box_str* lava1_d_box_gpu,
    FOUR_VECTOR* lava1_d_rv_gpu,
    float* lava1_d_qv_gpu,
    FOUR_VECTOR* lava1_d_fv_gpu,
    int lava1_grid_dimension_x,
    int lava1_grid_dimension_y,
    int lava1_grid_dimension_z,
    int lava1_block_dimension_x,
    int lava1_block_dimension_y,
    int lava1_block_dimension_z,
    int lava1_ptb_start_block_pos,
    int lava1_ptb_iter_block_step,
    int lava1_ptb_end_block_pos)
{
    (void)hot3d0_grid_dimension_z;
    (void)hot3d0_block_dimension_z;
    (void)hot3d0_ptb_iter_block_step;
    (void)lava1_grid_dimension_y;
    (void)lava1_grid_dimension_z;
    (void)lava1_block_dimension_x;
    (void)lava1_block_dimension_y;
    (void)lava1_block_dimension_z;
    (void)lava1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::hot3d_role(hot3d0_p, hot3d0_tIn, hot3d0_tOut, hot3d0_sdc, hot3d0_nx, hot3d0_ny, hot3d0_nz, hot3d0_ce, hot3d0_cw, hot3d0_cn, hot3d0_cs, hot3d0_ct, hot3d0_cb, hot3d0_cc, hot3d0_grid_dimension_x, hot3d0_grid_dimension_y, hot3d0_block_dimension_x, hot3d0_block_dimension_y, sp.role_block, sp.role_blocks, hot3d0_ptb_start_block_pos, hot3d0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::lava_role<4>(lava1_d_par_gpu, lava1_d_dim_gpu, lava1_d_box_gpu, lava1_d_rv_gpu, lava1_d_qv_gpu, lava1_d_fv_gpu, lava1_grid_dimension_x, sp.role_block, sp.role_blocks, lava1_ptb_start_block_pos, lava1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// hot3d-lava  workgroup split  2 hot3d : 1 lava workgroups per group
extern "C" __global__ __launch_bounds__(256) void hot3d_lava_mix_wg_2_1(
    float* hot3d0_p,
    float* hot3d0_tIn,
    float* hot3d0_tOut,
    float hot3d0_sdc,
    int hot3d0_nx,
    int hot3d0_ny,
    int hot3d0_nz,
    float hot3d0_ce,
    float hot3d0_cw,
    float hot3d0_cn,
    float hot3d0_cs,
    float hot3d0_ct,
    float hot3d0_cb,
    float hot3d0_cc,
    int hot3d0_grid_dimension_x,
    int hot3d0_grid_dimension_y,
    int hot3d0_grid_dimension_z,
    int hot3d0_block_dimension_x,
    int hot3d0_block_dimension_y,
    int hot3d0_block_dimension_z,
    int hot3d0_ptb_start_block_pos,
    int hot3d0_ptb_iter_block_step,
    int hot3d0_ptb_end_block_pos,
    par_str lava1_d_par_gpu,
    dim_str lava1_d_dim_gpu,
    box_str* lava1_d_box_gpu,
    FOUR_VECTOR* lava1_d_rv_gpu,
    float* lava1_d_qv_gpu,
    FOUR_VECTOR* lava1_d_fv_gpu,
    int lava1_grid_dimension_x,
    int lava1_grid_dimension_y,
    int lava1_grid_dimension_z,
    int lava1_block_dimension_x,
    int lava1_block_dimension_y,
    int lava1_block_dimension_z,
    int lava1_ptb_start_block_pos,
    int lava1_ptb_iter_block_step,
    int lava1_ptb_end_block_pos)
{
    (void)hot3d0_grid_dimension_z;
    (void)hot3d0_block_dimension_z;
    (void)hot3d0_ptb_iter_block_step;
    (void)lava1_grid_dimension_y;
    (void)lava1_grid_dimension_z;
    (void)lava1_block_dimension_x;
    (void)lava1_block_dimension_y;
    (void)lava1_block_dimension_z;
    (void)lava1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    if (sp.role == 0) {
        tk::hot3d_role(hot3d0_p, hot3d0_tIn, hot3d0_tOut, hot3d0_sdc, hot3d0_nx, hot3d0_ny, hot3d0_nz, hot3d0_ce, hot3d0_cw, hot3d0_cn, hot3d0_cs, hot3d0_ct, hot3d0_cb, hot3d0_cc, hot3d0_grid_dimension_x, hot3d0_grid_dimension_y, hot3d0_block_dimension_x, hot3d0_block_dimension_y, sp.role_block, sp.role_blocks, hot3d0_ptb_start_block_pos, hot3d0_ptb_end_block_pos, (int)threadIdx.x, 256);
    } else {
        tk::lava_role<4>(lava1_d_par_gpu, lava1_d_dim_gpu, lava1_d_box_gpu, lava1_d_rv_gpu, lava1_d_qv_gpu, lava1_d_fv_gpu, lava1_grid_dimension_x, sp.role_block, sp.role_blocks, lava1_ptb_start_block_pos, lava1_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// hot3d-lava  order split  1 of 2 workgroups start with hot3d, the others with lava
extern "C" __global__ __launch_bounds__(256) void hot3d_lava_mix_ord_1_1(
    float* hot3d0_p,
    float* hot3d0_tIn,
    float* hot3d0_tOut,
    float hot3d0_sdc,
    int hot3d0_nx,
    int hot3d0_ny,
    int hot3d0_nz,
    float hot3d0_ce,
    float hot3d0_cw,
    float hot3d0_cn,
    float hot3d0_cs,
    float hot3d0_ct,
    float hot3d0_cb,
    float hot3d0_cc,
    int hot3d0_grid_dimension_x,
    int hot3d0_grid_dimension_y,
    int hot3d0_grid_dimension_z,
    int hot3d0_block_dimension_x,
    int hot3d0_block_dimension_y,
    int hot3d0_block_dimension_z,
    int hot3d0_ptb_start_block_pos,
    int hot3d0_ptb_iter_block_step,
    int hot3d0_ptb_end_block_pos,
    par_str lava1_d_par_gpu,
    dim_str lava1_d_dim_gpu,
    box_str* lava1_d_box_gpu,
    FOUR_VECTOR* lava1_d_rv_gpu,
    float* lava1_d_qv_gpu,
    FOUR_VECTOR* lava1_d_fv_gpu,
    int lava1_grid_dimension_x,
    int lava1_grid_dimension_y,
    int lava1_grid_dimension_z,
    int lava1_block_dimension_x,
    int lava1_block_dimension_y,
    int lava1_block_dimension_z,
    int lava1_ptb_start_block_pos,
    int lava1_ptb_iter_block_step,
    int lava1_ptb_end_block_pos)
{
    (void)hot3d0_grid_dimension_z;
    (void)hot3d0_block_dimension_z;
    (void)hot3d0_ptb_iter_block_step;
    (void)lava1_grid_dimension_y;
    (void)lava1_grid_dimension_z;
    (void)lava1_block_dimension_x;
    (void)lava1_block_dimension_y;
    (void)lava1_block_dimension_z;
    (void)lava1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::hot3d_role(hot3d0_p, hot3d0_tIn, hot3d0_tOut, hot3d0_sdc, hot3d0_nx, hot3d0_ny, hot3d0_nz, hot3d0_ce, hot3d0_cw, hot3d0_cn, hot3d0_cs, hot3d0_ct, hot3d0_cb, hot3d0_cc, hot3d0_grid_dimension_x, hot3d0_grid_dimension_y, hot3d0_block_dimension_x, hot3d0_block_dimension_y, (int)blockIdx.x, (int)gridDim.x, hot3d0_ptb_start_block_pos, hot3d0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::lava_role<4>(lava1_d_par_gpu, lava1_d_dim_gpu, lava1_d_box_gpu, lava1_d_rv_gpu, lava1_d_qv_gpu, lava1_d_fv_gpu, lava1_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava1_ptb_start_block_pos, lava1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// hot3d-lava  order split  1 of 3 workgroups start with hot3d, the others with lava
extern "C" __global__ __launch_bounds__(256) void hot3d_lava_mix_ord_1_2(
    float* hot3d0_p,
    float* hot3d0_tIn,
    float* hot3d0_tOut,
    float hot3d0_sdc,
    int hot3d0_nx,
    int hot3d0_ny,
    int hot3d0_nz,
    float hot3d0_ce,
    float hot3d0_cw,
    float hot3d0_cn,
    float hot3d0_cs,
    float hot3d0_ct,
    float hot3d0_cb,
    float hot3d0_cc,
    int hot3d0_grid_dimension_x,
    int hot3d0_grid_dimension_y,
    int hot3d0_grid_dimension_z,
    int hot3d0_block_dimension_x,
    int hot3d0_block_dimension_y,
    int hot3d0_block_dimension_z,
    int hot3d0_ptb_start_block_pos,
    int hot3d0_ptb_iter_block_step,
    int hot3d0_ptb_end_block_pos,
    par_str lava1_d_par_gpu,
    dim_str lava1_d_dim_gpu,
    box_str* lava1_d_box_gpu,
    FOUR_VECTOR* lava1_d_rv_gpu,
    float* lava1_d_qv_gpu,
    FOUR_VECTOR* lava1_d_fv_gpu,
    int lava1_grid_dimension_x,
    int lava1_grid_dimension_y,
    int lava1_grid_dimension_z,
    int lava1_block_dimension_x,
    int lava1_block_dimension_y,
    int lava1_block_dimension_z,
    int lava1_ptb_start_block_pos,
    int lava1_ptb_iter_block_step,
    int lava1_ptb_end_block_pos)
{
    (void)hot3d0_grid_dimension_z;
    (void)hot3d0_block_dimension_z;
    (void)hot3d0_ptb_iter_block_step;
    (void)lava1_grid_dimension_y;
    (void)lava1_grid_dimension_z;
    (void)lava1_block_dimension_x;
    (void)lava1_block_dimension_y;
    (void)lava1_block_dimension_z;
    (void)lava1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::hot3d_role(hot3d0_p, hot3d0_tIn, hot3d0_tOut, hot3d0_sdc, hot3d0_nx, hot3d0_ny, hot3d0_nz, hot3d0_ce, hot3d0_cw, hot3d0_cn, hot3d0_cs, hot3d0_ct, hot3d0_cb, hot3d0_cc, hot3d0_grid_dimension_x, hot3d0_grid_dimension_y, hot3d0_block_dimension_x, hot3d0_block_dimension_y, (int)blockIdx.x, (int)gridDim.x, hot3d0_ptb_start_block_pos, hot3d0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::lava_role<4>(lava1_d_par_gpu, lava1_d_dim_gpu, lava1_d_box_gpu, lava1_d_rv_gpu, lava1_d_qv_gpu, lava1_d_fv_gpu, lava1_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava1_ptb_start_block_pos, lava1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}

// hot3d-lava  order split  2 of 3 workgroups start with hot3d, the others with lava
extern "C" __global__ __launch_bounds__(256) void hot3d_lava_mix_ord_2_1(
    float* hot3d0_p,
    float* hot3d0_tIn,
    float* hot3d0_tOut,
    float hot3d0_sdc,
    int hot3d0_nx,
    int hot3d0_ny,
    int hot3d0_nz,
    float hot3d0_ce,
    float hot3d0_cw,
    float hot3d0_cn,
    float hot3d0_cs,
    float hot3d0_ct,
    float hot3d0_cb,
    float hot3d0_cc,
    int hot3d0_grid_dimension_x,
    int hot3d0_grid_dimension_y,
    int hot3d0_grid_dimension_z,
    int hot3d0_block_dimension_x,
    int hot3d0_block_dimension_y,
    int hot3d0_block_dimension_z,
    int hot3d0_ptb_start_block_pos,
    int hot3d0_ptb_iter_block_step,
    int hot3d0_ptb_end_block_pos,
    par_str lava1_d_par_gpu,
    dim_str lava1_d_dim_gpu,
    box_str* lava1_d_box_gpu,
    FOUR_VECTOR* lava1_d_rv_gpu,
    float* lava1_d_qv_gpu,
    FOUR_VECTOR* lava1_d_fv_gpu,
    int lava1_grid_dimension_x,
    int lava1_grid_dimension_y,
    int lava1_grid_dimension_z,
    int lava1_block_dimension_x,
    int lava1_block_dimension_y,
    int lava1_block_dimension_z,
    int lava1_ptb_start_block_pos,
    int lava1_ptb_iter_block_step,
    int lava1_ptb_end_block_pos)
{
    (void)hot3d0_grid_dimension_z;
    (void)hot3d0_block_dimension_z;
    (void)hot3d0_ptb_iter_block_step;
    (void)lava1_grid_dimension_y;
    (void)lava1_grid_dimension_z;
    (void)lava1_block_dimension_x;
    (void)lava1_block_dimension_y;
    (void)lava1_block_dimension_z;
    (void)lava1_ptb_iter_block_step;
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 2, 1);
    for (int phase = 0; phase < 2; ++phase) {
        if ((sp.role ^ phase) == 0) {
            tk::hot3d_role(hot3d0_p, hot3d0_tIn, hot3d0_tOut, hot3d0_sdc, hot3d0_nx, hot3d0_ny, hot3d0_nz, hot3d0_ce, hot3d0_cw, hot3d0_cn, hot3d0_cs, hot3d0_ct, hot3d0_cb, hot3d0_cc, hot3d0_grid_dimension_x, hot3d0_grid_dimension_y, hot3d0_block_dimension_x, hot3d0_block_dimension_y, (int)blockIdx.x, (int)gridDim.x, hot3d0_ptb_start_block_pos, hot3d0_ptb_end_block_pos, (int)threadIdx.x, 256);
        } else {
            tk::lava_role<4>(lava1_d_par_gpu, lava1_d_dim_gpu, lava1_d_box_gpu, lava1_d_rv_gpu, lava1_d_qv_gpu, lava1_d_fv_gpu, lava1_grid_dimension_x, (int)blockIdx.x, (int)gridDim.x, lava1_ptb_start_block_pos, lava1_ptb_end_block_pos, (int)threadIdx.x, 256);
        }
    }
}
