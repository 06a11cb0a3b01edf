// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of tzgemm with mrif; parameter order = mrif's GPTB list,
// then tzgemm's (the concatenation MixKernel::initParams builds).

// mrif-tzgemm  wave split  256 tzgemm threads + 256 mrif threads per workgroup
extern "C" __global__ __launch_bounds__(512) void mrif_tzgemm_mix_wave_256(
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
    _Float16* tzgemm1_A,
    _Float16* tzgemm1_B,
    float* tzgemm1_C,
    int tzgemm1_NORMAL_M,
    int tzgemm1_NORMAL_N,
    int tzgemm1_NORMAL_K,
    int tzgemm1_grid_dimension_x,
    int tzgemm1_grid_dimension_y,
    int tzgemm1_grid_dimension_z,
    int tzgemm1_block_dimension_x,
    int tzgemm1_block_dimension_y,
    int tzgemm1_block_dimension_z,
    int tzgemm1_ptb_start_block_pos,
    int tzgemm1_ptb_iter_block_step,
    int tzgemm1_ptb_end_block_pos)
{
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)tzgemm1_grid_dimension_x;
    (void)tzgemm1_grid_dimension_y;
    (void)tzgemm1_grid_dimension_z;
    (void)tzgemm1_block_dimension_x;
    (void)tzgemm1_block_dimension_y;
    (void)tzgemm1_block_dimension_z;
    // One LDS object on purpose (ring + the arrival counter behind it): with two, the
    // compiler tags LDS accesses per object and then waits for every LDS-direct load in
    // flight before each read of the ring.
    __shared__ __align__(16) char tz_lds[TZ_LDS_BYTES + 16];
    unsigned *tz_arrivals = reinterpret_cast<unsigned *>(tz_lds + TZ_LDS_BYTES);
    if (threadIdx.x == 0) tk::RoleHandoverSync::init(tz_arrivals, 4);
    __syncthreads();   // the only barrier of all waves: before the roles part ways
    if (threadIdx.x < 256) {
        // One tzgemm wave per SIMD shares it with mrif waves: let the MFMA stream issue
        // whenever it is ready and the mrif waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while mrif waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the mrif blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = mrif0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, be_block, be_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x - 256, 256);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// mrif-tzgemm  wave split  256 tzgemm threads + 512 mrif threads per workgroup
extern "C" __global__ __launch_bounds__(768) void mrif_tzgemm_mix_wave_512(
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
    _Float16* tzgemm1_A,
    _Float16* tzgemm1_B,
    float* tzgemm1_C,
    int tzgemm1_NORMAL_M,
    int tzgemm1_NORMAL_N,
    int tzgemm1_NORMAL_K,
    int tzgemm1_grid_dimension_x,
    int tzgemm1_grid_dimension_y,
    int tzgemm1_grid_dimension_z,
    int tzgemm1_block_dimension_x,
    int tzgemm1_block_dimension_y,
    int tzgemm1_block_dimension_z,
    int tzgemm1_ptb_start_block_pos,
    int tzgemm1_ptb_iter_block_step,
    int tzgemm1_ptb_end_block_pos)
{
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)tzgemm1_grid_dimension_x;
    (void)tzgemm1_grid_dimension_y;
    (void)tzgemm1_grid_dimension_z;
    (void)tzgemm1_block_dimension_x;
    (void)tzgemm1_block_dimension_y;
    (void)tzgemm1_block_dimension_z;
    // One LDS object on purpose (ring + the arrival counter behind it): with two, the
    // compiler tags LDS accesses per object and then waits for every LDS-direct load in
    // flight before each read of the ring.
    __shared__ __align__(16) char tz_lds[TZ_LDS_BYTES + 16];
    unsigned *tz_arrivals = reinterpret_cast<unsigned *>(tz_lds + TZ_LDS_BYTES);
    if (threadIdx.x == 0) tk::RoleHandoverSync::init(tz_arrivals, 8);
    __syncthreads();   // the only barrier of all waves: before the roles part ways
    if (threadIdx.x < 256) {
        // One tzgemm wave per SIMD shares it with mrif waves: let the MFMA stream issue
        // whenever it is ready and the mrif waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while mrif waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the mrif blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = mrif0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::mrif_role<8>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, be_block, be_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x - 256, 512);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// mrif-tzgemm  workgroup split  1 tzgemm : 1 mrif workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_tzgemm_mix_wg_1_1(
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
    _Float16* tzgemm1_A,
    _Float16* tzgemm1_B,
    float* tzgemm1_C,
    int tzgemm1_NORMAL_M,
    int tzgemm1_NORMAL_N,
    int tzgemm1_NORMAL_K,
    int tzgemm1_grid_dimension_x,
    int tzgemm1_grid_dimension_y,
    int tzgemm1_grid_dimension_z,
    int tzgemm1_block_dimension_x,
    int tzgemm1_block_dimension_y,
    int tzgemm1_block_dimension_z,
    int tzgemm1_ptb_start_block_pos,
    int tzgemm1_ptb_iter_block_step,
    int tzgemm1_ptb_end_block_pos)
{
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)tzgemm1_grid_dimension_x;
    (void)tzgemm1_grid_dimension_y;
    (void)tzgemm1_grid_dimension_z;
    (void)tzgemm1_block_dimension_x;
    (void)tzgemm1_block_dimension_y;
    (void)tzgemm1_block_dimension_z;
    (void)tzgemm1_ptb_iter_block_step;
    __shared__ __align__(16) char tz_lds[TZ_LDS_BYTES_WG];
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 1);
    if (sp.role == 0) {
        tk::WorkgroupSync sync;
        tk::tzgemm_role<TZ_STAGES_WG, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), sp.role_block, sp.role_blocks, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x, tz_lds, sync);
    } else {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mrif-tzgemm  workgroup split  1 tzgemm : 2 mrif workgroups per group
extern "C" __global__ __launch_bounds__(256) void mrif_tzgemm_mix_wg_1_2(
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
    _Float16* tzgemm1_A,
    _Float16* tzgemm1_B,
    float* tzgemm1_C,
    int tzgemm1_NORMAL_M,
    int tzgemm1_NORMAL_N,
    int tzgemm1_NORMAL_K,
    int tzgemm1_grid_dimension_x,
    int tzgemm1_grid_dimension_y,
    int tzgemm1_grid_dimension_z,
    int tzgemm1_block_dimension_x,
    int tzgemm1_block_dimension_y,
    int tzgemm1_block_dimension_z,
    int tzgemm1_ptb_start_block_pos,
    int tzgemm1_ptb_iter_block_step,
    int tzgemm1_ptb_end_block_pos)
{
    (void)mrif0_kGlobalIndex;
    (void)mrif0_grid_dimension_z;
    (void)mrif0_block_dimension_x;
    (void)mrif0_block_dimension_y;
    (void)mrif0_block_dimension_z;
    (void)mrif0_ptb_iter_block_step;
    (void)tzgemm1_grid_dimension_x;
    (void)tzgemm1_grid_dimension_y;
    (void)tzgemm1_grid_dimension_z;
    (void)tzgemm1_block_dimension_x;
    (void)tzgemm1_block_dimension_y;
    (void)tzgemm1_block_dimension_z;
    (void)tzgemm1_ptb_iter_block_step;
    __shared__ __align__(16) char tz_lds[TZ_LDS_BYTES_WG];
    const tk::WgSplit sp = tk::wg_split((int)blockIdx.x, (int)gridDim.x, 1, 2);
    if (sp.role == 0) {
        tk::WorkgroupSync sync;
        tk::tzgemm_role<TZ_STAGES_WG, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), sp.role_block, sp.role_blocks, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x, tz_lds, sync);
    } else {
        tk::mrif_role<4>(mrif0_numK, mrif0_x, mrif0_y, mrif0_z, mrif0_outR, mrif0_outI, mrif0_grid_dimension_x, mrif0_grid_dimension_y, sp.role_block, sp.role_blocks, mrif0_ptb_start_block_pos, mrif0_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}
