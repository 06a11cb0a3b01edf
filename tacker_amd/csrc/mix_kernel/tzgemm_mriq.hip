// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of tzgemm with mriq; parameter order = mriq's GPTB list,
// then tzgemm's (the concatenation MixKernel::initParams builds).

// mriq-tzgemm  wave split  256 tzgemm threads + 256 mriq threads per workgroup
extern "C" __global__ __launch_bounds__(512) void mriq_tzgemm_mix_wave_256(
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
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
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
        // One tzgemm wave per SIMD shares it with mriq waves: let the MFMA stream issue
        // whenever it is ready and the mriq waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while mriq waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the mriq blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = mriq0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, be_block, be_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x - 256, 256);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// mriq-tzgemm  wave split  256 tzgemm threads + 512 mriq threads per workgroup
extern "C" __global__ __launch_bounds__(768) void mriq_tzgemm_mix_wave_512(
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
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
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
        // One tzgemm wave per SIMD shares it with mriq waves: let the MFMA stream issue
        // whenever it is ready and the mriq waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while mriq waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the mriq blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = mriq0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::mriq_role<8>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, be_block, be_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x - 256, 512);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// mriq-tzgemm  workgroup split  1 tzgemm : 1 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_tzgemm_mix_wg_1_1(
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
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
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
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-tzgemm  workgroup split  1 tzgemm : 2 mriq workgroups per group
extern "C" __global__ __launch_bounds__(256) void mriq_tzgemm_mix_wg_1_2(
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
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
    (void)mriq0_ptb_iter_block_step;
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
        tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, sp.role_block, sp.role_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// mriq-tzgemm  wave split  256 tzgemm threads + 256 mriq threads per workgroup
extern "C" __global__ __launch_bounds__(512) void mriq_tzgemm_mix_wave_256_large(
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
    (void)mriq0_kGlobalIndex;
    (void)mriq0_grid_dimension_z;
    (void)mriq0_block_dimension_x;
    (void)mriq0_block_dimension_y;
    (void)mriq0_block_dimension_z;
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
        // One tzgemm wave per SIMD shares it with mriq waves: let the MFMA stream issue
        // whenever it is ready and the mriq waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while mriq waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        if (tz_large_fused_fits(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K))
            tk::tzgemm_role_large_rot(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, true, sync);
        else
            tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the mriq blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = mriq0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::mriq_role<4>(mriq0_numK, mriq0_x, mriq0_y, mriq0_z, mriq0_Qr, mriq0_Qi, mriq0_grid_dimension_x, mriq0_grid_dimension_y, be_block, be_blocks, mriq0_ptb_start_block_pos, mriq0_ptb_end_block_pos, (int)threadIdx.x - 256, 256);
        }
        tk::role_wave_done(tz_arrivals);
    }
}
