// Generated by fusion/code/gen_run.py -- do not edit.
// Fused launches of tzgemm with cutcp; parameter order = cutcp's GPTB list,
// then tzgemm's (the concatenation MixKernel::initParams builds).

// cutcp-tzgemm  wave split  256 tzgemm threads + 128 cutcp threads per workgroup
extern "C" __global__ __launch_bounds__(384) void cutcp_tzgemm_mix_wave_128(
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
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
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
    if (threadIdx.x == 0) tk::RoleHandoverSync::init(tz_arrivals, 2);
    __syncthreads();   // the only barrier of all waves: before the roles part ways
    if (threadIdx.x < 256) {
        // One tzgemm wave per SIMD shares it with cutcp waves: let the MFMA stream issue
        // whenever it is ready and the cutcp waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while cutcp waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the cutcp blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = cutcp0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::cutcp_role<2>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, be_block, be_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x - 256, 128);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// cutcp-tzgemm  wave split  256 tzgemm threads + 256 cutcp threads per workgroup
extern "C" __global__ __launch_bounds__(512) void cutcp_tzgemm_mix_wave_256(
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
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
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
        // One tzgemm wave per SIMD shares it with cutcp waves: let the MFMA stream issue
        // whenever it is ready and the cutcp waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while cutcp waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the cutcp blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = cutcp0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, be_block, be_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x - 256, 256);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// cutcp-tzgemm  wave split  256 tzgemm threads + 384 cutcp threads per workgroup
extern "C" __global__ __launch_bounds__(640) void cutcp_tzgemm_mix_wave_384(
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
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
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
    if (threadIdx.x == 0) tk::RoleHandoverSync::init(tz_arrivals, 6);
    __syncthreads();   // the only barrier of all waves: before the roles part ways
    if (threadIdx.x < 256) {
        // One tzgemm wave per SIMD shares it with cutcp waves: let the MFMA stream issue
        // whenever it is ready and the cutcp waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while cutcp waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the cutcp blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = cutcp0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::cutcp_role<6>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, be_block, be_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x - 256, 384);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// cutcp-tzgemm  wave split  256 tzgemm threads + 512 cutcp threads per workgroup
extern "C" __global__ __launch_bounds__(768) void cutcp_tzgemm_mix_wave_512(
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
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
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
        // One tzgemm wave per SIMD shares it with cutcp waves: let the MFMA stream issue
        // whenever it is ready and the cutcp waves fill the slots it leaves.
        __builtin_amdgcn_s_setprio(TK_GEMM_WAVE_PRIORITY);
        // role barrier: an arrival counter in LDS while cutcp waves run, the hardware barrier once they have ended
        tk::RoleHandoverSync sync(tz_arrivals, 4, (int)threadIdx.x - 0, &tk_spin_fail);
        tk::tzgemm_role<TZ_STAGES, true>(tzgemm1_A, tzgemm1_B, tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, tk::tz_workspace_of(tzgemm1_C, tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K), (int)blockIdx.x, tzgemm1_ptb_iter_block_step, tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos, (int)threadIdx.x - 0, tz_lds, sync);
    } else {
        // A GEMM that leaves at least half of the workgroups without a tile: the cutcp blocks go
        // to those workgroups only, where nothing competes with them, and the workgroups that
        // hold the latency-critical tiles run them undisturbed.
        const int launched = cutcp0_ptb_iter_block_step;
        const int tz_busy = tk::tz_busy_workgroups(tzgemm1_NORMAL_M, tzgemm1_NORMAL_N, tzgemm1_NORMAL_K, launched,
                                                   tzgemm1_ptb_start_block_pos, tzgemm1_ptb_end_block_pos);
        const bool apart = 2 * tz_busy <= launched;
        const int be_block = apart ? (int)blockIdx.x - tz_busy : (int)blockIdx.x;
        const int be_blocks = apart ? launched - tz_busy : launched;
        if (be_block >= 0) {
            tk::cutcp_role<8>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, be_block, be_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x - 256, 512);
        }
        tk::role_wave_done(tz_arrivals);
    }
}

// cutcp-tzgemm  workgroup split  1 tzgemm : 1 cutcp workgroups per group
extern "C" __global__ __launch_bounds__(256) void cutcp_tzgemm_mix_wg_1_1(
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
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
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
        tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}

// cutcp-tzgemm  workgroup split  1 tzgemm : 2 cutcp workgroups per group
extern "C" __global__ __launch_bounds__(256) void cutcp_tzgemm_mix_wg_1_2(
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
    (void)cutcp0_zRegionIndex_t;
    (void)cutcp0_block_dimension_x;
    (void)cutcp0_block_dimension_y;
    (void)cutcp0_block_dimension_z;
    (void)cutcp0_ptb_iter_block_step;
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
        tk::cutcp_role<4>(cutcp0_binDim_x, cutcp0_binDim_y, cutcp0_binZeroAddr, cutcp0_h, cutcp0_cutoff2, cutcp0_inv_cutoff2, cutcp0_regionZeroAddr, cutcp0_grid_dimension_x, cutcp0_grid_dimension_y, cutcp0_grid_dimension_z, sp.role_block, sp.role_blocks, cutcp0_ptb_start_block_pos, cutcp0_ptb_end_block_pos, (int)threadIdx.x, 256);
    }
}
