"""GPU parity of the cutoff Coulomb potential partner (src/ori_kernel/cutcp_kernel.cu,
src/gptb_kernel/cutcp_kernel.cu, src/mix_kernel/tzgemm_cutcp.cu): against the oracle's walk through the
bins within |d| <= 2e-4 + 2e-5 |ref| (the hardware's reciprocal square root here, 1 / sqrtf there, CUDA's
rsqrtf in the reference: approximations of an ulp each, summed over hundreds of atoms) and against the
float64 sum over the atom list; the natural launch, the GPTB form over any tiling of its positions and
every fused variant give the same bits as each other (positions = regions x parts of the neighbour list); the host's binning equals the oracle's exactly."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
import tacker_amd as ta
from gpu_util import dev, gemm_inputs, gemm_tolerance_ok, host, launch, setup

pytestmark = pytest.mark.gpu
H, CUTOFF = 0.5, 12.0
C2, INV_C2 = 144.0, 0.006944            # as the reference types them (src/ori_kernel/cutcp_kernel.cu:226-227)


@pytest.fixture(scope="module", autouse=True)
def _init():
    setup()


def atoms_in_box(n, box, seed):
    rng = np.random.default_rng(seed)
    a = np.empty((n, 4), np.float32)
    a[:, :3] = rng.uniform(0, box, (n, 3))
    a[:, 3] = rng.uniform(-1, 1, n)
    a[a[:, 3] == 0, 3] = 0.5
    return a


def close(got, want):
    return bool(np.all(np.abs(got.astype(np.float64) - want.astype(np.float64)) <= 2e-4 + 2e-5 * np.abs(want)))


def bits(t):
    return host(t).view(np.uint32)


def case(points=(24, 24, 16), natoms=500, seed=4):
    nx, ny, nz = points
    atoms = atoms_in_box(natoms, (min(points) - 1) * H, seed)
    inp = ta.CutcpInput(atoms, (0, 0, 0), nx, ny, nz, H, CUTOFF)
    prep = oracle.cutcp_prepare(atoms, (0, 0, 0), nx, ny, nz, H, CUTOFF)
    return atoms, inp, prep


def test_host_binning_equals_the_oracles():
    atoms = atoms_in_box(5000, 19.5, seed=8)          # dense: some bins overflow
    atoms[3, 3] = 0.0
    inp = ta.CutcpInput(atoms, (0.25, -0.5, 0.0), 40, 40, 40, H, CUTOFF)
    prep = oracle.cutcp_prepare(atoms, (0.25, -0.5, 0.0), 40, 40, 40, H, CUTOFF)
    assert inp.binDim == prep["binDim"] and inp.padding == prep["padding"]
    assert np.array_equal(inp.host_bins, prep["bins"]) and np.array_equal(inp.nbr, prep["nbr"])
    assert (inp.extra, inp.excluded) == (prep["extra"], prep["excluded"]) and inp.extra > 0 and inp.excluded >= 1


def test_ori_and_gptb_forms_match_the_oracle_and_the_float64_sum():
    atoms, inp, prep = case()
    want = oracle.cutcp(prep, H, C2, INV_C2, inp.regions)
    e_ori, e_gptb, e_small = (torch.zeros_like(inp.energies) for _ in range(3))
    ta.ori_cutcp(inp, C2, INV_C2, e_ori)
    ta.gptb_cutcp(inp, C2, INV_C2, e_gptb)
    ta.gptb_cutcp(inp, C2, INV_C2, e_small, launch_grid=3, launch_block=64)
    assert close(host(e_ori), want) and np.abs(want).max() > 1.0
    assert np.array_equal(bits(e_gptb), bits(e_ori)) and np.array_equal(bits(e_small), bits(e_ori))
    # float64, no bins: every binned atom against every lattice point
    b = prep["bins"].reshape(-1, 4)
    b = b[b[:, 3] != 0].astype(np.float64)
    rx, ry, rz = inp.regions
    zs, ys, xs = np.arange(8 * rz) * H, np.arange(8 * ry) * H, np.arange(8 * rx) * H
    pot = np.zeros((8 * rz, 8 * ry, 8 * rx))
    for ax, ay, az, q in b:
        r2 = (az - zs)[:, None, None] ** 2 + (ay - ys)[None, :, None] ** 2 + (ax - xs)[None, None, :] ** 2
        with np.errstate(divide="ignore", invalid="ignore"):
            pot += np.where(r2 < C2, q / np.sqrt(r2) * (1.0 - r2 * INV_C2) ** 2, 0.0)
    truth = pot.reshape(rz, 8, ry, 8, rx, 8).transpose(0, 2, 4, 1, 3, 5)
    assert close(host(e_ori), truth)
    assert ta.spin_fail_flag() == 0


@pytest.mark.parametrize("seed", range(4))
def test_any_tiling_of_the_positions_gives_the_one_kernel(seed):
    rng = np.random.default_rng(800 + seed)
    atoms, inp, prep = case(points=[(24, 16, 16), (16, 24, 8), (8, 8, 40), (32, 16, 16)][seed], natoms=300, seed=seed)
    whole = torch.zeros_like(inp.energies)
    ta.ori_cutcp(inp, C2, INV_C2, whole)
    n = inp.blocks()
    cuts = sorted(set(rng.integers(0, n + 1, 3).tolist()) | {0, n})
    e = torch.full_like(inp.energies, -3.0)
    for a, b in zip(cuts, cuts[1:]):
        ta.gptb_cutcp(inp, C2, INV_C2, e, a, b, launch_grid=int(rng.choice([1, 5, 64, 256])),
                      launch_block=int(rng.choice([64, 128, 256])))
    assert np.array_equal(bits(e), bits(whole))
    assert n == oracle.cutcp_positions(inp.regions, len(inp.nbr)) == inp.regions[0] * inp.regions[1] * inp.regions[2] * 11
    # a partial range touches its regions only, in the reference's position order (x slowest); positions 1 and 2
    # are the first part of the neighbour list (entries 0, 11, 22, ...) of regions 1 and 2
    e = torch.full_like(inp.energies, -3.0)
    ta.gptb_cutcp(inp, C2, INV_C2, e, 1, 3)
    want = oracle.cutcp(prep, H, C2, INV_C2, inp.regions, 1, 3, out=np.full(tuple(e.shape), -3.0, np.float32),
                        parts="chunks")
    got = host(e)
    assert np.array_equal(got == -3.0, want == -3.0) and close(got, want)


# one point a thread in pieces dealt one and two to a workgroup (up to and from 256 regions on 256 CUs), two points (from 513)
@pytest.mark.parametrize("regions", [(16, 16, 1), (257, 1, 1), (16, 16, 2), (19, 27, 1)])
def test_pieces_of_every_size_give_the_same_bits(regions):
    rng = np.random.default_rng(sum(regions))
    atoms = atoms_in_box(6000, 1.0, seed=9)
    atoms[:, :3] *= [(8 * r - 1) * H for r in regions]
    inp = ta.CutcpInput(atoms, (0, 0, 0), *(8 * r for r in regions), H, CUTOFF, regions=regions)
    e_ori, e_gptb, e_small, e_cut = (torch.zeros_like(inp.energies) for _ in range(4))
    ta.ori_cutcp(inp, C2, INV_C2, e_ori)
    ta.gptb_cutcp(inp, C2, INV_C2, e_gptb)
    ta.gptb_cutcp(inp, C2, INV_C2, e_small, launch_grid=40, launch_block=256)
    cuts = [0, int(rng.integers(1, inp.blocks())), inp.blocks()]
    for a, b in zip(cuts, cuts[1:]):
        ta.gptb_cutcp(inp, C2, INV_C2, e_cut, a, b)
    for e in (e_gptb, e_small, e_cut):
        assert np.array_equal(bits(e), bits(e_ori))
    if regions[2] == 1:
        prep = oracle.cutcp_prepare(atoms, (0, 0, 0), *(8 * r for r in regions), H, CUTOFF)
        assert close(host(e_ori), oracle.cutcp(prep, H, C2, INV_C2, inp.regions))


@pytest.mark.parametrize("length", [1, 7, 8, 9, 31, 32, 33, 47, 64, 65, 97, 334])
def test_neighbour_lists_of_any_length(length):
    # eight bins are looked at at a time and the atoms found used four at a time: lists that end inside a batch, of one part and
    # of several (from 33 on), bins of none to eight atoms
    atoms, inp, prep = case(points=(24, 16, 16), natoms=400 + 37 * (length % 8), seed=length)
    full = inp.nbr
    try:
        inp.nbr = np.ascontiguousarray(np.random.default_rng(length).permutation(full)[:length])
        inp.load_neighbours()
        prep["nbr"] = inp.nbr
        for inv in (1 / 144.0, 0.0065):
            want = oracle.cutcp(prep, H, C2, inv, inp.regions)
            e = [torch.zeros_like(inp.energies) for _ in range(3)]
            ta.ori_cutcp(inp, C2, inv, e[0])
            ta.gptb_cutcp(inp, C2, inv, e[1])
            ta.gptb_cutcp(inp, C2, inv, e[2], launch_grid=2, launch_block=64)
            assert close(host(e[0]), want)
            assert np.array_equal(bits(e[1]), bits(e[0])) and np.array_equal(bits(e[2]), bits(e[0]))
    finally:
        inp.nbr = full
        inp.load_neighbours()


def test_a_grid_of_bins_too_long_for_products_of_24_bits():
    # the same two rows of bins, 4 and 600000 bins apart
    atoms, inp, _ = case(points=(8, 8, 8), natoms=20, seed=3)
    full = inp.nbr
    rows = np.random.default_rng(5).uniform(0.5, 3, (2, 4, 8, 4)).astype(np.float32)
    got = []
    try:
        inp.nbr = np.array([[0, 0, 0], [1, 0, 0], [2, 0, 0], [0, 1, 0], [1, 1, 0], [3, 1, 0]], np.int32)
        inp.load_neighbours()
        for length in (4, 600000):
            inp.bins = torch.zeros((2, length, 8, 4), device="cuda:0")
            inp.bins[:, :4] = dev(rows)
            inp.binDim, inp.bin_zero = (length, 2, 1), inp.bins.data_ptr()
            e = torch.zeros_like(inp.energies)
            ta.gptb_cutcp(inp, C2, 1 / 144.0, e)
            got.append(bits(e))
        assert np.array_equal(got[0], got[1]) and np.abs(got[0].view(np.float32)).min() > 1
    finally:
        inp.nbr = full
        inp.load_neighbours()


@pytest.mark.parametrize("inv", [1 / 144.0, 0.0065, 0.008])
@pytest.mark.parametrize("regions,natoms", [((1, 1, 1), 1), ((2, 1, 1), 64), ((1, 3, 2), 2000), ((9, 8, 3), 900), ((8, 9, 7), 1500)])
def test_cut_of_the_regions_and_meaning_of_the_cutoff(inv, regions, natoms):
    # the launch's wavefronts decide how regions are cut into pieces (1 or 2 points a lane); inv_cutoff2 need not be
    # 1 / cutoff2, and then the cutoff is a comparison; full bins, empty bins, a charge of zero inside a bin (it ends the bin)
    nx, ny, nz = (8 * r for r in regions)
    atoms = atoms_in_box(natoms, (min(nx, ny, nz) - 1) * H, seed=natoms)
    inp = ta.CutcpInput(atoms, (0, 0, 0), nx, ny, nz, H, CUTOFF)
    prep = oracle.cutcp_prepare(atoms, (0, 0, 0), nx, ny, nz, H, CUTOFF)
    filled = np.argwhere(prep["bins"][..., 3] != 0)
    for where in filled[::7]:
        prep["bins"][tuple(where)][3] = 0.0
    inp.bins.copy_(torch.from_numpy(prep["bins"]).cuda())
    want = oracle.cutcp(prep, H, C2, inv, inp.regions, parts="chunks")
    out = [torch.zeros_like(inp.energies) for _ in range(3)]
    ta.gptb_cutcp(inp, C2, inv, out[0])
    ta.gptb_cutcp(inp, C2, inv, out[1], launch_grid=1, launch_block=64)
    ta.ori_cutcp(inp, C2, inv, out[2])
    assert np.array_equal(bits(out[1]), bits(out[0])) and np.array_equal(bits(out[2]), bits(out[0]))
    assert close(host(out[0]), want)


@pytest.mark.parametrize("inv", [1 / 144.0, 0.0069])
def test_four_points_a_lane_give_the_bits_of_one_and_two(inv):
    # more than 2048 regions take four points a lane, one layer of them takes one and twelve take two; 0.0069: the cutoff is
    # compared, point by point, and a term that rounding moves across it is below 1e-5
    n = 8 * 13
    atoms = atoms_in_box(1500, (n - 1) * H, seed=13)
    prep = oracle.cutcp_prepare(atoms, (0, 0, 0), n, n, n, H, CUTOFF)
    got = {}
    for layers in (13, 12, 1):
        inp = ta.CutcpInput(atoms, (0, 0, 0), n, n, n, H, CUTOFF, regions=(13, 13, layers))
        out = [torch.zeros_like(inp.energies) for _ in range(2)]
        ta.gptb_cutcp(inp, C2, inv, out[0])
        ta.ori_cutcp(inp, C2, inv, out[1])
        assert np.array_equal(bits(out[0]), bits(out[1]))
        got[layers] = host(out[0])
    for layers in (12, 1):
        assert np.array_equal(got[layers].view(np.uint32), got[13][:layers].view(np.uint32))
    assert close(got[13], oracle.cutcp(prep, H, C2, inv, (13, 13, 13), parts="chunks"))


@pytest.mark.parametrize("inv", [1 / 144.0, 0.0069])
@pytest.mark.parametrize("regions,natoms", [((1, 6, 2), 300), ((8, 9, 7), 3000)])
@pytest.mark.parametrize("what", ["inf", "-inf", "nan", "both", "position"])
def test_charges_and_positions_that_are_not_finite_reach_the_points_within_the_cutoff_only(inv, regions, natoms, what):
    # an infinite charge, or one that is no number, shows at the points within its cutoff and nowhere else; an atom whose
    # position is not finite shows nowhere.  0.0069: the cutoff is compared, and a term that rounding moves across it is
    # below 1e-5
    nx, ny, nz = (8 * r for r in regions)
    atoms = atoms_in_box(natoms, (min(nx, ny, nz) - 1) * H, seed=natoms + 1)
    inp = ta.CutcpInput(atoms, (0, 0, 0), nx, ny, nz, H, CUTOFF)
    prep = oracle.cutcp_prepare(atoms, (0, 0, 0), nx, ny, nz, H, CUTOFF)
    filled = np.argwhere(prep["bins"][..., 3] != 0)
    values = {"inf": [np.inf], "-inf": [-np.inf], "nan": [np.nan], "both": [np.inf, -np.inf],
              "position": [np.inf, -np.inf, np.nan]}[what]
    for j, v in enumerate(values):
        prep["bins"][tuple(filled[(3 * j) % len(filled)])][j if what == "position" else 3] = v
    inp.bins.copy_(torch.from_numpy(prep["bins"]).cuda())
    want = oracle.cutcp(prep, H, C2, inv, inp.regions, parts="chunks")
    ta.gptb_cutcp(inp, C2, inv)
    got = host(inp.energies)
    ok = np.isfinite(want)
    assert ok.any() and (what == "position") == ok.all()
    assert np.array_equal(got[~ok], want[~ok], equal_nan=True)
    assert np.isfinite(got[ok]).all() and close(got[ok], want[ok])


@pytest.mark.parametrize("threads", [64, 192, 256, 320, 512, 1024])
@pytest.mark.parametrize("grid", [1, 3, 40])
def test_workgroups_of_any_size_give_the_same_bits(threads, grid):
    # the kernel launched by its handle: a workgroup has LDS for four wavefronts, further ones must not use any behind it
    atoms, inp, prep = case(points=(40, 32, 16), natoms=700, seed=9)
    want = torch.zeros_like(inp.energies)
    ta.gptb_cutcp(inp, C2, INV_C2, want)
    out = torch.zeros_like(want)
    i, f, p = C.c_int, C.c_float, C.c_void_p
    rx, ry, rz = inp.regions
    parts = inp.blocks() // (rx * ry * rz)
    launch("gptb_cutcp", grid, threads,
           [i(inp.binDim[0]), i(inp.binDim[1]), p(inp.bin_zero), f(H), f(C2), f(INV_C2), p(out.data_ptr()), i(0), i(rx), i(ry),
            i(rz * parts), i(8), i(2), i(8), i(0), i(grid), i(inp.blocks()), i(0)])
    assert np.array_equal(bits(out), bits(want)) and np.abs(host(want)).max() > 0


@pytest.mark.parametrize("variant", [None, "wave_128", "wave_256", "wave_512", "wg_1_1", "wg_1_2"])
def test_mix_tzgemm_cutcp(variant):
    M, N, K = 256, 256, 256
    A, B = gemm_inputs(M, N, K, seed=31)
    atoms, inp, prep = case(natoms=400, seed=6)
    solo_c = torch.zeros((M, N), device="cuda:0")
    ta.gptb_tzgemm(dev(A), dev(B), solo_c)
    solo_e = torch.zeros_like(inp.energies)
    ta.gptb_cutcp(inp, C2, INV_C2, solo_e)
    mix_c = torch.zeros((M, N), device="cuda:0")
    mix_e = torch.zeros_like(inp.energies)
    ta.mix_tzgemm_cutcp(inp, C2, INV_C2, dev(A), dev(B), mix_c, mix_e, variant=variant)
    assert np.array_equal(host(mix_c), host(solo_c))
    assert np.array_equal(bits(mix_e), bits(solo_e))
    assert close(host(mix_e), oracle.cutcp(prep, H, C2, INV_C2, inp.regions))
    ok, fro, dmax = gemm_tolerance_ok(host(mix_c), oracle.tzgemm(A, B, f64=True), K)
    assert ok and fro <= 1e-5
    n = inp.blocks()
    mix_e.zero_()
    mix_c.zero_()
    ta.mix_tzgemm_cutcp(inp, C2, INV_C2, dev(A), dev(B), mix_c, mix_e, be_start=0, be_end=5, tile_start=0, tile_end=5,
                        variant=variant)
    ta.mix_tzgemm_cutcp(inp, C2, INV_C2, dev(A), dev(B), mix_c, mix_e, be_start=5, be_end=n, tile_start=5, tile_end=16,
                        variant=variant)
    assert np.array_equal(bits(mix_e), bits(solo_e)) and np.array_equal(host(mix_c), host(solo_c))
    assert ta.spin_fail_flag() == 0


def test_creator_object_is_the_references_instance_on_seeded_atoms():
    # createKernel("cutcp"): 208^3 lattice points, spacing 0.5, cutoff 12, bins 32 x 32, grid (26, 26, 2)
    # (src/ori_kernel/cutcp_kernel.cu:181-263)
    k = ta.create_kernel("cutcp")
    info = k.info()
    assert (info["ptb_start"], info["ptb_end"], info["ori_grid_x"], info["ori_grid_y"]) == (0, 26 * 26 * 2 * 11, 26, 26)
    assert (k.param(0, "int"), k.param(1, "int")) == (32, 32)
    assert abs(k.param(3, "float") - 0.5) < 1e-7 and abs(k.param(4, "float") - 144.0) < 1e-4
    assert abs(k.param(5, "float") - 0.006944) < 1e-8
    k.execute()
    torch.cuda.synchronize()
    bins = ta.device_to_host(k.param(2) - (((3 * 32 + 3) * 32 + 3) * 32) * 4, (32, 32, 32, 8, 4), np.float32)
    assert 60000 < np.count_nonzero(bins[..., 3]) <= 70000
    got = ta.device_to_host(k.param(6), (2, 26, 26, 8, 8, 8), np.float32)
    prep = {"bins": bins, "padding": 3, "binDim": (32, 32, 32),
            "nbr": oracle.cutcp_prepare(np.zeros((0, 4), np.float32), (0, 0, 0), 208, 208, 208, H, CUTOFF)["nbr"]}
    for pos in (0, 700, 1351):                                   # x slowest: region (pos // 52, (pos // 2) % 26, pos % 2)
        want = oracle.cutcp(prep, H, C2, INV_C2, (26, 26, 2), pos, pos + 1)
        x, y, z = pos // 52, (pos // 2) % 26, pos % 2
        assert close(got[z, y, x], want[z, y, x]) and np.abs(want[z, y, x]).max() > 0.1
    assert ta.spin_fail_flag() == 0


def test_bad_arguments_are_refused():
    lib = ta.lib()
    atoms, inp, prep = case(natoms=10)
    a = inp.args(C2, INV_C2)
    assert lib.tacker_ori_cutcp(*((a[0], a[1], None) + a[3:]), None) == 1
    assert lib.tacker_gptb_cutcp(*(a[:7] + (0, 2, 2)), 0, 1, 0, 0, None) == 1
    assert lib.tacker_cutcp_set_neighbours(None, 5) == 1 and lib.tacker_cutcp_set_neighbours(inp.nbr.ctypes.data, 2000) == 1
    inp.load_neighbours()
