"""The work this framework is timed on: what its users run through the public entry points.

Kinds of case, each over the range its `draw` branch states:

  query          VGG16 at batch 1, the latency-critical job of the scheduler: image in host memory, logits on
                 the GPU
  gemm           tzgemm by itself through the one-shot call
  fused_stencil  tzgemm + 7-point stencil sweep in one launch
  fused_lbm      tzgemm + D3Q19 lattice-Boltzmann step in one launch
  fused_mriq     tzgemm + MRI-Q in one launch
  cutcp          a best-effort kernel alone: Parboil's cutoff Coulomb potential
  lava           a best-effort kernel alone: Rodinia's lavaMD
  path           a best-effort kernel alone: Rodinia's pathfinder

A best-effort kernel runs by itself whenever the scheduler has no query to put it next to; fused launches are
what it runs in otherwise.
"""
import math

import numpy as np
import torch

import tacker_amd as ta

DENSITY = 70000 / 104.0 ** 3     # cutcp: atoms per cubic Angstrom of the framework's own instance
SPACING, CUTOFF = 0.5, 12.0      # cutcp: lattice spacing and cutoff of the same instance
ATOMS_IN_REACH = DENSITY * 4.0 / 3.0 * math.pi * CUTOFF ** 3
STENCIL_C0, STENCIL_C1 = 1.0 / 6.0, 1.0 / 36.0
VGG16_CHANNELS = (64, 64, 0, 128, 128, 0, 256, 256, 256, 0, 512, 512, 512, 0, 512, 512, 512, 0)   # 0 = pooling


def listed():
    return [
        # one query of the co-location benchmark
        {"name": "query_224x224", "kind": "query", "height": 224, "width": 224},
        # a small, oblong image: most layers have few pixels, launches count
        {"name": "query_64x96", "kind": "query", "height": 64, "width": 96},
        # one small layer's worth of GEMM: the smallest call
        {"name": "gemm_256x384x512", "kind": "gemm", "M": 256, "N": 384, "K": 512},
        # a shape nobody tuned for: tile counts that divide neither the CUs nor the XCDs
        {"name": "gemm_1664x2432x896", "kind": "gemm", "M": 1664, "N": 2432, "K": 896},
        # the largest GEMM of the benchmark's shape table
        {"name": "gemm_4096x4096x4096", "kind": "gemm", "M": 4096, "N": 4096, "K": 4096},
        # the headline pair
        {"name": "fused_stencil_512x512x64", "kind": "fused_stencil", "M": 2048, "N": 2048, "K": 2048,
         "nx": 512, "ny": 512, "nz": 64},
        # the same pair small and ragged
        {"name": "fused_stencil_150x70x22", "kind": "fused_stencil", "M": 640, "N": 384, "K": 768,
         "nx": 150, "ny": 70, "nz": 22},
        # the memory-bound pair of the benchmark
        {"name": "fused_lbm_120x120x150", "kind": "fused_lbm", "M": 4096, "N": 4096, "K": 1024,
         "sx": 120, "sy": 120, "sz": 150},
        # the compute-bound pair of the benchmark
        {"name": "fused_mriq_2048x262144", "kind": "fused_mriq", "M": 2048, "N": 2048, "K": 2048,
         "numK": 2048, "numX": 262144},
        # best-effort kernels by themselves: the framework's own instance of cutcp, ...
        {"name": "cutcp_208", "kind": "cutcp", "points": 208, "layers": 2},
        # ... lavaMD on a domain of ordinary size, ...
        {"name": "lava_24", "kind": "lava", "boxes1d": 24},
        # ... and pathfinder's own instance
        {"name": "path_1200x125", "kind": "path", "cols": 1200, "iteration": 125},
    ]


def draw(rng):
    def spread(lo, hi, step=1):
        """a multiple of step in [lo, hi], even over the logarithm"""
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(hi, max(lo, int(round(v / step)) * step))

    def gemm(largest):
        """dimensions of 128 .. 4096 whose product is at most `largest`"""
        while True:
            d = {"M": spread(128, 4096, 128), "N": spread(128, 4096, 128), "K": spread(128, 4096, 128)}
            if d["M"] * d["N"] * d["K"] <= largest:
                return d

    kind = rng.choice(["query", "gemm", "gemm", "fused_stencil", "fused_lbm", "fused_mriq", "cutcp", "lava", "path"])
    c = {"kind": kind}
    if kind == "query":
        c.update(height=32 * rng.randint(1, 7), width=32 * rng.randint(1, 7))
    elif kind == "gemm":
        c.update(gemm(4096 ** 3))
    elif kind == "fused_stencil":
        c.update(gemm(2048 ** 3), nx=spread(32, 512), ny=spread(32, 512), nz=spread(6, 64))
        if rng.random() < 0.5:
            c["nx"] = c["nx"] // 4 * 4       # aligned rows are as common as odd ones
    elif kind == "fused_lbm":
        c.update(gemm(4096 * 4096 * 1024), sx=spread(24, 128), sy=spread(24, 128), sz=spread(24, 128))
    elif kind == "fused_mriq":
        c.update(gemm(2048 ** 3), numK=spread(128, 2048), numX=spread(8192, 262144, 256))
    elif kind == "cutcp":
        c.update(points=spread(48, 208, 8))
        c["layers"] = rng.randint(1, 2)
    elif kind == "lava":
        c.update(boxes1d=spread(2, 24))
    else:
        c.update(cols=spread(300, 20000), iteration=spread(5, 125))
    return c


class _Task(ta.LcTask):
    def __del__(self):
        self.close()


class _DeviceArray:
    """a device buffer as torch.as_tensor takes it; the tensor keeps it, and with it the buffer's owner"""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


class _Query:
    def __init__(self, case, rng):
        self.task = _Task("vgg16", case["height"], case["width"])
        image = self.task.host_input()
        image[:] = rng.random(image.size, dtype=np.float32)
        ptr, stride, n = self.task.logits()
        self.logits = torch.as_tensor(_DeviceArray(ptr, (n * stride,), self.task), device="cuda:0")[::stride]

    def __call__(self):
        self.task.execute()
        return self.logits


def _gemm_operands(case, gen):
    M, N, K = case["M"], case["N"], case["K"]
    A = torch.rand((M, K), device="cuda:0", generator=gen).mul_(2).sub_(1).half()
    B = torch.rand((N, K), device="cuda:0", generator=gen).mul_(2).sub_(1).half()
    return A, B, torch.zeros((M, N), device="cuda:0")


def _fused(case, gen, be_ori, blocks):
    """the fused-launch object of a best-effort kernel's whole grid and a whole GEMM, and the GEMM's output"""
    A, B, C = _gemm_operands(case, gen)
    tiles = (case["M"] // 64) * (case["N"] // 64)
    tz = ta.gptb_create(ta.ori_tzgemm_create(A, B, C), 0, 0, 0, tiles)
    be = ta.gptb_create(be_ori, 0, 0, 0, blocks)
    return ta.mix_create(be, tz, 0, blocks, 0, tiles), C


def prepare(case, seed):
    ta.init()
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda:0").manual_seed(seed)

    def uniform(lo, hi, shape):
        return torch.rand(shape, device="cuda:0", generator=gen).mul_(hi - lo).add_(lo)

    if kind == "query":
        return _Query(case, rng)
    if kind == "gemm":
        A, B, C = _gemm_operands(case, gen)

        def call():
            ta.gptb_tzgemm(A, B, C)
            return C
        return call
    if kind == "fused_stencil":
        grid = uniform(0, 1, (case["nz"], case["ny"], case["nx"]))
        nxt = grid.clone()
        if grid.numel() < 1 << 20:           # small: the one-shot call
            A, B, C = _gemm_operands(case, gen)

            def call():
                ta.mix_tzgemm_stencil(STENCIL_C0, STENCIL_C1, grid, nxt, A, B, C)
                return C, nxt
            return call
        mix, C = _fused(case, gen, ta.ori_stencil_create(STENCIL_C0, STENCIL_C1, grid, nxt),
                        ta.stencil_blocks(case["nx"], case["ny"], case["nz"]))
        out = (C, nxt)
    elif kind == "fused_lbm":
        # rest equilibrium with noise, 5 % obstacle cells
        cells = case["sx"] * case["sy"] * case["sz"]
        weights = torch.tensor([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12, device="cuda:0")
        src = torch.empty((20, cells), device="cuda:0")
        src[:19] = weights[:, None] + uniform(0, 1e-3, (19, cells))
        src[19] = (uniform(0, 1, cells) < 0.05).to(torch.int32).view(torch.float32)
        dst = src.clone()
        mix, C = _fused(case, gen, ta.ori_lbm_create(src, dst, case["sx"], case["sy"], case["sz"]),
                        case["sy"] * case["sz"])
        out = (C, dst[:19])
    elif kind == "fused_mriq":
        # the scanner's trajectory is the same for every scan; the voxels are the input
        scan = np.random.default_rng(1337)
        k = scan.uniform(-0.5, 0.5, (case["numK"], 3))
        phi = scan.uniform(0, 1, (2, case["numK"]))
        ta.mriq_set_kvalues(np.concatenate([k, (phi[0] ** 2 + phi[1] ** 2)[:, None]], 1).astype(np.float32))
        x, y, z = (uniform(-0.5, 0.5, case["numX"]) for _ in range(3))
        Qr, Qi = torch.zeros_like(x), torch.zeros_like(x)
        mix, C = _fused(case, gen, ta.ori_mriq_create(case["numK"], x, y, z, Qr, Qi),
                        ta.mriq_blocks(case["numK"], case["numX"]))
        out = (C, Qr, Qi)
    elif kind == "cutcp":
        n = case["points"]
        edge = (n - 1) * SPACING
        atoms = np.empty((int(DENSITY * edge ** 3), 4), np.float32)
        atoms[:, :3] = rng.uniform(0, edge, (len(atoms), 3))
        atoms[:, 3] = rng.uniform(0.1, 1, len(atoms)) * rng.choice([-1, 1], len(atoms))
        inp = ta.CutcpInput(atoms, (0, 0, 0), n, n, n, SPACING, CUTOFF, regions=(n // 8, n // 8, case["layers"]))
        mix = ta.gptb_create(ta.ori_cutcp_create(inp, CUTOFF ** 2, 1 / CUTOFF ** 2), 0, 0, 0, inp.blocks())
        out = inp.energies
    elif kind == "lava":
        n = 100 * case["boxes1d"] ** 3
        rv, qv = uniform(0.1, 1, (n, 4)), uniform(0.1, 1, n)
        fv = torch.zeros((n, 4), device="cuda:0")
        mix = ta.gptb_create(ta.ori_lava_create(0.5, rv, qv, fv), 0, 0, 0, ta.lava_blocks(case["boxes1d"]))
        out = fv
    else:
        cols, height = case["cols"], case["iteration"]
        wall = torch.randint(0, 10, (height, cols), device="cuda:0", dtype=torch.int32, generator=gen)
        src = torch.randint(0, 10, (cols,), device="cuda:0", dtype=torch.int32, generator=gen)
        result = torch.zeros(cols, dtype=torch.int32, device="cuda:0")
        mix = ta.gptb_create(ta.ori_path_create(height, wall, src, result), 0, 0, 0, ta.path_blocks(cols, height))
        out = result

    def launch():
        mix.execute()
        return out
    return launch


def run(state):
    return state()


def work(case):
    kind = case["kind"]
    bytes_, flops = 0.0, 0.0
    if kind == "query":
        h, w, c = case["height"], case["width"], 3
        params, macs = 0, 0
        for out in VGG16_CHANNELS:
            if out == 0:
                h, w = h // 2, w // 2
                continue
            params += 9 * c * out
            macs += h * w * 9 * c * out
            c = out
        for i, o in ((h * w * c, 4096), (4096, 4096), (4096, 1000)):
            params += i * o
            macs += i * o
        return {"bytes": 2.0 * params + 12.0 * case["height"] * case["width"] + 4000, "flops": 2.0 * macs}
    if "M" in case:
        M, N, K = case["M"], case["N"], case["K"]
        bytes_ += 2.0 * (M * K + N * K) + 4.0 * M * N
        flops += 2.0 * M * N * K
    if kind == "fused_stencil":
        points = case["nx"] * case["ny"] * case["nz"]
        bytes_ += 8.0 * points
        flops += 8.0 * points
    elif kind == "fused_lbm":
        cells = case["sx"] * case["sy"] * case["sz"]
        bytes_ += 4.0 * (20 + 19) * cells
        flops += 250.0 * cells
    elif kind == "fused_mriq":
        bytes_ += 16.0 * case["numK"] + 4.0 * 7 * case["numX"]
        flops += 12.0 * case["numK"] * case["numX"]
    elif kind == "cutcp":
        n, layers = case["points"] // 8, case["layers"]
        points = 512.0 * n * n * layers
        edge = (case["points"] - 1) * SPACING
        bytes_ += 4.0 * points + 16.0 * DENSITY * edge * edge * min(edge, 4.0 * layers + CUTOFF)
        flops += 14.0 * points * ATOMS_IN_REACH / 2      # the lowest layers have neighbours on one side only
    elif kind == "lava":
        b = case["boxes1d"]
        bytes_ += 100.0 * b ** 3 * (16 + 4 + 32)
        flops += 24.0 * 100 * 100 * float(3 * b - 2) ** 3
    elif kind == "path":
        bytes_ += 4.0 * case["cols"] * (case["iteration"] + 2)
        flops += 3.0 * case["cols"] * case["iteration"]
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times what the outputs differ by from the same path with its sums in 64 bits: tzgemm 0.9e-7 (K = 512) to
# 4.1e-7 (K = 4096); mri-q 1.2e-6; lavaMD 7.3e-7; cutcp 3.1e-7; the query 3.4e-4 (largest 1.5e-3), whose activations are
# rounded to f16 between the layers, so that a sum in another order now and then rounds to the next value.  Stencil, lbm
# and pathfinder have one order of operations.
TOLERANCE = {
    "query": {"rel": 1.4e-3, "max": 6e-3},
    "gemm": {"rel": 2e-6},
    "fused_stencil": {"rel": 2e-6},
    "fused_lbm": {"rel": 2e-6},
    "fused_mriq": {"rel": 5e-6},
    "cutcp": {"rel": 2e-6},
    "lava": {"rel": 4e-6},
    "path": "exact",
}
