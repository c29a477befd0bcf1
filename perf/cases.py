"""The work that this framework does for its users, as cases that can be timed.

A case is one pass through the public entry points of fastrecon_amd.hip on
inputs that are resident on the GPU, as a reconstruction program holds them:

  recon      gridding, then transforms + shift + crop + coil sum of squares
             (with `graph`, the same pass replayed as a captured graph)
  grid       gridding alone
  degrid     the forward operator: a grid sampled along the trajectory
  iterative  10 Pipe-Menon iterations for the density, then the recon
  learned    the density from the shipped network, then the recon
  scan       a trajectory seen for the first time: upload from device memory,
             gridding plan, gridding, image
  pils       the sensitivity-weighted recon: gridding, low-pass copy, both
             transforms, map normalisation, map-weighted sum
  gradient   loss gradient of one training batch of the density network

Trajectories are those of fastrecon_amd.synthetic (golden-angle radial,
Fibonacci kooshball, variable-density spirals), turned by an angle that comes
from the seed.
"""
import math
import os

import numpy as np
import torch

from fastrecon_amd import hip

L = 512                       # entries of the kernel table, as the program plans it
GOLDEN = math.pi * (math.sqrt(5.0) - 1.0) / 2.0
PACKAGE = os.path.dirname(os.path.abspath(hip.__file__))


def case(kind, traj, dim, image, og, coils, shots, readout, name=None, half=False, deapod=False, frames=0,
         graph=False):
    c = dict(kind=kind, traj=traj, dim=dim, image=image, og=og, coils=coils, shots=shots, readout=readout, half=half,
             deapod=deapod, frames=frames, graph=graph)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a calibration or navigator image: one coil, few spokes; latency and launches are all of it
        case("recon", "radial", 2, 48, 2.0, 1, 101, 96, "recon_radial2d_c1_n96"),
        # the reference program's own 2D case: golden-angle radial, 8 coils, 256^2 image
        case("recon", "radial", 2, 256, 2.0, 8, 402, 512, "recon_radial2d_c8_n512"),
        # a dynamic series: 64 frames of 8 to 48 spiral interleaves, replayed as one graph
        case("recon", "spiral", 2, 192, 2.0, 12, 48, 4096, "series_spiral2d_c12_n384", frames=64, graph=True),
        # a small 3D scan with odd sizes throughout and a deapodised image
        case("recon", "kooshball", 3, 90, 2.0, 5, 6007, 191, "recon_kooshball3d_c5_n180", deapod=True),
        # the headline workload: 32 coils of a 3D kooshball, gridding alone
        case("grid", "kooshball", 3, 128, 2.0, 32, 51200, 256, "grid_kooshball3d_c32_n256"),
        # high-resolution 3D with samples kept as FP16 pairs and a smaller oversampling
        case("grid", "kooshball", 3, 256, 1.5, 16, 100000, 384, "grid_kooshball3d_c16_half_n384", half=True),
        # the forward operator of an iterative reconstruction, one application
        case("degrid", "kooshball", 3, 64, 2.0, 8, 12800, 128, "degrid_kooshball3d_c8_n128"),
        # a trajectory without an analytic density: Pipe-Menon, then the image
        case("iterative", "kooshball", 3, 128, 2.0, 8, 51200, 256, "iterative_kooshball3d_c8_n256"),
        # the same with the shipped network in place of the iterations
        case("learned", "kooshball", 3, 128, 2.0, 32, 51200, 256, "learned_kooshball3d_c32_n256"),
        # one scan from its trajectory to its image, as the command-line program does once per run
        case("scan", "kooshball", 3, 96, 2.0, 8, 20000, 192, "scan_kooshball3d_c8_n192"),
        # the program's --pils path on its 2D case
        case("pils", "radial", 2, 256, 2.0, 8, 402, 512, "pils_radial2d_c8_n512"),
        # a training batch of the density network
        case("gradient", "none", 3, 128, 2.0, 1, 65536, 1, "gradient_b65536"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["recon", "recon", "grid", "grid", "degrid", "iterative", "learned", "scan", "pils", "gradient"])
    if kind == "gradient":
        return case(kind, "none", 3, 128, 2.0, 1, _log(rng, 1000, 200000), 1)
    dim = 2 if kind == "pils" else rng.choice([2, 3])
    og = rng.choice([1.25, 1.5, 2.0, 2.0])
    coils = _log(rng, 1, 32)
    half = kind in ("recon", "grid") and rng.random() < 0.25
    deapod = kind == "recon" and rng.random() < 0.4
    if dim == 3:
        image = 4 * _log(rng, 6, 36)
        while round(image * og) % 2:
            image += 2
        shots = _log(rng, 400, {"degrid": 10000, "iterative": 20000}.get(kind, 40000))
        return case(kind, "kooshball", 3, image, og, coils, shots, _log(rng, 48, 320), None, half, deapod)
    image = 4 * _log(rng, 12, 80)
    while round(image * og) % 2:
        image += 2
    if kind in ("recon", "grid") and rng.random() < 0.5:
        frames = rng.randrange(2, 65)
        return case(kind, "spiral", 2, min(image, 192), 2.0, min(coils, 16), rng.randrange(9, 49),
                    _log(rng, 512, 4096), None, half, deapod, frames, kind == "recon" and rng.random() < 0.5)
    if rng.random() < 0.5 and kind != "pils":
        return case(kind, "spiral", 2, image, og, coils, rng.randrange(8, 65), _log(rng, 512, 8192), None, half, deapod)
    return case(kind, "radial", 2, image, og, coils, _log(rng, 32, 1024), _log(rng, 64, 768), None, half, deapod)


# ------------------------------------------------------------------ inputs
def grid_size(c):
    return int(np.float32(c["image"]) * np.float32(c["og"]))


def crop(c):
    return (c["image"], c["image"], c["image"] if c["dim"] == 3 else 1)


def kernel_table(og, width=4.0):
    """Radial Kaiser-Bessel table (Beatty's beta), as the program's ConvKernel makes it."""
    beta = np.float32(math.pi * math.sqrt((width / og) ** 2 * (og - 0.5) ** 2 - 0.8))
    t = np.arange(L, dtype=np.float64) / (L - 1)
    return (np.i0(np.float64(beta) * np.sqrt(1.0 - t * t)) / np.i0(np.float64(beta))).astype(np.float32)


def frame_shots(c):
    """Interleaves of each frame of a series: 8 up to c["shots"], fixed by the case."""
    return np.random.default_rng(4 + c["frames"]).integers(8, c["shots"] + 1, c["frames"])


def spiral(n, readout, turn):
    t = torch.arange(readout, dtype=torch.float64, device="cuda") / readout
    ta = t ** 1.5
    ph = 2 * math.pi * (16.0 * ta[None, :] + torch.arange(n, dtype=torch.float64, device="cuda")[:, None] / n) + turn
    return torch.stack([0.5 * ta * torch.cos(ph), 0.5 * ta * torch.sin(ph)], -1).reshape(-1, 2)


def k_space(c, turn):
    """Sample positions in [-0.5, 0.5)^dim, FP64."""
    n, r = c["shots"], c["readout"]
    if c["traj"] == "spiral":
        return spiral(n, r, turn)
    j = (torch.arange(r, dtype=torch.float64, device="cuda") - r / 2) / r
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    if c["traj"] == "radial":
        u = torch.stack([torch.cos(i * GOLDEN + turn), torch.sin(i * GOLDEN + turn)], -1)
    else:
        z = 1 - (2 * i + 1) / n
        s = torch.sqrt(1 - z * z)
        phi = i * math.pi * (3 - math.sqrt(5.0)) + turn
        u = torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], -1)
    return (j[None, :, None] * u[:, None, :]).reshape(-1, u.shape[1])


def to_grid(k, N):
    """Grid units with the bounds of the first component, as the program normalises."""
    lo, hi = k[:, 0].min(), k[:, 0].max()
    return ((k - lo) / (hi - lo) * (N - 1)).float()


def inputs(c, seed):
    """(trajectory in grid units [M, dim], density [M], samples [M, coils], frame sizes or None), on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    N, turn = grid_size(c), float((seed * 0.6180339887) % 1.0) * math.pi
    sizes = None
    if c["frames"]:
        ks = [spiral(int(n), c["readout"], turn) for n in frame_shots(c)]
        sizes = np.array([k.shape[0] for k in ks], np.int64)
        t, k = torch.cat([to_grid(k, N) for k in ks]), torch.cat(ks)
    else:
        k = k_space(c, turn)
        t = to_grid(k, N)
    rho = k.norm(dim=1).float()
    dcf = (rho ** (c["dim"] - 1)).contiguous()
    # noise on an object's spectrum: large near the centre, a few per cent of that at the edge
    data = torch.randn(t.shape[0], 2 * c["coils"], generator=gen, device="cuda")
    data *= (0.05 + 1.0 / (1.0 + 40.0 * rho))[:, None]
    return t.contiguous(), dcf, torch.view_as_complex(data.view(t.shape[0], c["coils"], 2)), sizes


def batch(c, seed):
    """A feature table with targets, and the row indices of one batch."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    B = c["shots"]
    rows = 2 * B
    x = torch.rand(rows, 8, generator=gen, device="cuda")
    x[:, 1] = 2 * x[:, 1] - 1
    y = torch.sin(3 * x[:, 0]) + x[:, 3] - 0.5 * x[:, 7] + 0.1 * torch.randn(rows, generator=gen, device="cuda")
    return x, y.contiguous(), torch.randperm(rows, generator=gen, device="cuda")[:B].contiguous()


def network(dim):
    z = np.load(os.path.join(PACKAGE, "ldcf_kooshball.npz" if dim == 3 else "ldcf_radial2d.npz"), allow_pickle=False)
    return z["params"], float(z["mu"]), float(z["sigma"]), int(z["base"])


# --------------------------------------------------------------- the passes
_context = None


def context():
    """One context for the process, as a program holds it."""
    global _context
    if _context is None:
        torch.cuda.init()
        _context = hip.Context(0)
    return _context


class View:
    """A device buffer of the library, for torch.as_tensor; keeps its owner alive."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (int(ptr), False), "version": 2}


def view(owner, shape, kind):
    return torch.as_tensor(View(owner, owner.ptr, shape, kind), device="cuda")


def prepare(c, seed):
    ctx = context()
    if c["kind"] == "gradient":
        x, y, idx = batch(c, seed)
        mlp = hip.MLP(ctx)
        params, mu, sigma, base = network(3)
        mlp.set_params(params, mu, sigma)
        mlp.base = base
        buffers = []
        for t in (x, y, idx):
            b = hip.DeviceBuffer(ctx, t.numel() * t.element_size())
            view(b, tuple(t.shape), "<i8" if t.dtype == torch.int64 else "<f4").copy_(t)
            buffers.append(b)
        torch.cuda.synchronize()
        return dict(kind="gradient", mlp=mlp, x=buffers[0], y=buffers[1], idx=buffers[2], B=c["shots"])
    N, rc, dim, C, F = grid_size(c), crop(c), c["dim"], c["coils"], c["frames"]
    t, dcf, data, sizes = inputs(c, seed)
    torch.cuda.synchronize()
    M = t.shape[0]
    s = hip.Samples(ctx, dim, M, C, hip.FR_SAMPLES_C16 if c["half"] else hip.FR_SAMPLES_C64, sizes)
    g = hip.Grids(ctx, dim, N, C, F)
    lut = kernel_table(c["og"])
    S = dict(kind=c["kind"], ctx=ctx, s=s, g=g, N=N, rc=rc, lut=lut, grid=view(g, (C, g.cells), "<c8"))
    if c["kind"] == "scan":
        S.update(t=t, dcf=dcf, data=data, dim=dim)
    else:
        s.set_traj_device(t.data_ptr(), dim)
        s.set_dcf_device(dcf.data_ptr())
        s.set_data_device(data.data_ptr(), hip.FR_LAYOUT_SAMPLE_MAJOR)
        S["plan"] = hip.Plan(ctx, s, N, 4.0, lut)
    if c["kind"] == "degrid":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed + 1)
        S["grid"].copy_(torch.view_as_complex(torch.randn(C, g.cells, 2, generator=gen, device="cuda")))
        S["out"] = hip.DeviceBuffer(ctx, 8 * M * C)
        S["samples"] = view(S["out"], (M, C), "<c8")
    elif c["kind"] != "grid":
        S["fft"] = hip.FFT(ctx, dim, N, C * max(F, 1), +1)
        S["img"] = hip.DeviceBuffer(ctx, 4 * rc[0] * rc[1] * rc[2] * max(F, 1))
        S["image"] = view(S["img"], (max(F, 1) * rc[2], rc[1], rc[0]), "<f4")
        centre = np.full(dim, (N - 1) / 2.0, np.float32)
        S["deapod"] = hip.deapod_map(ctx, dim, N, 4.0, lut, centre, rc) if c["deapod"] else None
    if c["kind"] == "learned":
        S["mlp"] = hip.MLP(ctx)
        params, mu, sigma, base = network(dim)
        S["mlp"].set_params(params, mu, sigma)
        S["mlp"].base = base
    if c["kind"] == "pils":
        S["map"] = hip.Grids(ctx, dim, N, C)
    ctx.sync()
    if c["graph"]:
        S["graph"] = hip.Graph(S["plan"], s, g, S["fft"], rc, True, S["deapod"], S["img"])
    torch.cuda.synchronize()
    return S


def run(S):
    kind = S["kind"]
    if kind == "gradient":
        gradient, loss = S["mlp"].grad(S["x"], S["y"], S["B"], S["idx"])
        return {"gradient": gradient, "loss": loss}
    ctx, s, g = S["ctx"], S["s"], S["g"]
    if kind == "grid":
        hip.grid_execute(S["plan"], s, g)
        return S["grid"]
    if kind == "degrid":
        hip.degrid_execute(S["plan"], s, g, S["out"])
        return S["samples"]
    if "graph" in S:
        S["graph"].launch()
        return S["image"]
    if kind == "pils":
        hip.grid_execute(S["plan"], s, g)
        hip.grids_copy(ctx, g, S["map"])
        S["fft"](g)
        hip.lowfilter(ctx, S["map"], 22)
        S["fft"](S["map"])
        hip.normalize(ctx, S["map"])
        out = hip.sos_map(ctx, g, S["map"], S["rc"], True)
        return view(out, (S["rc"][2], S["rc"][1], S["rc"][0]), "<c8")
    plan = S.get("plan")
    if kind == "scan":
        s.set_traj_device(S["t"].data_ptr(), S["dim"])
        s.set_dcf_device(S["dcf"].data_ptr())
        s.set_data_device(S["data"].data_ptr(), hip.FR_LAYOUT_SAMPLE_MAJOR)
        plan = hip.Plan(ctx, s, S["N"], 4.0, S["lut"])
    elif kind == "iterative":
        hip.pipe_menon(plan, s, 10, True)
    elif kind == "learned":
        S["mlp"].dcf_from_traj(s, S["N"])
    hip.grid_execute(plan, s, g)
    hip.fft_sos(S["fft"], g, S["rc"], True, S["deapod"], S["img"])
    return S["image"]


# ------------------------------------------------------------------- sizes
def sample_count(c):
    return int(frame_shots(c).sum()) * c["readout"] if c["frames"] else c["shots"] * c["readout"]


def work(c):
    if c["kind"] == "gradient":
        B, weights = c["shots"], 8 * 64 + 64 * 64 + 64
        return {"bytes": B * (32 + 4 + 8), "flops": 6.0 * B * weights}
    N, C, M, dim = grid_size(c), c["coils"], sample_count(c), c["dim"]
    F = max(c["frames"], 1)
    cells, image = F * N ** dim, F * c["image"] ** dim
    value = 4 if c["half"] else 8
    taps = 4.0 / 3.0 * math.pi * 8.0 if dim == 3 else math.pi * 4.0       # of a kernel of width 4
    samples = M * (4 * dim + 4) + M * C * value
    gridding = 4.0 * M * C * taps
    transform = 5.0 * C * cells * dim * math.log2(N)
    kind = c["kind"]
    if kind == "grid":
        return {"bytes": samples + 8 * C * cells, "flops": gridding}
    if kind == "degrid":
        return {"bytes": 4 * dim * M + 8 * C * cells + 8 * M * C, "flops": gridding}
    w = {"bytes": samples + 4 * image, "flops": gridding + transform}
    if kind == "iterative":
        # each iteration reads the trajectory and the density and writes the density
        w = {"bytes": w["bytes"] + 10 * M * (4 * dim + 8), "flops": w["flops"] + 10 * 8.0 * M * taps}
    elif kind == "learned":
        w = {"bytes": w["bytes"] + M * (4 * dim + 4), "flops": w["flops"] + 2.0 * M * (8 * 64 + 64 * 64 + 64)}
    elif kind == "pils":
        w = {"bytes": samples + 8 * image, "flops": gridding + 2 * transform}
    return w


# --------------------------------------------------------- values in 64 bits
def taps_of(t, N, z_frame, lut):
    """For each kernel offset: accepted samples, their cells and their weights.  Which cells a sample reaches and
    which table entry it takes are decided in FP32, as the gridding is defined; the weights are then 64-bit."""
    dim, two = t.shape[1], torch.tensor(2.0, device="cuda")
    start = torch.ceil(t - two)
    table = torch.from_numpy(lut).double().cuda()
    for o in np.ndindex(*([4] * dim)):
        cell = [start[:, d] + o[d] for d in range(dim)]
        sq = [(cell[d] - t[:, d]) ** 2 for d in range(dim)]
        d2 = sq[1] + sq[0] if dim == 2 else (sq[2] + sq[1]) + sq[0]
        dist = d2.double().sqrt().float()
        keep = dist < 2.0
        for d in range(dim):
            keep &= (cell[d] >= 0) & (cell[d] <= N - 1)
        i = keep.nonzero().squeeze(1)
        q = ((dist[i].double() / 2.0).float() * float(L - 1)).double()
        at = cell[1][i].long() * N + cell[0][i].long()
        if dim == 3:
            at += cell[2][i].long() * (N * N)
        if z_frame is not None:
            at += z_frame[i] * (N * N)
        yield i, at, table[torch.floor(q + 0.5).long()]


def grid64(t, w, data, N, cells, z_frame, lut):
    """[coils, cells] complex128: the sums that gridding defines."""
    M, C = data.shape
    out = torch.zeros(cells, 2 * C, dtype=torch.float64, device="cuda")
    step = max(1, 40_000_000 // (2 * C))
    for a in range(0, M, step):
        b = min(M, a + step)
        v = torch.view_as_real(data[a:b].to(torch.complex128)).reshape(b - a, 2 * C) * w[a:b, None].double()
        for i, at, weight in taps_of(t[a:b], N, None if z_frame is None else z_frame[a:b], lut):
            out.index_add_(0, at, v[i] * weight[:, None])
    return torch.view_as_complex(out.view(cells, C, 2)).T


def degrid64(t, grid, N, lut):
    """[M, coils] complex128."""
    rows = grid.T.contiguous()
    M, C = t.shape[0], rows.shape[1]
    out = torch.zeros(M, C, dtype=torch.complex128, device="cuda")
    step = max(1, 20_000_000 // C)
    for a in range(0, M, step):
        b = min(M, a + step)
        for i, at, weight in taps_of(t[a:b], N, None, lut):
            out[a:b].index_add_(0, i, rows[at].to(torch.complex128) * weight[:, None])
    return out


def transform64(grid, c, N):
    """[coils, (frames or z), y, x]: the unnormalised transform, shifted and cropped."""
    dim, C, F, n = c["dim"], grid.shape[0], c["frames"], c["image"]
    axes = (-3, -2, -1) if dim == 3 else (-2, -1)
    a = (N - n) // 2
    out = []
    for k in range(C):
        g = grid[k].contiguous().view((N, N, N) if dim == 3 else (max(F, 1), N, N))
        v = torch.fft.fftshift(torch.fft.ifftn(g, dim=axes, norm="forward"), dim=axes)
        out.append((v[a:a + n] if dim == 3 else v)[:, a:a + n, a:a + n].clone())
    return torch.stack(out)


def density64(t, N, lut):
    """10 Pipe-Menon iterations from ones.  Each offset's taps are sorted by cell once, and a cell's sum is the
    difference of two running sums."""
    M, dim = t.shape
    taps = []
    for i, at, weight in taps_of(t, N, None, lut):
        at, order = at.sort()
        cells, counts = torch.unique_consecutive(at, return_counts=True)
        taps.append((i[order].int(), at.int(), weight[order], cells, counts.cumsum(0)))
    w = torch.ones(M, dtype=torch.float64, device="cuda")
    for _ in range(10):
        g = torch.zeros(N ** dim, dtype=torch.float64, device="cuda")
        for i, at, weight, cells, ends in taps:
            g[cells] += torch.diff((w[i] * weight).cumsum(0)[ends - 1], prepend=g.new_zeros(1))
        d = torch.zeros(M, dtype=torch.float64, device="cuda")
        for i, at, weight, cells, ends in taps:
            d[i] += g[at] * weight
        w = torch.where(d > 0, w / d, torch.zeros_like(w))
    return w


def box_count(h, r):
    """Samples within r cells of each cell (a cube of 2 r + 1), from the histogram h."""
    for d in range(h.dim()):
        n = h.shape[d]
        s = torch.cat([torch.zeros_like(h.narrow(d, 0, 1)), h.cumsum(d)], d)
        i = torch.arange(n, device="cuda")
        h = s.index_select(d, (i + r + 1).clamp(max=n)) - s.index_select(d, (i - r).clamp(min=0))
    return h


def features64(t, N):
    """The eight features of the density network; cells and shells are decided in FP32."""
    M, dim = t.shape
    u = ((t - 0.5 * (N - 1)).double() / (0.5 * N)).float()
    r2 = u[:, 0] * u[:, 0] + u[:, 1] * u[:, 1]
    r2 = r2 + u[:, 2] * u[:, 2] if dim == 3 else r2
    r = r2.double().sqrt().float()
    rho = r * (0.5 * N)
    cell = torch.floor(t + 0.5).clamp(0, N - 1).long()
    at = cell[:, 1] * N + cell[:, 0] + (cell[:, 2] * N * N if dim == 3 else 0)
    h = torch.bincount(at, minlength=N ** dim).view((N,) * dim)
    shells = int(math.ceil(N * math.sqrt(dim))) + 2
    b = torch.floor(2 * rho).clamp(0, shells - 1).long()
    lo = b.double() / 2
    hi = lo + 0.5
    cells = 4.0 / 3.0 * math.pi * (hi ** 3 - lo ** 3) if dim == 3 else math.pi * (hi ** 2 - lo ** 2)
    u, r = u.double(), r.double()
    f = torch.zeros(M, 8, dtype=torch.float64, device="cuda")
    f[:, 0] = torch.log1p(rho.double()) / 5
    f[:, 1] = torch.atan2(u[:, 1], u[:, 0]) / math.pi
    f[:, 2] = 0.5
    if dim == 3:
        f[:, 2] = torch.where(r > 0, torch.acos((u[:, 2] / r.clamp(min=1e-30)).clamp(-1, 1)) / math.pi, f[:, 2])
    for q, radius in enumerate((1, 2, 4)):
        f[:, 3 + q] = torch.log1p((box_count(h, radius).view(-1)[at] - 1).double()) / 8
    f[:, 6] = (rho.max() - rho).clamp(max=4.0).double() / 4
    f[:, 7] = torch.log1p(torch.bincount(b, minlength=shells)[b].double() / cells) / 8
    return f


def layers64(params):
    """W1, b1, W2, b2, w3, b3 in 64 bits, the weight matrices with their BF16 values."""
    p, parts, a = torch.from_numpy(np.asarray(params, np.float32)).cuda(), [], 0
    for shape in ((8, 64), (64,), (64, 64), (64,), (64,), (1,)):
        n = int(np.prod(shape))
        v = p[a:a + n].view(shape)
        parts.append((v.bfloat16() if len(parts) in (0, 2, 4) else v).double())
        a += n
    return parts


def network64(x, layers):
    W1, b1, W2, b2, w3, b3 = layers
    h = torch.nn.functional.silu(x @ W1 + b1)
    return torch.nn.functional.silu(h @ W2 + b2) @ w3 + b3


def exact(c, seed):
    if c["kind"] == "gradient":
        x, y, idx = batch(c, seed)
        layers = [v.requires_grad_() for v in layers64(network(3)[0])]
        loss = ((network64(x[idx].double(), layers) - y[idx].double()) ** 2).mean()
        loss.backward()
        return {"gradient": torch.cat([v.grad.reshape(-1) for v in layers]), "loss": loss.detach()}
    N, C = grid_size(c), c["coils"]
    t, dcf, data, sizes = inputs(c, seed)
    lut = kernel_table(c["og"])
    if c["kind"] == "degrid":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed + 1)
        return degrid64(t, torch.view_as_complex(torch.randn(C, N ** c["dim"], 2, generator=gen, device="cuda")), N, lut)
    if c["half"]:
        data = torch.view_as_complex(torch.view_as_real(data).half().float())
    w = dcf
    if c["kind"] == "iterative":
        w = density64(t, N, lut)
    elif c["kind"] == "learned":
        params, mu, sigma, base = network(c["dim"])
        layers, w = layers64(params), []
        f = features64(t, N)
        for a in range(0, f.shape[0], 1 << 20):
            x = f[a:a + (1 << 20)]
            w.append(torch.exp(mu + sigma * network64(x, layers) - (8 * x[:, base] if base >= 0 else 0)))
        w = torch.cat(w)
        del f
    frame = None if sizes is None else torch.repeat_interleave(torch.arange(len(sizes), device="cuda"),
                                                               torch.from_numpy(sizes).cuda())
    g = grid64(t, w, data, N, max(c["frames"], 1) * N ** c["dim"], frame, lut)
    del t, data
    if c["kind"] == "grid":
        return g
    if c["kind"] == "pils":
        i = torch.arange(N, device="cuda")
        r = ((i - N // 2) ** 2)[:, None] + ((i - N // 2) ** 2)[None, :]
        at = ((r.double() / (2.0 * 22 * 22 / 4.0)).float().double() * 100).long()
        low = torch.where(at < 2000, torch.exp(-at.double() / 100), torch.zeros(1, dtype=torch.float64, device="cuda"))
        v, m = transform64(g, c, N), transform64(g * low.view(-1), c, N)
        return (v * (m / (m.abs() ** 2).sum(0).sqrt()).conj()).sum(0)
    v = (transform64(g, c, N).abs() ** 2).sum(0).sqrt()
    if c["deapod"]:
        centre = torch.full((1, c["dim"]), (N - 1) / 2.0, device="cuda")
        one = torch.ones(1, 1, dtype=torch.complex64, device="cuda")
        flat = dict(c, frames=0)
        v = v / transform64(grid64(centre, torch.ones(1, device="cuda"), one, N, N ** c["dim"], None, lut), flat, N)[0].abs()
    return v
