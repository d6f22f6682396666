"""The work a user of this package has it do, as cases that a timing program can run.

``listed()`` holds one case per kind of work, from the smallest call to the largest; ``draw(rng)`` gives
more cases of the same kinds over the whole range of sizes, ragged ones among them.  A case is prepared
once (inputs on the GPU, made from a seed, and the network or view sets a program keeps), then ``run`` makes one
pass through the package's public entry points.  ``exact`` states the outputs in 64 bits with plain torch, from
the definitions of the operators, without this package.

Kinds:
  siddon, interpolated   forward projection (tigre_amd.Ax) of a volume stored as float32, bfloat16 or float16
  fdk_bp, matched        backprojection (tigre_amd.Atb)
  tv, awtv, piccs        the TV steps of the POCS algorithms (minTV, AwminTV, minPICCS)
  rof                    the ROF denoiser of SART-TV and FISTA (tvdenoise)
  fdk                    a whole FDK reconstruction (algorithms.fdk): weights, ramp filter, backprojection
  ossart                 a whole OS-SART reconstruction (algorithms.ossart), set-up of the weights included
  cnn, cnn_grad          the learned proximal network: inference on a volume, gradients on a batch of crops
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tigre_amd
from tigre_amd.algorithms import fdk, ossart
from tigre_amd.geometry import cone_geometry
from tigre_amd.learned import ResidualCNN

DEV = "cuda"
DSO, DSD = 1000.0, 1536.0  # the source distances of the package's default geometry
CHUNK = 1 << 25            # elements of the largest temporaries of exact()
TYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def _scan(name, kind, volume, detector, views, dtype="float32", off_u=0.0, off_v=0.0, **more):
    nz, ny, nx = volume
    case = {"kind": kind, "nz": nz, "ny": ny, "nx": nx, "nv": detector[0], "nu": detector[1], "views": views,
            "dtype": dtype, "off_u": off_u, "off_v": off_v, **more}
    return {"name": name, **case} if name else case


def _image(name, kind, volume, iterations):
    nz, ny, nx = volume
    case = {"kind": kind, "nz": nz, "ny": ny, "nx": nx, "iterations": iterations}
    return {"name": name, **case} if name else case


def _net(name, kind, batch, volume):
    nz, ny, nx = volume
    case = {"kind": kind, "batch": batch, "nz": nz, "ny": ny, "nx": nx}
    return {"name": name, **case} if name else case


def listed():
    return [
        # the smallest call: the low-resolution preset, one subset of views of an iterative reconstruction
        _scan("siddon_64_subset", "siddon", (64, 64, 64), (128, 128), 20),
        # the headline projection: the high-resolution preset, a full turn in one-degree steps
        _scan("siddon_512", "siddon", (512, 512, 512), (512, 512), 360),
        # ragged volume and detector, detector offset, the narrow storage of the Krylov solvers
        _scan("siddon_ragged_bf16", "siddon", (170, 230, 201), (190, 243), 97, "bfloat16", 7.3, -3.1),
        # the smooth projector of FISTA, at an ordinary size
        _scan("interpolated_256", "interpolated", (256, 256, 256), (256, 256), 180),
        # the headline backprojection
        _scan("fdk_bp_512", "fdk_bp", (512, 512, 512), (512, 512), 360),
        # the adjoint-weighted backprojection of the Krylov solvers, ragged sizes
        _scan("matched_ragged", "matched", (191, 256, 237), (250, 301), 180, "float32", 4.0, 2.5),
        # the TV step of one ASD-POCS iteration
        _image("tv_256", "tv", (256, 256, 256), 20),
        # the denoising step of one SART-TV iteration, ragged
        _image("rof_ragged", "rof", (150, 181, 170), 50),
        # a whole analytic reconstruction
        _scan("fdk_256", "fdk", (256, 256, 256), (256, 256), 180),
        # a whole iterative reconstruction: six subsets of twenty views
        _scan("ossart_96", "ossart", (96, 96, 96), (96, 96), 120, iterations=3),
        # the learned step on a volume
        _net("cnn_128", "cnn", 1, (128, 128, 128)),
        # one training step's gradients: the default minibatch of 32^3 crops
        _net("cnn_grad_8x32", "cnn_grad", 8, (32, 32, 32)),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _volume(rng, lo, hi):
    n = _log(rng, lo, hi)
    return tuple(max(lo // 2, int(n * rng.uniform(0.6, 1.0))) for _ in range(3))


def draw(rng):
    kind = rng.choice(("siddon", "siddon", "interpolated", "fdk_bp", "matched", "matched", "tv", "awtv", "piccs", "rof",
                       "fdk", "ossart", "cnn", "cnn_grad"))
    if kind in ("tv", "awtv", "piccs"):
        return _image(None, kind, _volume(rng, 40, 400), rng.choice((5, 10, 20)))
    if kind == "rof":
        return _image(None, kind, _volume(rng, 40, 256), rng.choice((20, 50)))
    if kind == "cnn":
        return _net(None, kind, 1, _volume(rng, 24, 200))
    if kind == "cnn_grad":
        return _net(None, kind, rng.choice((4, 8, 16)), tuple(rng.randint(17, 40) for _ in range(3)))
    top = {"siddon": 448, "interpolated": 288, "fdk_bp": 448, "matched": 448, "fdk": 320, "ossart": 112}[kind]
    vol = _volume(rng, 40, top)
    n = max(vol)
    det = tuple(max(32, int(n * rng.uniform(0.8, 1.3))) for _ in range(2))
    views = _log(rng, 18, 200) if kind != "ossart" else rng.randint(50, 130)
    offsets = {}
    dtype = "float32"
    if kind in ("siddon", "interpolated", "fdk_bp", "matched"):
        dtype = rng.choice(("float32", "float32", "bfloat16", "float16"))
        if rng.random() < 0.5:
            offsets = {"off_u": round(rng.uniform(-8, 8), 2), "off_v": round(rng.uniform(-8, 8), 2)}
    more = {"iterations": rng.randint(1, 3)} if kind == "ossart" else {}
    return _scan(None, kind, vol, det, views, dtype, **offsets, **more)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _voxel(case):
    """Voxel size in mm: a 256 mm field of view."""
    return 256.0 / max(case["nz"], case["ny"], case["nx"])


def _pixel(case):
    """Pixel size in mm: a 409.6 mm detector."""
    return 409.6 / max(case["nv"], case["nu"])


def _geometry(case):
    n = (case["nz"], case["ny"], case["nx"])
    d, p = _voxel(case), _pixel(case)
    geo = cone_geometry(n, tuple(k * d for k in n), (case["nv"], case["nu"]), (p, p), DSO, DSD)
    geo.offDetector = np.array([case["off_v"], case["off_u"]])
    return geo, _angles(case)


def _angles(case):
    return np.linspace(0, 2 * np.pi, case["views"], endpoint=False)


def _ellipsoids(case, seed, count=12):
    """Rows (z, y, x centre, z, y, x semi-axis, attenuation per mm), mm."""
    g = torch.Generator().manual_seed(int(seed))
    r = torch.rand(count, 7, generator=g, dtype=torch.float64)
    d = _voxel(case)
    half = torch.tensor([case["nz"], case["ny"], case["nx"]], dtype=torch.float64) * d / 2
    e = torch.empty(count, 7, dtype=torch.float64)
    e[:, :3] = (r[:, :3] - 0.5) * 1.2 * half
    e[:, 3:6] = (0.08 + 0.4 * r[:, 3:6]) * half
    e[:, 6] = 0.002 + 0.02 * r[:, 6]
    return e


def _phantom(case, seed, noise):
    d = _voxel(case)
    n = (case["nz"], case["ny"], case["nx"])
    z, y, x = [(torch.arange(k, device=DEV, dtype=torch.float32) + (0.5 - k / 2)) * d for k in n]
    vol = torch.zeros(n, dtype=torch.float32, device=DEV)
    for c in _ellipsoids(case, seed).tolist():
        r = (((z - c[0]) / c[3]) ** 2)[:, None, None] + (((y - c[1]) / c[4]) ** 2)[None, :, None] \
            + (((x - c[2]) / c[5]) ** 2)[None, None, :]
        vol += (r <= 1.0) * c[6]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    vol += noise * torch.randn(n, generator=g, device=DEV)
    return vol


def _sinogram(case, seed, noise=0.005):
    """Line integrals of the ellipsoids in closed form, with noise; (views, nv, nu)."""
    d, p = _voxel(case), _pixel(case)
    nv, nu = case["nv"], case["nu"]
    out = torch.empty(case["views"], nv, nu, dtype=torch.float32, device=DEV)
    a = torch.as_tensor(_angles(case), device=DEV, dtype=torch.float32)
    ud = (torch.arange(nu, device=DEV, dtype=torch.float32) + (0.5 - nu / 2)) * p + case["off_u"]
    vd = (torch.arange(nv, device=DEV, dtype=torch.float32) + (0.5 - nv / 2)) * p + case["off_v"]
    ca, sa = torch.cos(a)[:, None], torch.sin(a)[:, None]
    dx, dy, dz = -DSD * ca - ud * sa, -DSD * sa + ud * ca, vd          # source to pixel
    length = torch.sqrt((DSD ** 2 + ud ** 2)[None, :] + (vd ** 2)[:, None])
    rows = max(1, CHUNK // (nv * nu))
    for i in range(0, case["views"], rows):
        s = slice(i, i + rows)
        acc = torch.zeros(len(a[s]), nv, nu, device=DEV)
        for cz, cy, cx, az, ay, ax, w in _ellipsoids(case, seed).tolist():
            ox, oy, oz = (DSO * ca[s] - cx) / ax, (DSO * sa[s] - cy) / ay, -cz / az
            qa = ((dx[s] / ax) ** 2 + (dy[s] / ay) ** 2)[:, None, :] + ((dz / az) ** 2)[None, :, None]
            qb = (ox * dx[s] / ax + oy * dy[s] / ay)[:, None, :] + (oz * dz / az)[None, :, None]
            qc = (ox ** 2 + oy ** 2 + oz * oz - 1.0)[:, :, None]
            disc = torch.clamp(qb * qb - qa * qc, min=0.0)
            acc += (2.0 * w) * torch.sqrt(disc) / qa
        out[s] = acc * length
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    out += noise * torch.randn(out.shape, generator=g, device=DEV)
    return out


def _weights(seed):
    """Weights and biases of the network, as a trained one would be loaded."""
    g = torch.Generator().manual_seed(int(seed))
    shapes = [(27, 32, 1)] + [(27, 32, 32)] * 4 + [(27, 1, 32)]
    W = [torch.randn(s, generator=g) * (2.0 / (27 * s[2])) ** 0.5 for s in shapes]
    b = [0.05 * torch.randn(s[1], generator=g) for s in shapes]
    return [w.numpy() for w in W], [v.numpy() for v in b]


def _net_input(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    n = (case["batch"], case["nz"], case["ny"], case["nx"])
    x = torch.rand(n, generator=g, device=DEV)
    for dim in (1, 2, 3):  # smooth on the scale of a few voxels, as an image is
        x = (x + torch.roll(x, 1, dim) + torch.roll(x, 2, dim)) / 3
    return x.contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("siddon", "interpolated"):
        geo, angles = _geometry(case)
        return {"case": case, "x": _phantom(case, seed, 0.0005).to(TYPES[case["dtype"]]), "geo": geo, "angles": angles}
    if kind in ("fdk_bp", "matched", "fdk", "ossart"):
        geo, angles = _geometry(case)
        return {"case": case, "x": _sinogram(case, seed).to(TYPES[case["dtype"]]), "geo": geo, "angles": angles}
    if kind in ("tv", "awtv", "piccs", "rof"):
        state = {"case": case, "x": _phantom(case, seed, 0.001 if kind != "rof" else 0.0005)}
        if kind == "piccs":
            state["prior"] = _phantom(case, seed, 0.0)
        if kind == "rof":  # im3ddenoise hands the denoiser an image between 0 and 1
            state["x"] -= state["x"].min()
            state["x"] /= state["x"].max()
        return state
    W, b = _weights(seed)
    net = ResidualCNN(seed=0)
    net.load({"W": W, "b": b, "data_scale": 1.0})
    state = {"case": case, "x": _net_input(case, seed), "net": net}
    if kind == "cnn_grad":
        state["dout"] = (_net_input(case, seed + 1) - 0.5) / state["x"].numel() ** 0.5
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "siddon":
        return tigre_amd.Ax(x, state["geo"], state["angles"])
    if kind == "interpolated":
        return tigre_amd.Ax(x, state["geo"], state["angles"], "interpolated")
    if kind == "fdk_bp":
        return tigre_amd.Atb(x, state["geo"], state["angles"], "FDK")
    if kind == "matched":
        return tigre_amd.Atb(x, state["geo"], state["angles"], "matched")
    if kind == "fdk":
        return fdk(x, state["geo"], state["angles"], return_tensor=True)
    if kind == "ossart":
        return ossart(x, state["geo"], state["angles"], case["iterations"], return_tensor=True)
    if kind == "tv":
        return tigre_amd.minTV(x, _step(case), case["iterations"])
    if kind == "awtv":
        return tigre_amd.AwminTV(x, _step(case), case["iterations"], delta=-0.02)
    if kind == "piccs":
        return tigre_amd.minPICCS(x, state["prior"], _step(case), case["iterations"])
    if kind == "rof":
        return tigre_amd.tvdenoise(x, case["iterations"], 50.0)
    net = state["net"]
    if kind == "cnn":
        return net.forward(x[0])
    out = net.forward(x, keep=True)
    dW, db = net.backward(state["dout"])
    return {"out": out, "dW": dW, "db": db}


def _step(case):
    """Step length of the TV descent: 0.002 of a typical change of the image (its norm grows with the voxel count)."""
    return 2e-5 * (case["nz"] * case["ny"] * case["nx"]) ** 0.5


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    vox = case["nz"] * case["ny"] * case["nx"]
    if kind in ("tv", "awtv", "piccs", "rof"):
        # per voxel and iteration: three differences, their norm, the divergence and the update; piccs twice
        ops = {"tv": 22, "awtv": 34, "piccs": 44, "rof": 30}[kind]
        reads = 2 if kind == "piccs" else 1
        return {"bytes": 4.0 * vox * (reads + 1), "flops": float(ops) * vox * case["iterations"]}
    if kind in ("cnn", "cnn_grad"):
        vox *= case["batch"]
        macs = 27 * (32 + 4 * 32 * 32 + 32)
        weights = 4.0 * (macs + 5 * 32 + 1)
        if kind == "cnn":
            return {"bytes": 8.0 * vox + weights, "flops": 2.0 * macs * vox}
        # forward, weight gradients of every layer, data gradients of all but the first
        return {"bytes": 12.0 * vox + 2 * weights, "flops": 2.0 * vox * (2 * macs + 27 * (4 * 32 * 32 + 32))}
    item = 4.0 if case["dtype"] == "float32" else 2.0
    pix = case["views"] * case["nv"] * case["nu"]
    nbytes = item * (vox + pix)
    n = (case["nx"] + case["ny"]) / 2
    if kind == "siddon":        # about 1.5 n crossings a ray, one multiply-add each
        return {"bytes": nbytes, "flops": 2 * 1.5 * n * pix}
    if kind == "interpolated":  # two samples a voxel, seven interpolations and a sum each
        return {"bytes": nbytes, "flops": 2 * n * 22.0 * pix}
    update = 12.0 if kind != "matched" else 20.0  # projection of the voxel, bilinear sample, weight
    back = update * vox * case["views"]
    if kind == "fdk":
        length = 2 * 2 ** math.ceil(math.log2(2 * case["nu"]))
        back += 5.0 * length * math.log2(length) * case["views"] * case["nv"]
    if kind == "ossart":
        back = case["iterations"] * (back + 2 * 1.5 * n * pix + 5.0 * pix)
    return {"bytes": nbytes, "flops": back}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
_F32 = np.float32


class _Exact:
    """The scan of a case in 64 bits, from the single-precision values the operators are given."""

    def __init__(self, case, voxel=None, size=None, volume=None):
        d, p = _voxel(case), _pixel(case)
        self.n = volume or (case["nz"], case["ny"], case["nx"])
        self.d = tuple(float(_F32(v)) for v in ((d, d, d) if voxel is None else voxel))  # z, y, x
        self.s = tuple(float(_F32(v)) for v in ([k * d for k in self.n] if size is None else size))
        self.nv, self.nu = case["nv"], case["nu"]
        self.dp = float(_F32(p))
        self.off_u, self.off_v = float(_F32(case["off_u"])), float(_F32(case["off_v"]))
        self.angles = _F32(_angles(case)).astype(np.float64)

    def rays(self, a, centre):
        """Source and source-to-pixel vectors (x, y, z) of one view in voxels, the volume's corner (or, with
        centre, its first voxel's centre) at the origin.  Vectors are (nv, nu)."""
        ca, sa = math.cos(a), math.sin(a)
        u = (torch.arange(self.nu, device=DEV, dtype=torch.float64) + (0.5 - self.nu / 2)) * self.dp + self.off_u
        v = (torch.arange(self.nv, device=DEV, dtype=torch.float64) + (0.5 - self.nv / 2)) * self.dp + self.off_v
        sz, sy, sx = [s / 2 - (d / 2 if centre else 0.0) for s, d in zip(self.s, self.d)]
        dz, dy, dx = self.d
        src = ((DSO * ca + sx) / dx, (DSO * sa + sy) / dy, sz / dz)
        o = torch.zeros(self.nv, self.nu, device=DEV, dtype=torch.float64)
        return src, (o + (-DSD * ca - u * sa) / dx, o + (-DSD * sa + u * ca) / dy, o + (v / dz)[:, None])

    def siddon(self, vol, a):
        """One view: all plane crossings of a ray inside the volume sorted, each segment in its midpoint's voxel."""
        nz, ny, nx = self.n
        src, dirs = self.rays(a, False)
        out = torch.zeros(self.nv * self.nu, device=DEV, dtype=torch.float64)
        flat = vol.reshape(-1)
        rows = max(1, CHUNK // (nx + ny + nz + 5))
        for i in range(0, out.numel(), rows):
            r = [torch.where(c.abs() < 1e-3, 0.0, c) for c in (q.reshape(-1)[i:i + rows] for q in dirs)]
            lo = torch.full_like(r[0], -math.inf)
            hi = torch.full_like(r[0], math.inf)
            cross = []
            for c, s, n in zip(r, src, (nx, ny, nz)):
                flat_axis = c == 0
                inv = 1.0 / torch.where(flat_axis, 1.0, c)
                t0, t1 = (0.0 - s) * inv, (n - s) * inv
                out_of = not 0.0 < s < n
                lo = torch.maximum(lo, torch.where(flat_axis, math.inf if out_of else -math.inf, torch.minimum(t0, t1)))
                hi = torch.minimum(hi, torch.where(flat_axis, -math.inf if out_of else math.inf, torch.maximum(t0, t1)))
                k = (torch.arange(n + 1, device=DEV, dtype=torch.float64) - s)[None, :] * inv[:, None]
                cross.append(torch.where(flat_axis[:, None], math.inf, k))
            hit = lo < hi
            lo, hi = torch.where(hit, lo, 0.0), torch.where(hit, hi, 0.0)
            t = torch.cat(cross + [lo[:, None], hi[:, None]], 1)
            t = torch.sort(torch.minimum(torch.maximum(t, lo[:, None]), hi[:, None]), 1).values
            mid = 0.5 * (t[:, 1:] + t[:, :-1])
            idx = torch.zeros(mid.shape, device=DEV, dtype=torch.int64)
            for c, s, n, step in zip(r, src, (nx, ny, nz), (1, nx, nx * ny)):
                idx += (s + mid * c[:, None]).floor_().clamp_(0, n - 1).long() * step
            part = ((t[:, 1:] - t[:, :-1]) * flat[idx]).sum(1)
            dz, dy, dx = self.d
            out[i:i + rows] = part * torch.sqrt((r[0] * dx) ** 2 + (r[1] * dy) ** 2 + (r[2] * dz) ** 2)
        return out.reshape(self.nv, self.nu)

    def interpolated(self, pad, a, accuracy=0.5):
        """One view: trilinear samples every `accuracy` voxels; pad is the volume with two zero layers around."""
        nz, ny, nx = self.n
        dz, dy, dx = self.d
        src, dirs = self.rays(a, True)
        r = [q.reshape(-1) for q in dirs]
        count = torch.ceil(torch.sqrt(r[0] ** 2 + r[1] ** 2 + r[2] ** 2) / accuracy)
        st = [c / count for c in r]
        ex, ey = DSO / dx, DSO / dy
        skip = ex * ey / math.sqrt((ex * math.sin(a)) ** 2 + (ey * math.cos(a)) ** 2) - math.hypot(nx // 2, ny // 2)
        crop = math.floor(max(skip, 0.0))
        first = math.floor(crop / accuracy)
        cap = (2.0 * DSO / min(dx, dy) + crop) / accuracy
        last = torch.where(count > cap, math.ceil(cap), count)
        lo = torch.full_like(r[0], float(first))
        hi = last.clone()
        for c, s, n in zip(st, src, (nx, ny, nz)):
            inv = 1.0 / torch.where(c == 0, 1e-300, c)
            t0, t1 = (-1.0 - s) * inv, (n - s) * inv
            lo = torch.maximum(lo, torch.floor(torch.minimum(t0, t1)))
            hi = torch.minimum(hi, torch.ceil(torch.maximum(t0, t1)))
        total = torch.zeros_like(r[0])
        live = lo <= hi
        if not bool(live.any()):
            return total.reshape(self.nv, self.nu)
        m0, m1 = int(lo[live].min()), int(hi[live].max())
        flat = pad.reshape(-1)
        px, py = nx + 4, ny + 4
        step = max(1, CHUNK // (4 * total.numel()))
        for m in range(m0, m1 + 1, step):
            k = torch.arange(m, min(m + step, m1 + 1), device=DEV, dtype=torch.float64)[:, None]
            on = (k >= lo) & (k <= hi)
            w, idx = [], torch.zeros(on.shape, device=DEV, dtype=torch.int64)
            for c, s, n, stride in zip(st, src, (nx, ny, nz), (1, px, px * py)):
                q = (s + k * c).clamp_(-1.5, n + 0.5)  # beyond the border every tap is zero
                f = q.floor()
                w.append(q - f)
                idx += (f.long() + 2) * stride
            c = [flat[idx + o] for o in (0, 1, px, px + 1, px * py, px * py + 1, px * py + px, px * py + px + 1)]
            c = [c[j] + w[0] * (c[j + 1] - c[j]) for j in (0, 2, 4, 6)]
            c = [c[j] + w[1] * (c[j + 1] - c[j]) for j in (0, 2)]
            total += torch.where(on, c[0] + w[2] * (c[1] - c[0]), 0.0).sum(0)
        dl = torch.sqrt((st[0] * dx) ** 2 + (st[1] * dy) ** 2 + (st[2] * dz) ** 2)
        return (total * dl).reshape(self.nv, self.nu)

    def back(self, proj, views, matched):
        """Backprojection of the views listed (indices), proj (len(views), nv, nu) in 64 bits."""
        nz, ny, nx = self.n
        dz, dy, dx = self.d
        sz, sy, sx = self.s
        out = torch.zeros(self.n, device=DEV, dtype=torch.float64)
        y = (torch.arange(ny, device=DEV, dtype=torch.float64) * dy - sy / 2 + dy / 2)[:, None]
        x = (torch.arange(nx, device=DEV, dtype=torch.float64) * dx - sx / 2 + dx / 2)[None, :]
        z = torch.arange(nz, device=DEV, dtype=torch.float64) * dz - sz / 2 + dz / 2
        pu = self.nu + 4
        slab = max(1, CHUNK // (2 * ny * nx))
        for i, view in enumerate(views):
            a = self.angles[view]
            ca, sa = math.cos(a), math.sin(a)
            pad = torch.zeros(self.nv + 4, pu, device=DEV, dtype=torch.float64)
            pad[2:-2, 2:-2] = proj[i]
            flat = pad.reshape(-1)
            depth = DSO - (x * ca + y * sa)                     # distance to the source along the central ray
            mag = DSD / depth
            ur = ((y * ca - x * sa) * mag - self.off_u) / self.dp + (self.nu / 2 - 0.5)
            u = ur.clamp(-2.0, self.nu + 0.5)
            fu = u.floor()
            wu, iu = u - fu, fu.long() + 2
            w2 = (DSO / depth) ** 2
            # the matched weight's in-plane detector coordinate, from the texture coordinate (half a pixel on)
            day = (ur + 0.5 + 0.5 - self.nu / 2) * self.dp + self.off_u
            rho = (DSO * ca - x) ** 2 + (DSO * sa - y) ** 2
            for k in range(0, nz, slab):
                zz = z[k:k + slab, None, None]
                vr = (zz * mag - self.off_v) / self.dp + (self.nv / 2 - 0.5)
                v = vr.clamp(-2.0, self.nv + 0.5)
                fv = v.floor()
                wv = v - fv
                idx = (fv.long() + 2) * pu + iu
                t = flat[idx]
                t = t + wu * (flat[idx + 1] - t)
                idx += pu
                b = flat[idx]
                b = b + wu * (flat[idx + 1] - b)
                t = t + wv * (b - t)
                if matched:
                    zd = (vr + 0.5 + 0.5 - self.nv / 2) * self.dp + self.off_v
                    t = t * ((DSD ** 2 + day ** 2 + zd ** 2) ** 1.5 / (DSD * (rho + zz ** 2)))
                else:
                    t = t * w2
                out[k:k + slab] += t
        return out * (dx * dy * dz / self.dp ** 2) if matched else out


def _ramp(x, case):
    """Cosine weight and ramp filter of FDK."""
    p = _pixel(case)
    nu, nv = case["nu"], case["nv"]
    length = 64
    while length <= 2 * nu:
        length *= 2
    k = np.arange(-length // 2, length // 2)
    h = np.zeros(length)
    h[k == 0] = 0.25
    h[k % 2 == 1] = -1.0 / (np.pi * k[k % 2 == 1]) ** 2
    resp = torch.as_tensor(2 * np.abs(np.fft.fft(h))[: length // 2 + 1], device=DEV)
    u = (torch.arange(nu, device=DEV, dtype=torch.float64) + (0.5 - nu / 2)) * p
    v = (torch.arange(nv, device=DEV, dtype=torch.float64) + (0.5 - nv / 2)) * p
    x = x * (DSD / torch.sqrt(DSD ** 2 + u[None, :] ** 2 + v[:, None] ** 2))
    pad = (length - nu) // 2
    rows = torch.nn.functional.pad(x, (pad, length - nu - pad))
    out = torch.fft.irfft(torch.fft.rfft(rows) * resp, n=length)[..., pad:pad + nu]
    return out * (DSD / DSO * (2 * math.pi / case["views"]) / (4 * p))


def _exact_ossart(case, proj):
    nz, ny, nx = case["nz"], case["ny"], case["nx"]
    d, p = _voxel(case), _pixel(case)
    g = _Exact(case)
    # ray weights: chords through a volume of 2^3 voxels, a tenth wider and as high as the detector
    size = (max(case["nv"] * p, nz * d), 1.1 * ny * d, 1.1 * nx * d)
    e = _Exact(case, [s / 2 for s in size], size, (2, 2, 2))
    ones = torch.ones(2, 2, 2, device=DEV, dtype=torch.float64)
    W = torch.stack([e.siddon(ones, a) for a in g.angles])
    W = 1.0 / torch.where(W <= d / 2, math.inf, W)
    # voxel weights: backprojected ones on a shrunk volume, averaged over z
    s = np.array([nz * d, ny * d, nx * d])
    s = s * np.max(s[1:] / np.linalg.norm(s[1:])) * 0.9
    f = _Exact(case, s / np.array([nz, ny, nx]), s)
    blocks = [list(range(i, min(i + 20, case["views"]))) for i in range(0, case["views"], 20)]
    unit = torch.ones(20, case["nv"], case["nu"], device=DEV, dtype=torch.float64)
    V = [f.back(unit[: len(b)], b, False).mean(0) for b in blocks]
    V = [torch.where(v == 0, math.inf, v) for v in V]
    x = torch.zeros(nz, ny, nx, device=DEV, dtype=torch.float64)
    for _ in range(case["iterations"]):
        for b, v in zip(blocks, V):
            r = torch.stack([W[i] * (proj[i] - g.siddon(x, g.angles[i])) for i in b])
            x = (x + g.back(r, b, False) / v).clamp_(min=0)
    return x


def _tv_direction(f, pad_z, inv_delta, eps):
    """Sum of a voxel's normalised backward differences minus its upper neighbours' components."""
    g = torch.nn.functional.pad(f[None, None], (0, 0, 0, 0, 1, 1))[0, 0] if pad_z else f
    dz, dy, dx = torch.zeros_like(g), torch.zeros_like(g), torch.zeros_like(g)
    dz[1:] = g[1:] - g[:-1]
    dy[:, 1:] = g[:, 1:] - g[:, :-1]
    dx[:, :, 1:] = g[:, :, 1:] - g[:, :, :-1]
    w = [torch.exp(-(q * inv_delta) ** 2) if inv_delta else 1.0 for q in (dz, dy, dx)]
    norm = torch.sqrt(w[0] * dz ** 2 + w[1] * dy ** 2 + w[2] * dx ** 2) + eps
    dz, dy, dx = w[0] * dz / norm, w[1] * dy / norm, w[2] * dx / norm
    v = dz + dy + dx
    v[:-1] -= dz[1:]
    v[:, :-1] -= dy[:, 1:]
    v[:, :, :-1] -= dx[:, :, 1:]
    return v[1:-1] if pad_z else v


def _exact_tv(case, x, prior):
    kind = case["kind"]
    step = float(_F32(_step(case)))
    ratio = float(_F32(0.95))
    for _ in range(case["iterations"]):
        if kind == "piccs":
            g = (1 - ratio) * _tv_direction(x, False, 0.0, 1e-6) + ratio * _tv_direction(x - prior, False, 0.0, 1e-6)
            x = x - g * (step / torch.sqrt((g * g).sum()))
        else:
            g = _tv_direction(x, True, 1.0 / float(_F32(-0.02)) if kind == "awtv" else 0.0, 1e-8)
            x = x - g * (step / torch.sqrt((g * g).sum() + 1e-7))
    return x


def _exact_rof(case, x):
    """Primal-dual iteration on the image between a mirrored slice below and a zero slice above."""
    z = torch.zeros_like(x[:1])
    f = torch.cat((x[1:2] if len(x) > 1 else z, x, z))
    u = f.clone()
    p = [torch.zeros_like(f) for _ in range(3)]
    for it in range(case["iterations"]):
        tau2 = 0.3 + 0.02 * it
        tau1 = (1.0 / tau2) * (1.0 / 6.0 - 5.0 / (15.0 + it))
        div = p[0] + p[1] + p[2]
        div[1:] -= p[0][:-1]
        div[:, 1:] -= p[1][:, :-1]
        div[:, :, 1:] -= p[2][:, :, :-1]
        u = u * (1.0 - tau1) + tau1 * (f + div / 50.0)
        p[0][:-1] += tau2 * (u[1:] - u[:-1])
        p[1][:, :-1] += tau2 * (u[:, 1:] - u[:, :-1])
        p[2][:, :, :-1] += tau2 * (u[:, :, 1:] - u[:, :, :-1])
        norm = torch.sqrt(p[0] ** 2 + p[1] ** 2 + p[2] ** 2).clamp_(min=1.0)
        p = [q / norm for q in p]
    return u[1:-1]


def _bf16(x):
    return x.float().to(torch.bfloat16).double()


def _taps(x):
    """x (N, D, H, W, C) shifted by each of the 27 taps, zeros outside."""
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    n, d, h, w, _ = x.shape
    for t in range(27):
        yield p[:, t // 9:t // 9 + d, t // 3 % 3:t // 3 % 3 + h, t % 3:t % 3 + w]


def _conv(x, w):
    n, d, h, wd, c = x.shape
    return sum(s.reshape(-1, c) @ k.T for s, k in zip(_taps(x), w)).reshape(n, d, h, wd, -1)


def _exact_cnn(case, x, W, b, dout):
    """The network with its storage types (bfloat16 weights, activations and activation gradients), 64-bit sums."""
    W = [_bf16(torch.as_tensor(w, device=DEV)) for w in W]
    b = [torch.as_tensor(v, device=DEV).double() for v in b]
    h = [_bf16(x)[..., None]]
    for l in range(5):
        h.append(_bf16(torch.relu(_conv(h[-1], W[l]) + b[l])))
        if dout is None:
            h = h[-1:]
    out = x + (_conv(h[-1], W[5])[..., 0] + b[5])
    if dout is None:
        return out[0]
    dW, db = [None] * 6, [None] * 6
    g = _bf16(dout)[..., None]
    for l in range(5, -1, -1):
        flat = g.reshape(-1, g.shape[-1])
        dW[l] = torch.stack([flat.T @ s.reshape(-1, s.shape[-1]) for s in _taps(h[l])])
        db[l] = flat.sum(0)
        if l:  # the adjoint: taps mirrored, channels swapped
            g = _bf16(_conv(g, W[l].flip(0).transpose(1, 2).contiguous()) * (h[l] > 0))
    return {"out": out, "dW": dW, "db": db}


def exact(case, seed):
    kind = case["kind"]
    state = prepare(case, seed)
    x = state["x"].double()
    if kind in ("tv", "awtv", "piccs"):
        return _exact_tv(case, x, state["prior"].double() if kind == "piccs" else None)
    if kind == "rof":
        return _exact_rof(case, x)
    if kind in ("cnn", "cnn_grad"):
        W, b = _weights(seed)
        return _exact_cnn(case, x, W, b, state["dout"].double() if kind == "cnn_grad" else None)
    g = _Exact(case)
    pix = case["views"] * case["nv"] * case["nu"]
    if kind == "siddon":
        if pix * (case["nx"] + case["ny"] + case["nz"]) > 4e9:
            return None  # too long in 64 bits
        return torch.stack([g.siddon(x, a) for a in g.angles])
    if kind == "interpolated":
        if pix * (case["nx"] + case["ny"]) > 8e9:
            return None
        pad = torch.nn.functional.pad(x[None, None], (2, 2, 2, 2, 2, 2))[0, 0].contiguous()
        return torch.stack([g.interpolated(pad, a) for a in g.angles])
    if kind == "ossart":
        return _exact_ossart(case, x)
    if case["views"] * case["nz"] * case["ny"] * case["nx"] > 2e10:
        return None
    if kind == "fdk":
        x = _ramp(x, case)
    return g.back(x, range(case["views"]), kind == "matched")
