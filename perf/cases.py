"""Performance cases of the tubular-segmentation path on one GPU.

Each case is one call (or the short chain of calls) that a program using this
framework makes on device-resident data: the anisotropic-TV cut alone, its
grid search and its ragged sets, the vesselness filter, the direction
adjustment, the gradient vector flow, and a volume's whole segmentation. The
volumes are noisy helix phantoms as in the reference experiment; frames are
those of smooth direction fields along the tube.
"""
import math

import numpy as np
import torch

from miccai2016_amd.device import default_context
from miccai2016_amd.phantom import A_ATV, GRID_DECAYS, GRID_WEIGHTINGS
from miccai2016_amd.pipeline import PipelineConfig, prepare_device, cut_parameters
from miccai2016_amd.processing.adjust_directions import AdvancedAdjuster
from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
from miccai2016_amd.processing.gradient_vector_flow import GvfGpu, GvfParameters
from miccai2016_amd.processing.qfrangi_gpu import FeatureFilter, VesselnessCalculation

WEIGHTING, DECAY = 10 ** -1.625, 10 ** 1.5   # the experiment's plain cell
MU = 0.1                                     # the experiment's flow regularisation


def _cut(name, d0, d1, d2, iters, update, bound, kind="atv", noise=1.5, aniso=1.0):
    return dict(name=name, path="cut", d0=d0, d1=d1, d2=d2, iters=iters, update=update,
                bound=bound, kind=kind, noise=noise, aniso=aniso)


def listed():
    return [
        # a region of interest cut with the class's own defaults: the criterion
        # every iteration, a stop at 1e-4
        _cut("cut_roi_default_stop", 24, 30, 37, 1000, 1, 1e-4, noise=1.0),
        # the 64^3 pipeline's cut
        _cut("cut_64", 64, 64, 64, 500, 30, 0.0),
        # one cell of the experiment's 128^3 grid, on its own
        _cut("cut_128", 128, 128, 128, 500, 30, 0.0),
        # the large single volume
        _cut("cut_256", 256, 256, 256, 1000, 30, 0.0, noise=1.0),
        # an interactive cut with foreground and background seeds
        _cut("cut_seeded_odd", 101, 117, 90, 300, 30, 0.0, kind="seeded", noise=1.0),
        # eigenvalues that differ from voxel to voxel, anisotropic voxels
        _cut("cut_pointwise", 80, 96, 72, 300, 10, 0.0, kind="pointwise", noise=1.0, aniso=2.0),
        # a row of the parameter grid on one 128^3 volume
        dict(name="grid_128", path="grid", d0=128, d1=128, d2=128, solves=16, iters=500,
             update=30, noise=1.5),
        # volumes of many shapes in one call
        dict(name="ragged_16", path="ragged", volumes=16, lo=40, hi=160, iters=300, update=30),
        # vesselness at three scales, odd sides
        dict(name="frangi_3_scales", path="frangi", d0=160, d1=131, d2=150, lo=1.0, hi=2.0,
             scales=3, noise=1.0, aniso=1.0),
        # main directions made consistent along the ridge
        dict(name="adjust_128", path="adjust", d0=128, d1=128, d2=128, noise=1.5),
        # the flow of the response-weighted directions
        dict(name="gvf_odd", path="gvf", d0=150, d1=128, d2=141, iters=200, aniso=1.0),
        # one noisy volume from image to labelling
        dict(name="segment_volume", path="segment", d0=96, d1=96, d2=96, iters=500, noise=1.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi):
    """Three sides around a common log-uniform length, each up to a third off it."""
    m = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [max(8, int(round(min(1.15 * hi, m * rng.uniform(0.7, 1.3))))) for _ in range(3)]


def draw(rng):
    path = rng.choice(["cut", "cut", "cut", "cut", "grid", "ragged", "frangi", "adjust", "gvf",
                       "segment"])
    noise = round(rng.uniform(0.5, 1.5), 2)
    aniso = rng.choice([1.0, 1.0, 1.0, 2.0])
    if path == "cut":
        d = _sides(rng, 20, 220)
        c = _cut("", *d, _log_int(rng, 100, 800), rng.choice([1, 10, 30, 30]),
                 rng.choice([0.0, 0.0, 1e-4]),
                 rng.choice(["atv", "atv", "tv", "seeded", "pointwise"]), noise, aniso)
        del c["name"]
        return c
    if path == "grid":
        d = _sides(rng, 24, 110)
        return dict(path=path, d0=d[0], d1=d[1], d2=d[2], solves=rng.randint(2, 20),
                    iters=_log_int(rng, 100, 500), update=30, noise=noise)
    if path == "ragged":
        lo = rng.randint(20, 60)
        return dict(path=path, volumes=rng.randint(3, 20), lo=lo, hi=lo + rng.randint(10, 90),
                    iters=_log_int(rng, 100, 400), update=30)
    if path == "frangi":
        d = _sides(rng, 24, 200)
        lo = round(rng.uniform(0.8, 2.0), 2)
        return dict(path=path, d0=d[0], d1=d[1], d2=d[2], lo=lo, hi=round(lo * rng.uniform(1.5, 3), 2),
                    scales=rng.randint(1, 4), noise=noise, aniso=aniso)
    if path == "adjust":
        d = _sides(rng, 32, 160)
        return dict(path=path, d0=d[0], d1=d[1], d2=d[2], noise=noise)
    if path == "gvf":
        d = _sides(rng, 20, 220)
        return dict(path=path, d0=d[0], d1=d[1], d2=d[2], iters=_log_int(rng, 40, 400), aniso=aniso)
    d = _sides(rng, 32, 140)
    return dict(path=path, d0=d[0], d1=d[1], d2=d[2], iters=_log_int(rng, 100, 600), noise=noise)


# ------------------------------------------------------------------ inputs ---

def _shape(case):
    return case["d0"], case["d1"], case["d2"]


def _voxel_size(case):
    """Slices `aniso` times as thick as the in-plane spacing."""
    return case.get("aniso", 1.0), 1.0, 1.0


def _phantom(shape, noise, gen, dev):
    """(noisy image, truth, axis-order tangent field) of a helix tube along
    axis 0, its phase drawn from the generator."""
    z, y, x = (torch.arange(s, device=dev, dtype=torch.float32) for s in shape)
    z, y, x = z[:, None, None], y[None, :, None], x[None, None, :]
    radius, pitch = 0.25 * min(shape), 0.375 * max(shape)
    tube = max(2.0, min(shape) / 16)
    w = 2 * math.pi / pitch
    phase = 2 * math.pi * torch.rand(1, generator=gen, device=dev) + w * z
    cy = (shape[1] - 1) / 2 + radius * torch.sin(phase)
    cx = (shape[2] - 1) / 2 + radius * torch.cos(phase)
    # the slice through a tube that rises at this slope is wider by its inverse cosine
    slope = math.sqrt(1 + (radius * w) ** 2)
    dy, dx = y - cy, x - cx
    along = dy * torch.cos(phase) - dx * torch.sin(phase)
    across = dy * torch.sin(phase) + dx * torch.cos(phase)
    truth = (across ** 2 + (along / slope) ** 2) <= tube ** 2
    img = truth + noise * torch.randn(shape, generator=gen, device=dev)
    tan = torch.stack([torch.ones_like(img), (radius * w * torch.cos(phase)).expand(shape),
                       (-radius * w * torch.sin(phase)).expand(shape)], -1)
    return img.float().contiguous(), truth, tan / tan.norm(dim=-1, keepdim=True)


def _smooth_directions(shape, tan, truth, gen, dev):
    """Unit vectors: the tangent inside the tube, a smooth random field beyond it."""
    coarse = torch.randn((1, 3) + tuple(max(2, s // 8) for s in shape), generator=gen, device=dev)
    v = torch.nn.functional.interpolate(coarse, size=shape, mode="trilinear", align_corners=True)
    v = torch.where(truth[..., None], tan, v[0].permute(1, 2, 3, 0))
    return v / v.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _frames(v):
    """Squeezed z-x-z angles (phi, theta, psi) of an orthonormal frame whose
    first column is v."""
    v = v.double()
    helper = torch.zeros_like(v)
    helper.scatter_(-1, v.abs().argmin(-1, keepdim=True), 1.0)
    b = torch.linalg.cross(v, helper)
    b = b / b.norm(dim=-1, keepdim=True)
    c = torch.linalg.cross(v, b)
    return torch.stack([torch.atan2(c[..., 0], -c[..., 1]), torch.acos(c[..., 2].clamp(-1, 1)),
                        torch.atan2(v[..., 2], b[..., 2])], -1).float()


def _capacities(img, noise):
    """Terminal capacities from the log-likelihood ratio of N(1, s^2) against N(0, s^2)."""
    x, var, eps = img.double(), noise ** 2, 1e-9
    pdf = lambda m: torch.exp(-(x - m) ** 2 / (2 * var)) / math.sqrt(2 * math.pi * var)
    r = torch.log((pdf(1) + eps) / (pdf(0) + eps))
    rq = 1 / math.log((1 / math.sqrt(2 * math.pi * var) + eps) / eps)
    return (rq * r.clamp_min(0)).float(), (rq * (-r).clamp_min(0)).float()


def _grad_mag_sq(img):
    return sum(g ** 2 for g in torch.gradient(img))


def _cut_fields(shape, noise, gen, dev):
    img, truth, tan = _phantom(shape, noise, gen, dev)
    quats = _frames(_smooth_directions(shape, tan, truth, gen, dev))
    cs, ct = _capacities(img, noise)
    u0 = img / (img.max() + torch.finfo(torch.float32).tiny)
    return dict(u0=u0, quats=quats, cs=cs, ct=ct, gms=_grad_mag_sq(img), truth=truth)


def _eigs(kind):
    return (1.0, 1.0, 1.0) if kind == "tv" else (1.0, A_ATV, A_ATV)


def _cut_inputs(case, seed):
    """Device inputs of a cut: u0, the frame buffer, alpha, capacities, labels."""
    ctx = default_context()
    gen = torch.Generator(device=ctx.device).manual_seed(seed)
    shape = _shape(case)
    f = _cut_fields(shape, case["noise"], gen, ctx.device)
    f["alpha"] = WEIGHTING * torch.exp(-f["gms"] / DECAY ** 2)
    f["labels"] = None
    if case["kind"] == "seeded":
        marks = torch.rand(shape, generator=gen, device=ctx.device) < 0.02
        f["labels"] = (marks * torch.where(f["truth"], 1, 2)).to(torch.uint8)
    if case["kind"] == "pointwise":
        lam = torch.rand(shape + (3,), generator=gen, device=ctx.device) * 0.9 + 0.1
        lam[..., 0] = 1.0
        f["eigs"] = torch.cat([lam.sqrt(), f["quats"]], -1).contiguous()
    else:
        f["eigs"] = f["quats"]
    return f


def _grid_cells(count, rng):
    return (rng.choice(GRID_WEIGHTINGS, count).astype(np.float32),
            rng.choice(GRID_DECAYS, count).astype(np.float32))


def _ragged_shapes(case):
    """Shapes of the set: the same for every seed, so that a pass's work is too."""
    rng = np.random.default_rng([case["volumes"], case["lo"], case["hi"]])
    return [tuple(int(s) for s in rng.integers(case["lo"], case["hi"] + 1, 3))
            for _ in range(case["volumes"])]


def _ragged_inputs(case, seed):
    ctx = default_context()
    gen = torch.Generator(device=ctx.device).manual_seed(seed)
    rng = np.random.default_rng(seed)
    shapes = _ragged_shapes(case)
    fields = [_cut_fields(s, float(rng.uniform(0.5, 1.5)), gen, ctx.device) for s in shapes]
    w, d = _grid_cells(len(shapes), rng)
    for f, wi, di in zip(fields, w, d):
        f["alpha"] = float(wi) * torch.exp(-f["gms"] / float(di) ** 2)
    packed = {k: torch.cat([f[k].reshape(-1) for f in fields])
              for k in ("u0", "quats", "alpha", "cs", "ct")}
    sizes = [math.prod(s) for s in shapes]
    offsets = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    return shapes, offsets, packed


def _image(case, seed):
    ctx = default_context()
    gen = torch.Generator(device=ctx.device).manual_seed(seed)
    return _phantom(_shape(case), case["noise"], gen, ctx.device)[0]


def _flow_input(case, seed):
    """Response-weighted directions, one field per component."""
    ctx = default_context()
    gen = torch.Generator(device=ctx.device).manual_seed(seed)
    shape = _shape(case)
    _, truth, tan = _phantom(shape, 1.0, gen, ctx.device)
    v = _smooth_directions(shape, tan, truth, gen, ctx.device)
    resp = torch.where(truth, 0.3 + 0.7 * torch.rand(shape, generator=gen, device=ctx.device),
                       0.05 * torch.rand(shape, generator=gen, device=ctx.device))
    return (v * resp[..., None]).permute(3, 0, 1, 2).contiguous()


def _filter(case):
    p = VesselnessCalculation.Parameters()
    p.bright_objects = True
    p.scales = (case["lo"], case["hi"], case["scales"])
    return FeatureFilter(p, default_context())


def _cut_params(case):
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound = case["iters"], case["update"], case.get("bound", 0.0)
    p.steps, p.cc = 0.16, 0.2
    return p


def _padded(criteria, case):
    """A cut's criterion log, zero after the iteration that stopped it."""
    out = np.zeros(-(-case["iters"] // case["update"]), criteria.dtype)
    out[:len(criteria)] = criteria
    return out


# -------------------------------------------------------------------- cases ---

def prepare(case, seed):
    ctx, path = default_context(), case["path"]
    st = dict(case=case, shape=None if path == "ragged" else _shape(case))
    if path == "cut":
        st.update(_cut_inputs(case, seed))
        st["cutter"] = CmfCutQAnisotropicGpu(_cut_params(case), ctx)
    elif path == "grid":
        gen = torch.Generator(device=ctx.device).manual_seed(seed)
        st.update(_cut_fields(st["shape"], case["noise"], gen, ctx.device))
        st["w"], st["d"] = _grid_cells(case["solves"], np.random.default_rng(seed))
        st["cutter"] = CmfCutQAnisotropicGpu(_cut_params(case), ctx)
    elif path == "ragged":
        st["shapes"], st["offsets"], st["packed"] = _ragged_inputs(case, seed)
        st["cutter"] = CmfCutQAnisotropicGpu(_cut_params(case), ctx)
    elif path == "frangi":
        st["img"], st["filter"] = _image(case, seed), _filter(case)
    elif path == "adjust":
        cfg = PipelineConfig()
        ff = _filter(dict(lo=cfg.scales[0], hi=cfg.scales[1], scales=cfg.scales[2]))
        val, quat = ff.execute_tensor(_image(case, seed), st["shape"])
        lo, hi = val.min(), val.max()
        st["resp"], st["quats"] = (val - lo) / (hi - lo), quat.clone()
        st["thresholds"] = cfg.ridge_thresholds
    elif path == "gvf":
        st["v"] = _flow_input(case, seed)
    else:
        cfg = PipelineConfig()
        cfg.cut_iters = case["iters"]
        st["img"], st["cfg"] = _image(case, seed), cfg
    return st


def run(st):
    ctx, case, path = default_context(), st["case"], st["case"]["path"]
    if path == "cut":
        cutter, kind = st["cutter"], case["kind"]
        u = cutter.execute_device(
            st["u0"].clone(), st["eigs"], st["alpha"], st["cs"], st["ct"], labels=st["labels"],
            scaling=_voxel_size(case), shape=st["shape"],
            const_sqevals=None if kind == "pointwise" else np.sqrt(_eigs(kind)))
        return dict(u=u, criteria=_padded(cutter.last_criteria, case))
    if path == "grid":
        u = st["u0"].reshape(1, -1).repeat(case["solves"], 1)
        return st["cutter"].execute_batched_device(u, case["solves"], st["w"], st["d"],
                                                   st["quats"], st["gms"], st["cs"], st["ct"],
                                                   st["shape"], _eigs("atv"))
    if path == "ragged":
        p = st["packed"]
        return st["cutter"].execute_ragged_device(p["u0"].clone(), p["quats"], p["alpha"], p["cs"],
                                                  p["ct"], st["shapes"], st["offsets"],
                                                  _eigs("atv"))
    if path == "frangi":
        val, quat = st["filter"].execute_tensor(st["img"], st["shape"], _voxel_size(case))
        return dict(response=val, frames=quat)
    if path == "adjust":
        adj = AdvancedAdjuster(threshold=st["thresholds"], qeigs=None, response=None, loader=ctx)
        dirs = adj.execute_tensor(st["quats"], st["resp"], st["shape"])
        return dict(directions=dirs, ridge_voxels=int(adj.ridge_voxels))
    if path == "gvf":
        p = GvfParameters()
        p.mu, p.tol, p.maxiter, p.normalize = MU, 0, case["iters"], False
        return GvfGpu(st["v"], p, _voxel_size(case), cl_program_loader=ctx,
                      shape=st["shape"]).execute_device()
    cfg, shape = st["cfg"], st["shape"]
    prep = prepare_device(st["img"], shape, case["noise"], cfg, ctx)
    alpha = WEIGHTING * torch.exp(-prep.gms / DECAY ** 2)
    u0 = (st["img"] / (st["img"].max() + torch.finfo(torch.float32).tiny)).reshape(-1)
    cutter = CmfCutQAnisotropicGpu(cut_parameters(cfg), ctx)
    u = cutter.execute_device(u0, prep.quats, alpha, prep.cs, prep.ct, shape=shape,
                              const_sqevals=np.sqrt(_eigs("atv")))
    return dict(u=u, frames=prep.quats, cs=prep.cs, ct=prep.ct, gms=prep.gms)


# Operations of one voxel and iteration of the cut (p-step about 35, u-step
# about 20) and of one voxel, component and step of the flow.
_CUT_FLOPS, _FLOW_FLOPS = 55.0, 15.0


def work(case):
    path = case["path"]
    n = 0 if path == "ragged" else math.prod(_shape(case))
    if path == "cut":   # u0, alpha, cs, ct, frames (and eigenvalues, labels) in, u out
        per = 32 + (12 if case["kind"] == "pointwise" else 0) + (1 if case["kind"] == "seeded" else 0)
        # where the criterion may stop the solve, half of the iterations
        its = case["iters"] * (0.5 if case["bound"] > 0 else 1)
        return dict(bytes=per * n, flops=_CUT_FLOPS * n * its)
    if path == "grid":
        return dict(bytes=(24 + 8 * case["solves"]) * n,
                    flops=_CUT_FLOPS * n * case["iters"] * case["solves"])
    if path == "ragged":
        n = sum(math.prod(s) for s in _ragged_shapes(case))
        return dict(bytes=32 * n, flops=_CUT_FLOPS * n * case["iters"])
    if path == "frangi":
        # image in, response and frames out; 15 passes of 8 sigma taps and
        # about 400 operations of the eigensolver and the response per scale
        flops = 0.0
        for s in np.linspace(case["lo"], case["hi"], case["scales"]):
            flops += n * (15 * 2 * (8 * s + 1) + 400)
        return dict(bytes=20 * n, flops=flops)
    if path == "adjust":  # frames and response in, directions out
        return dict(bytes=28 * n, flops=200.0 * n)
    if path == "gvf":
        return dict(bytes=24 * n, flops=3 * _FLOW_FLOPS * n * case["iters"])
    cfg = PipelineConfig()
    flops = n * (_CUT_FLOPS * case["iters"] + 3 * _FLOW_FLOPS * cfg.gvf_iters + 2500.0)
    return dict(bytes=32 * n, flops=flops)


# ------------------------------------------------------- values in 64 bits ---

def _diff(x, axis):
    """Forward difference, zero at the end of the axis."""
    out = torch.zeros_like(x)
    m = x.shape[axis] - 1
    out.narrow(axis, 0, m).copy_(x.narrow(axis, 1, m) - x.narrow(axis, 0, m))
    return out


def _div(x, axis):
    """Negative adjoint of _diff."""
    m = x.shape[axis] - 1
    out = torch.zeros_like(x)
    out.narrow(axis, 0, m).copy_(x.narrow(axis, 0, m))
    out.narrow(axis, 1, m).sub_(x.narrow(axis, 0, m))
    return out


def _rotation(q):
    """Rz(phi) Rx(theta) Rz(psi) as nine fields."""
    phi, theta, psi = q.double().unbind(-1)
    cf, sf, ct, st, cp, sp = (phi.cos(), phi.sin(), theta.cos(), theta.sin(), psi.cos(), psi.sin())
    return [[cf * cp - sf * ct * sp, -cf * sp - sf * ct * cp, sf * st],
            [sf * cp + cf * ct * sp, -sf * sp + cf * ct * cp, -cf * st],
            [st * sp, st * cp, ct]]


def _cut_exact(u, quats, sq, alpha, cs, ct, labels, scaling, p):
    """The cut in 64 bits; sq: the eigenvalues' square roots, numbers or fields."""
    R = _rotation(quats)
    u, alpha, cs, ct = (x.double() for x in (u, alpha, cs, ct))
    u = u.clone()
    least = min(scaling)
    ss, rs = [p.steps * least ** 2 / s for s in scaling], [1 / s for s in scaling]
    rcc = 1 / (p.cc * least ** 2)
    uf = 0.0 if labels is None else (labels & 1).double()
    ub = 1.0 if labels is None else 1.0 - ((labels & 2) != 0).double()
    h = [torch.zeros_like(u) for _ in range(3)]
    pt, tmp, criteria = torch.minimum(cs, ct), -rcc * u, []
    for i in range(p.num_iter):
        g = [_diff(tmp, k) * ss[k] for k in range(3)]
        q = [sum(R[r][k] * h[r] for r in range(3)) / sq[k] +
             sum(R[r][k] * g[r] for r in range(3)) * sq[k] for k in range(3)]
        norm = (q[0] ** 2 + q[1] ** 2 + q[2] ** 2).sqrt()
        scale = torch.where(norm > alpha, alpha / norm, torch.ones_like(norm))
        q = [q[k] * scale * sq[k] for k in range(3)]
        h = [sum(R[r][k] * q[k] for k in range(3)) for r in range(3)]
        div = sum(_div(h[k], k) * rs[k] for k in range(3))
        ps = torch.minimum(div + pt - rcc * (u - ub), cs)
        pt = torch.minimum(ps - div + rcc * (u - uf), ct)
        err = div - ps + pt
        u -= err / rcc
        tmp = err - rcc * u
        if i % p.update == 0:
            criteria.append(err.abs().sum() / (u.numel() * rcc))
            if p.error_bound > 0 and float(criteria[-1]) < p.error_bound:
                break
    return u, torch.stack(criteria).cpu().numpy() if criteria else np.zeros(0)


def _mirrored(x, taps, axis):
    """True convolution along an axis, mirrored at its ends with period 2 (n - 1)."""
    n, r = x.shape[axis], len(taps) // 2
    at = torch.arange(n, device=x.device)
    out = torch.zeros_like(x)
    for j, t in enumerate(taps):
        k = (at - (j - r)) % (2 * (n - 1))
        out += float(t) * x.index_select(axis, torch.where(k < n, k, 2 * (n - 1) - k))
    return out


def _gauss(sigma, order):
    x = np.arange(-int(4 * sigma + 0.5), int(4 * sigma + 0.5) + 1, dtype=np.float64)
    g = np.exp(-0.5 * x ** 2 / sigma ** 2)
    g /= g.sum()
    g = [g, g * -x / sigma ** 2, g * (x ** 2 - sigma ** 2) / sigma ** 4][order]
    return g * sigma ** order


def _hessian(img, sigma):
    img = img.double()
    at = {}
    for o0 in range(3):
        a = _mirrored(img, _gauss(sigma[0], o0), 0)
        for o1 in range(3 - o0):
            b = _mirrored(a, _gauss(sigma[1], o1), 1)
            at[o0, o1] = _mirrored(b, _gauss(sigma[2], 2 - o0 - o1), 2)
    return at[2, 0], at[0, 2], at[0, 0], at[1, 1], at[1, 0], at[0, 1]


def _eigenvalues(a, b, c, ab, ac, bc):
    """Eigenvalues of symmetric 3 x 3 matrices, ascending by magnitude."""
    m = torch.stack([a, ab, ac, ab, b, bc, ac, bc, c], -1).reshape(-1, 3, 3)
    eye = torch.eye(3, dtype=m.dtype, device=m.device)
    q = (a + b + c).reshape(-1) / 3
    k = m - q[:, None, None] * eye
    p = (k.square().sum((1, 2)) / 6).sqrt().clamp_min(1e-300)
    k = k / p[:, None, None]
    det = (k[:, 0, 0] * (k[:, 1, 1] * k[:, 2, 2] - k[:, 1, 2] ** 2)
           - k[:, 0, 1] * (k[:, 0, 1] * k[:, 2, 2] - k[:, 1, 2] * k[:, 0, 2])
           + k[:, 0, 2] * (k[:, 0, 1] * k[:, 1, 2] - k[:, 1, 1] * k[:, 0, 2]))
    f = torch.acos((det / 2).clamp(-1, 1)) / 3
    top, low = q + 2 * p * f.cos(), q + 2 * p * (f + 2 * math.pi / 3).cos()
    lam = torch.stack([top, 3 * q - top - low, low], -1)
    return lam.gather(-1, lam.abs().argsort(-1)).unbind(-1)


def _response_exact(img, case):
    """The multi-scale response (bright tubes, alpha = beta = 0.5, c half the
    largest eigenvalue norm of each scale)."""
    best = torch.full((img.numel(),), -math.inf, dtype=torch.float64, device=img.device)
    for s in np.linspace(case["lo"], case["hi"], case["scales"]):
        l1, l2, l3 = _eigenvalues(*_hessian(img, [s / v for v in _voxel_size(case)]))
        norm2 = l1 ** 2 + l2 ** 2 + l3 ** 2
        c2 = norm2.max() / 4
        tiny = torch.finfo(torch.float32).tiny
        rb = l1.abs() / ((l2 * l3).abs().sqrt() + tiny)
        ra = l2.abs() / (l3.abs() + tiny)
        v = (1 - torch.exp(-2 * ra ** 2)) * torch.exp(-2 * rb ** 2) * (1 - torch.exp(-norm2 / (2 * c2)))
        best = torch.maximum(best, torch.where((l2 < 0) & (l3 < 0), v, torch.zeros_like(v)))
    return best


def _flow_exact(v, case):
    size = np.asarray(_voxel_size(case))
    dt = min(0.99, size.min() ** 3 / (2.01 ** 3 * MU))
    v = v.double()
    r = v.square().sum(0)
    g = torch.zeros_like(v)
    for _ in range(case["iters"]):
        lap = torch.zeros_like(g)
        for k in range(3):
            n = g.shape[k + 1]
            t = torch.empty_like(g)
            t.narrow(k + 1, 1, n - 2).copy_(g.narrow(k + 1, 0, n - 2) + g.narrow(k + 1, 2, n - 2))
            t.select(k + 1, 0).copy_(2 * g.select(k + 1, 1))
            t.select(k + 1, n - 1).copy_(2 * g.select(k + 1, n - 2))
            lap += (t - 2 * g) / size[k] ** 2
        g = g - dt * (r * (g - v) - MU * lap)
    return g.reshape(-1)


def exact(case, seed):
    path, p = case["path"], None
    if path in ("cut", "grid", "ragged"):
        p = _cut_params(case)
    if path == "cut":
        f = _cut_inputs(case, seed)
        if case["kind"] == "pointwise":
            sq = f["eigs"][..., :3].double().unbind(-1)
        else:
            sq = np.sqrt(_eigs(case["kind"]))
        u, criteria = _cut_exact(f["u0"], f["quats"], sq, f["alpha"], f["cs"], f["ct"], f["labels"],
                                 _voxel_size(case), p)
        return dict(u=u, criteria=_padded(criteria, case))
    if path == "grid":
        st = prepare(case, seed)
        us = []
        for w, d in zip(st["w"], st["d"]):
            alpha = float(w) * torch.exp(-st["gms"].double() / float(d) ** 2)
            us.append(_cut_exact(st["u0"], st["quats"], np.sqrt(_eigs("atv")), alpha, st["cs"],
                                 st["ct"], None, (1.0, 1.0, 1.0), p)[0].reshape(-1))
        return torch.stack(us)
    if path == "ragged":
        shapes, offsets, packed = _ragged_inputs(case, seed)
        out = torch.empty_like(packed["u0"], dtype=torch.float64)
        for s, o in zip(shapes, offsets):
            n = math.prod(s)
            f = {k: packed[k][o:o + n].reshape(s) for k in ("u0", "alpha", "cs", "ct")}
            q = packed["quats"][3 * o:3 * (o + n)].reshape(s + (3,))
            out[o:o + n] = _cut_exact(f["u0"], q, np.sqrt(_eigs("atv")), f["alpha"], f["cs"],
                                      f["ct"], None, (1.0, 1.0, 1.0), p)[0].reshape(-1)
        return out
    if path == "frangi":  # the frames of near-equal eigenvalues have no value of their own
        return dict(response=_response_exact(_image(case, seed), case), frames=None)
    if path == "gvf":
        return _flow_exact(_flow_input(case, seed), case)
    return None  # decisions at ridges: a rounding apart is another direction
