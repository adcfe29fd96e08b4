"""The work that users of this package have it do, as measurable cases.

Six paths, each through its public entry points:

  image   one pattern of a parameter set whose tables are on the device (a viewer, a series of
          exposures): SasCalc.doCalculationDevice
  whole   one pattern from the parameters to the image in host memory, as a script or the
          console takes it: SasCalc.set_params + doCalculation
  batch   many small patterns of one lattice with varied parameters, the training images of a
          network: SasCalc.stage_points + csx_render_batch_run
  fits    the objective of many independent 2D fits at several points each, one round of the
          batched simplex and the exact scoring of proposed starts: nm_eval
  post    what a training image goes through afterwards: linear scaling, r,phi resampling, log
          scaling, FFT: aidata.post_*
  train / predict   the surrogate network: loss and gradients of one minibatch; scores of the
          proposals of many fits

exact() gives the same values in FP64 with torch and numpy alone: the reflection tables,
series and sums of the simulator, the orientation average by a converged quadrature, and the
network in FP64.  It follows the simulator's definitions where they decide the result (tables
stored in FP32, the switch points and exit rule of the power series, the rod factor's 1e-9).
"""
import ctypes
import math

import numpy as np
import torch

from crystalscatter_amd import Context, SasCalc, _lib, aidata, nm_eval
from crystalscatter_amd.surrogate import BCT_BASE, FIT_HI, FIT_KEYS, FIT_LO, MLP, draw_parameters, params_dict

LATTICES = {"none": 12, "bcc": 4, "fcc": 5, "sc": 7, "bct": 8}
SHAPES = {"lorentz": 0, "gauss": 1, "mod1": 2, "mod2": 3, "pvoigt": 4, "pearson": 5}
BATCH_KEYS = ["EditRadius", "EditSigma", "uca,ucb,ucc", "I0", "EditDomainSize", "EditDebyeWaller"]
BATCH_MID = [8.0, 0.08, 30.0, 1.0, 200.0, 1.5]
BATCH_SPAN = [0.1, 0.2, 0.05, 0.3, 0.4, 0.5]   # relative variation of the training images


# ---- the cases ---------------------------------------------------------------------------
def _image(name, particle, lattice, grid, **kw):
    c = dict(name=name, kind="image", particle=particle, lattice=lattice, shape="gauss", precision="mixed", grid=grid,
             qmax=1.0, beam=False)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: a pattern of dissolved spheres for a viewer, FP64, launch latency
        _image("spheres-128", "sphere", "none", 64, precision="ref64", qmax=2.0),
        # the headline: FCC spheres on the full detector, every reflection of HKLmax 5
        _image("fcc-1024", "sphere", "fcc", 512),
        # a measured detector: beam position, pixel size and distance give q; odd edge tiles
        _image("fcc-beam-500", "sphere", "fcc", 250, beam=True),
        # oriented cylinders on a BCT lattice, the pattern that the fits are made to
        _image("bct-512", "cylinder", "bct", 256),
        # a peak shape other than the Gaussian: Lorentzian tails reach every pixel
        _image("fcc-lorentz-512", "sphere", "fcc", 256, shape="lorentz"),
        # cylinders with a distribution of directions: an orientation average per pixel
        _image("cyl-gauss-512", "cylinder", "none", 256, qmax=1.5),
        # a script's whole call: parameters in, image in host memory out, ragged size
        _image("bcc-whole-666", "sphere", "bcc", 333, kind="whole"),
        # training images of one parameter line, varied like the console's AI-data loop
        dict(name="train-images-512x128", kind="batch", lattice="fcc", grid=64, n=512),
        # their post-processing
        dict(name="post-256x128", kind="post", grid=64, size=128, n=256),
        # one round of the batched fits over uneven detectors
        dict(name="fits-96x4", kind="fits", nfits=96, nv=4, grid_lo=64, grid_hi=256),
        # one minibatch of the surrogate's training
        dict(name="mlp-gradient-65536", kind="train", rows=65536),
        # the proposals of a set of fits scored by the network
        dict(name="mlp-predict-2M", kind="predict", nsets=8192, px=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["image", "image", "image", "image", "whole", "batch", "fits", "post", "train", "predict"])
    if kind in ("image", "whole"):
        what = rng.choice(["sphere", "lattice", "lattice", "beam", "bct", "shape", "gauss"])
        prec = "mixed"
        if what == "sphere":
            c = _image("", "sphere", "none", _log_int(rng, 32, 512), precision=rng.choice(["ref64", "mixed"]),
                       qmax=rng.choice([1.0, 1.5, 2.0]))
        elif what in ("lattice", "beam"):
            g = _log_int(rng, 32, 512) if what == "lattice" else _log_int(rng, 32, 300)
            if what == "lattice" and g <= 256 and rng.random() < 0.25:
                prec = "ref64"
            c = _image("", "sphere", rng.choice(["fcc", "bcc", "sc"]), g, beam=what == "beam", precision=prec)
        elif what == "bct":
            c = _image("", "cylinder", "bct", _log_int(rng, 32, 300))
        elif what == "shape":
            c = _image("", "sphere", rng.choice(["fcc", "bcc", "sc"]), _log_int(rng, 32, 256),
                       shape=rng.choice(["lorentz", "mod1", "mod2", "pvoigt", "pearson"]))
        else:
            c = _image("", "cylinder", "none", _log_int(rng, 32, 256), qmax=rng.choice([0.8, 1.0, 1.5]))
        c["kind"] = kind
    elif kind == "batch":
        g = _log_int(rng, 24, 128)
        c = dict(kind=kind, lattice=rng.choice(["fcc", "bcc", "sc"]), grid=g,
                 n=_log_int(rng, 16, max(17, min(512, 512 * 64 * 64 // (g * g)))))
    elif kind == "post":
        size = rng.choice([64, 128, 256])
        c = dict(kind=kind, grid=_log_int(rng, 24, 100), size=size, n=_log_int(rng, 16, 256 * 128 * 128 // size ** 2))
    elif kind == "fits":
        lo = _log_int(rng, 32, 128)
        nv = rng.choice([1, 2, 3, 4, 8])
        c = dict(kind=kind, nfits=_log_int(rng, 4, 384 // nv), nv=nv, grid_lo=lo, grid_hi=min(256, 2 * lo + 1))
    elif kind == "train":
        c = dict(kind=kind, rows=_log_int(rng, 1000, 65536))
    else:
        px = rng.choice([100, 256, 1000])
        c = dict(kind=kind, nsets=_log_int(rng, 16, 2000000 // px), px=px)
    c.pop("name", None)
    return c


# ---- parameters of a case ----------------------------------------------------------------
def _rng(case, seed):
    return np.random.default_rng([int(seed), case.get("grid", 0), case.get("n", 0), case.get("rows", 0),
                                  case.get("nfits", 0), case.get("nsets", 0)])


def _image_params(case, seed):
    """The key=value parameters of an image case (the package's names), drawn like the fit
    workload (cylinders) or around the headline's values (spheres)."""
    r = _rng(case, seed)
    p = dict(LType=LATTICES[case["lattice"]], ComboBoxInterior=0, HKLmax=5, GridPoints=case["grid"],
             EditQmax=case["qmax"], I0=1, Base=0, RadButDebyeScherrer=1, ComboBoxPeak=SHAPES[case["shape"]],
             ignore_cbs=1)
    if case["particle"] == "sphere":
        a = float(r.uniform(27, 33))
        p.update(ComboBoxParticle=0, Ordis=7 if case["lattice"] == "none" else 0, EditSigma=float(r.uniform(0.07, 0.1)),
                 EditRadius=float(r.uniform(4, 6) if case["lattice"] == "none" else r.uniform(7, 9)), uca=a, ucb=a,
                 ucc=a, EditDomainSize=float(r.uniform(150, 250)), EditDebyeWaller=float(r.uniform(1.2, 1.8)),
                 EditAzi=float(r.uniform(4, 6)))
        if case["shape"] in ("pvoigt", "pearson"):
            p["EditPeakPar"] = float(r.uniform(30, 70) if case["shape"] == "pvoigt" else r.uniform(2.2, 6.8))
    elif case["lattice"] == "none":
        p.update(ComboBoxParticle=1, Ordis=0, EditRadius=float(r.uniform(2.5, 3.5)), Length=float(r.uniform(30, 50)),
                 EditSigma=0.06, SigmaL=0.06, EditDbeta=float(r.uniform(8, 12)), theta=float(r.uniform(20, 40)),
                 phi=45, fix_orcase=1)
    else:
        x = draw_parameters(r, 1)[0]
        p.update(BCT_BASE, EditRadius=float(x[0]), Length=float(x[1]), uca=float(x[2]), ucb=float(x[2]),
                 ucc=float(x[3]), EditDomainSize=float(x[4]), EditAzi=float(x[5]))
    if case["beam"]:
        n = 2 * case["grid"]
        # pixel size and distance as they put the detector's edge near qmax, the beam off centre
        p.update(CenterBeam=1, EditPixelNoX=n, EditPixelNoY=n, EditPixelX=240.0 / n, EditPixelY=240.0 / n, EditDet=5,
                 EditWavelength=0.154, BeamPosX=float(r.uniform(-0.1, 0.1) * n),
                 BeamPosY=float(r.uniform(-0.1, 0.1) * n))
    return p


def _batch_params(case, seed):
    base = dict(LType=LATTICES[case["lattice"]], ComboBoxParticle=0, Ordis=0, ComboBoxPeak=1, ComboBoxInterior=0,
                RadButDebyeScherrer=1, EditAzi=5, HKLmax=5, GridPoints=case["grid"], EditQmax=1, I0=1, Base=0,
                ignore_cbs=1)
    r = _rng(case, seed)
    X = np.array(BATCH_MID) * (1 + np.array(BATCH_SPAN) * r.uniform(-1, 1, (case["n"], len(BATCH_MID))))
    for j, k in enumerate(BATCH_KEYS):
        for kk in k.split(","):
            base[kk] = BATCH_MID[j]
    return base, X


def _fit_inputs(case, seed):
    """Per fit: its detector size (2 grid pixels), count scale and data (Poisson counts of a
    decaying pattern with rings, up to 1e4, an 8-pixel beam stop without data), and the points."""
    r = _rng(case, seed)
    grids = [int(r.integers(case["grid_lo"], case["grid_hi"] + 1)) for _ in range(case["nfits"])]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 1000003 + case["nfits"])
    datas, scales = [], []
    for g in grids:
        ax = torch.arange(-g, g, dtype=torch.float64, device="cuda") / g
        q = torch.sqrt(ax[:, None] ** 2 + ax[None, :] ** 2)
        a = float(r.uniform(15, 40))
        lam = 1e4 * (1 + (q / 0.05) ** 2) ** -2 * (1 + 0.8 * torch.cos(q * a))
        d = torch.poisson(lam, generator=gen)
        d[q < 8.0 / g] = 0.0
        datas.append(d.reshape(-1).contiguous())
        scales.append(float(r.uniform(0.5e4, 2e4)))
    X = np.stack([draw_parameters(r, case["nv"]) for _ in grids])
    return grids, scales, datas, np.clip(X, FIT_LO * 1.0001, FIT_HI * 0.9999)


def _fit_params(grid, scale, x):
    return dict(params_dict(x, grid), I0=scale, ignore_cbs=1)


def _post_images(case, seed):
    """Scattering images as the training loop gets them: six decades, rings, noise."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 1009 + case["n"])
    g = case["grid"]
    ax = torch.arange(-g, g, dtype=torch.float64, device="cuda") / g
    q = torch.sqrt(ax[:, None] ** 2 + ax[None, :] ** 2)
    a = 20 + 20 * torch.rand(case["n"], 1, 1, dtype=torch.float64, device="cuda", generator=gen)
    noise = torch.rand(case["n"], 2 * g, 2 * g, dtype=torch.float64, device="cuda", generator=gen)
    img = (1 + (q / 0.05) ** 2) ** -2 * (1.05 + torch.cos(q * a)) * (0.9 + 0.2 * noise)
    return img.reshape(case["n"], -1).contiguous()


def _net(r):
    """Weights (He-uniform, as a fresh network has them) and input phases of a surrogate."""
    nin, npad, h, layers = 70, 128, 256, 4
    parts = []
    for l in range(layers):
        k = nin if l == 0 else h
        w = np.zeros((h, npad if l == 0 else h), dtype=np.float32)
        w[:, :k] = r.uniform(-1, 1, (h, k)) * math.sqrt(6.0 / k)
        parts += [w.ravel(), r.uniform(-0.1, 0.1, h).astype(np.float32)]
    parts += [(r.uniform(-1, 1, h) * math.sqrt(3.0 / h)).astype(np.float32), np.zeros(1, dtype=np.float32)]
    F = np.zeros((32, 3), dtype=np.float32)
    pidx = np.full(32, -1, dtype=np.int32)
    for k in range(24):
        F[k, 2] = [0.25, 0.5, 0.75, 1.0, 1.25, 1.5, 2.0, 2.5][k % 8]
        pidx[k] = [2, 3, 0][k // 8]
    mag, ang = 0.5 * 32.0 ** r.uniform(0, 1, 8), 2 * math.pi * r.uniform(0, 1, 8)
    F[24:, 0], F[24:, 1] = mag * np.cos(ang), mag * np.sin(ang)
    affine = np.stack([0.5 * (FIT_LO + FIT_HI), 0.5 * (FIT_HI - FIT_LO)], axis=1).astype(np.float32)
    return np.concatenate(parts), F, pidx, affine


def _rows(case, seed):
    """Rows of the network: normalised parameter sets, each row's set and pixel (qx, qy), and
    for training the normalised log intensity."""
    r = _rng(case, seed)
    net = _net(r)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 1)
    if case["kind"] == "train":
        n, ns = case["rows"], max(1, case["rows"] // 16)
        sets = torch.randint(0, ns, (n,), device="cuda", generator=gen).to(torch.int32)
    else:
        ns = case["nsets"]
        n = ns * case["px"]
        sets = torch.arange(ns, dtype=torch.int32, device="cuda").repeat_interleave(case["px"])
    par = 2 * torch.rand(ns, 6, device="cuda", generator=gen) - 1
    q = 2 * torch.rand(n, 2, device="cuda", generator=gen) - 1
    t = torch.randn(n, device="cuda", generator=gen)
    return net, par, sets, q, t


# ---- preparation and one pass ------------------------------------------------------------
def _engine(p, device):
    e = SasCalc(device=device, params={k: v for k, v in p.items() if k != "ignore_cbs"})
    e.set("ignore_cbs", 1)
    return e


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("image", "whole"):
        p = _image_params(case, seed)
        st["calc"] = _engine(p, 0)
        if kind == "whole":
            st["params"] = {k: v for k, v in p.items() if k != "ignore_cbs"}
        else:
            st["calc"].prepare()
            st["out"] = torch.empty(4 * case["grid"] ** 2, dtype=torch.float64, device="cuda")
    elif kind == "batch":
        p, st["X"] = _batch_params(case, seed)
        st["engine"], st["ctx"] = _engine(p, -1), Context(0)
        st["out"] = torch.empty((case["n"], 4 * case["grid"] ** 2), dtype=torch.float64, device="cuda")
    elif kind == "fits":
        grids, scales, st["data"], st["X"] = _fit_inputs(case, seed)
        st["ctx"] = Context(0)
        st["fits"] = []
        for g, sc, d, x in zip(grids, scales, st["data"], st["X"]):
            st["fits"].append(dict(engine=_engine(_fit_params(g, sc, x[0]), -1), d_data=d.data_ptr(), w=2 * g, h=2 * g,
                                   lo=FIT_LO, hi=FIT_HI))
    elif kind == "post":
        st["imgs"], st["ctx"] = _post_images(case, seed), Context(0)
    else:
        (w, F, pidx, affine), st["par"], st["sets"], st["q"], st["t"] = _rows(case, seed)
        st["net"] = MLP(device=0, max_batch=case["rows"] if kind == "train" else 128, seed=1)
        st["net"].set_params(w)
        st["net"].set_features(F, pidx, affine)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "image":
        st["calc"].doCalculationDevice(st["out"].data_ptr(), case["precision"])
        return st["out"]
    if kind == "whole":
        st["calc"].set_params(st["params"])
        return st["calc"].doCalculation(case["precision"])
    if kind == "batch":
        ctx, L = st["ctx"], _lib.lib()
        ctx._chk(L.csx_fit_batch_begin(ctx._h), "csx_fit_batch_begin")
        st["engine"].stage_points(ctx, BATCH_KEYS, st["X"], st["out"].data_ptr(), st["out"].shape[1])
        ctx._chk(L.csx_render_batch_run(ctx._h, _lib.CSX_PREC_MIXED), "csx_render_batch_run")
        return st["out"]
    if kind == "fits":
        return nm_eval(st["ctx"], st["fits"], FIT_KEYS, st["X"])
    if kind == "post":
        ctx, g, s = st["ctx"], case["grid"], case["size"]
        img = st["imgs"].clone()
        aidata.post_scale_intensity(ctx, img, 1)
        rphi = aidata.post_rphi(ctx, img, (-g, g, -g, g), (2, -3), s)
        aidata.post_scale_clip(ctx, rphi, genlog=True)
        return img, rphi, aidata.post_ifft(ctx, rphi, s, out_type=2, scale=True, swap=True)
    if kind == "train":
        loss = st["net"].gradient(st["par"], st["sets"], st["q"], st["t"])
        return loss, st["net"].get_grads()
    return st["net"].predict(st["par"], st["sets"], st["q"])


# ---- the work of one pass ----------------------------------------------------------------
FLOP_PAIR = 40      # one Friedel pair at one pixel: cosine, angle, two exponents, two weights
FLOP_PX = 250       # one pixel outside the sum: q, P(q), <F>^2, S(q)
MLP_FWD = 2 * (70 * 256 + 3 * 256 * 256 + 256)
MLP_TRAIN = 2 * MLP_FWD + 2 * 3 * 256 * 256 + 2 * 256


def _lattice_flops(p, npx):
    """Peak-sum operations of npx pixels: the pairs whose Gaussian reaches 2^-32 of its weight at
    a pixel (mean over a coarse grid); every pair for the shapes with long tails."""
    tab = _lattice_tables(p)
    qh = tab["L3"][:, 5]
    if p["ComboBoxPeak"] == 1:
        ax = (np.arange(32) + 0.5) / 32 * p["EditQmax"]
        q = np.sqrt(ax[:, None] ** 2 + ax[None, :] ** 2).reshape(-1, 1)
        reach = math.sqrt(32 * math.log(2) * math.pi / 4) * 4.0 / p["EditDomainSize"]
        pairs = 0.5 * (np.abs(q - qh[None, :]) < reach).sum() / len(q)
    else:
        pairs = 0.5 * len(qh)
    return npx * (pairs * FLOP_PAIR + FLOP_PX)


def work(case):
    kind = case["kind"]
    if kind in ("image", "whole"):
        npx = 4 * case["grid"] ** 2
        p = _image_params(case, 1)
        if case["lattice"] != "none":
            flops = _lattice_flops(p, npx)
        elif case["particle"] == "cylinder":
            # the average's phase q L spans up to ~q L sin(34 deg) / pi periods in each of the two
            # angles, two nodes a period: about 16 x 16 nodes of 20 operations at the mean pixel
            flops = npx * (256 * 20 + FLOP_PX)
        else:
            flops = npx * FLOP_PX
        return {"bytes": 8 * npx, "flops": flops}
    if kind == "batch":
        npx = 4 * case["grid"] ** 2 * case["n"]
        return {"bytes": 8 * npx, "flops": _lattice_flops(_batch_params(case, 1)[0], npx)}
    if kind == "fits":
        r = _rng(case, 1)
        grids = [int(r.integers(case["grid_lo"], case["grid_hi"] + 1)) for _ in range(case["nfits"])]
        px = sum(4 * g * g for g in grids)
        p = _fit_params(grids[0], 1.0, 0.5 * (FIT_LO + FIT_HI))
        return {"bytes": 8 * px, "flops": _lattice_flops(p, px * case["nv"])}
    if kind == "post":
        n, g, s = case["n"], case["grid"], case["size"]
        return {"bytes": 8 * n * (2 * 4 * g * g + 2 * s * s),
                "flops": n * (10 * s * s * math.log2(s * s) + 10 * 4 * g * g + 30 * s * s)}
    n = case["rows"] if kind == "train" else case["nsets"] * case["px"]
    if kind == "train":
        return {"bytes": 16 * n + 4 * 215809 * 2, "flops": n * MLP_TRAIN}
    return {"bytes": 16 * n + 4 * 215809, "flops": n * MLP_FWD}


# ---- the same values in FP64 -------------------------------------------------------------
LD = np.longdouble
NC = 120  # terms of the power series


def _f32(x):
    return np.float32(x)


def _libm(name, x):
    """The C library's FP32 function (the tables are rounded with it)."""
    f = getattr(ctypes.CDLL("libm.so.6"), name)
    f.restype, f.argtypes = ctypes.c_float, [ctypes.c_float]
    return _f32(f(float(x)))


def _recip_basis(a, b, c):
    """Rotated reciprocal basis (rows a*, b*, c*) of an orthogonal cell with [111] along the
    beam; cell vectors, rotation and their products rounded to FP32 as the tables define them."""
    cb = math.cos(90 * math.pi / 180)
    sb = math.sin(90 * math.pi / 180)
    m1 = (cb - cb * cb) / sb
    m2 = math.sqrt(1.0 - m1 * m1 - cb * cb)
    S = [a * sb, 0.0, a * cb, b * m1, b * m2, b * cb, 0.0, 0.0, c * 1.0]

    def inv3(A):
        d = (A[0] * A[4] * A[8] + A[1] * A[5] * A[6] + A[2] * A[3] * A[7] - A[6] * A[4] * A[2] - A[7] * A[5] * A[0]
             - A[8] * A[3] * A[1])
        return [(A[4] * A[8] - A[5] * A[7]) / d, (A[2] * A[7] - A[1] * A[8]) / d, (A[1] * A[5] - A[2] * A[4]) / d,
                (A[5] * A[6] - A[3] * A[8]) / d, (A[0] * A[8] - A[2] * A[6]) / d, (A[2] * A[3] - A[0] * A[5]) / d,
                (A[3] * A[7] - A[4] * A[6]) / d, (A[1] * A[6] - A[0] * A[7]) / d, (A[0] * A[4] - A[1] * A[3]) / d]

    T = lambda A: [A[3 * j + i] for i in range(3) for j in range(3)]
    M = T(inv3(T(inv3(S))))
    cell = [[_f32(M[i] if k == 0 else M[1 + i] if k == 1 else M[2 + i]) for i in (0, 3, 6)] for k in range(3)]
    ae, be, ce = cell
    vol = float(ae[0] * (be[1] * ce[2] - be[2] * ce[1]) + ae[1] * (be[2] * ce[0] - be[0] * ce[2])
                + ae[2] * (be[0] * ce[1] - be[1] * ce[0]))
    n = [_f32(M[3 * i] + M[3 * i + 1] + M[3 * i + 2]) for i in range(3)]
    ln = _f32(math.sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]))
    nx, nz = n[0] / ln, n[2] / ln
    th = _libm("acosf", -nz)
    sth, cth = _libm("sinf", th), _libm("cosf", th)
    ep = _libm("asinf", nx / sth)
    sep, cep = _libm("sinf", ep), _libm("cosf", ep)
    r = [cep, _f32(-float(sep * cth)), sep * sth, sep, _f32(float(cep * cth)), -cep * sth, _f32(0.0), sth, cth]
    dr = float(r[0] * r[4] * r[8] + r[1] * r[5] * r[6] + r[2] * r[3] * r[7] - r[6] * r[4] * r[2] - r[7] * r[5] * r[0]
               - r[8] * r[3] * r[1])
    q = [float(v) / dr for v in (r[4] * r[8] - r[5] * r[7], r[2] * r[7] - r[1] * r[8], r[1] * r[5] - r[2] * r[4],
                                 r[5] * r[6] - r[3] * r[8], r[0] * r[8] - r[2] * r[6], r[2] * r[3] - r[0] * r[5],
                                 r[3] * r[7] - r[4] * r[6], r[1] * r[6] - r[0] * r[7], r[0] * r[4] - r[1] * r[3])]
    rot = lambda x: [_f32(q[3 * i] * float(x[0]) + q[3 * i + 1] * float(x[1]) + q[3 * i + 2] * float(x[2]))
                     for i in range(3)]
    ad, bd, cd = rot(ae), rot(be), rot(ce)
    R = [bd[1] * cd[2] - bd[2] * cd[1], bd[2] * cd[0] - bd[0] * cd[2], bd[0] * cd[1] - bd[1] * cd[0],
         ad[2] * cd[1] - ad[1] * cd[2], ad[0] * cd[2] - ad[2] * cd[0], ad[1] * cd[0] - ad[0] * cd[1],
         ad[1] * bd[2] - ad[2] * bd[1], ad[2] * bd[0] - ad[0] * bd[2], ad[0] * bd[1] - ad[1] * bd[0]]
    return np.array([float(v) for v in R]) / vol, vol


def _allowed(lt, h, k, l):
    if lt == 5:
        return ((h + k) % 2 == 0) & ((h + l) % 2 == 0)
    if lt in (4, 8):
        return (h + k + l) % 2 == 0
    return np.ones(h.shape, dtype=bool)


def _gamma(z):
    """Gamma of 1 < z <= 1000 as the simulator defines it: a product and an 8-term polynomial."""
    bm = [-0.577191652, 0.988205891, -0.897056937, 0.918206857, -0.756704078, 0.482199394, -0.193527818, 0.035868343]
    if math.modf(z)[0] < 1e-9:
        return LD(math.factorial(int(z) - 1))
    y, x = z - 1, z - math.trunc(z)
    fak = LD(y if math.trunc(y) else 1.0)
    for i in range(1, math.trunc(y)):
        fak *= y - i
    return fak * (1 + sum(b * x ** (i + 1) for i, b in enumerate(bm)))


def _gauss_norm(a):
    """Norms of the angular peak shapes for a > 0.01 (wider peaks are not among the cases)."""
    p2 = math.pi ** 2
    e = np.exp(-a * p2)
    return ((1 - e) / 2 / a - (1 - e * (1 + a * p2)) / 12 / a ** 2 + (2 - e * (2 + 2 * a * p2 + a * a * p2 ** 2)) / 240
            / a ** 3 - (6 - e * (6 + 6 * a * p2 + 3 * a * a * p2 ** 2 + a ** 3 * p2 ** 3)) / 10080 / a ** 4)


def _lorentz_norm(a):
    p2 = math.pi ** 2
    lg = np.log(1 + a * p2)
    return (lg / 2 / a - (a * p2 - lg) / 12 / a ** 2 + (-2 * a * p2 + a * a * p2 ** 2 + 2 * lg) / 480 / a ** 3
            - (a * p2 * (6 - 3 * a * p2 + 2 * a * a * p2 ** 2) - 6 * lg) / 60480 / a ** 4)


def _pearson_norm(a, b):
    b += 1e-6
    out = np.empty(a.shape)
    for i, v in enumerate(a):
        if v > 20:
            out[i] = (1 - math.exp((1 - b) * math.log(1 + v * math.pi ** 2))) / (2 * (b - 1)) / v
            continue
        f = lambda x: np.sin(x) / np.exp(b * np.log(1 + v * x * x))
        n, s = 1, 0.5 * math.pi * float(f(0.0) + f(math.pi))
        old = s
        for _ in range(9):
            s = 0.5 * (s + math.pi * float(f(math.pi / n * (np.arange(n) + 0.5)).sum()) / n)
            n *= 2
            if abs(1 - s / old) < 0.001:
                break
            old = s
        out[i] = s
    return out


def _lattice_tables(p):
    """Reflections (unit multiplicity) of the box |h|, |k|, |l| <= HKLmax: q_hkl, |q_hkl|, g3 and
    the peak norm in FP32 (columns 2, 3, 4, 5, 10, 11), the structure factor, V times the number
    of particles of the cell."""
    lt, H = int(p["LType"]), int(p["HKLmax"])
    g = np.arange(-H, H + 1)
    h, k, l = (v.ravel() for v in np.meshgrid(g, g, g, indexing="ij"))
    keep = _allowed(lt, h, k, l) & ((h != 0) | (k != 0) | (l != 0))
    h, k, l = h[keep], k[keep], l[keep]
    R, vol = _recip_basis(p["uca"], p["ucb"], p["ucc"])
    tp = 2 * math.pi
    qx, qy, qz = (tp * (R[i] * h + R[3 + i] * k + R[6 + i] * l) for i in range(3))
    qh = np.sqrt(qx * qx + qy * qy + qz * qz)
    a = 4 * qh * qh / (math.pi * (4.0 / p["EditAzi"]) ** 2)
    shape = int(p["ComboBoxPeak"]) + 1
    norm = (_gauss_norm(a) if shape == 2 else _lorentz_norm(a) if shape in (1, 5)
            else _pearson_norm(a, {3: 2, 4: 1.5, 6: p.get("EditPeakPar", 0)}[shape]))
    L3 = np.zeros((len(h), 17))
    for col, v in ((2, qx), (3, qy), (4, qz), (5, qh), (10, 4 * math.pi ** 2 / (tp * qh * qh)), (11, norm)):
        L3[:, col] = v.astype(np.float32)
    cell = {4: 2, 5: 4, 7: 1, 8: 2}[lt]
    return {"L3": L3, "mf": float(cell * cell), "v": vol * cell}


def _switch(c, first_negative=False):
    """Where a series gives way to its closed form: |c_n|^(-1/2n) at the last usable term."""
    n = NC
    if first_negative:
        n = 1
    else:
        small = np.nonzero(np.abs(c[1:]) < 1e-30)[0]
        if len(small):
            n = int(small[0]) + 1
    while n > 1 and (not np.isfinite(c[n]) or abs(c[n]) < 1e-99):
        n -= 1
    return float(abs(c[n]) ** (-1 / (2.0 * n)))


_TABLES = {}


def _schulz(z, *sums):
    """Running products of the coefficient recurrences for one width parameter, and the named
    inner sums of the <F>^2 series (kept: they do not depend on the sizes)."""
    if len(_TABLES) > 2048:
        _TABLES.clear()
    t = _TABLES.setdefault(z, {})
    n = np.arange(NC + 1)
    if not t:
        z12, f, f2, g3 = (np.ones(NC + 1, dtype=LD) for _ in range(4))
        g3[0] = math.sqrt(math.pi) / 2
        for i in range(1, NC + 1):
            z12[i] = z12[i - 1] * LD((z + 1) - 2 + 2 * i) * LD((z + 1) - 1 + 2 * i)
            f[i] = f[i - 1] * i
            f2[i] = f2[i - 1] * (2 * i - 1) * (2 * i)
            g3[i] = g3[i - 1] * LD(2 * i + 1) / 2
        t.update(z12=z12, f=f, f2=f2, g3=g3, four=LD(4) ** n)
    z12, f, g3, h = t["z12"], t["f"], t["g3"], LD(1.5)
    for name in sums:
        if name in t:
            continue
        t[name] = np.empty(NC + 1)
        for i in n:
            m, k = n[:i + 1], n[i::-1]
            if name == "sphere":
                terms = z12[m] * z12[k] / ((m + h) * g3[m] * (k + h) * g3[k] * f[m] * f[k])
            elif name == "rod":
                terms = z12[m] * z12[k] / (g3[m] * g3[k] * f[m] * f[k] * f[m] * f[k])
            else:
                with np.errstate(over="ignore"):
                    top = z12[m].astype(np.float64) * z12[k].astype(np.float64)
                terms = top / ((m + 1) * f[m] * (k + 1) * f[k] * f[m] * f[k])
            # accumulated in FP64 in order: where the series cancels, its rounding is the value
            acc = np.float64(0)
            for v in terms:
                acc = np.float64(acc + v)
            t[name][i] = acc
    return t


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _series(c, x):
    """sum c_n x^2n with the exit rule (relative change < 1e-4), elementwise."""
    s, old, xn = torch.ones_like(x), torch.zeros_like(x), torch.ones_like(x)
    on = torch.ones_like(x, dtype=torch.bool)
    for n in range(1, len(c)):
        if not bool(on.any()):
            break
        xn = xn * x * x
        s = torch.where(on, s + float(c[n]) * xn, s)
        on = on & ~(((s - old) / s).abs() < 1e-4)
        old = torch.where(on, s, old)
    return s


def _sphere_factors(p, q):
    z = (1 - p["EditSigma"] ** 2) / p["EditSigma"] ** 2
    R = p["EditRadius"]
    t, n = _schulz(z, "sphere"), np.arange(NC + 1)
    xr = (-LD((R / (2.0 * (z + 1))) ** 2)) ** n
    c4p = (9 * LD(math.sqrt(math.pi)) * t["four"] * t["z12"] * xr
           / (2 * (n + LD(3)) * (n + 2) * (n + LD(1.5)) * t["g3"] * t["f"])).astype(np.float64)
    c4f = (9 * LD(math.pi) * xr * t["sphere"] / 16).astype(np.float64)
    x = q * R / (z + 1)
    at, b = torch.atan(2 * x), 1 + 4 * x * x
    c = 1 / (2.0 * z * (z - 1) * (z - 2) * (z - 3)) * x ** -4
    p3 = c / ((z - 4) * (z - 5) * x * x) * (1 - torch.cos((z - 5) * at) / b ** (z - 5) / 2)
    pq = 9 * (c * (1 + torch.cos((z - 3) * at) / b ** ((z - 3) / 2))
              - 2 * c / ((z - 4) * x) * torch.sin((z - 4) * at) / b ** ((z - 4) / 2) + p3)
    at, b = torch.atan(x), 1 + x * x
    c = 1 / (z * (z - 1)) * x ** -2
    fq = (3 * (c / ((z - 2) * x) * torch.sin((z - 2) * at) / b ** ((z - 2) / 2)
               - c * torch.cos((z - 1) * at) / b ** ((z - 1) / 2))) ** 2
    lo = 0.4 * _switch(c4p)
    pq = torch.where(q < lo, _series(c4p, q.clamp(max=lo)), pq)
    lo = 0.4 * _switch(c4f)
    return pq, torch.where(q < lo, _series(c4f, q.clamp(max=lo)), fq)


def _rod(zl, arg):
    """The rod factor as written; on the line qx + qy = 0 (arg ~ 1e-10) the rounding of its cosine
    decides the value, so that one is taken correctly rounded."""
    x = (zl - 1) * torch.atan(2 * arg)
    c = torch.cos(x)
    m = x.abs() < 1e-6
    c[m] = torch.tensor([math.cos(v) for v in x[m].tolist()], dtype=torch.float64, device=x.device)
    return (1 / (2 * zl * (zl - 1))) * (1 / (arg * arg)) * (1 - c / (1 + 4 * arg * arg) ** ((zl - 1) / 2))


def _disk_p(zr, R, q, c4p, lo):
    x = q * R / (zr + 1)
    at, b = torch.atan(2 * x), 1 + 4 * x * x
    c = 1 / (zr * (zr - 1) * (zr - 2)) * x ** -3
    pq = (4 / math.pi) * (c - c * torch.sin((zr - 2) * at) / b ** ((zr - 2) / 2)
                          - (9 / 8) * c / ((zr - 3) * x) * torch.cos((zr - 3) * at) / b ** ((zr - 3) / 2))
    return torch.where(q < lo, _series(c4p, q.clamp(max=lo)), pq)


def _cylinder_factors(p, qx, qy, q):
    """P(q) and <F>^2 of cylinders along z: rod factor of qx + qy times the disk's."""
    zr = zl = (1 - 0.06 ** 2) / 0.06 ** 2
    R, Lc = p["EditRadius"], p["Length"]
    t, n = _schulz(zr, "rod", "disk"), np.arange(NC + 1)
    xl, xr = (-LD((Lc / (2.0 * (zl + 1))) ** 2)) ** n, (-LD((R / (2.0 * (zr + 1))) ** 2)) ** n
    c1p = (LD(math.sqrt(math.pi)) * t["four"] * t["z12"] * xl / (2 * (n + LD(1)) * t["g3"] * t["f"])).astype(np.float64)
    c4p = (4 * (n + LD(0.5)) * t["f2"] * t["z12"] * xr
           / ((n + LD(2)) * (n + 1) * t["f"] ** 2 * (n + 1) * t["f"])).astype(np.float64)
    c1f = (LD(math.pi) * xl * t["rod"] / 4).astype(np.float64)
    c4f = (xr * t["disk"]).astype(np.float64)
    s = qx + qy
    rod = _rod(zl, (s + 1e-9) * Lc / (zl + 1))
    lo1, lo1f = 0.6 * _switch(c1p, True), 0.6 * _switch(c1f)
    pl = torch.where(q < lo1, _series(c1p, torch.where(q < lo1, s, torch.zeros_like(s))), rod)
    fl = torch.where(q < lo1f, _series(c1f, torch.where(q < lo1f, s, torch.zeros_like(s))), rod)
    # short cylinders (L/R < 2) have no transverse factor
    pt = _disk_p(zr, R, q, c4p, 0.65 * _switch(c4p, True)) if Lc / R >= 2 else torch.ones_like(q)
    x = q * R / (zr + 1)
    at, b = torch.atan(x), 1 + x * x
    f1, f2 = (float(_gamma(zr - d) / _gamma(zr + 1)) for d in (0.5, 1.5))
    a1 = f1 * x ** -1.5 * (torch.sin((zr - 0.5) * at) - torch.cos((zr - 0.5) * at)) / b ** ((zr - 0.5) / 2)
    a2 = f2 * x ** -2.5 * (torch.sin((zr - 1.5) * at) + torch.cos((zr - 1.5) * at)) / b ** ((zr - 1.5) / 2)
    fr = ((2 / math.sqrt(math.pi)) * (a1 + (9 / 16) * a2)) ** 2
    lo = _switch(c4f)
    fr = torch.where(q < lo, _series(c4f, q.clamp(max=lo)), fr)
    return pl * pt, fl * fr


def _pixels(p):
    g = int(p["GridPoints"])
    ax = torch.arange(-g, g, dtype=torch.float64, device=_dev())
    i, j = ax[:, None].expand(2 * g, 2 * g).reshape(-1), ax[None, :].expand(2 * g, 2 * g).reshape(-1)
    if p.get("CenterBeam"):
        x = p["EditPixelX"] / 1000 * (i * p["EditPixelNoX"] / (2.0 * g) - p["BeamPosX"])
        y = p["EditPixelY"] / 1000 * (j * p["EditPixelNoY"] / (2.0 * g) - p["BeamPosY"])
        phi, th = torch.atan2(y, x), torch.atan2(torch.sqrt(x * x + y * y), torch.full_like(x, float(p["EditDet"])))
        k = 2 * math.pi / p["EditWavelength"]
        return k * torch.cos(phi) * torch.sin(th), k * torch.sin(phi) * torch.sin(th), k * (1 - torch.cos(th))
    qx, qy = p["EditQmax"] * i / g, p["EditQmax"] * j / g
    return qx, qy, torch.full_like(qx, 1e-20)


def _peak_sum(p, tab, qx, qy, qz, q):
    """Sum over the reflections of radial peak times angular peak times weight."""
    width, phiw = 4.0 / p["EditDomainSize"], 4.0 / p["EditAzi"]
    shape = int(p["ComboBoxPeak"]) + 1
    L = torch.tensor(tab["L3"], device=q.device)
    out = torch.empty_like(q)
    step = max(1, (1 << 25) // len(L))
    ln2 = math.log(2.0)
    c2, c3 = 4 * (math.sqrt(2) - 1), 4 * (math.exp(2 * ln2 / 3) - 1)
    eta, beta = p.get("EditPeakPar", 0) / 100.0, p.get("EditPeakPar", 0)
    if shape == 6:
        c4 = math.exp(ln2 / beta) - 1
        lead = float(_gamma(beta) / _gamma(beta - 0.5)) * c4 * 2 / (math.pi * width)
    for s in range(0, len(q), step):
        e = slice(s, s + step)
        Q = q[e, None]
        c = qx[e, None] * L[None, :, 2] + qy[e, None] * L[None, :, 3] + qz[e, None] * L[None, :, 4]
        c = c / (Q * L[None, :, 5])
        y2 = torch.where(c < -1, 0.0, torch.where(c > 1, math.pi, torch.acos(c.clamp(-1, 1)))) ** 2
        x2 = ((Q - L[None, :, 5]) / width) ** 2
        if shape == 2:
            t = torch.exp(-4 / math.pi * x2 - 4 * Q * Q / (math.pi * phiw ** 2) * y2) / (math.pi * width / 2)
        else:
            l2 = 1 + 4 * Q * Q / phiw ** 2 * y2
            if shape == 1:
                t = 2 / (math.pi * width * (1 + 4 * x2)) / l2
            elif shape == 3:
                t = 2 * math.sqrt(c2) / (math.pi * width * (1 + 4 * x2) ** 2) / (l2 * l2)
            elif shape == 4:
                t = math.sqrt(c3) / (2 * width * (1 + 4 * x2) ** 1.5) / l2 ** 1.5
            elif shape == 5:
                sq = eta * 2 / (math.pi * width * (1 + 4 * x2))
                sq = sq + (1 - eta) * torch.exp(-x2) / (math.sqrt(math.pi) * width)
                t = (sq * (eta / l2 + (1 - eta) * torch.exp(-4 * Q * Q / (math.pi * phiw ** 2) * y2)) / eta)
            else:
                t = lead / (1 + 4 * c4 * x2) ** beta / l2 ** beta
        out[e] = (t * (tab["mf"] * L[None, :, 10] / L[None, :, 11])).sum(dim=1)
    return out


def _gauss_cylinder(p, qx, qy, q):
    """P(q) of cylinders with Gaussian-distributed directions about (theta, 0): the rod factor
    averaged over polar (Gauss-Legendre) and azimuth (trapezoid, spectral) angles."""
    zl = zr = (1 - 0.06 ** 2) / 0.06 ** 2
    Lc, th, db = p["Length"], p["theta"] * math.pi / 180, p["EditDbeta"] * math.pi / 180
    top = float(np.float32(min(db * math.sqrt(math.log(1e5)), math.pi / 2)))
    x, w = np.polynomial.legendre.leggauss(96)
    d = 0.5 * top * (x + 1)
    w = w * np.sin(d) * np.exp(-d * d / db ** 2)
    w = w / w.sum()
    c1 = qx * float(np.float32(math.sin(th)))
    rq = torch.sqrt((qx * float(np.float32(-math.cos(th)))) ** 2 + qy * qy)
    psi = (np.arange(160) + 0.5) * math.pi / 160
    t = torch.tensor(np.cos(psi), device=q.device)
    pl = torch.zeros_like(q)
    step = max(1, (1 << 25) // len(t))
    for s in range(0, len(q), step):
        e = slice(s, s + step)
        acc = torch.zeros_like(q[e])
        for dk, wk in zip(d, w):
            arg = (c1[e] * math.cos(dk))[:, None] + (rq[e] * math.sin(dk))[:, None] * t[None, :] + 1e-10
            arg = arg * Lc / (zl + 1)
            # 1 - e^A cos B without cancellation at small arguments
            A, B = -(zl - 1) / 2 * torch.log1p(4 * arg * arg), (zl - 1) * torch.atan(2 * arg)
            rod = (-torch.expm1(A) + 2 * torch.exp(A) * torch.sin(B / 2) ** 2) / (2 * zl * (zl - 1) * arg * arg)
            acc += wk * rod.mean(dim=1)
        pl[e] = acc
    # below 0.4 of the switch point: the double series, in the simulator's coefficients
    m = 24
    f = [math.factorial(k) for k in range(2 * m + 3)]
    zv, c1p, c4 = 1.0, [1.0], 0.0
    for n in range(1, m + 1):
        zv *= ((zr + 1) - 2 + 2 * n) * ((zr + 1) - 1 + 2 * n)
        c1p.append(16.0 ** n * zv * (-(Lc / (2.0 * (zl + 1))) ** 2) ** n / ((2.0 * n + 1) * (n + 1)))
        if n == 1:
            c4 = 4 * 1.5 * 2 * zv * -(p["EditRadius"] / (2.0 * (zr + 1))) ** 2 / (3 * 2 * 2)
    lo = 0.4 * abs(c1p[1]) ** -0.5
    small = q < lo
    if bool(small.any()):
        X, Y = (qx[small] ** 2).cpu().numpy(), (qy[small] ** 2).cpu().numpy()
        p11, p13 = math.cos(th) ** 2, math.sin(th) ** 2
        tot, old = np.ones(len(X)), np.zeros(len(X))
        on = np.ones(len(X), dtype=bool)
        for n in range(1, m + 1):
            inner = np.zeros(len(X))
            for k in range(n + 1):
                # entry [n-k][k] of the table; entries above its diagonal keep their initial 1
                row, col = n - k, k
                v = 1.0 if col > row else 4.0 ** col / f[row - col] * sum(
                    p11 ** l * p13 ** (col - l) / (4.0 ** l * f[2 * (col - l)] * f[row - col + l] * f[l])
                    for l in range(col + 1))
                inner += v * X ** k * Y ** (n - k)
            tot = np.where(on, tot + c1p[n] * inner, tot)
            on &= ~(np.abs((tot - old) / tot) < 1e-4)
            old = np.where(on, tot, old)
        pl[small] = torch.tensor(tot, device=q.device)
    t, n = _schulz(zr), np.arange(NC + 1)
    c4p = (4 * (n + LD(0.5)) * t["f2"] * t["z12"] * (-LD((p["EditRadius"] / (2.0 * (zr + 1))) ** 2)) ** n
           / ((n + LD(2)) * (n + 1) * t["f"] ** 2 * (n + 1) * t["f"])).astype(np.float64)
    return pl * _disk_p(zr, p["EditRadius"], q, c4p, 0.65 * abs(c4) ** -0.5)


def _exact_image(p):
    qx, qy, qz = _pixels(p)
    q = torch.sqrt(qx * qx + qy * qy + qz * qz) + 1e-9
    if p["LType"] == 12:
        return p["I0"] * (_sphere_factors(p, q)[0] if p["ComboBoxParticle"] == 0 else _gauss_cylinder(p, qx, qy, q))
    tab = _lattice_tables(p)
    pq, fq = _sphere_factors(p, q) if p["ComboBoxParticle"] == 0 else _cylinder_factors(p, qx, qy, q)
    dw = torch.exp(-p.get("EditDebyeWaller", 2.0) ** 2 / 3 * q * q)
    s = 1 + fq / pq * (2 * math.pi * _peak_sum(p, tab, qx, qy, qz, q) / tab["v"] - 1) * dw
    return p["I0"] * s * pq


def _exact_net(case, seed):
    (w, F, pidx, affine), par, sets, q, t = _rows(case, seed)
    w = torch.tensor(w, dtype=torch.float64, device=q.device).requires_grad_(case["kind"] == "train")
    F, pidx = torch.tensor(F, device=q.device).double(), torch.tensor(pidx, device=q.device).long()
    affine = affine.astype(np.float64)
    par, q = par.double(), q.double()
    phys = par * torch.tensor(affine[:, 1], device=q.device) + torch.tensor(affine[:, 0], device=q.device)
    phys = torch.cat([phys, torch.ones_like(phys[:, :1])], dim=1)[:, pidx]     # index -1: the column of ones

    def net(lo, hi):
        s, qq = sets[lo:hi].long(), q[lo:hi]
        ph = 2 * math.pi * (qq @ F[:, :2].T) + F[:, 2] * qq.norm(dim=1, keepdim=True) * phys[s]
        pad = torch.zeros(len(s), 58, dtype=torch.float64, device=q.device)
        x = torch.cat([par[s], torch.sin(ph), torch.cos(ph), pad], dim=1)
        at = 0
        for k in (128, 256, 256, 256):
            x = torch.nn.functional.silu(x @ w[at:at + 256 * k].reshape(256, k).T + w[at + 256 * k:at + 256 * k + 256])
            at += 256 * k + 256
        return x @ w[at:at + 256] + w[at + 256]

    n, step = len(q), 1 << 17
    if case["kind"] == "predict":
        with torch.no_grad():
            return torch.cat([net(s, min(n, s + step)) for s in range(0, n, step)])
    loss = 0.0
    for s in range(0, n, step):
        e = min(n, s + step)
        part = ((net(s, e) - t[s:e].double()) ** 2).sum() / n
        part.backward()
        loss += float(part.detach())
    return loss, w.grad.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("image", "whole"):
        return _exact_image(_image_params(case, seed))
    if kind == "batch":
        base, X = _batch_params(case, seed)
        out = []
        for x in X:
            p = dict(base)
            for k, v in zip(BATCH_KEYS, x):
                p.update({kk: float(v) for kk in k.split(",")})
            out.append(_exact_image(p))
        return torch.stack(out)
    if kind == "fits":
        grids, scales, datas, X = _fit_inputs(case, seed)
        out = np.empty(X.shape[:2])
        for f, (g, sc, d) in enumerate(zip(grids, scales, datas)):
            for v in range(X.shape[1]):
                img = _exact_image(_fit_params(g, sc, X[f, v]))
                ok = (img > 0) & (d > 0)
                out[f, v] = float(((torch.log10(img[ok]) - torch.log10(d[ok])) ** 2).sum())
        return out
    if kind in ("train", "predict"):
        return _exact_net(case, seed)
    return None   # post: scans and resampling of given images, bound to the start's values
