"""Mirror images of the lattice kinds in mixed precision: one peak sum serves (ihex, i) and
(-ihex, -i) of the midpoint grid.  Sizes around the 16-pixel tiles and the 256-pixel
workgroups of the axis row and edge column, against the FP64 mode (which takes every pixel on
its own), and the fit objective under masks without the symmetry against the image's own terms."""
import numpy as np
import pytest

from helpers import CFG3, manifest, rel_err

from crystalscatter_amd import Context, SasCalc, nm_eval, render_batch

pytestmark = pytest.mark.gpu

BCT = manifest()["fixtures"]["cfg4_bct.npz"]["params"][0]
KINDS = {
    "fcc": CFG3,
    "bct_cylinder": BCT,
    "bct_cylinder_x": dict(BCT, theta=90, phi=0),
    "fcc_iso_cylinder": dict(CFG3, ComboBoxParticle=1, Ordis=7, EditRadius=3, Length=30, EditSigma=0.08, SigmaL=0.1),
    "hex_cylinder": dict(BCT, LType=1),   # unpaired reflections: every pixel on its own
}
SIZES = [1, 2, 7, 8, 9, 16, 17, 33, 130]


def _engine(p, z, device=0):
    e = SasCalc(device=device, params=dict(p, GridPoints=z))
    e.set("ignore_cbs", 1)
    e.prepare()
    return e


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("z", SIZES)
def test_image_against_fp64(kind, z):
    print(kind, z, flush=True)
    e = _engine(KINDS[kind], z)
    r = e.doCalculation("ref64")
    ok = np.isfinite(r) & (r != 0)
    batch = render_batch(Context(0), [_engine(KINDS[kind], z, -1)], "mixed")[0].cpu().numpy()
    for m in (e.doCalculation("mixed"), batch):   # the two-pass and the one-pass kernel
        assert np.array_equal(np.isfinite(m), np.isfinite(r))
        assert rel_err(m[ok], r[ok]).max() <= 1e-4   # the mixed mode's bar for every pixel


@pytest.mark.parametrize("theta,phi", [(30, 45), (60, 90), (30, 135), (90, 45), (60, -45), (45, 90), (180, 0), (37, 20),
                                       (0, 0), (60, 0)])
@pytest.mark.parametrize("length,sigmal", [(3, 0.06), (10, 0.06), (30, 0.06), (40, 0.3), (65, 0.46), (75, 0.4)])
def test_cylinders_off_the_axes(theta, phi, length, sigmal):
    """Cylinders whose projection vanishes on a line of pixels only up to rounding (the cosine and
    sine of 45 degrees differ by one ulp, the cosine of 90 is 6e-17; at theta = 180 on every
    pixel), or exactly: both images of each pixel against the FP64 mode.  Long polydisperse rods
    leave the power of the rod factor a few units in the last place off 1 on that line."""
    print(theta, phi, length, sigmal, flush=True)
    p = dict(BCT, theta=theta, phi=phi, Length=length, SigmaL=sigmal)
    e = _engine(p, 64)
    r = e.doCalculation("ref64")
    ok = np.isfinite(r) & (r != 0)
    batch = render_batch(Context(0), [_engine(p, 64, -1)], "mixed")[0].cpu().numpy()
    for m in (e.doCalculation("mixed"), batch):
        assert np.array_equal(np.isfinite(m), np.isfinite(r))
        err = rel_err(m[ok], r[ok])
        at = np.flatnonzero(ok)[err.argmax()]
        assert err.max() <= 1e-4, (err.max(), at % 128 - 64, at // 128 - 64, m[at], r[at])


@pytest.mark.parametrize("kind", ["fcc", "bct_cylinder"])
@pytest.mark.parametrize("z", [1, 8, 17, 33])
def test_objective_terms(kind, z):
    import torch
    n = 2 * z
    ctx, base = Context(0), _engine(KINDS[kind], z, -1)
    # the batch's image: the batched objective's own arithmetic
    img = render_batch(ctx, [base], "mixed")[0].cpu().numpy().reshape(n, n)
    rng = np.random.default_rng(z)
    data = rng.uniform(0.5, 2.0, (n, n)) * np.abs(img) * (rng.random((n, n)) > 0.2)
    keep = np.ones((n, n), dtype=bool)
    keep[:n // 2 + 1, :z // 3 + 1] = False   # a no-fit rectangle on one side only
    d = torch.tensor(data.ravel(), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    r = base.get("EditRadius")
    fit = dict(engine=base, d_data=d.data_ptr(), w=n, h=n, lo=[0.5 * r], hi=[2 * r], rects=[(0, 0, z // 3, n // 2)])
    s = nm_eval(ctx, [fit], ["EditRadius"], [[[r]]])[0, 0]
    ok = keep & (img > 0) & (data > 0)
    t = (np.log10(img[ok]) - np.log10(data[ok])) ** 2
    # terms to rounding: |log10| < 20, so each difference is good to about 1e-14
    assert abs(s - t.sum()) <= 1e-12 * max(1.0, t.sum())
