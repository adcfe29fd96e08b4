"""Values that depend on |qx| and |qy| only, evaluated on a quarter of the midpoint grid."""
import numpy as np
import pytest

from helpers import CFG1, CFG2, rel_err

from crystalscatter_amd import SasCalc

pytestmark = pytest.mark.gpu


def _image(p, z, prec, **kw):
    e = SasCalc(device=0, params=dict(p, GridPoints=z, **kw))
    e.set("ignore_cbs", 1)
    return e.doCalculation(prec).reshape((-1, e.bounds()[1] - e.bounds()[0]))


@pytest.mark.parametrize("z", [1, 2, 8, 9, 16, 17, 33, 130])
@pytest.mark.parametrize("kind", ["sphere", "cube", "cyl_iso", "cyl_gauss"])
def test_quarter_equals_first_quadrant(kind, z):
    """The whole image's first quadrant is the first-quadrant render (which evaluates every pixel
    on its own), and the image is even in both axes (Gaussian cylinders: in qy)."""
    p, prec = {"sphere": (CFG1, "ref64"), "cube": (dict(CFG1, ComboBoxParticle=4, EditRadius=4), "ref64"),
               "cyl_iso": (dict(CFG1, ComboBoxParticle=1, EditRadius=3, Length=30, SigmaL=0.1), "ref64"),
               "cyl_gauss": (dict(CFG2, fix_orcase=1), "mixed")}[kind]
    full = _image(p, z, prec)
    q1 = _image(p, z, prec, RadioButtonQ1=1, RadioButtonQ4=0)
    print(kind, z, flush=True)
    assert np.array_equal(full[z:, z:], q1, True)   # (cyl_gauss: the small-q series is NaN at one pixel of z = 130)
    inner = full[1:, 1:]
    assert np.array_equal(inner, inner[:, ::-1], True)
    # the first row and column have no positive counterpart in the image
    assert np.array_equal(full[0, 1:], full[0, :0:-1], True)
    if kind != "cyl_gauss":   # even in qy only
        assert np.array_equal(inner, inner[::-1]) and np.array_equal(full[1:, 0], full[:0:-1, 0])


@pytest.mark.parametrize("z", [1, 9, 17])
@pytest.mark.parametrize("reach", [0.5, 2.0])
def test_gauss_series_region(oracle_lib, z, reach):
    """Gaussian cylinders in their small-q series, alone (reach 0.5 of its limit: the other kernel on
    a quarter) and around the middle of a pattern (2.0): every form of the series evaluates the same
    terms in the same order, so the shared and the single waves, the quarter and the first quadrant
    agree bit for bit; the oracle's power tables round each of up to 16 terms differently."""
    p = dict(CFG2, fix_orcase=1)
    e = SasCalc(device=-1, params=dict(p, GridPoints=z))
    e.prepare()
    lim = 0.4 * e.scalars().limq[0]
    p["EditQmax"] = reach * lim
    i = np.arange(-z, z) / z
    series = np.hypot(i[:, None], i[None, :]) * reach < 1 - 1e-6
    if reach < 0.7:
        assert series.all()
    mixed, ref = _image(p, z, "mixed"), _image(p, z, "ref64")
    print(z, reach, int(series.sum()), flush=True)
    assert np.array_equal(mixed[series], ref[series], True)
    q1 = _image(p, z, "mixed", RadioButtonQ1=1, RadioButtonQ4=0)
    assert np.array_equal(mixed[z:, z:], q1, True)
    if reach < 1:
        o = oracle_lib.OracleEngine(dict(p, GridPoints=z))
        o.prepare()
        assert rel_err(mixed.ravel(), o.image(nthreads=4)).max() <= 1e-12
