"""The branch-free device transcendentals and the radiation state built on
them where their selects decide: results at the ends of the exponent range,
subnormal operands, zero field, zero and negative energies.  GPU equals the
oracle bit for bit (radiation states: values, NaN for NaN)."""
import numpy as np
import pytest

import kzo
from goldens import geoms, read_kgld
from koral_zig_amd import abi_types as T
from koral_zig_amd import hip

pytestmark = pytest.mark.gpu
GAM = 5.0 / 3.0
TINY = 2.0 ** -1074
# operands next to every threshold of kz_math.h: overflow, underflow and the
# subnormal results of exp; subnormals, the sqrt(2) fold and 1 for log and cbrt
EDGES = {
    "exp": np.concatenate([np.linspace(-746.0, -707.0, 4001), np.linspace(709.0, 710.0, 501),
                           np.nextafter(709.782712893384, [0, 1e9]), np.nextafter(-745.1332191019412, [0, -1e9]),
                           np.arange(-1080, 1030) * np.log(2.0) / 2.0]),
    "log": np.concatenate([TINY * 2.0 ** np.arange(60), TINY * np.arange(1, 200), 2.0 ** np.arange(-1022.0, 1024.0),
                           np.nextafter(np.sqrt(2.0) * 2.0 ** np.arange(-20.0, 20.0), 0),
                           np.sqrt(0.5) * 2.0 ** np.arange(-20.0, 20.0), 1.0 + np.arange(-50, 51) * 2.0 ** -52]),
    "cbrt": np.concatenate([TINY * np.arange(-200, 200), 2.0 ** np.arange(-1074.0, 1024.0),
                            -(3.0 ** np.arange(-600.0, 600.0)), np.nextafter(np.arange(1.0, 9.0) ** 3, 0)]),
    "log1p": np.concatenate([TINY * np.arange(-3, 4), 2.0 ** np.arange(-60.0, 1024.0), -(2.0 ** np.arange(-60.0, 0.0)),
                             [-1.0, -1.5, np.inf, -np.inf, np.nan, 0.0, -0.0]]),
}


@pytest.mark.parametrize("fn", sorted(EDGES))
def test_math_edges(fn):
    x = np.ascontiguousarray(EDGES[fn], np.float64)
    c, g = kzo.math_fn(fn, x), hip.math_fn(fn, x)
    bad = np.nonzero(c.view(np.int64) != g.view(np.int64))[0]
    assert bad.size == 0, (fn, x[bad[:5]], c[bad[:5]], g[bad[:5]])


@pytest.mark.parametrize("channels", ["all", "no-kn", "bridge"])
def test_radstate_corners(channels):
    """One golden state with each slot in turn set to values that reach the
    selects: no field, tiny and huge densities and energies, zero and negative
    internal and radiation energy, infinity and NaN."""
    op = T.opac_params_puffy()
    if channels == "no-kn":
        op.kleinnishina = 0  # one channel off: the code with run-time tests
    if channels == "bridge":
        op.synchrotron_bridge = 1
    inp, _ = read_kgld("rad/rad_thermo.kgld", 36, 13)
    pp = np.ascontiguousarray(inp[:8, 23:36])
    g = geoms(inp[:8])
    rows, geo = [], []
    for i in range(len(pp)):
        for slots in ((0,), (1,), (9,), (6, 7, 8), (0, 1), (1, 9)):
            for v in (0.0, 1e-300, 1e-120, 1e-30, 1e30, 1e120, -1e-10, np.inf, np.nan):
                q = pp[i].copy()
                q[list(slots)] = v
                rows.append(q)
                geo.append(g[i])
    rows, geo = np.array(rows), np.array(geo)
    for full in (0, 1):
        c = kzo.radstate(rows, geo, GAM, op, full)[:, [0, 1, 3, 4, 5, 6, 7, 11, 13]]
        z = hip.radstate(rows, geo, GAM, op, full)[:, :9]
        if not full:  # the entropy column
            c, z = c[:, :8], z[:, :8]
        bad = np.nonzero(~((c == z) | (np.isnan(c) & np.isnan(z))).all(axis=1))[0]
        assert bad.size == 0, (full, rows[bad[0]], c[bad[0]], z[bad[0]])


def test_exp_outside_the_integers():
    """Operands whose quotient by ln 2 no integer holds: NaN, infinities and
    everything past 1.5e9."""
    x = np.array([np.nan, np.inf, -np.inf, 1e9, -1e9, 1.5e9, -1.5e9, 2e9, -2e9, 1e19, -1e19, 1e300, -1e300,
                  np.finfo(float).max, -np.finfo(float).max])
    c, g = kzo.math_fn("exp", x), hip.math_fn("exp", x)
    assert np.array_equal(c, g, equal_nan=True), (c, g)


@pytest.mark.parametrize("y", [0.2, 0.86, 4.0 / 3.0, 1.0 / 3.0, 0.69, 1.69, 0.463, -0.463, 1.5, 2.5, -7.5, 40.5])
def test_pow_edges(y):
    """The exponents of the opacities and of the entropy, and two whose results
    over- and underflow: subnormal, zero, negative, infinite and NaN bases."""
    x = np.concatenate([EDGES["log"], EDGES["cbrt"], [1.0, -1.0, 0.0, -0.0, np.inf, -np.inf, np.nan, 1.7976931348623157e308],
                        10.0 ** np.linspace(-323.0, 308.0, 4001)])
    c, g = kzo.math_fn("pow", x, y), hip.math_fn("pow", x, y)
    bad = np.nonzero(~((c.view(np.int64) == g.view(np.int64)) | (np.isnan(c) & np.isnan(g))))[0]
    assert bad.size == 0, (y, x[bad[:5]], c[bad[:5]], g[bad[:5]])


@pytest.mark.parametrize("gam", [5.0 / 3.0, 4.0 / 3.0, 1.5, 2.0, 1.2])
def test_entropy_edges(gam):
    """The entropy of a state over densities and internal energies from
    subnormal to huge, zero, negative, infinite and NaN; 1.5 and 2 make its
    exponent 1 / (gam - 1) an integer, which takes the general power."""
    v = np.concatenate([[0.0, -0.0, 5e-324, 2.0 ** -1022, 1.0, -1e-10, -1e30, np.inf, -np.inf, np.nan,
                         1.7976931348623157e308], 10.0 ** np.arange(-320.0, 308.0, 23.0),
                        10.0 ** np.linspace(-30.0, 30.0, 25)])
    inp, _ = read_kgld("rad/rad_thermo.kgld", 36, 13)
    pp = np.repeat(inp[:1, 23:36], v.size ** 2, axis=0)
    pp[:, 0], pp[:, 1] = np.repeat(v, v.size), np.tile(v, v.size)
    geo = np.repeat(geoms(inp[:1]), len(pp), axis=0)
    op = T.opac_params_puffy()
    c, g = kzo.radstate(pp, geo, gam, op, 1)[:, 13], hip.radstate(pp, geo, gam, op, 1)[:, 8]
    bad = np.nonzero(~((c == g) | (np.isnan(c) & np.isnan(g))))[0]
    assert bad.size == 0, (gam, pp[bad[0], :2], c[bad[0]], g[bad[0]])
    assert np.isfinite(c).sum() > 100
