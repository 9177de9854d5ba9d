"""The branch-free device transcendentals (koral-zig_amd/csrc/kz_dev_math.h)
compiled for the host, with the C library's frexp and ldexp for the gfx950
builtins and a saturating conversion for the instruction that dm_int names:
every result has the bits of kz_math.h (NaN for
NaN) at every special operand and threshold, and no operand, NaN, infinity and
the largest magnitudes included, is converted to an integer that cannot hold
it (the build traps there)."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "koral-zig_amd" / "csrc"

SOURCE = r"""
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#define __device__
#define __forceinline__ inline
#define KZM_QUAL static inline
static inline double __builtin_amdgcn_ldexp(double x, int e) { return ldexp(x, e); }
static inline double __builtin_amdgcn_frexp_mant(double x) { int e; return isfinite(x) ? frexp(x, &e) : x; }
static inline int __builtin_amdgcn_frexp_exp(double x) { int e = 0; if (isfinite(x)) frexp(x, &e); return e; }
// v_cvt_i32_f64: saturates, 0 for NaN
static inline int cvt_i32(double x) { return x != x ? 0 : x >= 2147483647.0 ? 2147483647 : x <= -2147483648.0 ? -2147483647 - 1 : (int)x; }
#include "dev_math.h"
using namespace kzd;
static double entropy(double p, double rho, double n) { return kzm_log(kzm_pow(p, n) / kzm_pow(rho, n + 1.0)); }
static double from_log(double x, double y) { double h, l; dm_log_dd(x, &h, &l); return dm_pow_from_log(h, l, y); }
// argv[1]: function; stdin: rows of three doubles; stdout: rows of (device, kz_math.h)
int main(int, char **argv) {
  double a[3], o[2];
  const char *f = argv[1];
  while (fread(a, sizeof a, 1, stdin) == 1) {
    if (!strcmp(f, "exp")) o[0] = dm_exp(a[0]), o[1] = kzm_exp(a[0]);
    else if (!strcmp(f, "log")) o[0] = dm_log(a[0]), o[1] = kzm_log(a[0]);
    else if (!strcmp(f, "log1p")) o[0] = dm_log1p(a[0]), o[1] = kzm_log1p(a[0]);
    else if (!strcmp(f, "cbrt")) o[0] = dm_cbrt(a[0]), o[1] = kzm_cbrt(a[0]);
    else if (!strcmp(f, "pow_frac")) o[0] = dm_pow_frac(a[0], a[1]), o[1] = kzm_pow(a[0], a[1]);
    else if (!strcmp(f, "pow_from_log")) o[0] = from_log(a[0], a[1]), o[1] = kzm_pow(a[0], a[1]);
    else if (!strcmp(f, "log_entropy")) o[0] = dm_log_entropy(a[0], a[1], a[2]), o[1] = entropy(a[0], a[1], a[2]);
    else return 3;
    fwrite(o, sizeof o, 1, stdout);
  }
  return 0;
}
"""

HUGE = np.finfo(np.float64).max
TINY = 2.0 ** -1074
SPECIAL = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1.0, -1.0, TINY, -TINY, 2.0 ** -1022, HUGE, -HUGE, 1e10, -1e10,
                    3e9, -3e9, 0.5, 2.0, np.nextafter(1, 0), np.nextafter(1, 2)])
RNG = np.random.default_rng(41)
WIDE = np.concatenate([SPECIAL, 10.0 ** RNG.uniform(-323, 308, 4000), -(10.0 ** RNG.uniform(-323, 308, 500)),
                       2.0 ** np.arange(-1074.0, 1024.0)])
POSITIVE = WIDE[(WIDE > 0) & np.isfinite(WIDE)]


def _grid(x, *more):
    """Every combination of the operands as rows of three."""
    cols = np.meshgrid(x, *(more + ([0.0],) * (2 - len(more))), indexing="ij")
    return np.stack([c.ravel() for c in cols], axis=1)


ROWS = {
    "exp": _grid(np.concatenate([WIDE, RNG.uniform(-760, 720, 4000), np.linspace(-746, -707, 2001),
                                 np.nextafter(709.782712893384, [0, 1e9]), [709.782712893384, -745.1332191019412],
                                 np.nextafter(-745.1332191019412, [0, -1e9])])),
    "log": _grid(WIDE),
    "log1p": _grid(np.concatenate([WIDE, RNG.uniform(-1, 1, 2000)])),
    "cbrt": _grid(WIDE),
    # the exponents of the opacities; results over- and underflow at the ends
    "pow_frac": _grid(WIDE, (0.2, 0.86, 4.0 / 3.0, 1.0 / 3.0, 0.69, 1.69, 0.463, 7.5)),
    "pow_from_log": _grid(POSITIVE, (0.69, -0.463, 1.69, 0.463, -7.5)),
    # 1 / (gam - 1) for gam = 5/3, 4/3, 3/2, 2 and the values that take the general way
    "log_entropy": _grid(np.concatenate([SPECIAL, POSITIVE[::40]]), np.concatenate([SPECIAL, POSITIVE[::60]]),
                         (1.0 / (5.0 / 3.0 - 1.0), 1.0 / (4.0 / 3.0 - 1.0), 2.0, 1.0, 0.0, -1.0, -2.5, np.inf, np.nan)),
}


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("dev_math")
    text = (CSRC / "kz_dev_math.h").read_text()
    (d / "dev_math.h").write_text(text.replace('asm("v_cvt_i32_f64 %0, %1" : "=v"(k) : "v"(x));', "k = cvt_i32(x);"))
    (d / "m.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-mfma", "-I", str(CSRC),
                    "-fsanitize=float-cast-overflow,shift,signed-integer-overflow", "-fsanitize-undefined-trap-on-error",
                    "-o", str(d / "m"), str(d / "m.cpp")], check=True)
    return d / "m"


@pytest.mark.parametrize("fn", sorted(ROWS))
def test_device_math(program, fn):
    rows = np.ascontiguousarray(ROWS[fn])
    r = subprocess.run([str(program), fn], input=rows.tobytes(), capture_output=True)
    assert r.returncode == 0, (r.returncode, "an operand was converted to an integer that cannot hold it")
    out = np.frombuffer(r.stdout).reshape(-1, 2)
    assert len(out) == len(rows)
    dev, ref = out[:, 0], out[:, 1]
    bad = np.nonzero((dev.view(np.int64) != ref.view(np.int64)) & ~(np.isnan(dev) & np.isnan(ref)))[0]
    assert bad.size == 0, (fn, bad.size, rows[bad[:4]], dev[bad[:4]], ref[bad[:4]])
