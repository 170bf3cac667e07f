"""x**(1/3) of dgswem_amd/csrc/dg_crmath.hpp over every exponent of a double: the host build against the double
nearest to the exact value, around the ends of the reduction's exponent classes and at arguments whose exact value
lies close to a midpoint between two doubles."""
import math
import random

import pytest

from test_crmath_cpu import exact_pow3, lib  # noqa: F401  (lib: the fixture)

# arguments whose exact value lies within 2^-71 of a midpoint
HARD = ["0x1.c3f6a44128e51p+383", "0x1.9d6e2e9efe09ap+641", "0x1.93a5c4fbbe881p-762", "0x1.38714129fe26p+639",
        "0x1.9ea5fd473c11ap+708", "0x1.1bdbda99692a8p+966", "0x1.694403c7f806bp+709", "0x1.aa5d674fc9bccp-763",
        "0x1.37da414a06cedp+687", "0x1.2c2fb43d9a462p+703", "0x1.762f7d2891c74p-646", "0x1.3a15c9f8b90dcp+860",
        "0x1.dd402d3500f76p+836"]


@pytest.mark.parametrize("x", [float.fromhex(h) for h in HARD])
def test_near_midpoints(lib, x):  # noqa: F811
    assert lib.t_pow3(x) == exact_pow3(x)


def test_every_exponent(lib):  # noqa: F811
    """One argument of every exponent, and the ends of each exponent class (powers of two with their neighbours),
    which the reduction's x = 2^3k m has to put into [1/2, 4)."""
    rng = random.Random(17)
    args = [math.ldexp(rng.uniform(0.5, 1.0), e) for e in range(-1073, 1025)]
    for e in list(range(-30, 31)) + [-1074, -1073, -1022, -1021, -1020, 1021, 1022, 1023]:
        x = math.ldexp(1.0, e)
        args += [x, math.nextafter(x, 0.0), math.nextafter(x, math.inf)]
    bad = [x.hex() for x in args if x > 0.0 and lib.t_pow3(x) != exact_pow3(x)]
    assert not bad, bad[:5]


def test_depths_of_every_class(lib):  # noqa: F811
    rng = random.Random(23)
    bad = [x.hex() for x in (2.0 ** rng.uniform(-12.0, 14.0) for _ in range(1500)) if lib.t_pow3(x) != exact_pow3(x)]
    assert not bad, bad[:5]
    assert lib.t_pow3(math.inf) == math.inf and math.isnan(lib.t_pow3(math.nan)) and math.isnan(lib.t_pow3(-math.inf))
