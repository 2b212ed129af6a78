"""The shortcuts of csrc/exact.hpp and the literal forms behind them: states
where a face or a zone is not ordinary (negative, zero, tiny or huge pressure
and density, NaN and infinite zones, Alfven and sound speeds that coincide)
stepped beside ordinary ones, bit for bit against the oracle in every kernel
that evaluates them (pencils, 2-D and 3-D tiles, flux arrays, 2-D MHD tiles)."""
import numpy as np
import pytest

import oracle
from mara2_amd import abi, problems
from mara2_amd.runtime import Block

pytestmark = pytest.mark.gpu

# every mesh takes another kernel: pencils, 2-D tiles, 3-D tiles
MESHES = {"1d": (70, 1, 1), "2d": (67, 9, 1), "3d": (66, 7, 6)}
# (density factor, pressure factor) of the planted zones; None: as it is
PLANTED = {"negative_pressure": (None, -0.3), "zero_pressure": (None, 0.0), "tiny": (1e-210, 1e-200),
           "huge": (1e70, 1e65), "nan": (np.nan, None), "infinite": (np.inf, None), "near_limits": (1e-39, 1e-45)}


def _state(desc, seed=11):
    rng = np.random.default_rng(seed)
    P = problems.empty(desc)
    P[..., 0] = 1 + 0.3 * rng.random(P.shape[:3])
    P[..., 4] = 1 + 0.3 * rng.random(P.shape[:3])
    P[..., 1:4] = 0.5 * rng.standard_normal(P.shape[:3] + (3,))
    if P.shape[3] >= 8:
        P[..., 5:8] = 0.4 * rng.standard_normal(P.shape[:3] + (3,))
    return P


def _compare(desc, P, steps=2, dt=1e-3):
    problems.apply_bc(desc, P)
    Po = P.copy()
    with Block(desc) as blk:
        blk.upload(P)
        for _ in range(steps):
            blk.advance(dt, check=False)
            oracle.advance(desc, Po, 0.0, dt)
        Pg = blk.download()
    assert np.array_equal(Pg, Po, equal_nan=True)


@pytest.mark.parametrize("planted", list(PLANTED))
@pytest.mark.parametrize("riemann", ["hlle", "hllc"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_hydro_zones_that_are_not_ordinary(mesh, riemann, planted):
    desc = abi.make_desc(law="hydro", riemann=riemann, bc="periodic", cells=MESHES[mesh])
    P = _state(desc)
    rho, p = PLANTED[planted]
    for at in (8, 33, 34, 60):  # alone and side by side
        z = P[at, P.shape[1] // 2, P.shape[2] // 2]
        z[0] = z[0] if rho is None else z[0] * rho
        z[4] = z[4] if p is None else z[4] * p
    with np.errstate(all="ignore"):
        _compare(desc, P, steps=1)


@pytest.mark.parametrize("field", ["aligned", "none", "weak"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_mhd_fields_without_an_ordinary_discriminant(mesh, field):
    """aligned: the Alfven speed along the normal equals the sound speed, so
    the discriminant is zero or rounds below it; none and weak: B = 0, or too
    small for its square."""
    desc = abi.make_desc(law="mhd", riemann="hlle", bc="periodic", cells=MESHES[mesh], pressure_floor=1e-6)
    P = _state(desc)
    half = P.shape[0] // 2
    P[:half, ..., 5:8] = 0.0
    if field == "aligned":
        P[:half, ..., 5] = np.sqrt(desc.gamma * P[:half, ..., 4])
    elif field == "weak":
        P[:half, ..., 6] = 1e-165
    _compare(desc, P)
