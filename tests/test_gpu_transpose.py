"""The tiles that move a state between MeshData's order and the device's
(csrc/kernels.hpp k_transpose): meshes with partial tiles along x and z, planes,
lines and every number of fields.  A state comes back as it went, and one step
of it equals the oracle's bit for bit, so every zone was where it belongs."""
import numpy as np
import pytest

import oracle
from mara2_amd import abi, problems
from mara2_amd.runtime import Block

pytestmark = pytest.mark.gpu

# with two guards a side: tiles are 32 zones along x by 16 along z (or y of a plane)
CELLS = [(28, 12, 1), (29, 13, 1), (61, 40, 1), (28, 3, 12), (30, 5, 13), (4, 6, 29), (70, 4, 4), (257, 1, 1)]


@pytest.mark.parametrize("law,cooling", [("hydro", 0.0), ("mhd", 0.0), ("mhd", 0.1)])
@pytest.mark.parametrize("cells", CELLS)
def test_zones_go_where_they_belong(cells, law, cooling):
    desc = abi.make_desc(law=law, recon="plm", riemann="hlle", bc="outflow", cells=cells, cooling_rate=cooling)
    rng = np.random.default_rng(5)
    P = 0.1 * rng.random(abi.array_shape(desc))
    P[..., 0] += 1.0
    P[..., 4] += 1.0
    problems.apply_bc(desc, P)
    Po = P.copy()
    with Block(desc) as blk:
        blk.upload(P)
        assert np.array_equal(blk.download(), P)
        blk.advance(1e-4)
        oracle.advance(desc, Po, 0.0, 1e-4)
        assert np.array_equal(blk.download(), Po)
