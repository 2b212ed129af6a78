"""The z planes a fused 3-D block marches per work-group while no shape was set
(fused_planes in csrc/fused.hpp): the result is the one of every set shape, bit
for bit, for a block of its own, a group of blocks and the no-allocation
step's size, and the shape a block reports stays the documented default."""
import numpy as np
import pytest

from mara2_amd import abi, problems
from mara2_amd.runtime import Block, Group

pytestmark = pytest.mark.gpu


def _random(desc, seed=3):
    rng = np.random.default_rng(seed)
    P = problems.empty(desc)
    P[..., 0] = 1 + 0.2 * rng.random(P.shape[:3])
    P[..., 4] = 1 + 0.2 * rng.random(P.shape[:3])
    P[..., 1:4] = 0.3 * rng.standard_normal(P.shape[:3] + (3,))
    return problems.apply_bc(desc, P)


@pytest.mark.parametrize("recon", ["pcm", "plm", "weno5"])
@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed"])
@pytest.mark.parametrize("cells", [(8, 8, 3), (66, 9, 5), (65, 33, 50), (40, 70, 131)])
def test_unset_planes_equal_set_ones(cells, precision, recon):
    desc = abi.make_desc(law="hydro", recon=recon, riemann="hllc", cells=cells, precision=precision)
    P = _random(desc)
    out = []
    for planes in (None, 16, 3):
        with Block(desc) as blk:
            assert blk.get_shape().zplanes == 16
            if planes:
                blk.set_shape(abi.make_shape(zplanes=planes))
            blk.upload(P)
            blk.run(0.3, 1e300, 3)
            out.append(blk.download())
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_a_groups_members_equal_the_block():
    desc = abi.make_desc(law="hydro", riemann="hllc", cells=(48, 40, 36))
    P = _random(desc)
    with Block(desc) as blk, Group(desc, (2, 2, 2)) as grp:
        blk.upload(P)
        grp.upload(P)
        for _ in range(2):
            blk.advance(1e-3)
            grp.advance(1e-3)
        assert np.array_equal(blk.download(), grp.download())
