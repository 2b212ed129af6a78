"""Uploads and downloads of every size class (csrc/transfer.hpp): below and
above the size where several host threads share a copy, with whole and partial
chunks, from several threads at once, and again after the last block released
the pinned chunks.  A state comes back as it went, bit for bit."""
import threading

import numpy as np
import pytest

from mara2_amd import abi
from mara2_amd.runtime import Block

pytestmark = pytest.mark.gpu

# 8 372 160 and 8 390 400 bytes lie either side of the threshold of 8 MiB;
# then a ragged copy, more chunks than lanes, and one of whole chunks only
CELLS = [(60, 31, 1), (452, 455, 1), (452, 456, 1), (701, 663, 1), (118, 97, 85), (508, 1020, 1)]


def _roundtrip(cells, seed):
    desc = abi.make_desc(law="hydro", bc="outflow", cells=cells)
    P = np.random.default_rng(seed).random(abi.array_shape(desc))
    with Block(desc) as blk:
        for _ in range(2):
            blk.upload(P)
            Q = blk.download()
            assert np.array_equal(P, Q)


@pytest.mark.parametrize("cells", CELLS)
def test_roundtrip(cells):
    _roundtrip(cells, 1)


def test_several_threads_at_once():
    errors = []

    def work(k):
        try:
            for n in range(3):
                _roundtrip(CELLS[2 + (k + n) % 3], 10 * k + n)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
