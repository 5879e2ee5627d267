"""The whole-GPU path's control values come back through host memory lent to
each call: calls from several threads and streams at once, and one after another
on changing streams, give what a single call gives."""

import threading

import numpy as np
import pytest
import torch

from dxtb_amd import workloads
from dxtb_amd.engine import ScfOptions
from dxtb_amd.large import LargeSystem
from helpers import TIGHT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [1, 3])
def test_calls_from_threads_and_streams(threads):
    """Bitwise: every sum of the SCF has a fixed order (the forces' atomic
    sums do not, so the potential is compared)."""
    mols = [workloads.water_cluster(np.random.default_rng(k), 6 + 5 * k) for k in range(3)]
    opts = ScfOptions(**TIGHT)

    def run(z, p):
        big = LargeSystem(z, "cuda:0", opts=opts)
        e = big.run(p, forces=False)["energy"]
        torch.cuda.current_stream().synchronize()
        return e, big.pipe.pot.cpu().numpy()

    ref = [run(*m) for m in mols]
    got, errors = {}, []

    def work(t):
        try:
            for rep in range(3):
                with torch.cuda.stream(torch.cuda.Stream()):
                    i = (t + rep) % 3
                    got[t, rep] = (i, run(*mols[i]))
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors and len(got) == 3 * threads
    for i, (e, v) in got.values():
        assert e == ref[i][0] and np.array_equal(v, ref[i][1])
