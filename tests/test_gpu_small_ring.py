"""Transforms of the rings that one workgroup can hold: around the batch size
at which 2^13 changes from two passes to whole limbs, at the thread counts'
edges, with primes of both arithmetic paths, random and extreme words."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")
import oracle as orc  # noqa: E402


def _note(msg):
    print("[case]", msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("logn,polys,limbs", [(11, 2, 3), (12, 2, 1), (12, 3, 5), (13, 2, 1), (13, 2, 32), (13, 3, 22),
                                              (13, 2, 33)])
def test_transforms(logn, polys, limbs):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    _note("small ring logn=%d limbs=%dx%d" % (logn, polys, limbs))
    bits = [60, 51, 46, 58, 40, 50]
    ctx = nx.Context(logn, [bits[i % len(bits)] for i in range(limbs)] + [60])
    rng = np.random.default_rng(logn * 100 + limbs)
    data = np.stack([np.stack([rng.integers(0, q, ctx.n, dtype=np.uint64) for q in ctx.moduli[:limbs]])
                     for _ in range(polys)])
    data[0, 0] = ctx.moduli[0] - 1
    fwd = nx.transform_to_ntt(nx.Ciphertext.from_array(ctx, data, 1, 2.0 ** 30, ntt_form=False))
    got = fwd.to_array()
    for p in range(polys):
        for i in range(limbs):
            assert np.array_equal(got[p, i], orc.ntt_forward(data[p, i].copy(), logn, ctx.moduli[i])), (p, i)
    assert np.array_equal(nx.transform_from_ntt(fwd).to_array(), data)
