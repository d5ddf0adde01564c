"""Transforms of the rings that one workgroup can hold: around the batch size
at which 2^13 changes from two passes to whole limbs, at the thread counts'
edges, with primes of both arithmetic paths, random and extreme words; and the
transforms that take words of another prime as they load them (the key switch's
ModUp, its ModDown and the rescale), in every kind of first pass."""
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


# one whole limb, two passes, a batch past the change, and the first ring that
# always runs in two; last and special primes larger and smaller than the others
@pytest.mark.parametrize("logn,chain,special", [(11, [60, 46, 46], 60), (12, [46, 60, 40], 46), (13, [60, 60, 60, 60], 60),
                                                (13, [46, 60] * 6, 51), (14, [60, 46, 60], 58)])
def test_lift_and_centre(logn, chain, special):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    _note("lift and centre logn=%d primes=%d" % (logn, len(chain) + 1))
    ctx = nx.Context(logn, chain + [special])
    sk = nx.SecretKey(ctx, seed=5)
    rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=6)
    rng = np.random.default_rng(logn)
    key = rk.key_array(0)
    data = np.stack([np.stack([rng.integers(0, q, ctx.n, dtype=np.uint64) for q in ctx.moduli[:len(chain)]])
                     for _ in range(3)])
    top = np.broadcast_to(np.array(ctx.moduli[:len(chain)], dtype=np.uint64)[None, :, None] - 1, data.shape).copy()
    for d in (data, top):
        ct = nx.relinearize(nx.Ciphertext.from_array(ctx, d, 1, 2.0 ** 40), rk)
        got = ct.to_array()
        assert np.array_equal(got, orc.switch_key(d[:2], d[2], ctx.moduli, key, logn))
        want = np.stack([orc.rescale_poly_ntt(p, ctx.moduli[:len(chain)], logn) for p in got])
        assert np.array_equal(nx.rescale_to_next(ct).to_array(), want)
