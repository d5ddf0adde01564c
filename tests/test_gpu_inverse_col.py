"""Batches large enough that the conversions of a hybrid key switch run the
inverse transform's column pass themselves, against the same operations one at a
time (where they do not): the products' ModUp and ModDown, and a hoisted
ModDown, with full and partial last digits and both column lengths.  (Where the
passes ran is read from the launches in test_gpu_inverse_fold.py: choices that
the autotuner made in this process may have moved them here.)"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")


def _rand(rng, ctx, polys, l):
    return np.stack([np.stack([rng.integers(0, q, ctx.n, dtype=np.uint64) for q in ctx.moduli[:l]])
                     for _ in range(polys)])


@pytest.mark.parametrize("logn,chain,alpha,count", [(16, [50, 46, 46, 46, 46, 51, 51], 2, 32),
                                                    (16, [46] * 5 + [47] * 3, 3, 33),
                                                    (17, [46] * 3 + [51] * 2, 2, 16)])
def test_batches(logn, chain, alpha, count):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    print("[case] inverse column logn=%d primes=%d alpha=%d count=%d" % (logn, len(chain), alpha, count), flush=True)
    sys.stdout.flush()
    ctx = nx.Context(logn, chain, special_primes=alpha)
    sk = nx.SecretKey(ctx, seed=8)
    rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=9)
    rng = np.random.default_rng(logn + alpha)
    l = ctx.L
    top = np.broadcast_to(np.array(ctx.moduli[:l], dtype=np.uint64)[None, :, None] - 1, (2, l, ctx.n)).copy()
    cts = [nx.Ciphertext.from_array(ctx, _rand(rng, ctx, 2, l), 1, 2.0 ** 40) for _ in range(3)]
    cts.append(nx.Ciphertext.from_array(ctx, top, 1, 2.0 ** 40))
    a = [cts[i % 4] for i in range(count)]
    b = [cts[(i + 1 + i // 4) % 4] for i in range(count)]
    many = nx.multiply_relin_rescale_many(a, b, rk)
    ones = {}
    for i in range(count):
        key = (i % 4, (i + 1 + i // 4) % 4)
        if key not in ones:
            ones[key] = nx.multiply_relin_rescale_many(a[i:i + 1], b[i:i + 1], rk)[0].to_array()
        assert np.array_equal(many[i].to_array(), ones[key]), i
    steps = [1 if i % 2 else -2 for i in range(count)]
    gk = nx.KSwitchKeys(ctx).generate_galois(sk, [ctx.elt_from_step(s) for s in (1, -2)], seed=10)
    got = nx.rotate_hoisted(cts[-1], steps, gk)
    for s in (1, -2):
        want = nx.rotate_hoisted(cts[-1], [s], gk)[0].to_array()
        for i in range(count):
            if steps[i] == s:
                assert np.array_equal(got[i].to_array(), want), i
