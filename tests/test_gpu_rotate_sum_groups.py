"""Sums of rotations whose key switches run together: many short sums take few
launches, sums that a chunk boundary cuts are added up, sums without a rotated
input and of more inputs than a launch takes, and chunks cut by the size of the
digits, word for word against each sum by itself and the oracle."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")
import oracle as orc  # noqa: E402
from oracle import hybrid  # noqa: E402

STEPS = (1, -2, 5)


def _note(msg):
    print("[case]", msg, flush=True)
    sys.stdout.flush()


def _rand(rng, ctx, polys, l):
    return np.stack([np.stack([rng.integers(0, q, ctx.n, dtype=np.uint64) for q in ctx.moduli[:l]])
                     for _ in range(polys)])


def _env(logn, chain, alpha, inputs):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    _note("rotation sums logn=%d primes=%d alpha=%d" % (logn, len(chain), alpha))
    ctx = nx.Context(logn, chain, special_primes=alpha)
    sk = nx.SecretKey(ctx, seed=41)
    gk = nx.KSwitchKeys(ctx).generate_galois(sk, [ctx.elt_from_step(s) for s in STEPS], seed=42)
    rng = np.random.default_rng(logn + alpha)
    data = [_rand(rng, ctx, 2, ctx.L) for _ in range(inputs)]
    data[0] = np.broadcast_to(np.array(ctx.moduli[:ctx.L], dtype=np.uint64)[None, :, None] - 1, data[0].shape).copy()
    return ctx, sk, gk, data, [nx.Ciphertext.from_array(ctx, d, 1, 2.0 ** 30) for d in data]


def _oracle(ctx, gk, alpha, datas, steps):
    el = [ctx.elt_from_step(s) if s else 0 for s in steps]
    arr = {e: gk.key_array(e) for e in set(el) if e}
    kk = [arr[e] if e else None for e in el]
    if alpha == 1:
        return orc.rotate_sum(datas, el, kk, ctx.moduli, ctx.log_n)
    return hybrid.rotate_sum_hybrid(datas, el, kk, ctx.moduli, ctx.L, alpha, ctx.log_n)


@pytest.mark.parametrize("logn,chain,alpha", [(14, [46, 60, 46], 1), (14, [51, 46, 46, 46, 51, 51], 2),
                                              (13, [46, 60, 46], 1)])
def test_groups(logn, chain, alpha):
    ctx, sk, gk, data, cts = _env(logn, chain, alpha, 4)
    # chunks of even size cut the sums of 31 and 20; 0: only inputs without a rotation
    sizes = [1, 2, 0, 31, 1, 20, 3, 40]
    groups, steps, k = [], [], 0
    for g, size in enumerate(sizes):
        groups.append([cts[(k + i) % 4] for i in range(max(size, 2))])
        steps.append([STEPS[(k + i) % 3] if size else 0 for i in range(max(size, 2))])
        if size > 2:
            steps[-1][size // 2] = 0
        k += size
    got = [c.to_array() for c in nx.rotate_sum_many(groups, steps, gk)]
    for g in range(len(sizes)):
        assert np.array_equal(got[g], nx.rotate_sum(groups[g], steps[g], gk).to_array()), g
    for g in (3, 7):
        want = _oracle(ctx, gk, alpha, [data[cts.index(c)] for c in groups[g]], steps[g])
        assert np.array_equal(got[g], want), g


def test_launches():
    """forty sums of one rotated input: one launch a chunk, not one a sum"""
    ctx, sk, gk, data, cts = _env(14, [46, 46, 46], 1, 4)
    groups = [[cts[i % 4]] for i in range(40)]
    steps = [[STEPS[i % 3]] for i in range(40)]
    ctx.synchronize()
    nx.profile_select("ks_lift_col,ks_row_inner_rot")
    try:
        nx.rotate_sum_many(groups, steps, gk)
        ctx.synchronize()
        counts = [nx.profile_read(c)[0] for c in ("ks_lift_col", "ks_row_inner_rot")]
    finally:
        nx.profile_select("")
    assert counts == [2, 2]


def test_chunks_of_digits():
    """20 limbs at N = 2^17: the digits of four inputs fill a chunk"""
    ctx, sk, gk, data, cts = _env(17, [40] * 20 + [46], 1, 5)
    steps = [STEPS[i % 3] for i in range(5)]
    assert np.array_equal(nx.rotate_sum(cts, steps, gk).to_array(), _oracle(ctx, gk, 1, data, steps))
    rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=43)
    many = nx.multiply_relin_rescale_many(cts, cts[1:] + cts[:1], rk)
    for i in range(5):
        one = nx.rescale_to_next(nx.relinearize(nx.multiply(cts[i], cts[(i + 1) % 5]), rk))
        assert np.array_equal(many[i].to_array(), one.to_array()), i
