"""Key switches with primes of 2^51 and above: few inputs take the stored ModUp,
many the kernel that multiplies the digits in its row pass, and both give the
oracle's words.  Which of them ran is read from the launch classes, on both
sides of the rule (workgroups of a launch, share of wide primes at N = 2^17);
primes below 2^51 alone never store a ModUp."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")
import oracle as orc  # noqa: E402

ROWS = ("ks_row_inner", "ks_row_inner_rot")


def _rand(rng, ctx, polys, l):
    return np.stack([np.stack([rng.integers(0, q, ctx.n, dtype=np.uint64) for q in ctx.moduli[:l]])
                     for _ in range(polys)])


def _ran(ctx, f):
    """f(), and whether a row kernel ran"""
    ctx.synchronize()
    nx.profile_select(",".join(ROWS))
    try:
        out = f()
        ctx.synchronize()
        return out, sum(nx.profile_read(c)[0] for c in ROWS) > 0
    finally:
        nx.profile_select("")


# (log2 N, chain, one input fused, inputs of a large call, the large call fused)
CASES = [(14, [60, 46, 47, 50, 51, 58, 60], False, 5, True), (14, [60, 46, 47, 50, 51, 58, 60], False, 4, False),
         (15, [60] * 7 + [60], False, 2, True), (16, [58, 46, 46, 46, 46, 46, 58], False, 2, True),
         (16, [60] * 8, True, 2, True), (17, [60, 46, 46, 46, 46, 46, 46, 60], True, 2, True),
         (17, [60, 60, 60, 60, 46, 46, 60], False, 3, False), (14, [46, 46, 50], True, 2, True)]


@pytest.mark.parametrize("logn,chain,one,count,many", CASES)
def test_paths(logn, chain, one, count, many):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    print("[case] wide key switch logn=%d primes=%d count=%d" % (logn, len(chain), count), flush=True)
    sys.stdout.flush()
    ctx = nx.Context(logn, chain)
    sk = nx.SecretKey(ctx, seed=51)
    rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=52)
    steps = (1, -3)
    el = [ctx.elt_from_step(s) for s in steps]
    gk = nx.KSwitchKeys(ctx).generate_galois(sk, el, seed=53)
    rng = np.random.default_rng(logn + count)
    l = ctx.L
    data = [_rand(rng, ctx, 2, l) for _ in range(count)]
    data[-1] = np.broadcast_to(np.array(ctx.moduli[:l], dtype=np.uint64)[None, :, None] - 1, data[-1].shape).copy()
    cts = [nx.Ciphertext.from_array(ctx, d, 1, 2.0 ** 20) for d in data]
    # one key: each input by itself and all together
    a, b = cts, cts[1:] + cts[:1]
    tensors = [nx.multiply(x, y) for x, y in zip(a, b)]
    t0 = tensors[0].to_array()
    first, ran = _ran(ctx, lambda: nx.relinearize(tensors[0], rk))
    assert ran == one
    assert np.array_equal(first.to_array(), orc.switch_key(t0[:2], t0[2], ctx.moduli, rk.key_array(0), logn))
    if l > 1:
        got, ran = _ran(ctx, lambda: nx.multiply_relin_rescale_many(a, b, rk))
        assert ran == many
        for i in range(count):
            want = nx.rescale_to_next(nx.relinearize(tensors[i], rk)).to_array()
            assert np.array_equal(got[i].to_array(), want), i
    # sums of rotations: one by itself and `count` of them together
    groups = [[cts[g], cts[(g + 1) % count]] for g in range(count)]
    summed, ran = _ran(ctx, lambda: nx.rotate_sum(groups[0], list(steps), gk))
    assert ran == one
    want = orc.rotate_sum([data[0], data[1 % count]], el, [gk.key_array(e) for e in el], ctx.moduli, logn)
    assert np.array_equal(summed.to_array(), want)
    sums, ran = _ran(ctx, lambda: nx.rotate_sum_many(groups, [list(steps)] * count, gk))
    assert ran == many
    for g in range(count):
        assert np.array_equal(sums[g].to_array(), nx.rotate_sum(groups[g], list(steps), gk).to_array()), g
