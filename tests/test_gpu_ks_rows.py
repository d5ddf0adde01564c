"""Key switches whose digits go from the column pass straight into the row pass
and inner product (rings 2^14 .. 2^17): relinearisation and sums of rotations,
word for word against the oracle.

The cases sit at the edges of the kernels: every pass split (7 + 7, 7 + 8,
8 + 8, 8 + 9 stages), primes just below the bounds that choose the form of a
sum of products (46 and 47 bits: unreduced digits or not; 50 and 51: the number
of terms between two reductions; 58 and 60, which calls as small as most of
these take through a stored ModUp: test_gpu_ks_wide.py has both), more digits
than terms between two reductions, short last digits, levels below the top, one
output prime past a chunk, and keys uploaded with extreme words."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")
import oracle as orc  # noqa: E402
from oracle import hybrid  # noqa: E402

CASES = [
    # (log2 N, chain, special primes, chain index)
    (14, [60, 46, 47, 50, 51, 58, 60], 1, 1),
    (14, [46] * 19 + [46], 1, 1),
    (14, [51] * 9 + [51], 1, 2),
    (14, [50] * 9 + [50], 1, 1),
    (15, [51, 46, 46, 51, 51], 1, 1),
    (16, [58, 40, 40, 58], 1, 1),
    (17, [47, 60, 51], 1, 1),
    (14, [51, 46, 46, 46, 46, 51, 51], 2, 1),
    (14, [51] + [46] * 12 + [51] * 8, 8, 1),
    (15, [51] + [46] * 7 + [51] * 5, 5, 2),
    (17, [46] * 4 + [51] * 3, 3, 1),
    (14, [45] * 13 + [50] * 12, 12, 1),
]


def _note(msg):
    print("[case]", msg, flush=True)
    sys.stdout.flush()


def _rand(rng, moduli, polys, limbs, n):
    return np.stack([np.stack([rng.integers(0, q, n, dtype=np.uint64) for q in moduli[:limbs]]) for _ in range(polys)])


def _key_primes(ctx):
    return np.array(ctx.moduli, dtype=np.uint64)


def _switch(ctx, alpha, data, key):
    """(c0, c1) + key switch of c2"""
    if alpha == 1:
        return orc.switch_key(data[:2], data[2], ctx.moduli, key, ctx.log_n)
    ks = np.stack(hybrid.switch_key_hybrid(data[2], key, ctx.moduli, ctx.L, alpha, ctx.log_n))
    mods = np.array(ctx.moduli[: data.shape[1]], dtype=np.uint64)[None, :, None]
    return (data[:2] + ks) % mods  # below 2^62


@pytest.mark.parametrize("logn,chain,alpha,ci", CASES)
def test_relinearize(logn, chain, alpha, ci):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    _note("relinearize logn=%d primes=%d alpha=%d level=%d" % (logn, len(chain), alpha, ci))
    ctx = nx.Context(logn, chain, special_primes=alpha)
    sk = nx.SecretKey(ctx, seed=11)
    rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=12)
    rng = np.random.default_rng(13)
    l = ctx.limbs_of(ci)
    q = np.array(ctx.moduli[:l], dtype=np.uint64)[None, :, None]
    data = _rand(rng, ctx.moduli, 3, l, ctx.n)
    top = np.broadcast_to(q - 1, data.shape).copy()
    key = rk.key_array(0)
    for d in (data, top):
        got = nx.relinearize(nx.Ciphertext.from_array(ctx, d, ci, 2.0 ** 40), rk).to_array()
        assert np.array_equal(got, _switch(ctx, alpha, d, key))
    # an uploaded key is read in full: every word at the top of its range
    ext = np.broadcast_to((_key_primes(ctx) - 1)[None, None, :, None], key.shape).copy()
    ext[:, 1, :, ::3] = 0
    rk2 = nx.KSwitchKeys(ctx)
    rk2.upload(0, ext)
    got = nx.relinearize(nx.Ciphertext.from_array(ctx, data, ci, 2.0 ** 40), rk2).to_array()
    assert np.array_equal(got, _switch(ctx, alpha, data, ext))


@pytest.mark.parametrize("logn,chain,alpha,ci", [c for c in CASES if c[0] != 17 or c[2] == 1])
def test_rotate_sum(logn, chain, alpha, ci):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    _note("rotate_sum logn=%d primes=%d alpha=%d level=%d" % (logn, len(chain), alpha, ci))
    ctx = nx.Context(logn, chain, special_primes=alpha)
    sk = nx.SecretKey(ctx, seed=21)
    steps = [1, 0, -5]
    el = [ctx.elt_from_step(s) if s else 0 for s in steps]
    gk = nx.KSwitchKeys(ctx).generate_galois(sk, [e for e in el if e], seed=22)
    kk = [gk.key_array(e) if e else None for e in el]
    rng = np.random.default_rng(23)
    l = ctx.limbs_of(ci)
    datas = [_rand(rng, ctx.moduli, 2, l, ctx.n) for _ in steps]
    cts = [nx.Ciphertext.from_array(ctx, d, ci, 2.0 ** 40) for d in datas]
    if alpha == 1:
        want = orc.rotate_sum(datas, el, kk, ctx.moduli, logn)
    else:
        want = hybrid.rotate_sum_hybrid(datas, el, kk, ctx.moduli, ctx.L, alpha, logn)
    assert np.array_equal(nx.rotate_sum(cts, steps, gk).to_array(), want)
    # a key without seeds among generated ones: all are read in full
    gk2 = nx.KSwitchKeys(ctx).generate_galois(sk, [el[0]], seed=22)
    gk2.upload(el[2], kk[2])
    kk2 = [gk2.key_array(e) if e else None for e in el]
    want2 = want if np.array_equal(kk2[0], kk[0]) else (
        orc.rotate_sum(datas, el, kk2, ctx.moduli, logn) if alpha == 1
        else hybrid.rotate_sum_hybrid(datas, el, kk2, ctx.moduli, ctx.L, alpha, logn))
    assert np.array_equal(nx.rotate_sum_many([cts, cts[:1]], [steps, steps[:1]], gk2)[0].to_array(), want2)


def test_batch_equals_single():
    """several targets under one key: each input's words are its own key switch's"""
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    for logn, chain, alpha in ((15, [51, 46, 46, 51], 1), (16, [51] + [46] * 9 + [51] * 4, 4)):
        _note("batch logn=%d alpha=%d" % (logn, alpha))
        ctx = nx.Context(logn, chain, special_primes=alpha)
        sk = nx.SecretKey(ctx, seed=31)
        rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=32)
        rng = np.random.default_rng(33)
        cts = [nx.Ciphertext.from_array(ctx, _rand(rng, ctx.moduli, 2, ctx.L, ctx.n), 1, 2.0 ** 40) for _ in range(6)]
        many = nx.multiply_relin_rescale_many(cts[:5], cts[1:], rk)
        for i in range(5):
            one = nx.rescale_to_next(nx.relinearize(nx.multiply(cts[i], cts[i + 1]), rk))
            assert np.array_equal(many[i].to_array(), one.to_array()), i
