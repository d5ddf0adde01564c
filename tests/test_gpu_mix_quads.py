"""Block mix four outputs at a time (tiles inside one block, primes below 2^51):
word for word the multiply-accumulate over the expanded plaintexts, with entry
steps of +1, -1 and others, ragged rows, output and input counts around
multiples of four, and primes of every form of the sums (46, 47, 50, 51 bits,
and 60 bits beside them)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")

LOGN, CHAIN = 14, [51, 46, 47, 50, 60, 60]


def _note(msg):
    print("[case]", msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def env():
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    ctx = nx.Context(LOGN, CHAIN)
    rng = np.random.default_rng(1)
    limbs = ctx.L
    q = np.array(ctx.moduli[:limbs], dtype=np.uint64)[None, :, None]
    cts = []
    for i in range(128):
        d = np.stack([np.stack([rng.integers(0, m, ctx.n, dtype=np.uint64) for m in ctx.moduli[:limbs]])
                      for _ in range(2)])
        if i % 5 == 0:
            d[:, :, ::2] = np.broadcast_to(q - 1, d.shape)[:, :, ::2]
        cts.append(nx.Ciphertext.from_array(ctx, d, 1, 2.0 ** 30))
    return ctx, cts


def _band(K, M, count, sign):
    index = np.full((M, K), -1, dtype=np.int32)
    for m in range(M):
        for k in range(K):
            e = m + k - K // 2 if sign > 0 else m - k + K // 2
            if 0 <= e < count:
                index[m, k] = e
    return index


def _rows(K, M):
    return np.arange(M * K, dtype=np.int32).reshape(M, K)


def _mixed(K, M, count):
    rng = np.random.default_rng(K + M)
    index = rng.integers(-1, count, (M, K)).astype(np.int32)
    index[: M // 2, : K // 2] = (np.arange(K // 2)[None, :] * 3 + np.arange(M // 2)[:, None]) % count
    index[M - 1] = -1  # an output without terms
    return index


@pytest.mark.parametrize("period,index", [
    (64, _band(127, 64, 64, -1)), (64, _band(64, 127, 64, +1)), (64, _band(5, 3, 64, +1)), (4, _band(9, 8, 16, -1)),
    (128, _rows(33, 7)), (1, _rows(4, 4)), (64, _mixed(45, 22, 32)), (2, np.zeros((1, 1), dtype=np.int32)),
], ids=["down", "up", "small", "short", "rows", "least", "mixed", "one"])
def test_quads_equal_plain_accumulate(env, period, index):
    ctx, cts = env
    M, K = index.shape
    _note("mix quads K=%d M=%d period=%d" % (K, M, period))
    count = max(int(index.max()) + 1, 1)
    W = nx.PeriodicPlaintexts(ctx, np.random.default_rng(K).uniform(-1, 1, (count, period)), 2.0 ** 30)
    pts = {}
    outs = nx.multiply_periodic_mix(cts[:K], W, index)
    for m, o in enumerate(outs):
        terms = [(k, int(e)) for k, e in enumerate(index[m]) if e >= 0]
        if not terms:
            assert not o.to_array().any()
            continue
        for _, e in terms:
            if e not in pts:
                pts[e] = W.expand(e)
        ref = nx.multiply_plain_accumulate([cts[k] for k, _ in terms], [pts[e] for _, e in terms])
        assert np.array_equal(o.to_array(), ref.to_array()), "output %d" % m
