"""Which kernel a periodic mix takes (four outputs a wave, or one): both sides of
the rule's lines -- inputs, outputs, share of terms that no group of four shares
-- word for word the multiply-accumulate over the expanded plaintexts, on chains
of each arithmetic path and of both."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")


CHAINS = {"mixed": [51, 46, 47, 50, 60, 60], "small": [51, 46, 47, 50], "wide": [60, 58, 60], "wide58": [58, 55, 58]}


@pytest.fixture(scope="module", params=list(CHAINS))
def env(request):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    ctx = nx.Context(14, CHAINS[request.param])
    rng = np.random.default_rng(3)
    q = np.array(ctx.moduli[:ctx.L], dtype=np.uint64)[None, :, None]
    cts = [nx.Ciphertext.from_array(ctx, rng.integers(0, 2 ** 63, (2, ctx.L, ctx.n), dtype=np.uint64) % q, 1,
                                    2.0 ** 30) for _ in range(40)]
    return ctx, cts, request.param in ("mixed", "small")


def _index(K, M, singles, step):
    """rows step k + m, in every row all but the first `singles` terms (of K)"""
    index = (step * np.arange(K)[None, :] + np.arange(M)[:, None] + (K if step < 0 else 0)) % 64
    index[:, :singles] = np.random.default_rng(K * M).integers(0, 64, (M, singles))
    return index.astype(np.int32)


@pytest.mark.parametrize("K,M,singles,step,quads", [
    (16, 16, 0, 1, True), (15, 16, 0, 1, False), (16, 15, 0, 1, False), (32, 16, 4, 1, True), (32, 16, 8, 1, False),
    (40, 17, 0, 1, True), (40, 19, 0, 1, False), (1, 1, 0, 1, False), (16, 64, 16, 1, False), (16, 16, 0, 3, True),
    (40, 16, 0, 0, True), (16, 16, 0, -1, True)])
def test_rule(env, K, M, singles, step, quads):
    ctx, cts, small = env
    print("[case] mix rule K=%d M=%d singles=%d" % (K, M, singles), flush=True)
    sys.stdout.flush()
    index = _index(K, M, singles, step)
    W = nx.PeriodicPlaintexts(ctx, np.random.default_rng(M).uniform(-1, 1, (64, 64)), 2.0 ** 30)
    ctx.synchronize()
    nx.profile_select("block_mix_quads")
    try:
        outs = nx.multiply_periodic_mix(cts[:K], W, index)
        ctx.synchronize()
        assert (nx.profile_read("block_mix_quads")[0] > 0) == (quads and small)
    finally:
        nx.profile_select("")
    pts = {int(e): W.expand(int(e)) for e in np.unique(index)}
    for m in sorted({0, M // 2, M - 1}):
        ref = nx.multiply_plain_accumulate(cts[:K], [pts[int(e)] for e in index[m]])
        assert np.array_equal(outs[m].to_array(), ref.to_array()), m
