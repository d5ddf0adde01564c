"""The matrix product's accumulation over operands that lie where they were
made: one term, terms past a fold and past a launch, columns past a launch,
columns that begin inside a batch, and more batches than a launch names, against
the sums in Python integers."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")
from nexus_amd import mm  # noqa: E402


def _note(msg):
    print("[case]", msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("inner,cols,sizes", [(1, 1, [1]), (33, 3, [64, 32, 4]), (257, 1, [256, 2]), (2, 65, [128, 4]),
                                              (7, 13, [2] * 49)])
def test_accumulate(inner, cols, sizes):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    _note("accumulate inner=%d cols=%d batches=%d" % (inner, cols, len(sizes)))
    ctx = nx.Context(11, [60, 40, 60])
    sk = nx.SecretKey(ctx, seed=1)
    gk = nx.KSwitchKeys(ctx).generate_galois(sk, mm.reference_elts(ctx.n, 11), seed=2)
    rng = np.random.default_rng(inner)
    ct = mm.compress(ctx, sk, rng.uniform(-1, 1, ctx.n), 1e10, seed=3)
    made = {m: mm.expand(ct, m, gk) for m in set(sizes)}
    q = ctx.moduli[:2]
    top = [q[0] - 1, q[1] - 1]
    arrays = [np.stack([np.full(ctx.n, top[i], dtype=np.uint64) if j == 0 else
                        rng.integers(0, q[i], ctx.n, dtype=np.uint64) for i in range(2)]) for j in range(inner)]
    pts = [nx.Plaintext.from_array(ctx, a, 1, 2.0 ** 40) for a in arrays]
    got = mm.accumulate(pts, [made[m] for m in sizes], cols)
    flat = [(m, k) for m in sizes for k in range(m)]
    for i in sorted({0, cols // 2, cols - 1}):
        want = 0
        for j in range(inner):
            m, k = flat[i * inner + j]
            want = want + made[m][k].to_array().astype(object) * arrays[j].astype(object)[None]
        want = want % np.array(q, dtype=object)[None, :, None]
        assert np.array_equal(got[i].to_array(), want.astype(np.uint64)), i
