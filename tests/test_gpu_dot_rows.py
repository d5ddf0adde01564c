"""Rows of plaintext products over shared ciphertexts: every number of rows a
launch can take and one past it, with every plaintext there and with holes, one
term and a count past a launch's, at words of the full range, against Python
integers."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")


@pytest.mark.parametrize("logn,count", [(1, 1), (3, 33), (11, 3)])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_rows(logn, count, rows):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    print("[case] dot rows logn=%d count=%d rows=%d" % (logn, count, rows), flush=True)
    sys.stdout.flush()
    ctx = nx.Context(logn, [60, 46, 60])
    rng = np.random.default_rng(rows)
    q = np.array(ctx.moduli[:2], dtype=np.uint64)[:, None]

    def rand(*shape):
        return (rng.integers(0, 2 ** 63, shape + (2, ctx.n), dtype=np.uint64) % q).astype(np.uint64)

    c = rand(count, 2)
    p = rand(rows, count)
    c[0], p[0, 0] = q - 1, q - 1
    cts = [nx.Ciphertext.from_array(ctx, x, 1, 2.0 ** 30) for x in c]
    for holes in (False, True):
        keep = rng.random((rows, count)) < (0.6 if holes else 2.0)
        keep[:, rows % count] = True
        pts = [[nx.Plaintext.from_array(ctx, p[g, r], 1, 2.0 ** 30) if keep[g, r] else None for r in range(count)]
               for g in range(rows)]
        got = nx.multiply_plain_accumulate_multi(cts, pts)
        for g in range(rows):
            want = sum(c[r].astype(object) * p[g, r].astype(object)[None] for r in range(count) if keep[g, r])
            assert np.array_equal(got[g].to_array(), (want % q.astype(object)).astype(np.uint64)), g
