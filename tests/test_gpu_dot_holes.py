"""Rows of plaintext products with missing plaintexts: how many launches they
take (seven and eight rows: two, unless every plaintext is there), and their
words against the single sums."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")


@pytest.mark.parametrize("rows,hole,launches", [(6, 5, 1), (7, 0, 2), (7, None, 1), (8, 7, 2), (8, None, 1),
                                                (14, 0, 3), (14, 13, 2), (13, 12, 2)])
def test_launches(rows, hole, launches):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    print("[case] dot holes rows=%d hole=%s" % (rows, hole), flush=True)
    sys.stdout.flush()
    ctx = nx.Context(11, [60, 46, 60])
    rng = np.random.default_rng(rows)
    q = np.array(ctx.moduli[:2], dtype=np.uint64)[:, None]
    cts = [nx.Ciphertext.from_array(ctx, rng.integers(0, 2 ** 63, (2, 2, ctx.n), dtype=np.uint64) % q, 1, 2.0 ** 30)
           for _ in range(3)]
    pts = [[nx.Plaintext.from_array(ctx, rng.integers(0, 2 ** 63, (2, ctx.n), dtype=np.uint64) % q, 1, 2.0 ** 30)
            for _ in cts] for _ in range(rows)]
    if hole is not None:
        pts[hole][1] = None
    ctx.synchronize()
    nx.profile_select("dot_plain")
    try:
        got = nx.multiply_plain_accumulate_multi(cts, pts)
        ctx.synchronize()
        assert nx.profile_read("dot_plain")[0] == launches
    finally:
        nx.profile_select("")
    for g in range(rows):
        on = [r for r in range(3) if pts[g][r] is not None]
        want = nx.multiply_plain_accumulate([cts[r] for r in on], [pts[g][r] for r in on])
        assert np.array_equal(got[g].to_array(), want.to_array()), g
