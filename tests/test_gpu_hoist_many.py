"""Several inputs rotated by the same steps: one input to one past what a thread
and a launch take together, enough digits that sums of every prime size fold,
generated and uploaded keys, random and extreme words, against the oracle's
hoisted rotation of each."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")
import oracle as orc  # noqa: E402


@pytest.mark.parametrize("chain", [[46] * 18 + [47], [50] * 6 + [50], [51] * 4 + [51], [60, 46, 51, 60]],
                         ids=["46", "50", "51", "mixed"])
@pytest.mark.parametrize("inputs", [1, 2, 3, 4, 5, 33])
def test_rotations(chain, inputs):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    print("[case] hoisted many primes=%d inputs=%d" % (len(chain), inputs), flush=True)
    sys.stdout.flush()
    logn = 6
    ctx = nx.Context(logn, chain)
    steps = [1, 0, -3, 1]
    el = {s: ctx.elt_from_step(s) for s in steps if s}
    sk = nx.SecretKey(ctx, seed=3)
    gk = nx.KSwitchKeys(ctx).generate_galois(sk, list(el.values()), seed=4)
    rng = np.random.default_rng(inputs)
    q = np.array(ctx.moduli[:ctx.L], dtype=np.uint64)[None, :, None]
    data = [rng.integers(0, 2 ** 63, (2, ctx.L, ctx.n), dtype=np.uint64) % q for _ in range(inputs)]
    data[-1] = np.broadcast_to(q - 1, data[-1].shape).copy()
    # the first step's key replaced by words at the top of their range, read in full
    ext = gk.key_array(el[1])
    ext[:] = (np.array(ctx.moduli, dtype=np.uint64) - 1)[None, None, :ext.shape[2], None]
    gk2 = nx.KSwitchKeys(ctx).generate_galois(sk, [el[-3]], seed=4)
    gk2.upload(el[1], ext)
    cts = [nx.Ciphertext.from_array(ctx, d, 1, 2.0 ** 30) for d in data]
    for keys in (gk, gk2):
        got = nx.rotate_hoisted_many(cts, steps, keys)
        arr = {s: keys.key_array(el[s]) for s in el}
        for b in range(inputs):
            for k, s in enumerate(steps):
                want = data[b] if s == 0 else orc.rotate_hoisted(data[b], el[s], arr[s], ctx.moduli, logn)
                assert np.array_equal(got[b][k].to_array(), want), (b, s)
        one = nx.rotate_hoisted(cts[-1], steps, keys)
        for k in range(len(steps)):
            assert np.array_equal(one[k].to_array(), got[-1][k].to_array()), k
