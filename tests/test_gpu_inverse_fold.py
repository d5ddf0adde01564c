"""Where the inverse's column pass runs: large batches of a hybrid key switch fold
it into conversions of up to nine inputs, small ones launch it, and after autotuning the
key switch's digits follow the choice measured on them.
Fused products with a remainder chunk and the top word of every prime, against
the same products one at a time.

The tuner's choices are process-wide, so the checks run in a process of their
own (this file as a program)."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fold():
    nx = pytest.importorskip("nexus_amd")
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], cwd=ROOT, timeout=100, capture_output=True,
                       text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stderr[-3000:]


def _inverse_columns(nx, ctx, f):
    """f() and the column passes of inverse transforms that it launched"""
    ctx.synchronize()
    nx.profile_select("ntt_inv_col")
    try:
        out = f()
        ctx.synchronize()
        return out, nx.profile_read("ntt_inv_col")[0]
    finally:
        nx.profile_select("")


def main():
    sys.path.insert(0, ROOT)
    import nexus_amd as nx

    # the last: passes of a chunk of 32 and a remainder of 3, digits and ModDown of alpha + 1 inputs
    for logn, chain, alpha, passes in ((16, [46] * 5 + [47] * 3, 3, 2), (15, [51] + [46] * 9 + [51] * 8, 8, 2),
                                       (16, [46] * 9 + [47] * 9, 9, 3), (16, [46] * 10 + [47] * 10, 10, 4)):
        print("[case] inverse fold logn=%d alpha=%d" % (logn, alpha), flush=True)
        ctx = nx.Context(logn, chain, special_primes=alpha)
        sk = nx.SecretKey(ctx, seed=8)
        rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=9)
        rng = np.random.default_rng(alpha)
        l = ctx.L
        q = np.array(ctx.moduli[:l], dtype=np.uint64)[None, :, None]
        cts = [nx.Ciphertext.from_array(ctx, rng.integers(0, 2 ** 63, (2, l, ctx.n), dtype=np.uint64) % q, 1,
                                        2.0 ** 30) for _ in range(3)]
        cts.append(nx.Ciphertext.from_array(ctx, np.broadcast_to(q - 1, (2, l, ctx.n)).copy(), 1, 2.0 ** 30))
        count = 35  # a chunk of 32 and a remainder
        a = [cts[i % 4] for i in range(count)]
        b = [cts[(i + 1 + i // 4) % 4] for i in range(count)]
        many, cols = _inverse_columns(nx, ctx, lambda: nx.multiply_relin_rescale_many(a, b, rk, fused=True))
        assert cols == passes, cols
        ones = {}
        for i in range(count):
            key = (i % 4, (i + 1 + i // 4) % 4)
            if key not in ones:
                one, cols = _inverse_columns(nx, ctx, lambda: nx.multiply_relin_rescale_many(a[i:i + 1], b[i:i + 1], rk,
                                                                                          fused=True))
                assert cols == 2, cols
                ones[key] = one[0].to_array()
            assert np.array_equal(many[i].to_array(), ones[key]), i
        rep = nx.autotune(ctx, reps=2)
        digits = {e["batch"]: e["mode"] for e in rep["digits"]}[32]
        _, cols = _inverse_columns(nx, ctx, lambda: nx.multiply_relin_rescale_many(a[:32], b[:32], rk, fused=True))
        # the tuner's ModDowns end at 32 polys: these 64 keep the default rule
        assert cols == (alpha > 9 or digits != 0) + (alpha > 8), (cols, rep["digits"])
        del ctx, sk, rk, cts, a, b, many, one
    print("ok", flush=True)


if __name__ == "__main__":
    main()
