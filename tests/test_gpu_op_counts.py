"""The double-precision operations that the profiler records for the fused
conversions, against a count of what one output and one input word take, and the
bytes it records for the inner products, whose inputs share one key.

The autotuner's choices are process-wide and may replace these launches, so the
checks run in a process of their own (this file as a program)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRODUCT, REDUCE, TERM, QUOTIENT = 8, 4, 6, 6  # an FMA counts two


def test_relinearisation():
    nx = pytest.importorskip("nexus_amd")
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], cwd=ROOT, timeout=100, capture_output=True,
                       text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stderr[-3000:]


def _conversion(inputs):
    sums = -(-inputs // 8)  # terms share a quotient by eights
    return TERM * inputs + QUOTIENT * sums + (sums - 1) * (1 + REDUCE) + REDUCE


def main():
    sys.path.insert(0, ROOT)
    import nexus_amd as nx

    logn, l = 14, 9
    for alpha in (2, 8, 9):
        print("[case] operation counts alpha=%d" % alpha, flush=True)
        ctx = nx.Context(logn, [46] * l + [47] * alpha, special_primes=alpha)
        sk = nx.SecretKey(ctx, seed=1)
        rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=2)
        a = nx.encrypt(ctx, sk, nx.encode(ctx, [0.5], 2.0 ** 30), seed=3)
        t = nx.multiply(a, a)
        ctx.synchronize()
        nx.profile_select("ks_modup_col,ks_moddown_col,ks_row_inner")
        nx.relinearize(t, rk)
        ctx.synchronize()
        up, down = (nx.profile_read_flops(c) for c in ("ks_modup_col", "ks_moddown_col"))
        rows = nx.profile_read("ks_row_inner")
        nx.profile_select("")
        column = 7 * (PRODUCT + 2) / 2  # 2^7 rows: half a butterfly a word and stage
        # a partial digit is counted with a full one's terms
        outs = sum(l + alpha - min(alpha, l - j) for j in range(0, l, alpha))
        assert up == ctx.n * (l * (PRODUCT + REDUCE) + outs * (_conversion(alpha) + column)), (alpha, up)
        out = _conversion(alpha) + PRODUCT + 1 + REDUCE + column + REDUCE
        assert down == 2 * ctx.n * (alpha * (PRODUCT + REDUCE + 6) + l * out), (alpha, down)
        # one input: its key's uniform half comes from seeds
        digits = -(-l // alpha)
        word = 8 * ctx.n * (l + alpha)
        assert rows[0] == 1 and rows[2] == word * (digits + digits + 2), (alpha, rows)
        nx.profile_select("ks_row_inner")
        nx.multiply_relin_rescale_many([a] * 3, [a] * 3, rk)
        ctx.synchronize()
        rows = nx.profile_read("ks_row_inner")
        nx.profile_select("")
        assert rows[0] == 1 and rows[2] == word * (3 * digits + 2 * digits + 3 * 2), (alpha, rows)
        del ctx, sk, rk, a, t
    print("ok", flush=True)


if __name__ == "__main__":
    main()
