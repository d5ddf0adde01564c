"""The double-precision operations that the profiler records for the fused
conversions, against a count of what one output and one input word take."""
import sys

import pytest

pytestmark = pytest.mark.gpu

nx = pytest.importorskip("nexus_amd")

PRODUCT, REDUCE, TERM, QUOTIENT = 8, 4, 6, 6  # an FMA counts two


def _conversion(inputs):
    sums = -(-inputs // 8)  # terms share a quotient by eights
    return TERM * inputs + QUOTIENT * sums + (sums - 1) * (1 + REDUCE) + REDUCE


@pytest.mark.parametrize("alpha", [2, 8, 9])
def test_relinearisation(alpha):
    if nx.device_count() < 1:
        pytest.skip("no GPU visible")
    print("[case] operation counts alpha=%d" % alpha, flush=True)
    sys.stdout.flush()
    logn, l = 14, 9
    ctx = nx.Context(logn, [46] * l + [47] * alpha, special_primes=alpha)
    sk = nx.SecretKey(ctx, seed=1)
    rk = nx.KSwitchKeys(ctx).generate_relin(sk, seed=2)
    a = nx.encrypt(ctx, sk, nx.encode(ctx, [0.5], 2.0 ** 30), seed=3)
    t = nx.multiply(a, a)
    ctx.synchronize()
    nx.profile_select("ks_modup_col,ks_moddown_col")
    try:
        nx.relinearize(t, rk)
        ctx.synchronize()
        up, down = (nx.profile_read_flops(c) for c in ("ks_modup_col", "ks_moddown_col"))
    finally:
        nx.profile_select("")
    column = 7 * (PRODUCT + 2) / 2  # 2^7 rows: half a butterfly a word and stage
    digits = [min(alpha, l - j) for j in range(0, l, alpha)]
    outs = sum(l + alpha - s for s in digits)
    # a partial digit is counted as a full one's terms
    assert up == ctx.n * (l * (PRODUCT + REDUCE) + outs * (_conversion(alpha) + column))
    out = _conversion(alpha) + PRODUCT + 1 + REDUCE + column + REDUCE
    assert down == 2 * ctx.n * (alpha * (PRODUCT + REDUCE + 6) + l * out)
