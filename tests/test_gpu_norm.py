"""RMSNorm over rows of more than one 64-token tile (one octet of tokens per workgroup) at the edges of
its channels per thread and token octets, against a float64 norm of the fp16 input; its sums of
squares are exact, bit for bit the scales of the kernel for up to 64 tokens."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plan(wavec, D, T, gamma):
    g = wavec.WaveGraph(kv_cache_max_seq=0, fold_rmsnorm_gamma=False)
    g.add_input("x", D, 1, T, is_1d=True)
    g.add_rmsnorm("n", "x", "y", D, gamma)
    g.set_output("y")
    return g.compile()


@pytest.mark.parametrize("D,T", [(1024, 65), (1025, 100), (2048, 2048), (3000, 777), (4097, 130),
                                 (8192, 72), (8193, 70), (768, 200), (767, 200), (2048, 8190),
                                 (768, 8200), (5000, 8224)])
def test_middling_token_counts(wavec, D, T):
    rng = np.random.default_rng(D + T)
    gamma = (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    plan = _plan(wavec, D, T, gamma)
    # magnitudes from the smallest subnormal to the largest fp16, a constant and a zero token
    x = (rng.standard_normal((D, T)) * 2.0 ** rng.integers(-24, 13, (1, T))).astype(np.float16)
    x[:, 0] = np.float16(65504.0)
    x[:, 1] = 0.0
    y, _ = plan.infer_f32(x.astype(np.float32)[:, None, :])
    x64 = x.astype(np.float64)
    ref = x64 / np.sqrt((x64 ** 2).mean(0) + 1e-5) * gamma.astype(np.float16).astype(np.float64)[:, None]
    # one fp16 rounding (half an ulp, 2^-11 relative, 2^-25 for subnormals) after three fp32
    # roundings of the scale and products (each 2^-24 relative)
    bound = np.abs(ref) * (2.0 ** -11 + 2.0 ** -21) + 2.0 ** -25
    assert np.all(np.abs(y[:, 0, :] - ref) <= bound)


def test_infinities_and_nans(wavec):
    """A token with an infinite channel scales to zeros and one NaN (inf * 0); one with a NaN is
    all NaN; the tokens beside them are not touched."""
    D, T = 1500, 80
    x = np.ones((D, 1, T), np.float32)
    x[7, 0, 3] = np.inf
    x[8, 0, 12] = np.nan
    y, _ = _plan(wavec, D, T, np.ones(D, np.float32)).infer_f32(x)
    assert np.isnan(y[7, 0, 3]) and np.all(np.delete(y[:, 0, 3], 7) == 0.0)
    assert np.all(np.isnan(y[:, 0, 12]))
    rest = np.delete(y[:, 0, :], [3, 12], axis=1)
    assert np.all(np.abs(rest - 1.0) < 2e-3)


def _tie_token(rng, D):
    """D fp16 values whose sum of squares lies 2^-48 beside the middle of two fp32 values."""
    x = rng.permutation(np.concatenate([rng.standard_normal(D - 64), np.zeros(64)])).astype(np.float16)
    units = lambda v: int(round(float(v) * 2.0 ** 24))  # exact: fp16 values are multiples of 2^-24
    free = list(np.flatnonzero(x == 0))
    total = sum(units(v) ** 2 for v in x)
    ulp = 1 << (total.bit_length() - 24)
    target = total // ulp * ulp + ulp // 2 + ulp + int(rng.choice([-1, 1]))
    while total < target:  # the rest as squares, largest first (11-bit significands)
        m = math.isqrt(target - total)
        drop = max(0, m.bit_length() - 11)
        m = m >> drop << drop
        x[free.pop()] = np.float16(m * 2.0 ** -24)
        total += m * m
    assert sum(units(v) ** 2 for v in x) == target and target.bit_length() - 24 == ulp.bit_length() - 1
    return x


@pytest.mark.parametrize("D", [768, 2048, 4096, 8192])
def test_sums_are_exact(wavec, D):
    """Sums next to the middle of two fp32 values, where a sum rounded on the way gives the other
    one: the outputs are those of the exact integer sums that run up to 64 tokens."""
    rng = np.random.default_rng(D)
    T = 640
    x = np.stack([_tie_token(rng, D) for _ in range(T)], 1)
    gamma = (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    y, _ = _plan(wavec, D, T, gamma).infer_f32(x.astype(np.float32)[:, None, :])
    few = _plan(wavec, D, 64, gamma)
    for t in range(0, T, 64):
        want, _ = few.infer_f32(x[:, t:t + 64].astype(np.float32)[:, None, :])
        assert np.array_equal(y[:, 0, t:t + 64].view(np.uint32), want[:, 0].view(np.uint32)), t
