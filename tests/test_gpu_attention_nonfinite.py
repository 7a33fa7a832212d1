"""GPU: attention over scores that are not finite, whole and in key chunks,
prompts and decode steps. A NaN or +inf score, and a query whose admitted
scores are all -inf, give NaN (the oracle's three passes: exp(x - max) / sum);
the other rows stay within the error bound of finite attention."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_prefill_split import attend, check, inputs

pytestmark = pytest.mark.gpu

PLANTS = ["nan q", "inf q", "nan k", "inf k", "scores -inf", "first scores -inf"]


def plant(what, q, k, s, kv):
    """Plants it; the first row of q that meets it (s: none)."""
    if what == "nan q":
        q[s - 1, :] = np.nan
        return s - 1
    if what == "inf q":
        q[s - 1, :] = np.inf  # scores of +inf and -inf
        return s - 1
    if what in ("nan k", "inf k"):
        k[kv - 1, :] = np.nan if what == "nan k" else np.inf  # admitted by the last query only
        q[s - 1, :] = np.abs(q[s - 1, :])
        return s - 1
    q[:] = np.abs(q)
    k[: kv if what == "scores -inf" else kv // 2, :] = -np.inf
    return 0 if what == "scores -inf" else s


def expect(got, want, q, k, v, s, kv, h, hkv, d, met):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    if met == s:
        lo = kv // 2  # the keys at -inf weigh nothing
        check(got, q, k[lo:], v[lo:], s, kv - lo, h, hkv, d, True)
    else:
        assert np.all(np.isnan(got[met:]))
        check(got, q, k, v, s, kv, h, hkv, d, True, rows=range(met))


def oracle(q, k, v, s, kv, h, hkv, d):
    out, st = orc.attention(q, k, v, orc.attention_params(s, kv, h, d, kv_head_count=hkv, causal=True))
    assert st == 0
    return out


@pytest.mark.parametrize("what", PLANTS)
@pytest.mark.parametrize("kv", [40, 300, 600])  # one chunk, two, four
@pytest.mark.parametrize("d", [32, 64, 80, 96, 112, 128])
def test_prompts(dev, d, kv, what):
    s, h, hkv = 5, 4, 2
    q, k, v = inputs(d + kv, s, kv, h, hkv, d)
    met = plant(what, q, k, s, kv)
    with np.errstate(all="ignore"):
        expect(attend(dev, q, k, v, s, kv, h, hkv, d, causal=True), oracle(q, k, v, s, kv, h, hkv, d),
               q, k, v, s, kv, h, hkv, d, met)


@pytest.mark.parametrize("what", PLANTS)
@pytest.mark.parametrize("kv", [40, 700])
@pytest.mark.parametrize("d", [8, 64, 96, 128, 256])
@pytest.mark.parametrize("hkv", [1, 4])
def test_decode_steps(dev, hkv, d, kv, what):
    h = 4
    q, k, v = inputs(d + kv, 1, kv, h, hkv, d)
    met = plant(what, q, k, 1, kv)
    with np.errstate(all="ignore"):
        expect(attend(dev, q, k, v, 1, kv, h, hkv, d, causal=True), oracle(q, k, v, 1, kv, h, hkv, d),
               q, k, v, 1, kv, h, hkv, d, met)
