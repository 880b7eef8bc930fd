"""GPU parity of attention over several query rows and an fp16 cache (the
matrix-core chunk path): rows and keys at the edges of its tiles (32 stacked
rows a wave, 128 a workgroup, 32 keys a tile, one and several key splits),
every head grouping, against float64. The query parts carry 2^-24 of the
row's elements and the sums are fp32: with scores of a few units 1e-6 holds
with room. Infinities and NaN reach exactly the rows that see them."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import fresh_thread, rel_l2, scratch_held

pytestmark = pytest.mark.gpu
F16 = 1


def _reference(q, k, v, causal):
    b, hq, sq, d = q.shape
    hkv, sk = k.shape[1:3]
    out = np.zeros(q.shape)
    for bi in range(b):
        for h in range(hq):
            s = q[bi, h].astype(np.float64) @ k[bi, h // (hq // hkv)].astype(np.float64).T / np.sqrt(d)
            if causal:
                s[np.arange(sk)[None] > (sk - sq + np.arange(sq))[:, None]] = -np.inf
            w = np.exp(s - s.max(1, keepdims=True))
            out[bi, h] = w / w.sum(1, keepdims=True) @ v[bi, h // (hq // hkv)].astype(np.float64)
    return out


def _run(rocm, dev, q, k, v, causal):
    b, hq, sq, d = q.shape
    hkv, sk = k.shape[1:3]
    out, qd, kd, vd = dev.empty(q.size), dev.put(q), dev.put(k), dev.put(v)
    rocm.call("aljabr_rocm_attention_gqa", dev.ptr(out), dev.ptr(qd), dev.ptr(kd), dev.ptr(vd), None, b, hq, hkv, sq,
              sk, d, F16, 0.0, causal)
    return dev.get(out).reshape(q.shape)


def _inputs(seed, b, hq, hkv, sq, sk, d):
    g = np.random.default_rng(seed)
    return (g.standard_normal((b, hq, sq, d), dtype=np.float32),
            g.standard_normal((b, hkv, sk, d), dtype=np.float32).astype(np.float16),
            g.standard_normal((b, hkv, sk, d), dtype=np.float32).astype(np.float16))


@pytest.mark.parametrize("b,hq,hkv,sq,sk,d", [
    (64, 32, 8, 33, 33, 64), (8, 48, 16, 11, 2047, 128), (4, 8, 8, 32, 8192 + 31, 64), (16, 8, 8, 129, 129, 128),
    (1, 16, 2, 17, 4100, 128), (2, 8, 4, 128, 1025, 64), (1, 5, 1, 127, 2111, 128), (1, 32, 8, 256, 2048, 128)])
@pytest.mark.parametrize("causal", [0, 1])
def test_chunk(rocm, dev, b, hq, hkv, sq, sk, d, causal):
    q, k, v = _inputs(sq + sk, b, hq, hkv, sq, sk, d)
    q[0, 0] *= 1e-3                          # rows of another magnitude
    assert rel_l2(_run(rocm, dev, q, k, v, causal), _reference(q, k, v, causal)) <= 1e-6


@pytest.mark.parametrize("b,sk", [(256, 70), (12, 1100)])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_rows_stay_apart(rocm, dev, b, sk, where, value):
    sq = 40
    q, k, v = _inputs(5, b, 4, 1, sq, sk, 64)
    want = _reference(q, k, v, 1)
    (k if where == "k" else v)[:, 0, sk - 10, 3] = value
    got = _run(rocm, dev, q, k, v, 1)
    assert rel_l2(got[:, :, :sq - 10], want[:, :, :sq - 10]) <= 1e-6
    if where == "v":
        hit = got[:, :, sq - 10:, 3]
        assert np.all(np.isnan(hit) if np.isnan(value) else hit == np.inf)
        assert rel_l2(got[:, :, sq - 10:, 4:], want[:, :, sq - 10:, 4:]) <= 1e-6
    elif np.isnan(value):
        assert np.isnan(got[:, :, sq - 10:]).all()
    else:                                    # +inf scores give NaN, -inf ones leave the key out
        up = q[:, :, sq - 10:, 3] > 0
        assert np.isnan(got[:, :, sq - 10:][up]).all() and np.isfinite(got[:, :, sq - 10:][~up]).all()


@pytest.mark.parametrize("hq,hkv,sq,sk,d", [(32, 8, 33, 2050, 128), (8, 8, 129, 1111, 64), (5, 1, 21, 8000, 128)])
@pytest.mark.parametrize("where", ["q", "v"])
def test_every_row_done_again(rocm, dev, hq, hkv, sq, sk, d, where):
    """An infinite V element that all rows of a KV head see, or one NaN row:
    the other elements, heads and rows keep their accuracy."""
    q, k, v = _inputs(7, 2, hq, hkv, sq, sk, d)
    want = _reference(q, k, v, 1)
    if where == "q":
        q[1, 1, 2, 5] = np.nan
    else:
        v[1, 0, 5, 3] = -np.inf
    got = _run(rocm, dev, q, k, v, 1)
    hit = np.zeros(got.shape, bool)
    if where == "q":
        hit[1, 1, 2] = True
        assert np.isnan(got[hit]).all()
    else:
        hit[1, :hq // hkv, :, 3] = True
        assert np.all(got[hit] == -np.inf)
    assert rel_l2(got[~hit], want[~hit]) <= 1e-6


# The chunk kernel's tile image (K, V^T, padded) is on the stream where it took
# the call; the split kernel's partials are smaller here.
@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,chunk", [
    (1, 32, 8, 32, 2048, 128, True), (1, 32, 8, 8, 4097, 128, True), (1, 32, 8, 7, 8192, 128, False),
    (1, 32, 8, 32, 1000, 128, False), (2, 8, 8, 64, 2048, 128, True), (16, 64, 8, 4, 2048, 64, True)])
def test_which_kernel(rocm, dev, b, hq, hkv, sq, sk, d, chunk):
    q, k, v = _inputs(3, b, hq, hkv, sq, sk, d)
    out, qd, kd, vd = dev.empty(q.size), dev.put(q), dev.put(k), dev.put(v)

    def body():
        rocm.call("aljabr_rocm_attention_gqa", dev.ptr(out), dev.ptr(qd), dev.ptr(kd), dev.ptr(vd), None, b, hq, hkv, sq,
                  sk, d, F16, 0.0, 1)
        return scratch_held(rocm)

    assert (fresh_thread(body) >= 2 * (k.size + v.size)) == chunk


def test_growing_calls_rarely_reallocate(rocm, dev):
    """A chunked prompt grows its keys with every call; the stream's scratch
    grows geometrically, not with each (a growth waits for the stream)."""
    import torch
    hq, hkv, sq, d = 32, 8, 128, 128
    q = torch.zeros(hq * sq * d, device="cuda:0")
    out = torch.empty_like(q)
    kv = torch.zeros(hkv * 8192 * d, dtype=torch.float16, device="cuda:0")
    torch.cuda.synchronize()

    def body():
        seen = []
        for sk in range(256, 8192 + 1, 128):
            rocm.call("aljabr_rocm_attention_gqa", dev.ptr(out), dev.ptr(q), dev.ptr(kv), dev.ptr(kv), None, 1, hq, hkv,
                      sq, sk, d, 1, 0.0, 1)
            seen.append(scratch_held(rocm))
        return seen

    seen = fresh_thread(body)
    assert seen[-1] >= 2 * 2 * hkv * 8192 * d
    assert len(set(seen)) <= 16
