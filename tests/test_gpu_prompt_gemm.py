"""GPU parity of the prompt GEMM (matmuls of more tokens than one pass of the
small-M kernels): every format at the edges of its tiles (32 tokens x 32 rows
a tile, 64 or 128 tokens and 256 rows a workgroup, 64-element chunks), against
the oracle. Tolerances: two fp16 activation parts carry 2^-22 an element, so
the fp32 sums' 2^-24 * sqrt(K) dominate and 2e-6 of a row holds with room. One
part (NF4 at K % 1024 == 0, Q4_K at the shapes whose passes round) is fp16(x)
times the exact weights: the reference multiplies fp16(x), so the same bound
holds (against x itself the rounding is 2^-12 of |w||x|, whatever cancels in
the row)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import fresh_thread, rel_l2, scratch_held

pytestmark = pytest.mark.gpu
Q4_0, Q8_0, Q4_K, Q6_K, NF4 = 2, 8, 12, 14, 100
TOL = 2e-6


def _weights(oracle, t, n, k, seed):
    if t in (Q4_K, Q6_K):
        return oracle.random_k_blocks(t, n * k // 256, seed, scale=0.5 / np.sqrt(k) / (200 if t == Q4_K else 1000))
    return oracle.quantize(t, oracle.normal(seed, n * k, 0.0, 0.5 / np.sqrt(k)))


def _decoded(oracle, t, raw, n, k):
    return oracle.dequant(t, raw, n * k).reshape(n, k).astype(np.float64)


def _parts(x, rounded):
    return (x.astype(np.float16) if rounded else x).astype(np.float64)


@pytest.mark.parametrize("t,n,k,m", [
    (Q4_0, 33, 32, 9), (Q4_0, 257, 1056, 65), (Q4_0, 64, 512, 128), (Q4_0, 300, 2048, 129),
    (Q8_0, 1, 96, 17), (Q8_0, 255, 640, 64), (Q8_0, 512, 2560, 197), (Q8_0, 31, 1024, 33),
    (Q4_K, 33, 256, 65), (Q4_K, 1000, 2304, 66), (Q4_K, 12300, 4096, 130), (Q4_K, 257, 4096, 300),
    (Q6_K, 7, 256, 65), (Q6_K, 1024, 2560, 97), (Q6_K, 300, 1280, 257)])
def test_gguf_prompt(rocm, dev, oracle, t, n, k, m):
    raw = _weights(oracle, t, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    x[1] *= 3e4 if k % 512 else 1.0          # past fp16's range: these shapes take any fp32 row
    y = dev.empty(m * n)
    w, xd = dev.put(raw), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, t, m)
    got = dev.get(y).reshape(m, n)
    rounded = t == Q4_K and k == 4096 and n > 8192
    ref = _parts(x, rounded) @ _decoded(oracle, t, raw, n, k).T
    for i in range(m):
        assert rel_l2(got[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("n,k,m", [(33, 192, 65), (257, 1280, 66), (300, 1024, 129), (2048, 2048, 256), (64, 4096, 145)])
def test_nf4_prompt(rocm, dev, oracle, n, k, m):
    codes, absmax = oracle.nf4_quantize(oracle.normal(5, n * k, 0.0, 0.02), 64)
    x = oracle.normal(6, m * k).reshape(m, k)
    y = dev.empty(m * n)
    c, a, xd = dev.put(codes), dev.put(absmax), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch_nf4", dev.ptr(y), dev.ptr(xd), dev.ptr(c), dev.ptr(a), k, n, 64, m)
    got = dev.get(y).reshape(m, n)
    ref = _parts(x, k % 1024 == 0) @ oracle.nf4_dequant(codes, absmax, n * k, 64).reshape(n, k).astype(np.float64).T
    for i in range(m):
        assert rel_l2(got[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("t,ns,k,m", [(Q8_0, (320, 64, 33), 640, 100), (Q4_K, (2048, 1024, 1056), 1024, 65),
                                      (Q4_0, (96, 32, 32), 1024, 40)])
def test_stacked_prompt(rocm, dev, oracle, t, ns, k, m):
    """Three matrices in one launch equal the oracle; repeats are identical."""
    raws = [_weights(oracle, t, n, k, 20 + i) for i, n in enumerate(ns)]
    x = oracle.normal(8, m * k).reshape(m, k)
    ws, xd = [dev.put(r) for r in raws], dev.put(x)
    outs = []
    for _ in range(2):
        ys = [dev.empty(m * n) for n in ns]
        rocm.call("aljabr_rocm_matvec_tb_triple_batch", *[dev.ptr(y) for y in ys], dev.ptr(xd),
                  *[dev.ptr(w) for w in ws], k, *ns, t, t, t, m)
        outs.append([dev.get(y).reshape(m, n) for y, n in zip(ys, ns)])
    for got, again, raw, n in zip(*outs, raws, ns):
        assert np.array_equal(got, again)
        assert rel_l2(got, x.astype(np.float64) @ _decoded(oracle, t, raw, n, k).T) <= TOL


def _put_at(dev, a, offset):
    """The bytes of `a` on the device, `offset` bytes past an aligned address."""
    import torch
    raw = np.ascontiguousarray(a).view(np.uint8).ravel()
    t = dev.empty(raw.size + offset, np.uint8)
    t[offset:] = torch.from_numpy(raw).to(t.device)
    torch.cuda.synchronize()
    return t, t.data_ptr() + offset


# Tokens that the passes run in fp32: weights off 16-byte alignment (4, 8), and
# the last single token of the passes of 8 (Q4_0, Q8_0) and 32 (K-quants).
# Elements past fp16's range and rows far below it keep their accuracy.
@pytest.mark.parametrize("t,n,k,m,offset,row", [
    (Q4_0, 96, 1024, 130, 4, 3), (Q8_0, 96, 512, 130, 8, 3), (Q4_0, 64, 1024, 129, 0, 128), (Q8_0, 96, 512, 193, 0, 192),
    (Q6_K, 300, 1024, 129, 0, 128), (Q4_K, 300, 1024, 193, 0, 192)])
@pytest.mark.parametrize("size", [1e5, 1e-5])
def test_gguf_prompt_keeps_fp32_range(rocm, dev, oracle, t, n, k, m, offset, row, size):
    raw = _weights(oracle, t, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    x[row] *= size
    w, wp = _put_at(dev, raw, offset)
    y, xd = dev.empty(m * n), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), wp, k, n, t, m)
    got = dev.get(y).reshape(m, n)
    ref = x.astype(np.float64) @ _decoded(oracle, t, raw, n, k).T
    for i in range(m):
        assert rel_l2(got[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("n,k,m", [(96, 1280, 130), (96, 1024, 130)])
@pytest.mark.parametrize("size", [1e5, 1e-5])
def test_nf4_prompt_with_absmax_off_8_bytes(rocm, dev, oracle, n, k, m, size):
    """The passes run these in fp32, whatever K: no rounding, fp32's range."""
    codes, absmax = oracle.nf4_quantize(oracle.normal(5, n * k, 0.0, 0.02), 64)
    x = oracle.normal(6, m * k).reshape(m, k)
    x[3] *= size
    a, ap = _put_at(dev, absmax, 4)
    y, c, xd = dev.empty(m * n), dev.put(codes), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch_nf4", dev.ptr(y), dev.ptr(xd), dev.ptr(c), ap, k, n, 64, m)
    got = dev.get(y).reshape(m, n)
    ref = x.astype(np.float64) @ oracle.nf4_dequant(codes, absmax, n * k, 64).reshape(n, k).astype(np.float64).T
    for i in range(m):
        assert rel_l2(got[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("n,k", [(12300, 4096), (300, 1024), (300, 1280)])
@pytest.mark.parametrize("size", [3e3, 6e4])
def test_q4_k_prompt_one_signed_rows(rocm, dev, oracle, n, k, size):
    """A sub-block's 32 activations are each in fp16's range, their sum is not."""
    m = 130
    raw = _weights(oracle, Q4_K, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    x[5] = size + x[5]
    y, w, xd = dev.empty(m * n), dev.put(raw), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, Q4_K, m)
    got = dev.get(y).reshape(m, n)
    ref = _parts(x, n > 8192) @ _decoded(oracle, Q4_K, raw, n, k).T
    for i in range(m):
        assert rel_l2(got[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("m", [65, 97, 129])
def test_last_q4_k_token_is_not_rounded(rocm, dev, oracle, m):
    """Where the passes round a Q4_K matrix's activations, a single token left
    over runs on the batch-1 kernel, in fp32."""
    n, k = 12300, 4096
    raw = _weights(oracle, Q4_K, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    x[-1] *= 1e5
    y, w, xd = dev.empty(m * n), dev.put(raw), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, Q4_K, m)
    got = dev.get(y).reshape(m, n)
    w64 = _decoded(oracle, Q4_K, raw, n, k)
    assert rel_l2(got[-1], x[-1].astype(np.float64) @ w64.T) <= TOL
    assert rel_l2(got[:-1], _parts(x[:-1], True) @ w64.T) <= TOL


def test_last_q4_k_token_of_a_stack_is_not_rounded(rocm, dev, oracle):
    ns, k, m = (12320, 12300, 64), 4096, 97
    raws = [_weights(oracle, Q4_K, n, k, 3 + i) for i, n in enumerate(ns)]
    x = oracle.normal(4, m * k).reshape(m, k)
    ys, ws, xd = [dev.empty(m * n) for n in ns], [dev.put(r) for r in raws], dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_triple_batch", *[dev.ptr(y) for y in ys], dev.ptr(xd), *[dev.ptr(w) for w in ws], k,
              *ns, Q4_K, Q4_K, Q4_K, m)
    for y, raw, n in zip(ys, raws, ns):
        got, w64 = dev.get(y).reshape(m, n), _decoded(oracle, Q4_K, raw, n, k)
        assert rel_l2(got[-1], x[-1].astype(np.float64) @ w64.T) <= TOL
        assert rel_l2(got[:-1], _parts(x[:-1], n > 8192) @ w64.T) <= TOL


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m", [8, 130])
def test_k_quants_need_16_byte_weights(rocm, dev, oracle, t, m):
    """Refused at every batch size, as the entry point says."""
    n, k = 64, 512
    w, wp = _put_at(dev, _weights(oracle, t, n, k, 3), 4)
    y, xd = dev.empty(m * n), dev.put(oracle.normal(4, m * k))
    with pytest.raises(rocm.RocmError) as e:
        rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), wp, k, n, t, m)
    assert e.value.status == rocm.ERR_BAD_ARGUMENT


def _random_blocks(t, n, k, seed):
    """Random Q4_0 / Q8_0 rows, made quickly."""
    g = np.random.default_rng(seed)
    b = np.empty((n * k // 32, 18 if t == Q4_0 else 34), np.uint8)
    b[:, 2:] = g.integers(0, 256, (b.shape[0], b.shape[1] - 2), np.uint8)
    b[:, :2] = (g.random(b.shape[0], np.float32) * (0.1 if t == Q4_0 else 0.01)).astype(np.float16).view(np.uint8).reshape(-1, 2)
    return b.reshape(n, -1)


@pytest.mark.parametrize("t,n,k,m", [(Q8_0, 4096, 14336, 512), (Q4_0, 4096, 14336, 512), (Q8_0, 2816, 1024, 1000),
                                     (Q8_0, 1024, 1024, 40), (Q4_0, 256, 14336, 64)])
def test_long_sums_keep_their_accuracy(rocm, dev, oracle, t, n, k, m):
    """The fp32 sums over K round no more than those of the passes of 8 tokens.
    A product's own rounding is 0.75e-7 and a chain of L additions adds 2.5e-8
    sqrt(L / 2): the passes' chains (of 8 to 16 blocks, then 8 waves or the
    slices) measure 0.97e-7 at K = 1024 and 1.19e-7 at K = 14336, one chain
    over all of K 1.25e-7 and 2.08e-7."""
    raw = _random_blocks(t, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    y, w, xd = dev.empty(m * n), dev.put(raw), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, t, m)
    step = 31 if n > 1024 else 3
    got = dev.get(y).reshape(m, n)[:, ::step]
    raw = np.ascontiguousarray(raw[::step])
    ref = x.astype(np.float64) @ _decoded(oracle, t, raw.ravel(), len(raw), k).T
    assert rel_l2(got, ref) <= (1.0e-7 if k == 1024 else 1.19e-7)


def test_q4_k_prompt_is_no_further_off_than_fp32(rocm, dev, oracle):
    """K % 512 != 0: the vector kernel's fp32 gives 1.13e-7 here; sub-block sums
    rounded to fp32 before their split gave 1.30e-7."""
    n, k, m = 2304, 2304, 512
    raw = _weights(oracle, Q4_K, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    y, w, xd = dev.empty(m * n), dev.put(raw), dev.put(x)
    vec = dev.empty(8 * n)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, Q4_K, m)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(vec), dev.ptr(xd), dev.ptr(w), k, n, Q4_K, 8)
    ref = x.astype(np.float64) @ _decoded(oracle, Q4_K, raw, n, k).T
    assert rel_l2(dev.get(y).reshape(m, n), ref) <= rel_l2(dev.get(vec).reshape(8, n), ref[:8])


def test_scratch_is_bounded_over_all_panels(rocm, dev):
    """The K slices' partial sums of all weight panels together keep to their bound."""
    import torch
    n, k, m = 152064, 8192, 384
    w = torch.zeros(n * k // 256 * 210, dtype=torch.uint8, device="cuda:0")
    x, y = torch.zeros(m * k, device="cuda:0"), torch.empty(m * n, device="cuda:0")
    torch.cuda.synchronize()

    def body():
        rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(x), dev.ptr(w), k, n, Q6_K, m)
        return scratch_held(rocm)

    assert 4 * m * k <= fresh_thread(body) <= 512 << 20
    assert not y.any()


# More than one panel of the weight image (128 MiB), segments that end inside
# a panel and one that crosses its end, with K slices (n small) and without.
@pytest.mark.parametrize("t,ns,k,m", [(Q8_0, (8032, 6016, 1001), 14336, 40), (Q4_0, (59008, 4032, 1003), 4096, 600)])
def test_prompt_panels(rocm, dev, oracle, t, ns, k, m):
    raws = [_random_blocks(t, n, k, 30 + i) for i, n in enumerate(ns)]
    x = oracle.normal(8, m * k).reshape(m, k)
    ws, xd, ys = [dev.put(r) for r in raws], dev.put(x), [dev.empty(m * n) for n in ns]

    def body():
        rocm.call("aljabr_rocm_matvec_tb_triple_batch", *[dev.ptr(y) for y in ys], dev.ptr(xd),
                  *[dev.ptr(w) for w in ws], k, *ns, t, t, t, m)
        return scratch_held(rocm)

    assert fresh_thread(body) >= (64 << 20) + 4 * m * k
    g = np.random.default_rng(1)
    for y, raw, n in zip(ys, raws, ns):
        got = dev.get(y).reshape(m, n)
        rows = np.unique(np.concatenate([np.arange(0, n, 257), np.arange(n - 40, n), g.integers(0, n, 64)]))
        ref = x.astype(np.float64) @ _decoded(oracle, t, np.ascontiguousarray(raw[rows]).ravel(), len(rows), k).T
        assert rel_l2(got[:, rows], ref) <= TOL
        assert np.abs(got[:, rows] - ref).max() <= 20 * TOL * np.abs(ref).max()


@pytest.mark.parametrize("m", [4097, 4100, 8192 + 33])
def test_prompt_token_passes(rocm, dev, oracle, m):
    """More tokens than one pass of 4096 takes."""
    n, k = 70, 512
    raw = _weights(oracle, Q8_0, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    y, w, xd = dev.empty(m * n), dev.put(raw), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, Q8_0, m)
    got = dev.get(y).reshape(m, n)
    ref = x.astype(np.float64) @ _decoded(oracle, Q8_0, raw, n, k).T
    for i in range(m):
        assert rel_l2(got[i], ref[i]) <= TOL, i


# Which path takes a call: the prompt GEMM holds its activation image (2 bytes
# an element and part) on a stream that had none; the passes' partial sums and
# images of 8 to 64 tokens are smaller. Both sides of the lines, single
# matrices and stacks.
@pytest.mark.parametrize("t,ns,k,m,prompt", [
    (Q4_0, (4096,), 4096, 17, False), (Q4_0, (4096,), 4096, 25, True), (Q8_0, (4096,), 4096, 9, False),
    (Q4_0, (4096, 1024, 1024), 4096, 9, True), (Q8_0, (2560, 640, 640), 2560, 17, True), (Q8_0, (1280,), 1280, 9, True), (Q8_0, (2560,), 2560, 9, False),
    (Q8_0, (3328,), 1280, 9, True), (Q4_K, (4096,), 4096, 32, False), (Q4_K, (4096,), 4096, 33, True),
    (Q4_K, (1024,), 1536, 64, False), (Q4_K, (1024,), 1024, 66, True), (Q4_K, (4096, 1024, 1024), 4096, 66, True),
    (Q6_K, (1024,), 1024, 33, False), (Q6_K, (1024,), 1024, 66, True), (Q6_K, (3328,), 1280, 24, True),
    (NF4, (4096,), 4096, 128, False), (NF4, (4096,), 4096, 160, True), (NF4, (14336,), 4096, 160, False),
    (NF4, (640,), 2560, 66, True)])
def test_which_path(rocm, dev, oracle, t, ns, k, m, prompt):
    import torch
    x = torch.zeros(m * k, device="cuda:0")
    ys = [torch.empty(m * n, device="cuda:0") for n in ns]
    ws = [torch.zeros(n * k * (2 if t == Q8_0 else 1), dtype=torch.uint8, device="cuda:0") for n in ns]
    absmax = torch.ones(ns[0] * k // 64, device="cuda:0")
    torch.cuda.synchronize()

    def body():
        if t == NF4:
            rocm.call("aljabr_rocm_matvec_tb_batch_nf4", dev.ptr(ys[0]), dev.ptr(x), dev.ptr(ws[0]), dev.ptr(absmax), k,
                      ns[0], 64, m)
        elif len(ns) == 1:
            rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(ys[0]), dev.ptr(x), dev.ptr(ws[0]), k, ns[0], t, m)
        else:
            rocm.call("aljabr_rocm_matvec_tb_triple_batch", *[dev.ptr(y) for y in ys], dev.ptr(x),
                      *[dev.ptr(w) for w in ws], k, *ns, t, t, t, m)
        return scratch_held(rocm)

    held = fresh_thread(body)
    # Weight image and activation image together.
    bytes_per = {Q4_0: 0.5625, Q8_0: 1.0625, Q4_K: 0.5625, Q6_K: 1.125, NF4: 0.5625}[t]
    image = min(sum(ns) * k * bytes_per, 100 << 20) + 2 * m * k
    assert (held >= image) == prompt, (held, image)


@pytest.mark.parametrize("t,k,m", [(Q8_0, 9472, 130), (Q4_0, 1280, 700), (Q8_0, 2560, 300)])
def test_infinite_activations_stay_infinite(rocm, dev, oracle, t, k, m):
    """An infinity times a weight is infinite (NaN where the weight is zero)
    through the folded sums and the slices; other tokens are not touched."""
    n = 96
    raw = _random_blocks(t, n, k, 3)
    raw.reshape(-1, 18 if t == Q4_0 else 34)[:, 1] |= 4          # no zero scales
    x = oracle.normal(4, m * k).reshape(m, k)
    x[7, 70] = -np.inf
    x[9, 3] = np.nan
    y, w, xd = dev.empty(m * n), dev.put(raw), dev.put(x)
    rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, t, m)
    got = dev.get(y).reshape(m, n)
    w64 = _decoded(oracle, t, raw.ravel(), n, k)
    with np.errstate(invalid="ignore"):
        want = -np.inf * np.sign(w64[:, 70])
    assert np.array_equal(got[7], want, equal_nan=True)
    assert np.isnan(got[9]).all()
    rest = np.r_[0:7, 8, 10:m]
    assert rel_l2(got[rest], x[rest].astype(np.float64) @ w64.T) <= TOL


def test_captured_call_keeps_the_passes(rocm, dev, oracle):
    """Under stream capture no scratch is taken: K % 512 != 0 runs in fp32 by 8
    tokens, and every replay equals the oracle."""
    import torch
    t, n, k, m = Q8_0, 255, 640, 64
    raw = _weights(oracle, t, n, k, 3)
    x = oracle.normal(4, m * k).reshape(m, k)
    w, xd, y = dev.put(raw), dev.put(x), dev.empty(m * n)
    ref = x.astype(np.float64) @ _decoded(oracle, t, raw, n, k).T

    def body():
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        rocm.call("aljabr_rocm_set_stream", stream.cuda_stream)
        rocm.call("aljabr_rocm_set_sync_mode", 0)
        with torch.cuda.graph(graph, stream=stream):
            rocm.call("aljabr_rocm_matvec_tb_batch", dev.ptr(y), dev.ptr(xd), dev.ptr(w), k, n, t, m)
        outs = []
        for _ in range(3):
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            outs.append(y.cpu().numpy().reshape(m, n))
        return outs, scratch_held(rocm)

    outs, held = fresh_thread(body)
    assert held == 0
    for got in outs:
        assert rel_l2(got, ref) <= TOL
