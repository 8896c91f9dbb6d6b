"""GPU parity: Q6_K weights with full-range int8 scales (as GGUF files hold
them) on the matrix cores, where sc * (q - 32) needs two exact f16 operands.

An operand rounded to one f16 would be off by one unit in up to 4096, about
1e-5 of an output, so the fast prefill kernel is compared against f64 sums of
the exact integers with the rounding bound of its f32 sums: per block three
roundings (dw * D, times dx, the running sum; each at most 2^-24 of the terms
so far), block ranges add one more each, so (3 nb + 8) 2^-24 sum_b |t_b|.  D
itself, a block's integer sum, is exact while its partial sums stay within
2^24; a block whose products add up to more (|p| summed, up to 2^27) rounds
at most once per four products of either operand, 128 times, each by 2^-24 of
that sum.
"""
import ctypes

import numpy as np
import pytest

from heliopause_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _full_range(seed, rows, k):
    """Q6_K blocks with scales over -128..127, extremes and quants of 0 and 63
    (q - 32 = -32, 31) planted."""
    w = S.q6_k_blocks(seed, rows, k).reshape(-1, 210).copy()
    w[:, 192:208] = S.random_bytes(S.derive(seed, "scales"), 16 * w.shape[0]).reshape(-1, 16)
    w[0, 192:196] = np.array([127, -127, -128, -67], dtype=np.int8).view(np.uint8)
    w[1, 0:192] = 0
    w[1, 192:208] = np.int8(-127).view(np.uint8)
    w[2, 0:192] = 255
    w[2, 192:208] = 127
    return w.reshape(rows, -1)


def _terms(oracle, w, x, rows):
    """Per-block f64 contributions [rows][m][nb] of the Q8_K input."""
    m, k = x.shape
    qs, d, _ = oracle.quantize_q8_k(x)
    xq = (qs.astype(np.float64).reshape(m, -1, 256) * d.astype(np.float64)[:, :, None])
    deq = np.stack([oracle.dequantize(3, w[r], k) for r in range(rows)]).astype(np.float64).reshape(rows, -1, 256)
    return np.einsum("rbe,mbe->rmb", deq, xq)


def _bound(oracle, w, x, rows):
    """(f64 sums, rounding bounds), [rows][m], of the module's first lines."""
    m, k = x.shape
    qs, d, _ = oracle.quantize_q8_k(x)
    xq = np.abs(qs.astype(np.float64)).reshape(m, -1, 256)
    b = w.reshape(rows, -1, 210)
    dw = b[:, :, 208:210].copy().view(np.float16).astype(np.float64)[:, :, 0]
    deq = np.stack([oracle.dequantize(3, w[r], k) for r in range(rows)]).astype(np.float64).reshape(rows, -1, 256)
    ints = np.abs(np.divide(deq, dw[:, :, None], out=np.zeros_like(deq), where=dw[:, :, None] != 0))  # |sc (q - 32)|
    p = np.matmul(ints.transpose(1, 0, 2), xq.transpose(1, 2, 0))  # [nb][rows][m], sums of |products|
    unit = np.abs(dw).T[:, :, None] * np.abs(d.astype(np.float64)).reshape(m, -1).T[:, None, :]
    t = _terms(oracle, w, x, rows)
    rounded = np.where(p > 2.0 ** 24 * (1 - 1e-9), p * unit, 0.0).sum(0)
    return t.sum(2), ((3 * (k // 256) + 8) * np.abs(t).sum(2) + 128 * rounded) * 2.0 ** -24


def _device(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(torch.device("cuda:0"))


@pytest.fixture(params=[True, False], ids=["both-layouts", "one-layout"])
def layouts(request, hip):
    hip.setWeightLayouts(request.param)
    yield request.param
    hip.setWeightLayouts(True)


@pytest.mark.parametrize("rows,k,m", [(16, 256, 64), (33, 2560, 65), (300, 2560, 130), (130, 10240, 100)])
def test_fast_prefill_full_range(hip, oracle, layouts, rows, k, m):
    """The automatic device kernel from 64 columns: alone, and in one launch
    with Q4_K weights (whose outputs do not change with the company)."""
    import torch

    print(f"full range fast rows={rows} k={k} m={m} both={layouts}", flush=True)
    seed = S.derive(S.BASE_SEED, "full-range", rows, k, m)
    w6, w4 = _full_range(seed, rows, k), S.q4_k_blocks(S.derive(seed, 4), 48, k)
    x = S.activations(seed, m, k)
    x[0] = 127.0  # every quant -127
    h6 = hip.createHipQuantizedWeightHandle("Q6_K", w6, k, rows)
    h4 = hip.createHipQuantizedWeightHandle("Q4_K", w4, k, 48)
    try:
        dx = _device(x.reshape(-1))
        alone, joined, q4, q4_alone = (torch.empty(n * m, dtype=torch.float32, device="cuda:0")
                                       for n in (rows, rows, 48, 48))
        hip.matmul_multi_device([h6.handle], dx.data_ptr(), k, m, [alone.data_ptr()], [alone.numel()])
        hip.matmul_multi_device([h4.handle, h6.handle], dx.data_ptr(), k, m, [q4.data_ptr(), joined.data_ptr()],
                                [q4.numel(), joined.numel()])
        hip.matmul_multi_device([h4.handle], dx.data_ptr(), k, m, [q4_alone.data_ptr()], [q4_alone.numel()])
        torch.cuda.synchronize()
    finally:
        hip.releaseHipQuantizedWeightHandle(h6)
        hip.releaseHipQuantizedWeightHandle(h4)
    want, bound = _bound(oracle, w6, x, rows)
    for got in (alone, joined):
        g = got.cpu().numpy().reshape(m, rows).T.astype(np.float64)
        assert np.all(np.abs(g - want) <= bound), np.max(np.abs(g - want) / np.maximum(bound, 1e-300))
    ref4 = oracle.matmul(1, w4, x, 48, threads=8)
    for got in (q4, q4_alone):
        g = got.cpu().numpy()
        assert np.max(np.abs(g - ref4.reshape(-1))) <= 1e-4 * np.abs(ref4).max()


def test_full_range_more_columns_than_a_prefill_launch(hip, oracle):
    """65,537 columns on the device: more than one launch of the prefill
    kernels takes, so the vector-ALU kernels run (the oracle's bits)."""
    import torch

    rows, k, m = 16, 256, 65537
    print(f"full range m={m}", flush=True)
    seed = S.derive(S.BASE_SEED, "full-range-many")
    w, part = _full_range(seed, rows, k), S.activations(seed, 64, k)
    x = np.resize(part, (m, k))  # column c is part[c % 64]
    h = hip.createHipQuantizedWeightHandle("Q6_K", w, k, rows)
    try:
        dx, out = _device(x.reshape(-1)), torch.empty(rows * m, dtype=torch.float32, device="cuda:0")
        hip.matmul_multi_device([h.handle], dx.data_ptr(), k, m, [out.data_ptr()], [out.numel()])
        torch.cuda.synchronize()
        got = out.cpu().numpy().reshape(m, rows)
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
    ref = oracle.matmul(3, w, part, rows).reshape(64, rows)
    assert np.array_equal(got.view(np.uint32), np.resize(ref, (m, rows)).view(np.uint32))


def test_full_range_capture_without_scratch(hip, oracle):
    """A captured call of 70 columns on a stream that no call has sized scratch
    for is accepted (the vector-ALU kernels: the oracle's bits on every
    replay); sized, the capture takes the fast prefill kernel."""
    import torch

    rows, k, m = 40, 768, 70
    seed = S.derive(S.BASE_SEED, "full-range-capture")
    w, x = _full_range(seed, rows, k), S.activations(seed, m, k)
    ref = oracle.matmul(3, w, x, rows)
    want, bound = _bound(oracle, w, x, rows)
    h = hip.createHipQuantizedWeightHandle("Q6_K", w, k, rows)
    stream = torch.cuda.Stream()
    print("full range capture", flush=True)
    try:
        dx, out = _device(x.reshape(-1)), torch.empty(rows * m, dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        run = lambda: hip.matmul_multi_device([h.handle], dx.data_ptr(), k, m, [out.data_ptr()],  # noqa: E731
                                              [out.numel()], stream.cuda_stream)
        for sized in (False, True):
            if sized:
                run()
                torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                run()
            for _ in range(3):
                out.zero_()
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                got = out.cpu().numpy()
                if sized:
                    assert np.all(np.abs(got.reshape(m, rows).T.astype(np.float64) - want) <= bound)
                else:
                    assert np.array_equal(got.view(np.uint32), ref.reshape(-1).view(np.uint32))
            del graph
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
        hip.lib().hp_hip_release_stream_scratch(ctypes.c_void_p(stream.cuda_stream))


def test_fast_prefill_full_range_geglu(hip, oracle, layouts):
    """gate and up as full-range Q6_K in one tile, GeGLU in its epilogue:
    elements within two f16 steps (gelu rounds its input and result to f16),
    and all but the few at a rounding boundary equal to f32."""
    import torch

    rows, k, m = 200, 2560, 70
    print(f"full range geglu both={layouts}", flush=True)
    seed = S.derive(S.BASE_SEED, "full-range-geglu")
    wg, wu = _full_range(S.derive(seed, 1), rows, k), _full_range(S.derive(seed, 2), rows, k)
    x = S.activations(seed, m, k) * 0.05
    hg = hip.createHipQuantizedWeightHandle("Q6_K", wg, k, rows)
    hu = hip.createHipQuantizedWeightHandle("Q6_K", wu, k, rows)
    try:
        dx, out = _device(x.reshape(-1)), torch.empty(rows * m, dtype=torch.float32, device="cuda:0")
        hip.matmul_geglu_device(hg.handle, hu.handle, dx.data_ptr(), k, m, out.data_ptr(), rows)
        torch.cuda.synchronize()
        got = out.cpu().numpy().astype(np.float64)
    finally:
        hip.releaseHipQuantizedWeightHandle(hg)
        hip.releaseHipQuantizedWeightHandle(hu)
    ref = oracle.geglu(oracle.matmul(3, wg, x, rows, threads=8).reshape(-1),
                       oracle.matmul(3, wu, x, rows, threads=8).reshape(-1)).astype(np.float64)
    rel = np.abs(got - ref) / np.maximum(np.abs(ref), 0.01 * np.sqrt(np.mean(ref * ref)))
    assert rel.max() <= 2 * 2.0 ** -10, rel.max()
    assert np.mean(rel <= 1e-4) >= 0.99
