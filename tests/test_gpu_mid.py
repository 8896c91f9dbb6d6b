"""GPU parity: the mid kernels (matrix cores, every column of a launch) are
bit-exact with the oracle at the edges of their segments (16 rows), column
groups (16, 32), block pipelines (5, 4, 3 and 2 blocks deep) and work items,
from segments and from tiles, with full-range Q6_K scales.

The row waves take launches of two segments per CU and more (8192 rows on 256
CUs), the class pairs the smaller ones and launches of mixed types.
"""
import ctypes

import numpy as np
import pytest

from heliopause_amd import synthetic as S

pytestmark = pytest.mark.gpu

TYPES = {"Q4_K": 1, "Q6_K": 3}


def _blocks(kind, seed, rows, k):
    w = S.weight_blocks(kind, seed, rows, k)
    if kind == "Q6_K":  # scales over all of int8
        w = w.reshape(-1, 210).copy()
        w[:, 192:208] = S.random_bytes(S.derive(seed, "scales"), 16 * w.shape[0]).reshape(-1, 16)
        w = w.reshape(rows, -1)
    return w


@pytest.fixture(params=[True, False], ids=["both-layouts", "one-layout"])
def layouts(request, hip):
    hip.setWeightLayouts(request.param)
    yield request.param
    hip.setWeightLayouts(True)


def _bits(a):
    return np.ascontiguousarray(a).reshape(-1).view(np.uint32)


@pytest.mark.parametrize("specs,k,m", [
    ([("Q4_K", 1)], 256, 5),
    ([("Q4_K", 17), ("Q6_K", 33), ("Q4_K", 16)], 1024, 16),
    ([("Q6_K", 40), ("Q4_K", 130)], 1536, 17),          # 6 blocks; 2 column groups of 16
    ([("Q4_K", 129), ("Q6_K", 15)], 2560, 33),
    ([("Q6_K", 100)], 2816, 63),                        # 11 blocks
    ([("Q4_K", 4000), ("Q6_K", 300)], 512, 49),         # class pairs of 32 columns
    ([("Q4_K", 8180)], 512, 7),                         # row waves: a rest of rows, 2 blocks
    ([("Q6_K", 8500)], 256, 16),                        # one block per item
    ([("Q6_K", 20000)], 768, 30),                       # several items per workgroup, 3 blocks
    ([("Q4_K", 9000), ("Q4_K", 8200)], 1280, 50),       # two weights; 2 column groups of 32
    ([("Q6_K", 66000)], 256, 2),                        # two columns of one block: vector ALU
    ([("Q4_K", 40)], 10240, 5), ([("Q6_K", 33)], 10240, 16),   # long rows: single classes, 16 columns
    ([("Q4_K", 24), ("Q6_K", 40)], 10240, 17), ([("Q6_K", 50)], 10240, 32), ([("Q4_K", 17)], 5120, 31),  # and 32
])
def test_mid_bit_exact(hip, oracle, layouts, specs, k, m):
    """Device and host calls."""
    import torch

    print(f"mid {specs} k={k} m={m} both={layouts}", flush=True)
    seed = S.derive(S.BASE_SEED, "mid", k, m)
    ws = [_blocks(t, S.derive(seed, i), r, k) for i, (t, r) in enumerate(specs)]
    x = S.activations(seed, m, k)
    x[0, :256] = 0.0
    refs = [oracle.matmul(TYPES[t], w, x, r, threads=8) for (t, r), w in zip(specs, ws)]
    hs = [hip.createHipQuantizedWeightHandle(t, w, k, r) for (t, r), w in zip(specs, ws)]
    try:
        dx = torch.from_numpy(x.reshape(-1)).to("cuda:0")
        outs = [torch.empty(r * m, dtype=torch.float32, device="cuda:0") for _, r in specs]
        hip.matmul_multi_device([h.handle for h in hs], dx.data_ptr(), k, m, [o.data_ptr() for o in outs],
                                [o.numel() for o in outs])
        torch.cuda.synchronize()
        got = [o.cpu().numpy() for o in outs]
        host = hip.matMulQuantizedHipResidentMulti(hs, x, k, m) if len(hs) > 1 else [
            hip.matMulQuantizedHipResident(hs[0], x, k, specs[0][1], m)]
    finally:
        for h in hs:
            hip.releaseHipQuantizedWeightHandle(h)
    for ref, g, hg in zip(refs, got, host):
        assert np.array_equal(_bits(g), _bits(ref))
        assert np.array_equal(_bits(hg), _bits(ref))


@pytest.mark.parametrize("gate,up,rows,k,m", [
    ("Q4_K", "Q4_K", 200, 768, 21), ("Q4_K", "Q6_K", 48, 1280, 40), ("Q6_K", "Q6_K", 4200, 256, 5),
    ("Q4_K", "Q4_K", 4112, 512, 40), ("Q4_K", "Q4_K", 17000, 256, 11),
    ("Q4_K", "Q4_K", 4080, 512, 33), ("Q6_K", "Q6_K", 2050, 768, 63), ("Q6_K", "Q4_K", 2049, 512, 50),  # pairs of 32
])
def test_mid_geglu_bit_exact(hip, oracle, layouts, gate, up, rows, k, m):
    import torch

    print(f"mid geglu {gate} {up} {rows} k={k} m={m} both={layouts}", flush=True)
    seed = S.derive(S.BASE_SEED, "mid-geglu", rows, k, m)
    wg, wu = _blocks(gate, S.derive(seed, 1), rows, k), _blocks(up, S.derive(seed, 2), rows, k)
    x = S.activations(seed, m, k) * 0.05
    hg = hip.createHipQuantizedWeightHandle(gate, wg, k, rows)
    hu = hip.createHipQuantizedWeightHandle(up, wu, k, rows)
    try:
        dx, out = torch.from_numpy(x.reshape(-1)).to("cuda:0"), torch.empty(rows * m, device="cuda:0")
        hip.matmul_geglu_device(hg.handle, hu.handle, dx.data_ptr(), k, m, out.data_ptr(), rows)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
    finally:
        hip.releaseHipQuantizedWeightHandle(hg)
        hip.releaseHipQuantizedWeightHandle(hu)
    ref = oracle.geglu(oracle.matmul(TYPES[gate], wg, x, rows, threads=8).reshape(-1),
                       oracle.matmul(TYPES[up], wu, x, rows, threads=8).reshape(-1))
    assert np.array_equal(_bits(got), _bits(ref))


@pytest.mark.parametrize("kind,full,rows,k,m,launches", [
    ("Q6_K", False, 65600, 256, 2, 1), ("Q4_K", False, 65600, 256, 4, 1),  # kquant_mfma
    ("Q6_K", True, 65530, 1024, 2, 2), ("Q6_K", True, 65600, 1024, 4, 2),  # activation tiles, row waves
    ("Q6_K", True, 65600, 1024, 2, 1),  # a 513th item: the last round is nearly empty, vector ALU
])
def test_two_to_four_columns_of_large_launches(hip, oracle, kind, full, rows, k, m, launches):
    """Weights of single f16 operands stay on the one-launch matrix-core
    kernel, full-range Q6_K weights go to the row waves."""
    print(f"mid few columns {kind} full={full} k={k} m={m}", flush=True)
    seed = S.derive(S.BASE_SEED, "mid-few", k, m)
    w = _blocks(kind, seed, rows, k) if full else S.weight_blocks(kind, seed, rows, k)
    x = S.activations(seed, m, k)
    h = hip.createHipQuantizedWeightHandle(kind, w, k, rows)
    try:
        before = hip.hipResidentWeightStats()["kernelLaunches"]
        got = hip.matMulQuantizedHipResident(h, x, k, rows, m)
        assert hip.hipResidentWeightStats()["kernelLaunches"] - before == launches
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
    assert np.array_equal(_bits(got), _bits(oracle.matmul(TYPES[kind], w, x, rows, threads=8)))


@pytest.mark.parametrize("specs,k,m,launches", [
    ([("Q4_K", 2560)], 256, 8, 1), ([("Q6_K", 300), ("Q4_K", 100)], 256, 5, 1), ([("Q6_K", 8200)], 512, 6, 1),
    ([("Q6_K", 8200)], 768, 5, 1), ([("Q6_K", 8200)], 768, 6, 2), ([("Q4_K", 2560)], 256, 9, 2),
])
def test_short_rows_of_five_to_eight_columns(hip, oracle, specs, k, m, launches):
    """Short rows in single f16 operands: kquant_mfma's one launch, or the
    activation tiles and the mid kernel."""
    print(f"mid short rows {specs} k={k} m={m}", flush=True)
    seed = S.derive(S.BASE_SEED, "mid-short", k, m)
    ws = [S.weight_blocks(t, S.derive(seed, i), r, k) for i, (t, r) in enumerate(specs)]
    x = S.activations(seed, m, k)
    hs = [hip.createHipQuantizedWeightHandle(t, w, k, r) for (t, r), w in zip(specs, ws)]
    try:
        before = hip.hipResidentWeightStats()["kernelLaunches"]
        got = hip.matMulQuantizedHipResidentMulti(hs, x, k, m) if len(hs) > 1 else [
            hip.matMulQuantizedHipResident(hs[0], x, k, specs[0][1], m)]
        assert hip.hipResidentWeightStats()["kernelLaunches"] - before == launches
    finally:
        for h in hs:
            hip.releaseHipQuantizedWeightHandle(h)
    for (t, r), w, g in zip(specs, ws, got):
        assert np.array_equal(_bits(g), _bits(oracle.matmul(TYPES[t], w, x, r, threads=8)))


@pytest.mark.parametrize("specs,k,m", [
    ([("Q4_K", 4100), ("Q6_K", 4100)], 256, 40), ([("Q4_K", 2560)], 256, 520),
    ([("Q6_K", 2000), ("Q4_K", 600)], 2560, 1540), ([("Q6_K", 2100)], 3840, 1030),
])
def test_many_columns_of_host_calls(hip, oracle, layouts, specs, k, m):
    """Host calls of the sizes that the bit-exact prefill kernel takes."""
    print(f"mid many columns {specs} k={k} m={m} both={layouts}", flush=True)
    seed = S.derive(S.BASE_SEED, "mid-many", k, m)
    ws = [S.weight_blocks(t, S.derive(seed, i), r, k) for i, (t, r) in enumerate(specs)]
    part = S.activations(seed, 40, k)
    x = np.resize(part, (m, k))  # column c is part[c % 40]
    hs = [hip.createHipQuantizedWeightHandle(t, w, k, r) for (t, r), w in zip(specs, ws)]
    try:
        got = hip.matMulQuantizedHipResidentMulti(hs, x, k, m) if len(hs) > 1 else [
            hip.matMulQuantizedHipResident(hs[0], x, k, specs[0][1], m)]
    finally:
        for h in hs:
            hip.releaseHipQuantizedWeightHandle(h)
    for (t, r), w, g in zip(specs, ws, got):
        ref = oracle.matmul(TYPES[t], w, part, r, threads=8).reshape(40, r)
        assert np.array_equal(_bits(g), _bits(np.resize(ref, (m, r))))


def test_capture_without_scratch(hip, oracle):
    """A captured call of eight columns on a stream that no call has sized
    scratch for is accepted (its kernels without activation tiles run), with
    the same bits on every replay; sized, the capture takes the mid kernel."""
    import torch

    rows, k, m = 64, 768, 8
    w, x = _blocks("Q6_K", 5, rows, k), S.activations(6, m, k)
    ref = oracle.matmul(3, w, x, rows)
    h = hip.createHipQuantizedWeightHandle("Q6_K", w, k, rows)
    stream = torch.cuda.Stream()
    try:
        dx, out = torch.from_numpy(x.reshape(-1)).to("cuda:0"), torch.empty(rows * m, device="cuda:0")
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
                assert np.array_equal(_bits(out.cpu().numpy()), _bits(ref)), sized
            del graph
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
        hip.lib().hp_hip_release_stream_scratch(ctypes.c_void_p(stream.cuda_stream))


def test_capture_of_40_columns_needs_scratch(hip, oracle):
    """From 32 columns of single-operand weights on, every kernel of the
    automatic choice needs scratch: a capture on a stream without is refused,
    one after an uncaptured call of the shape is not."""
    import torch

    rows, k, m = 64, 768, 40
    w, x = _blocks("Q4_K", 5, rows, k), S.activations(6, m, k)
    h = hip.createHipQuantizedWeightHandle("Q4_K", w, k, rows)
    stream = torch.cuda.Stream()
    try:
        dx, out = torch.from_numpy(x.reshape(-1)).to("cuda:0"), torch.empty(rows * m, device="cuda:0")
        torch.cuda.synchronize()
        run = lambda: hip.matmul_multi_device([h.handle], dx.data_ptr(), k, m, [out.data_ptr()],  # noqa: E731
                                              [out.numel()], stream.cuda_stream)
        refused, graph = None, torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out.zero_()
            try:
                run()
            except RuntimeError as e:
                refused = str(e)
        assert refused and "before graph capture" in refused
        run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            run()
        for _ in range(2):
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(_bits(out.cpu().numpy()), _bits(oracle.matmul(1, w, x, rows)))
        del graph
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
        hip.lib().hp_hip_release_stream_scratch(ctypes.c_void_p(stream.cuda_stream))


def test_capture_without_scratch_leaves_no_error(hip, oracle):
    """A call that runs other kernels for want of scratch has succeeded: the
    last-error text is still that of the last call that failed."""
    import torch

    rows, k, m = 64, 768, 8
    w, x = _blocks("Q6_K", 5, rows, k), S.activations(6, m, k)
    h = hip.createHipQuantizedWeightHandle("Q6_K", w, k, rows)
    stream = torch.cuda.Stream()
    try:
        dx, out = torch.from_numpy(x.reshape(-1)).to("cuda:0"), torch.empty(rows * m, device="cuda:0")
        torch.cuda.synchronize()
        with pytest.raises(Exception):
            hip.matmul_multi_device([h.handle], dx.data_ptr(), k, m, [out.data_ptr()], [out.numel() - 1])
        failed = hip.last_error()
        assert failed
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            hip.matmul_multi_device([h.handle], dx.data_ptr(), k, m, [out.data_ptr()], [out.numel()],
                                    stream.cuda_stream)
        assert hip.last_error() == failed
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(_bits(out.cpu().numpy()), _bits(oracle.matmul(3, w, x, rows)))
        del graph
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
        hip.lib().hp_hip_release_stream_scratch(ctypes.c_void_p(stream.cuda_stream))


def test_failed_allocation_is_not_the_next_calls_error(hip, oracle):
    """Every device allocation of the library, scratch among them, goes through one
    function.  After one has failed (a weight of 600 GB: refused before its
    bytes are read), the launches of the next call still succeed."""
    import torch

    rows, k, m = 32, 512, 9
    w, x = _blocks("Q4_K", 7, rows, k), S.activations(8, m, k)
    h = hip.createHipQuantizedWeightHandle("Q4_K", w, k, rows)
    try:
        small = torch.zeros(256, dtype=torch.uint8, device="cuda:0")
        big_k, big_rows = 1 << 20, 1 << 20
        out = ctypes.c_uint64(0)
        code = hip.lib().hp_hip_weight_upload_device(TYPES["Q4_K"], small.data_ptr(), big_k // 256 * 144 * big_rows,
                                                     big_k, big_rows, ctypes.byref(out))
        assert code != 0 and "allocation" in hip.last_error()
        got = hip.matMulQuantizedHipResident(h, x, k, rows, m)
        assert np.array_equal(_bits(got), _bits(oracle.matmul(1, w, x, rows)))
    finally:
        hip.releaseHipQuantizedWeightHandle(h)
