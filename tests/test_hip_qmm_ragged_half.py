"""The MFMA quantized matmul where its tiles end: K that is no multiple of
the 32-row chunk, N that is no multiple of a lane's four columns, row counts
around the 16- and 32-row tiles, and fp16 / bf16 activations and outputs with
scales of either type, against the product in 64 bits.

fp32 bound: A is split at 22 bits and 2 k products are summed in fp32, so
|err| <= (2^-22 + 2 k 2^-24) sum |a w|.  16-bit activations are used as they
are: k products summed in fp32, then one rounding of the output (2^-11 of it
for fp16, 2^-8 for bf16, half an ulp of 11 and 8 bits, and 2^-24 where fp16 is subnormal)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _weights(rng, kind, block, k, n):
    """(codes, scales, code values as float64, quant type)"""
    if kind == "int4":
        packed, s = O.quantize_int4((rng.standard_normal((k, n)) * 0.02).astype(np.float32), block)
        v = np.empty((2 * packed.shape[0], n), np.int8)
        v[0::2] = (packed.view(np.int8) << 4) >> 4
        v[1::2] = packed.view(np.int8) >> 4
        return packed, s, v[:k].astype(np.float64), 2
    if block == 0:
        q, s = O.quantize_int8((rng.standard_normal((k, n)) * 0.02).astype(np.float32))
        return q, s.reshape(1, n), q.astype(np.float64), 1
    q = rng.integers(-127, 128, (k, n), dtype=np.int8)
    return q, (rng.random((-(-k // block), n)) * 0.01 + 1e-4).astype(np.float32), q.astype(np.float64), 1


def _dense(values, scales, block):
    k = values.shape[0]
    return values * scales.astype(np.float64).repeat(block or k, 0)[:k]


KINDS = [("int8", 0), ("int8", 96), ("int4", 32), ("int4", 64)]


@pytest.mark.parametrize("kind,block", KINDS)
@pytest.mark.parametrize("m,k,n", [(5, 31, 16), (7, 33, 17), (16, 1001, 67), (17, 224, 131), (33, 1, 19), (40, 95, 1027),
                                   (100, 2047, 515), (129, 64, 130)])
def test_ragged_fp32(hip, kind, block, m, k, n):
    rng = np.random.default_rng(m * 1000 + k + n + block)
    q, s, v, qt = _weights(rng, kind, block, k, n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    print(f"case ragged {kind} block={block} m={m} k={k} n={n}", flush=True)
    out = hip.run_qmm(x, q, s, k, qt, block).astype(np.float64)
    wd = _dense(v, s, block)
    mag = np.abs(x.astype(np.float64)) @ np.abs(wd)
    assert np.all(np.abs(out - x.astype(np.float64) @ wd) <= (2.0 ** -22 + 2 * k * 2.0 ** -24) * 1.01 * mag + 1e-30)


@pytest.mark.parametrize("kind,block", KINDS)
@pytest.mark.parametrize("m,k,n", [(5, 1, 17), (33, 40, 130), (33, 46, 40), (33, 46, 41), (6, 48, 31), (6, 80, 40), (6, 49, 100), (8, 72, 80),
                                   (8, 73, 80), (900, 31, 151), (900, 31, 480)])
def test_ragged_small(hip, kind, block, m, k, n):
    # both sides of the sizes up to which a thread per output is the faster one
    test_ragged_fp32(hip, kind, block, m, k, n)


@pytest.mark.parametrize("kind,block", [("int8", 0), ("int8", 24), ("int4", 32), ("int4", 8)])
@pytest.mark.parametrize("m", [1, 3])
@pytest.mark.parametrize("k,n", [(31, 17), (64, 31), (576, 257), (2048, 515), (2048, 5633), (300, 26000 + 7), (5632, 2049)])
def test_ragged_gemv(hip, kind, block, m, k, n):
    # up to four rows: the 16-column groups of every tile width and split of
    # the decode kernel, the last one moved back inside the row
    rng = np.random.default_rng(m + k + n + block)
    q, s, v, qt = _weights(rng, kind, block, k, n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    print(f"case ragged gemv {kind} block={block} m={m} k={k} n={n}", flush=True)
    wd = _dense(v, s, block)
    bound = 2 * k * 2.0 ** -24 * 1.01 * (np.abs(x.astype(np.float64)) @ np.abs(wd)) + 1e-30
    for shift in (0, 1):   # codes at an odd address too
        buf = np.zeros(q.nbytes + 1, np.int8)
        buf[shift:shift + q.nbytes] = q.view(np.int8).reshape(-1)
        da, dq, ds, dc = (hip.DeviceBuffer.from_array(t) for t in (x, buf, s, np.zeros((m, n), np.float32)))
        hip.qmm_f32(da.addr, dq.addr + shift, ds.addr, dc.addr, m, k, n, qt, block)
        out = dc.download(np.float32, (m, n)).astype(np.float64)
        assert np.all(np.abs(out - x.astype(np.float64) @ wd) <= bound)


@pytest.mark.parametrize("m", [1, 3])
@pytest.mark.parametrize("k,n", [(64, 31), (2048, 515), (5632, 2049), (2048, 512)])
def test_ragged_gemv_large_values(hip, m, k, n):
    # sums of value times code that fill fp32 (at most 2e38), of either sign;
    # (512 columns: aligned width, codes at an odd address)
    rng = np.random.default_rng(k + n)
    q, s, v, qt = _weights(rng, "int4", 32, k, n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x *= np.float32(2e38 / np.abs((x[:, :k // 32 * 32].reshape(m, -1, 32, 1) * v[:k // 32 * 32].reshape(1, -1, 32, n))
                                  .cumsum(2)).max())
    print(f"case ragged gemv large m={m} k={k} n={n}", flush=True)
    wd = _dense(v, s, 32)
    shift = 1 if n == 512 else 0
    buf = np.zeros(q.nbytes + 1, np.int8)
    buf[shift:shift + q.nbytes] = q.view(np.int8).reshape(-1)
    da, dq, ds, dc = (hip.DeviceBuffer.from_array(t) for t in (x, buf, s, np.zeros((m, n), np.float32)))
    hip.qmm_f32(da.addr, dq.addr + shift, ds.addr, dc.addr, m, k, n, qt, 32)
    out, ref = dc.download(np.float32, (m, n)).astype(np.float64), x.astype(np.float64) @ wd
    fits = np.abs(ref) < 3.4e38
    assert np.all(np.abs(out - ref)[fits] <= (2 * k * 2.0 ** -24 * 1.01 * (np.abs(x.astype(np.float64)) @ np.abs(wd)))[fits])
    assert fits.all()


def _bits(x, bf16):
    return O.f32_to_bf16_bits(x) if bf16 else O.f32_to_f16_bits(x)


def _wide(bits, bf16):
    return (bits.astype(np.uint32) << 16).view(np.float32) if bf16 else bits.view(np.float16).astype(np.float32)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("half_scale", [False, True])
@pytest.mark.parametrize("kind,block", KINDS)
@pytest.mark.parametrize("m,k,n", [(1, 256, 96), (3, 2048, 515), (4, 33, 20), (16, 992, 336), (31, 224, 67), (70, 320, 258),
                                   (130, 1000, 132), (200, 2048, 1100)])
def test_half(hip, bf16, half_scale, kind, block, m, k, n):
    rng = np.random.default_rng(m + k + n + block)
    q, s, v, qt = _weights(rng, kind, block, k, n)
    # fp16 rows from 1e-7 (subnormal) to 1e3; a bf16 row of 1e30
    x = rng.standard_normal((m, k)).astype(np.float32)
    x *= np.float32(10.0) ** rng.integers(-3, 4, (m, 1)).astype(np.float32)
    x[0] *= np.float32(1e30 if bf16 else 1e-6)
    a = _bits(x, bf16)
    sb = _bits(s, bf16) if half_scale else s
    dt = hip.DTYPE_BF16 if bf16 else hip.DTYPE_F16
    da, dq, ds, dc = (hip.DeviceBuffer.from_array(t) for t in (a, q.view(np.int8), sb, np.zeros((m, n), np.uint16)))
    print(f"case half bf16={bf16} half_scale={half_scale} {kind} block={block} m={m} k={k} n={n}", flush=True)
    hip.qmm(da.addr, dt, dq.addr, ds.addr, dt if half_scale else hip.DTYPE_F32, dc.addr, dt, m, k, n, qt, block)
    out = _wide(dc.download(np.uint16, (m, n)), bf16).astype(np.float64)
    wd = _dense(v, _wide(sb, bf16) if half_scale else s, block)
    aw = _wide(a, bf16).astype(np.float64)
    ref, mag = aw @ wd, np.abs(aw) @ np.abs(wd)
    ulp = 2.0 ** -8 if bf16 else 2.0 ** -11
    fits = np.abs(ref) < (3e38 if bf16 else 65000)
    bound = ulp * 1.01 * np.abs(ref) + 2 * k * 2.0 ** -24 * mag + 2.0 ** -24 * (not bf16)
    assert np.all(np.abs(out - ref)[fits] <= bound[fits]), np.max((np.abs(out - ref) / bound)[fits])


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("m,k,n", [(1, 8192, 20480), (1, 8192, 18304), (2, 8192, 20480)])
def test_half_large_matrix(hip, captured, m, k, n):
    # one bf16 row of an INT4 matrix of 75 MB is widened for the decode GEMV (the
    # second matrix is just below, the third call has two rows); without memory
    # for the widened rows, as in a stream's first call when it is captured,
    # the MFMA kernel takes it
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    a = torch.randn(m, k, generator=g, device="cuda")
    q = torch.randint(-128, 128, (k // 2, n), generator=g, device="cuda", dtype=torch.int8)
    s = torch.rand(k // 32, n, generator=g, device="cuda") * 1e-3
    lo = ((q << 4) >> 4).double()
    wd = torch.stack([lo, (q >> 4).double()], 1).view(k, n) * s.double().repeat_interleave(32, 0)
    # up to where value times code fills fp32, not 16 times it
    a[0] *= 2e38 / (8 * 32 * a[0].abs().max())
    a = a.to(torch.bfloat16)
    out = torch.zeros(m, n, device="cuda", dtype=torch.bfloat16)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    print(f"case half large m={m} k={k} n={n} captured={captured}", flush=True)

    def call():
        hip.qmm(a.data_ptr(), hip.DTYPE_BF16, q.data_ptr(), s.data_ptr(), hip.DTYPE_F32, out.data_ptr(), hip.DTYPE_BF16,
                m, k, n, 2, 32, stream=stream.cuda_stream)

    graph = torch.cuda.CUDAGraph()
    if captured:
        with torch.cuda.graph(graph, stream=stream):
            call()
    ref = a.double() @ wd
    bound = 2.0 ** -8 * 1.01 * ref.abs() + 2 * k * 2.0 ** -24 * (a.double().abs() @ wd.abs())
    for _ in range(2):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay() if captured else call()
        torch.cuda.synchronize()
        assert torch.all((out.double() - ref).abs() <= bound)


@pytest.mark.parametrize("m,k,n", [(65537 * 32 + 5, 33, 16), (5, 65537 * 64 + 9, 16)])
def test_half_staging_of_many_blocks(hip, m, k, n):
    # more than 65535 blocks of 32 rows, or of 64 columns, are staged
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(m % 1000)
    a = torch.randn(m, k, generator=g, device="cuda", dtype=torch.float16)
    q = torch.randint(-127, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
    s = torch.full((1, n), 1e-3, device="cuda")
    out = torch.zeros(m, n, device="cuda", dtype=torch.float16)
    print(f"case half staging m={m} k={k} n={n}", flush=True)
    hip.qmm(a.data_ptr(), hip.DTYPE_F16, q.data_ptr(), s.data_ptr(), hip.DTYPE_F32, out.data_ptr(), hip.DTYPE_F16, m, k, n,
            1, 0)
    rows = torch.tensor(sorted({0, 1, min(m, 31), m // 2, max(m - 6, 0), m - 1} & set(range(m))), device="cuda")
    aw = a[rows].double()
    ref, mag = aw @ q.double() * 1e-3, aw.abs() @ q.double().abs() * 1e-3
    # (a sum is in many parts: no chain of additions is longer than 2^16)
    bound = 2.0 ** -11 * 1.01 * ref.abs() + 2 * min(k, 2 ** 16) * 2.0 ** -24 * mag + 2.0 ** -24
    assert torch.all((out[rows].double() - ref).abs() <= bound)


@pytest.mark.parametrize("bf16", [False, True])
def test_half_infinity_and_nan(hip, bf16):
    # 5 x 64 times 64 x 32 codes that are never zero: a row's infinity reaches
    # every output of the row, a NaN too, and other rows stay as they were
    m, k, n = 5, 64, 32
    rng = np.random.default_rng(3)
    q = rng.integers(1, 128, (k, n), dtype=np.int8)
    s = np.ones((1, n), np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1, 7], x[3, 60] = np.inf, np.nan
    dt = hip.DTYPE_BF16 if bf16 else hip.DTYPE_F16
    da, dq, ds, dc = (hip.DeviceBuffer.from_array(t) for t in (_bits(x, bf16), q, s, np.zeros((m, n), np.uint16)))
    hip.qmm(da.addr, dt, dq.addr, ds.addr, hip.DTYPE_F32, dc.addr, dt, m, k, n, 1, 0)
    out = _wide(dc.download(np.uint16, (m, n)), bf16)
    assert np.all(np.isposinf(out[1])) and np.all(np.isnan(out[3])) and np.all(np.isfinite(out[[0, 2, 4]]))


@pytest.mark.parametrize("m,k,n", [(5, 63, 17), (7, 2048, 515), (40, 96, 64), (6, 8192, 67)])
def test_fp32_infinity_beside_large_values(hip, m, k, n):
    # a row's infinity or NaN decides its outputs whatever the row's finite
    # values are (codes that are never zero), as in the reference's fp32 sums
    rng = np.random.default_rng(k)
    q = (rng.integers(1, 128, (k, n)) * rng.choice([-1, 1], (k, n))).astype(np.int8)
    s = np.full((1, n), 0.01, np.float32)
    x = (rng.standard_normal((m, k)) * 1e6).astype(np.float32)
    x[1, 7], x[2, k - 1], x[4, 0] = np.inf, -np.inf, np.nan
    print(f"case fp32 infinity m={m} k={k} n={n}", flush=True)
    out = hip.run_qmm(x, q, s, k, 1, 0)
    inf = np.float32(np.inf)
    assert np.array_equal(out[1], np.copysign(inf, q[7].astype(np.float32)))
    assert np.array_equal(out[2], np.copysign(inf, -q[k - 1].astype(np.float32)))
    assert np.isnan(out[4]).all() and np.isfinite(out[[0, 3]]).all() and np.isfinite(out[5:]).all()


@pytest.mark.parametrize("kind,block", [("int8", 0), ("int4", 32)])
@pytest.mark.parametrize("m,k,n", [(1, 2048, 5633), (4, 5632, 2049), (9, 2048, 515)])
def test_ragged_first_call_is_captured(hip, kind, block, m, k, n):
    # a stream whose first call is recorded has no split scratch: such widths
    # take the kernel that needs none, and every replay gives its result
    import torch

    rng = np.random.default_rng(m + n)
    q, s, v, qt = _weights(rng, kind, block, k, n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    da, dq, ds = (torch.from_numpy(np.ascontiguousarray(t)).cuda() for t in (x, q.view(np.int8), s))
    out = torch.zeros(m, n, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    print(f"case captured {kind} m={m} k={k} n={n}", flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        hip.qmm_f32(da.data_ptr(), dq.data_ptr(), ds.data_ptr(), out.data_ptr(), m, k, n, qt, block,
                    stream=stream.cuda_stream)
    wd = _dense(v, s, block)
    bound = (2.0 ** -22 + 2 * k * 2.0 ** -24) * 1.01 * (np.abs(x.astype(np.float64)) @ np.abs(wd)) + 1e-30
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.all(np.abs(out.cpu().numpy().astype(np.float64) - x.astype(np.float64) @ wd) <= bound)


@pytest.mark.parametrize("half_scale", [False, True])
@pytest.mark.parametrize("kind,block", KINDS)
@pytest.mark.parametrize("m,k,n", [(1, 2048, 515), (5, 992, 336), (17, 4096, 130), (40, 95, 67), (130, 1000, 132), (200, 2048, 1100)])
def test_bf16_products_beyond_fp32(hip, half_scale, kind, block, m, k, n):
    # rows whose products with the codes, or the sums of those, exceed fp32
    # although the outputs do not; rows of bf16 subnormals; a row that holds
    # an infinity; a row whose outputs do exceed bf16
    rng = np.random.default_rng(m + k + n + block)
    q, s, v, qt = _weights(rng, kind, block, k, n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    wd = _dense(v, s, block)
    top = np.abs(x.astype(np.float64) @ wd).max(1)   # outputs of a unit row
    x[0] *= np.float32(1e38 / max(top[0], 4.0))
    if m > 4:
        x[1] *= np.float32(2e-39)
        x[2, 3] = np.inf
        x[3] = np.where(v[:, 0] * s[0, 0] >= 0, 3e38, -3e38)
        x[4] *= np.float32(4e37 / max(top[4], 4.0))
    if m > 5:
        x[-1] *= np.float32(1e38 / max(top[-1], 4.0))
    a = _bits(x, True)
    sb = _bits(s, True) if half_scale else s
    da, dq, ds, dc = (hip.DeviceBuffer.from_array(t) for t in (a, q.view(np.int8), sb, np.zeros((m, n), np.uint16)))
    print(f"case bf16 large half_scale={half_scale} {kind} block={block} m={m} k={k} n={n}", flush=True)
    hip.qmm(da.addr, hip.DTYPE_BF16, dq.addr, ds.addr, hip.DTYPE_BF16 if half_scale else hip.DTYPE_F32, dc.addr,
            hip.DTYPE_BF16, m, k, n, qt, block)
    out = _wide(dc.download(np.uint16, (m, n)), True).astype(np.float64)
    wd = _dense(v, _wide(sb, True) if half_scale else s, block)
    aw = _wide(a, True).astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref, mag = aw @ wd, np.abs(aw) @ np.abs(wd)
        # a result within half an ulp of bf16's largest number may go either way
        fits, beyond = np.abs(ref) < 3.3e38, np.abs(ref) > 3.45e38
        bound = 2.0 ** -8 * 1.01 * np.abs(ref) + 2 * k * 2.0 ** -24 * mag + 2.0 ** -133
        assert np.all(np.abs(out - ref)[fits] <= bound[fits]), np.max((np.abs(out - ref) / bound)[fits])
    assert fits[0].all() and fits[-1].all()
    if m > 4:
        assert fits[1].all() and not np.isfinite(out[2]).any() and beyond[3].any()
        assert np.array_equal(out[beyond & np.isfinite(ref)], np.copysign(np.inf, ref[beyond & np.isfinite(ref)]))


@pytest.mark.parametrize("kind,block", [("int8", 0), ("int4", 32)])
@pytest.mark.parametrize("m,k,n", [(1, 2048, 5633), (4, 5632, 2049), (9, 2048, 515)])
def test_ragged_without_scratch_memory(hip, monkeypatch, kind, block, m, k, n):
    # device memory that runs out for a ragged call's scratch leaves the kernel
    # that needs none; an aligned call reports it
    import torch

    rng = np.random.default_rng(m + n)
    q, s, v, qt = _weights(rng, kind, block, k, n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    da, dq, ds = (torch.from_numpy(np.ascontiguousarray(t)).cuda() for t in (x, q.view(np.int8), s))
    out = torch.zeros(m, n, device="cuda")
    stream = torch.cuda.Stream()   # a new stream: no scratch yet
    torch.cuda.synchronize()
    monkeypatch.setenv("VELOMIND_FAIL_BACKEND", "HIP:Scratch:allocate")
    print(f"case no memory {kind} m={m} k={k} n={n}", flush=True)
    hip.qmm_f32(da.data_ptr(), dq.data_ptr(), ds.data_ptr(), out.data_ptr(), m, k, n, qt, block,
                stream=stream.cuda_stream)
    if m == 9:
        with pytest.raises(Exception):
            hip.qmm_f32(da.data_ptr(), dq.data_ptr(), ds.data_ptr(), out.data_ptr(), m, k, 512, qt, block,
                        stream=stream.cuda_stream)
    monkeypatch.delenv("VELOMIND_FAIL_BACKEND")
    torch.cuda.synchronize()
    wd = _dense(v, s, block)
    bound = (2.0 ** -22 + 2 * k * 2.0 ** -24) * 1.01 * (np.abs(x.astype(np.float64)) @ np.abs(wd)) + 1e-30
    assert np.all(np.abs(out.cpu().numpy().astype(np.float64) - x.astype(np.float64) @ wd) <= bound)
