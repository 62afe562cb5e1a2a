"""Every configuration of the MFMA GEMM (rows_m > 4, and 16-bit activations),
forced through the tuning override VELOMIND_GEMM_WIDE="BM,BN,S,D": row tiles of
16, 32 and (per-column INT8) 64, four waves or, with D = 2, eight, pairs of waves
side by side in N with BN = 256, and S splits of K.

Per-column INT8, blockwise INT8 and INT4; fp32, fp16 and bf16; one split and
three (deterministic split-K reduction), partial M and N tiles, every remainder
of the pipelined loop, block scales from 1e-7 to 1e3.  Where the oracle is the
reference the bound is 1e-3 * max|ref|; test_forced_config and
test_activation_magnitudes hold every kind to fp32 summation bounds.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _check(out, ref, tol=TOL):
    ref = np.asarray(ref, np.float64)
    err = np.abs(out.astype(np.float64) - ref).max()
    bound = tol * max(np.abs(ref).max(), 1e-30)
    assert err <= bound, f"max abs err {err:.3e} > {bound:.3e}"


def _weights(kind, k, n, rng, block):
    w = (rng.standard_normal((k, n)) * 0.02).astype(np.float32)
    if kind == "int8":
        q, s = O.quantize_int8(w)
        return q, s, 1, 0
    if kind == "int8_block":
        q = rng.integers(-127, 128, (k, n), dtype=np.int8)
        s = (rng.random(((k + block - 1) // block, n)) * 0.01 + 1e-4).astype(np.float32)
        return q, s, 1, block
    q, s = O.quantize_int4(w, block)
    return q, s, 2, block


# (BM, BN, D) of the override -> row tile, 32-row tiles of it, waves, waves side
# by side in N, and the loop's pipeline stages.
CONFIGS = {
    (16, 64, 1): (16, 1, 4, 1, 3), (16, 64, 2): (16, 1, 8, 1, 3), (32, 128, 1): (32, 1, 4, 1, 3), (32, 128, 2): (32, 1, 8, 1, 3),
    (128, 128, 1): (32, 2, 4, 1, 4), (128, 256, 1): (32, 2, 4, 2, 4),   # per-column INT8
    (32, 256, 1): (32, 1, 4, 2, 3),                                     # blockwise
}
KINDS = [("int8", 0), ("int8", 96), ("int4", 32), ("int4", 128)]


def _configs(kind, block, pieces=True):
    for cfg, (tile, mt, _, nw, _) in CONFIGS.items():
        if (mt == 1 or block == 0) and (nw == 1 or mt == 2 or block > 0) and (pieces or (mt == 1 and nw == 1)):
            yield cfg


def _forced_k(kind, block, cfg, splits, turns):
    """K for which every wave but the last runs `turns` chunks and the number
    of splits is the one asked for; the launcher's arithmetic, checked."""
    tile, _, waves, nw, _ = CONFIGS[cfg]
    chunk = 16 if block == 0 and tile == 32 else 32
    units = splits * (waves // nw)
    chunks = units * turns - 1
    per_wave = -(-chunks // units)
    assert per_wave == turns and -(-chunks // (per_wave * (waves // nw))) == splits
    return chunk * chunks


def _random_weights(rng, kind, block, k, n):
    """(codes, scales, dense weights in 64 bits, quant type)"""
    nb = -(-k // block) if block else 1
    s = (rng.random((nb, n)) * 0.01 + 1e-4).astype(np.float32)
    if kind == "int8":
        q = rng.integers(-127, 128, (k, n), dtype=np.int8)
        v = q
    else:
        q = rng.integers(0, 256, ((k + 1) // 2, n)).astype(np.uint8)
        v = np.empty((2 * q.shape[0], n), np.int8)
        v[0::2], v[1::2] = (q.view(np.int8) << 4) >> 4, q.view(np.int8) >> 4
        v = v[:k]
    return q, s, v.astype(np.float64) * s.astype(np.float64).repeat(block or k, 0)[:k], 2 if kind == "int4" else 1


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("kind,block,cfg", [(*kb, c) for kb in KINDS for c in _configs(*kb)])
def test_forced_config(hip, monkeypatch, kind, block, cfg, splits):
    m, n = 150, 531   # partial tiles of every width, a last quad that moves back
    stages = CONFIGS[cfg][4]
    for turns in range(stages + 1, 2 * stages + 1):   # the loop runs, then every remainder
        k = _forced_k(kind, block, cfg, splits, turns)
        rng = np.random.default_rng(k + cfg[0] + cfg[1] + splits)
        q, s, wd, qt = _random_weights(rng, kind, block, k, n)
        x = rng.standard_normal((m, k)).astype(np.float32)
        monkeypatch.setenv("VELOMIND_GEMM_WIDE", "%d,%d,%d,%d" % (cfg[0], cfg[1], splits, cfg[2]))
        print(f"case forced {kind} block={block} {cfg} S={splits} turns={turns} m={m} k={k} n={n}", flush=True)
        out = hip.run_qmm(x, q, s, k, qt, block).astype(np.float64)
        bound = (2.0 ** -22 + 2 * k * 2.0 ** -24) * 1.01 * (np.abs(x.astype(np.float64)) @ np.abs(wd))
        assert np.all(np.abs(out - x.astype(np.float64) @ wd) <= bound)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("half_scale", [False, True])
@pytest.mark.parametrize("m", [100, 150])   # rows as they lie, and staged in operand order
@pytest.mark.parametrize("kind,block", KINDS)
def test_forced_config_half(hip, monkeypatch, kind, block, m, half_scale, bf16):
    n = 531
    for cfg in _configs(kind, block, pieces=m > 128):
        for splits in (1, 3):
            k = _forced_k(kind, block, cfg, splits, CONFIGS[cfg][4] + 2)
            k -= k % 32 if m <= 128 else 0   # (rows are read as they lie in whole chunks only)
            rng = np.random.default_rng(k + cfg[0] + cfg[1] + m)
            q, s, wd, qt = _random_weights(rng, kind, block, k, n)
            wide = (lambda b: (b.astype(np.uint32) << 16).view(np.float32)) if bf16 else (
                lambda b: b.view(np.float16).astype(np.float32))
            bits = O.f32_to_bf16_bits if bf16 else O.f32_to_f16_bits
            a, sb = bits(rng.standard_normal((m, k)).astype(np.float32)), bits(s)
            if half_scale:
                wd *= (wide(sb).astype(np.float64) / s).repeat(block or k, 0)[:k]
            dt = hip.DTYPE_BF16 if bf16 else hip.DTYPE_F16
            da, dq, ds, dc = (hip.DeviceBuffer.from_array(t) for t in (a, q.view(np.int8), sb if half_scale else s,
                                                                       np.zeros((m, n), np.uint16)))
            monkeypatch.setenv("VELOMIND_GEMM_WIDE", "%d,%d,%d,%d" % (cfg[0], cfg[1], splits, cfg[2]))
            print(f"case forced half bf16={bf16} {kind} block={block} {cfg} S={splits} m={m} k={k} n={n}", flush=True)
            hip.qmm(da.addr, dt, dq.addr, ds.addr, dt if half_scale else hip.DTYPE_F32, dc.addr, dt, m, k, n, qt, block)
            out = wide(dc.download(np.uint16, (m, n))).astype(np.float64)
            aw = wide(a).astype(np.float64)
            ref = aw @ wd
            bound = (2.0 ** -8 if bf16 else 2.0 ** -11) * 1.01 * np.abs(ref) + 2 * k * 2.0 ** -24 * (
                np.abs(aw) @ np.abs(wd)) + 2.0 ** -24
            assert np.all(np.abs(out - ref) <= bound), (cfg, splits)


@pytest.mark.parametrize("mag", [1e-7, 1e-3, 1e3])
@pytest.mark.parametrize("qt", ["int4", "int8_block"])
def test_scale_magnitudes(hip, mag, qt):
    # Block scales spanning 3 orders of magnitude inside each column.
    m, k, n, block = 33, 256, 128, 32
    rng = np.random.default_rng(int(mag * 1e7) % 1000 + 3)
    nb = k // block
    spread = 10.0 ** rng.uniform(-1.5, 1.5, (nb, n))
    s = (mag * spread).astype(np.float32)
    if qt == "int4":
        codes = rng.integers(-8, 8, (k, n))
        packed = np.zeros(((k + 1) // 2, n), np.uint8)
        packed |= (codes[0::2] & 0xF).astype(np.uint8)
        packed |= ((codes[1::2] & 0xF) << 4).astype(np.uint8)
        q, hq, oq = packed, hip.QUANT_INT4, O.QUANT_INT4
    else:
        q, hq, oq = rng.integers(-127, 128, (k, n), dtype=np.int8), hip.QUANT_INT8, O.QUANT_INT8
    x = rng.standard_normal((m, k)).astype(np.float32)
    ref = O.qmm(x, q.view(np.int8), s, k, oq, block)
    out = hip.run_qmm(x, q, s, k, hq, block)
    # columns differ by orders of magnitude: hold each column to its own max
    ref64 = np.asarray(ref, np.float64)
    colmax = np.abs(ref64).max(axis=0)
    err = np.abs(out.astype(np.float64) - ref64).max(axis=0)
    assert np.all(err <= TOL * np.maximum(colmax, 1e-300)), f"worst column ratio {np.max(err / colmax):.3e}"


def test_split_k_deterministic(hip, monkeypatch):
    m, k, n = 24, 2048, 640
    rng = np.random.default_rng(5)
    q, s = O.quantize_int4((rng.standard_normal((k, n)) * 0.02).astype(np.float32), 32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    monkeypatch.setenv("VELOMIND_GEMM_WIDE", "32,128,8,2")   # eight K splits, eight waves
    outs = [hip.run_qmm(x, q, s, k, hip.QUANT_INT4, 32) for _ in range(3)]
    for o in outs[1:]:
        assert np.array_equal(o.view(np.uint32), outs[0].view(np.uint32))
    _check(outs[0], O.qmm(x, q.view(np.int8), s, k, O.QUANT_INT4, 32))


def _magnitude_rows(rng, k):
    """Rows of A at |a| ~ 1e-6, 1, 1e5, 1e6 and 1e30, and one row whose
    entries span 1e-6 .. 1e6 (the MFMA path stages each row with its own
    power-of-two scale, split into two fp16 parts)."""
    base = rng.standard_normal((6, k)).astype(np.float32)
    mags = np.array([1e-6, 1.0, 1e5, 1e6, 1e30], np.float32)
    x = base.copy()
    x[:5] *= mags[:, None]
    x[5] *= (10.0 ** rng.uniform(-6, 6, k)).astype(np.float32)
    return x


@pytest.mark.parametrize("kind,block", [("int8", 0), ("int8_block", 32), ("int4", 32)])
@pytest.mark.parametrize("reps", [1, 8, 30])      # m = 6, 48, 180: 16- and 32-row tiles
def test_activation_magnitudes(hip, kind, block, reps):
    import llama_oracle as LO

    k, n = 256, 320
    rng = np.random.default_rng(17 + reps)
    q, s, qt, blk = _weights(kind, k, n, rng, block)
    oq = O.QUANT_INT4 if qt == 2 else O.QUANT_INT8
    x = np.tile(_magnitude_rows(rng, k), (reps, 1))
    print(f"case magnitudes kind={kind} m={x.shape[0]} k={k} n={n}", flush=True)
    out = hip.run_qmm(x, q, s, k, qt, blk).astype(np.float64)
    assert np.isfinite(out).all()
    ref = np.asarray(O.qmm(x, q.view(np.int8), s, k, oq, blk), np.float64)
    rowmax = np.abs(ref).max(axis=1)
    err = np.abs(out - ref).max(axis=1)
    assert np.all(err <= TOL * rowmax), f"worst row ratio {np.max(err / rowmax):.3e}"
    # Against the model of what the MFMAs multiply (A split into two fp16
    # parts, the exact weights) the only difference left is fp32 summation
    # of 2k products and the chunk sums' scaling: |err| <= 2k * 2^-24 *
    # sum_k |a * w|.
    lin = LO.Linear(q=q, s=s, k=k, n=n, quant_type=oq, block=blk, mode=LO.LINEAR_DENSE)
    wd = lin.dense().astype(np.float64)
    model = LO.split_rows_fp16(x) @ wd
    mag = np.abs(x.astype(np.float64)) @ np.abs(wd)
    bound = 2 * k * 2.0 ** -24 * 1.01 * mag + 1e-300
    assert np.all(np.abs(out - model) <= bound), f"worst ratio {np.max(np.abs(out - model) / bound):.3e}"
    # every kind is fp32-equivalent against the reference loop itself
    bound = (2.0 ** -22 + 4 * k * 2.0 ** -24) * 1.01 * mag + 1e-300
    assert np.all(np.abs(out - ref) <= bound), f"worst ratio {np.max(np.abs(out - ref) / bound):.3e}"


@pytest.mark.parametrize("kind,block", [("int8", 0), ("int4", 32)])
def test_long_k(hip, kind, block):
    # K = 2048: the default rule's splits, every stage used several times
    m, k, n = 200, 2048, 512
    rng = np.random.default_rng(91 + block)
    q, s, qt, blk = _weights(kind, k, n, rng, block)
    x = rng.standard_normal((m, k)).astype(np.float32)
    print(f"case long k kind={kind} m={m} k={k} n={n}", flush=True)
    _check(hip.run_qmm(x, q, s, k, qt, blk), O.qmm(x, q.view(np.int8), s, k, O.QUANT_INT4 if qt == 2 else O.QUANT_INT8, blk))


@pytest.mark.parametrize("kind,block", [("int8", 0), ("int4", 32)])
@pytest.mark.parametrize("m,n", [(384, 300), (401, 4500), (700, 1100), (1025, 2600)])
def test_row_panels(hip, kind, block, m, n):
    # past 384 rows tiles are numbered in panels of rows, the last one shorter:
    # every tile of every panel is written
    k = 96
    rng = np.random.default_rng(m + n)
    q, s, qt, blk = _weights(kind, k, n, rng, block)
    x = rng.standard_normal((m, k)).astype(np.float32)
    print(f"case panels kind={kind} m={m} k={k} n={n}", flush=True)
    _check(hip.run_qmm(x, q, s, k, qt, blk), O.qmm(x, q.view(np.int8), s, k, O.QUANT_INT4 if qt == 2 else O.QUANT_INT8, blk))
