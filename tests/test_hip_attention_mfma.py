"""FusedAttention of several query rows on the matrix cores (head_dim 64 and
128): edges of the 16-row query tiles and of the key blocks (32 keys, 16 at
head_dim 128), two and four key groups, grouped heads, batches, values that a
mask has to keep apart, and the sizes from which a wave per row takes the call.

Bound: scores are fp32 dot products of d terms, |ds| <= d 2^-24 sum |q k|
scale, which the exponential turns into a relative error of each weight; the
weighted sum of sk values adds sk 2^-24.  Against the result in 64 bits:
|err| <= 2 (max |ds| + (sk + 8) 2^-24) sum p |v| / sum p."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(q, k, v, scale, causal):
    """(attention in 64 bits, error bound); a row uses its visible keys only."""
    b, hq, sq, d = q.shape
    rep, sk = hq // k.shape[1], k.shape[2]
    q, k, v = q.astype(np.float64), np.repeat(k, rep, 1).astype(np.float64), np.repeat(v, rep, 1).astype(np.float64)
    out, bound = np.empty(q.shape), np.empty(q.shape)
    for i in range(sq):
        n = sk - sq + i + 1 if causal else sk
        with np.errstate(all="ignore"):
            s = np.einsum("bhd,bhkd->bhk", q[:, :, i], k[:, :, :n]) * scale
            ds = np.einsum("bhd,bhkd->bhk", np.abs(q[:, :, i]), np.abs(k[:, :, :n])).max(-1) * scale * d * 2.0 ** -24
            p = np.exp(s - s.max(-1, keepdims=True))
            p /= p.sum(-1, keepdims=True)
            out[:, :, i] = np.einsum("bhk,bhkd->bhd", p, v[:, :, :n])
            bound[:, :, i] = 2 * (ds[..., None] + (n + 8) * 2.0 ** -24) * np.einsum("bhk,bhkd->bhd", p, np.abs(v[:, :, :n]))
    return out, bound


def _inputs(batch, hq, hk, sq, sk, d, seed):
    rng = np.random.default_rng(seed)
    return tuple(rng.standard_normal(s).astype(np.float32) for s in ((batch, hq, sq, d), (batch, hk, sk, d), (batch, hk, sk, d)))


@pytest.mark.parametrize("batch,hq,hk,sq,sk", [
    (1, 2, 1, 5, 48), (1, 3, 3, 7, 59), (1, 3, 3, 7, 60), (2, 10, 5, 48, 48), (1, 4, 4, 16, 64), (2, 4, 2, 17, 65), (1, 3, 1, 33, 127), (1, 5, 5, 64, 64), (2, 6, 3, 65, 129),
    (1, 2, 2, 100, 400), (1, 8, 2, 31, 300),
    (3, 15, 5, 130, 130),     # 405 tiles of 16 rows: four key groups, as all above
    (1, 64, 8, 150, 498),     # 640: two at head_dim 64
    (2, 40, 8, 450, 450),     # 2320: two at either
])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_tiles(hip, batch, hq, hk, sq, sk, d, causal):
    q, k, v = _inputs(batch, hq, hk, sq, sk, d, sq * 7 + sk + d)
    scale = 0.2 if sq == 33 else 0.0   # 0: 1 / sqrt(d)
    print(f"case attention tiles b={batch} hq={hq} hk={hk} sq={sq} sk={sk} d={d} causal={causal}", flush=True)
    out = hip.run_attention(q, k, v, scale, causal).astype(np.float64)
    ref, bound = _reference(q, k, v, scale or 1 / np.sqrt(d), causal)
    assert np.all(np.abs(out - ref) <= bound), np.max(np.abs(out - ref) / bound)


@pytest.mark.parametrize("hq,hk", [(2, 1), (416, 8)])   # four key groups, and two (2080 tiles of 16 rows)
@pytest.mark.parametrize("d", [64, 128])
def test_masked_values_do_not_reach_earlier_rows(hip, d, hq, hk):
    # infinities and NaN in V and K at positions that some rows of a tile see
    # and others do not; a score of -inf beside finite ones; a row whose
    # every score is -inf (no softmax: NaN, as one row's kernel gives)
    sq = sk = 70
    q, k, v = _inputs(1, hq, hk, sq, sk, d, d)
    v[:, :, 20, 3], v[:, :, 21, 5], v[:, :, 66, 0] = np.inf, np.nan, -np.inf
    k[:, :, 40, 7] = np.nan
    k[:, :, 50] = 0.0
    k[:, :, 50, 0] = np.inf
    q[..., 0] = -np.abs(q[..., 0])       # -inf scores at key 50
    print(f"case attention masked specials d={d} hq={hq}", flush=True)
    out = hip.run_attention(q, k, v, 0.0, True)
    ref, bound = _reference(q, k, v, 1 / np.sqrt(d), True)
    finite = np.isfinite(ref)
    assert np.array_equal(finite, np.isfinite(out)) and np.array_equal(np.isnan(ref), np.isnan(out))
    assert np.array_equal(ref[np.isinf(ref)], out[np.isinf(ref)].astype(np.float64))
    assert np.all(np.abs(out - ref)[finite] <= bound[finite])
    # rows before position 20 see nothing special, rows from 40 on a NaN score
    assert finite[:, :, :20].all() and np.isnan(ref[:, :, 40:]).all()
    k2 = np.zeros_like(k)
    k2[..., 0] = np.inf
    out = hip.run_attention(np.ascontiguousarray(np.where(np.arange(d) == 0, q, 0.0), np.float32), k2, np.ones_like(v), 0.0, True)
    assert np.isnan(out).all()
