"""The matrix-core prefill kernel (prefill.hip) over the sizes where it can go
wrong: every gqa factor (padding columns), both head dims, ragged row blocks,
stages that end inside the diagonal, launches without splits, with splits of
some row blocks only and with the most splits of one block. Each chunk is
large enough that the size rule sends it there."""
from __future__ import annotations

import numpy as np
import pytest

import pyoracle
from dbinfer_amd.kv import F32, INT8, HipKV
from helpers import assert_close, normal

pytestmark = pytest.mark.gpu


# sinks: -1 fp32, otherwise int8 with that many fp32 sinks
@pytest.mark.parametrize("sinks", [-1, 4])
@pytest.mark.parametrize("hd,nkv,G,n,pos0", [
    (64, 8, 1, 500, 6000), (64, 8, 2, 200, 4000), (64, 8, 3, 200, 3000),
    (64, 8, 4, 256, 1000), (64, 4, 5, 257, 1500), (64, 4, 6, 300, 1500),
    (64, 4, 7, 300, 1500), (64, 2, 8, 600, 900),
    (64, 8, 4, 64, 8000),      # one row block of 32 splits
    (128, 8, 1, 500, 4000), (128, 8, 2, 250, 3000), (128, 8, 3, 150, 2500),
    (128, 8, 4, 256, 1000), (128, 4, 5, 200, 2000), (128, 4, 6, 200, 1500),
    (128, 4, 7, 300, 300),     # blocks of 1 to 7 splits
    (128, 2, 8, 1100, 0),      # a prompt from position 0
    (128, 8, 4, 1100, 3),      # stages that end inside the diagonal
    (64, 16, 8, 1050, 0),      # more row blocks than splits have room for: none
])
def test_prefill_chunk(hd, nkv, G, n, pos0, sinks):
    run_chunk(hd, nkv, G, n, pos0, sinks)


@pytest.mark.parametrize("hd,nkv,G,n,pos0,sinks", [
    (64, 8, 4, 256, 2000, 0), (128, 8, 3, 256, 2000, 0),
    (64, 8, 4, 256, 2000, 70),    # sinks in three stages
    (128, 8, 3, 256, 2000, 33),
    (64, 8, 8, 900, 0, 100),      # rows that see some of the sinks only
    (128, 4, 7, 900, 0, 9),
])
def test_prefill_chunk_int8_sinks(hd, nkv, G, n, pos0, sinks):
    run_chunk(hd, nkv, G, n, pos0, sinks)


def run_chunk(hd, nkv, G, n, pos0, sinks):
    nh, cap, P = nkv * G, pos0 + n + 40, nkv * hd
    scale = np.float32(1.0) / np.sqrt(np.float32(hd))
    kind = (max(sinks, 0), 0, F32 if sinks < 0 else INT8)
    g, o = HipKV(1, cap, nkv, hd, *kind), pyoracle.OracleKV(1, cap, nkv, hd, *kind)
    K, V = normal(7 + n, pos0 + n, P), normal(8 + n, pos0 + n, P)
    if sinks < 0:
        # what lies past the chunk is not attended, whatever it holds
        bad = np.full((40, P), np.nan, np.float32)
        g.append_n(0, 0, np.concatenate([K, bad]), np.concatenate([V, bad]))
        g.truncate(pos0 + n)
    else:
        K[:, ::101] *= 8.0
        V[:, ::101] *= 8.0
        g.append_n(0, 0, K, V)
    o.append_n(0, 0, K, V)
    q = normal(9 + n, n, nh * hd)
    got = g.attend_chunk(0, pos0, q, nh, scale)
    # the oracle on the first and last rows and some between
    for r in sorted({0, 1, 31, 32, n // 2, n - 33, n - 2, n - 1}):
        want = o.attend(0, pos0 + r, q[r], nh, scale, n_threads=8)
        assert_close(got.reshape(n, -1)[r], want, what=f"row {r}")
    # every row against float64, over what the cache holds
    k, v = (a.reshape(pos0 + n, nkv, hd).astype(np.float64) for a in (K, V))
    if sinks >= 0:
        m = pos0 + n
        ks = np.repeat(g.export("k_scale", 0).reshape(-1, nkv, hd), 32, 0)[:m]
        vs = np.repeat(g.export("v_scale", 0).reshape(-1, nkv, hd // 32)[:m], 32, -1)
        kc = g.export("k8", 0).reshape(-1, nkv, hd)[:m]
        vc = g.export("v8", 0).reshape(-1, nkv, hd)[:m]
        sk = min(sinks, m)
        k[sk:] = (kc.astype(np.float64) * ks)[sk:]
        v[sk:] = (vc.astype(np.float64) * vs)[sk:]
    qd = q.reshape(n, nkv, G, hd).astype(np.float64) * float(scale)
    past = np.arange(pos0 + n)[None, :] > (pos0 + np.arange(n))[:, None]
    for h in range(nkv):
        s = np.einsum("ngd,kd->ngk", qd[:, h], k[:, h], optimize=True)
        s = np.where(past[:, None, :], -np.inf, s)
        s = np.exp(s - s.max(-1, keepdims=True))
        want = np.einsum("ngk,kd->ngd", s / s.sum(-1, keepdims=True), v[:, h], optimize=True)
        assert_close(got.reshape(n, nkv, G, hd)[:, h], want, what=f"kv head {h}")
    assert np.array_equal(g.attend_chunk(0, pos0, q, nh, scale), got)
