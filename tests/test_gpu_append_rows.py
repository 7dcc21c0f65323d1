"""The one-launch rows kernels (append.hip, rows_f32_kernel and rows_i8_kernel):
bias, rope, append and quantization of a chunk's rows, bit-exact with the
oracle's row-by-row flow at the edges of the 32-token groups and passes, with
sinks, staging rows left by earlier appends, and rows of any alignment."""
from __future__ import annotations

import numpy as np
import pytest

import pyoracle
from dbinfer_amd.kv import F32, INT8, HipKV
from helpers import assert_close, normal

pytestmark = pytest.mark.gpu

NAMES = {F32: ("k", "v"),
         INT8: ("k8", "v8", "k_scale", "v_scale", "k_raw", "k_sink", "v_sink")}


@pytest.mark.parametrize("dtype", [F32, INT8])
@pytest.mark.parametrize("hd,nkv,G,sink,steps", [
    # steps: (pos0, n) in turn; a pos0 below the rows seen is a rollback
    (64, 2, 3, 4, [(0, 1), (1, 30), (31, 1), (32, 33), (65, 5)]),
    (128, 2, 4, 4, [(0, 31), (31, 2), (33, 64), (97, 31)]),
    (128, 1, 8, 0, [(0, 100), (90, 5), (95, 64), (159, 7)]),   # rollbacks
    (64, 4, 1, 40, [(0, 37), (37, 70)]),                       # sinks past one group
    (128, 3, 5, 9, [(0, 8), (8, 16), (20, 12), (30, 1)]),
])
@pytest.mark.parametrize("bias,shift", [(False, 0), (True, 1)])
def test_append_rows(dtype, hd, nkv, G, sink, steps, bias, shift):
    torch = pytest.importorskip("torch")
    nh, theta = nkv * G, 1e4
    cap = max(p + n for p, n in steps) + 3
    ns = sink if dtype == INT8 else 0
    g = HipKV(1, cap, nkv, hd, ns, 0, dtype, theta)
    o = pyoracle.OracleKV(1, cap, nkv, hd, ns, 0, dtype, theta)
    scale = np.float32(1.0) / np.sqrt(np.float32(hd))
    stream = torch.cuda.Stream()
    g.set_stream(stream.cuda_stream)
    bs = [normal(5 + i, m * hd) if bias else None for i, m in enumerate((nh, nkv, nkv))]

    def dev(a):  # rows that start `shift` floats past an aligned address
        if a is None:
            return None
        t = torch.zeros(a.size + shift, device="cuda")
        t[shift:] = torch.from_numpy(a.reshape(-1)).cuda()
        return t

    for i, (pos0, n) in enumerate(steps):
        q, k, v = (normal(100 * i + j, n, m * hd) for j, m in enumerate((nh, nkv, nkv)))
        t = [dev(a) for a in (q, k, v, *bs)]
        out = torch.zeros(n * nh * hd, device="cuda")
        torch.cuda.synchronize()
        ptr = [None if a is None else a.data_ptr() + 4 * shift for a in t]
        g.chunk_qkv_async(0, pos0, n, nh, scale, *ptr, out.data_ptr())
        torch.cuda.synchronize()
        qr = np.empty_like(q)
        for c in range(n):
            qc, kc, vc = (a[c] if b is None else a[c] + b for a, b in zip((q, k, v), bs))
            qr[c] = pyoracle.rope(qc, [pos0 + c], theta, nh, 1, hd)
            o.append(0, pos0 + c, pyoracle.rope(kc, [pos0 + c], theta, nkv, 1, hd), vc)
        for name in NAMES[dtype]:
            if "sink" in name and ns == 0:
                continue
            a, b = g.export(name, 0), o.export(name, 0)
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (name, pos0, n)
        want = o.attend_chunk(0, pos0, qr, nh, scale)
        assert_close(out.cpu().numpy(), np.asarray(want).reshape(-1), what=f"rows {pos0}+{n}")
    # the same rows without the producer
    k, v = normal(901, 40, nkv * hd), normal(902, 40, nkv * hd)
    t = [dev(k), dev(v)]
    torch.cuda.synchronize()
    n = min(40, cap - 5)
    g.append_async(0, 5, n, t[0].data_ptr() + 4 * shift, t[1].data_ptr() + 4 * shift)
    o.append_n(0, 5, k[:n], v[:n])
    torch.cuda.synchronize()
    for name in NAMES[dtype]:
        if "sink" in name and ns == 0:
            continue
        assert np.array_equal(g.export(name, 0).view(np.uint8), o.export(name, 0).view(np.uint8)), name
    g.close()
