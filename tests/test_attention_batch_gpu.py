"""Batched decode attention (one new token per sequence) against a float64
attention, at the cache sizes where its number of position ranges changes (64,
128 with 8 sequences, 256) and one off them, with sequences at the first and
last position of their cache, at pass edges, and anywhere.  Tolerance and its
derivation: test_attention_gpu."""
import ctypes

import numpy as np
import pytest

from n550_qwen3_bringup_handover_amd import abi, runtime
from tests.test_attention_gpu import EPS, HD, LD, NKV, U, VP, bits, norm_rope

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq", [1, 7, 8, 33])
@pytest.mark.parametrize("max_seq", [2, 63, 64, 65, 127, 128, 129, 256, 257, 700])
def test_batch_attention(n_seq, max_seq):
    print(f"batch attention n_seq {n_seq} max_seq {max_seq}", flush=True)
    L = runtime.init()
    r = np.random.default_rng([n_seq, max_seq])
    pos = r.integers(0, max_seq, n_seq).astype(np.int32)
    pos[:5] = [min(p, max_seq - 1) for p in (max_seq - 1, 0, 63, 64, 127)][:len(pos[:5])]
    qkv = r.standard_normal((n_seq, LD)).astype(np.float32)
    qn, kn = (bits(1 + 0.1 * r.standard_normal(HD)) for _ in range(2))
    ang = r.uniform(0, 2 * np.pi, (max_seq, HD // 2))
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    k = r.standard_normal((n_seq, NKV, max_seq, HD)).astype(np.float32)
    v = r.standard_normal((n_seq, NKV, max_seq, HD)).astype(np.float32)
    for s in range(n_seq):
        k[s, :, pos[s]:] = v[s, :, pos[s]:] = np.nan          # unwritten entries must not matter
    kc = np.ascontiguousarray(k.reshape(n_seq, NKV, max_seq, HD // 4, 4).transpose(0, 1, 3, 2, 4))
    up = abi.DeviceBuffer.from_array
    att = up(np.full(n_seq * 2048, np.nan, np.float32))
    part = up(np.full(n_seq * 8 * 8 * 2 * (HD + 4), np.nan, np.float32))
    b = [up(x) for x in (qkv, kc, v, qn, kn, cos, sin, pos)]
    p = [VP(x.ptr) for x in b]
    rc = L.qm_attention_decode_batch(p[0], VP(att.ptr), VP(part.ptr), p[1], p[2], ctypes.c_size_t(NKV * max_seq * HD),
                                     *p[3:], ctypes.c_int(n_seq), ctypes.c_int(max_seq), ctypes.c_float(EPS))
    assert rc == 0
    abi.sync()
    got = att.download(np.float32, n_seq * 2048).reshape(n_seq, 16, HD)
    kgot = b[1].download(np.float32, kc.size).reshape(kc.shape).transpose(0, 1, 3, 2, 4).reshape(k.shape)
    vgot = b[2].download(np.float32, v.size).reshape(v.shape)
    f = lambda w: (w.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x = qkv.astype(np.float64)
    c, s_ = cos[pos].astype(np.float64), sin[pos].astype(np.float64)
    q = norm_rope(x[:, :2048].reshape(-1, 16, HD), f(qn), c, s_)
    knew = norm_rope(x[:, 2048:3072].reshape(-1, NKV, HD), f(kn), c, s_)
    vnew = qkv[:, 3072:].reshape(n_seq, NKV, HD)
    for s in range(n_seq):
        ks = np.concatenate([k[s, :, :pos[s]], knew[s][:, None]], 1)
        vs = np.concatenate([v[s, :, :pos[s]], vnew[s][:, None]], 1)
        vmax = np.abs(vs).max()
        tol = (6 * np.sqrt(HD + 16) + 8 + 2 * np.sqrt(pos[s] + 1)) * U * vmax
        for hd in range(16):
            sc = ks[hd // 2] @ q[s, hd] / np.sqrt(HD)
            e = np.exp(sc - sc.max())
            assert np.abs(got[s, hd] - (e / e.sum()) @ vs[hd // 2]).max() <= tol, (s, pos[s], hd)
        assert np.abs(kgot[s, :, pos[s]] - knew[s]).max() <= 32 * U * np.abs(knew[s]).max()
        assert np.array_equal(vgot[s, :, pos[s]], vnew[s])
        rest = np.arange(max_seq) != pos[s]                    # nothing else is written
        assert np.array_equal(kgot[s][:, rest], k[s][:, rest], equal_nan=True)
        assert np.array_equal(vgot[s][:, rest], v[s][:, rest], equal_nan=True)
