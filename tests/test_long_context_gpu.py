"""Decode across 1,024 positions, where a step's attention takes finer ranges: a
generate that crosses it equals its eager launches bit for bit, its persistent
mode (whose long steps are per-layer launches) gives the same bits, and the
logits of the last step equal those of forward() fed the same tokens; and the
long-context attention against a float64 one at the split's edges."""
import ctypes
import os

import numpy as np
import pytest

from n550_qwen3_bringup_handover_amd import abi, model as M, runtime
from tests.test_attention_gpu import EPS, HD, LD, NKV, U, VP, Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pos,max_seq", [(0, 16), (15, 2048), (1023, 1024), (1024, 2048), (1025, 4096), (1983, 2048),
                                         (8191, 8192)])
def test_long_attention(pos, max_seq):
    L = runtime.init()
    x = Case(1, pos, max_seq)
    want, _ = x.exact()
    up = abi.DeviceBuffer.from_array
    kc = np.full((NKV, HD // 4, max_seq, 4), np.nan, np.float32)
    vc = np.full((NKV, max_seq, HD), np.nan, np.float32)
    kc[:, :, :pos] = x.k.reshape(NKV, pos, HD // 4, 4).transpose(0, 2, 1, 3)
    vc[:, :pos] = x.v
    out, part = up(np.full(2048, np.nan, np.float32)), up(np.full(8 * 16 * 2 * (HD + 4), np.nan, np.float32))
    b = [up(t) for t in (x.qkv, kc, vc, x.qn, x.kn, x.cos, x.sin, np.array([pos], np.int32))]
    p = [VP(t.ptr) for t in b]
    assert L.qm_attention_decode_long(p[0], VP(out.ptr), VP(part.ptr), *p[1:], max_seq, ctypes.c_float(EPS)) == 0
    abi.sync()
    vmax = max(np.abs(x.qkv[:, 3072:]).max(), np.abs(x.v).max() if pos else 0)
    tol = (6 * np.sqrt(HD + 16) + 8 + 2 * np.sqrt(pos + 1)) * U * vmax       # as in test_attention_gpu
    assert np.abs(out.download(np.float32, 2048).reshape(1, 16, HD) - want).max() <= tol


def test_generate_across_1024():
    blob = M.qw3m_random(3, M.LAYOUT_ROW, threads=16)
    m = M.Model(blob, max_seq=1100)
    del blob
    prompt = np.random.default_rng(5).integers(0, M.VOCAB, 1018).astype(np.int32)
    res = []
    for graph, persist in ((True, False), (False, False), (True, True), (True, False)):
        if persist and runtime.lib().qwen3_hip_model_set_persistent(m._h, 1) != 0:
            continue
        m.set_graph(graph)
        res.append((m.generate(prompt, 12), m.logits()))
        m.set_persistent(False)
    for t, l in res[1:]:
        assert np.array_equal(t, res[0][0]) and np.array_equal(l, res[0][1])
    toks = res[0][0]
    m.generate(prompt, 0)
    for i, t in enumerate(toks[:-1]):
        m.forward(np.array([t], np.int32), 1018 + i)
    assert np.array_equal(m.logits(), res[0][1])
    m.close()
