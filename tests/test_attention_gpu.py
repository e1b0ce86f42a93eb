"""The chunk attention (qm_attention: RoPE and cache write, causal attention
on the matrix cores) against a float64 attention over the same inputs.

The sizes are where its launch changes shape or its tiles are ragged: 8- and
16-token blocks (nt 496 / 497 is where one turns into the other), chunks and
contexts one off a tile, contexts long enough that the key range is split
over blocks and merged (a few tokens behind 300 .. 8,000 positions), one
token, and the end of the cache.

Tolerance.  Roundings add like a random walk.  A score (rms 1 here, its sum
of HD products scaled by 1 / sqrt(HD)) carries HD + 16 of them, of sums no
larger than 3: sqrt(HD + 16) * 3 * 2^-24, which moves a weight by as much,
relative; normalising may double it; exp and the divisions add 8 units and the
weighted sum sqrt(ctx) (twice that at two sigma): |err| <= (6 sqrt(HD + 16) + 8 +
2 sqrt(ctx)) 2^-24 max|v|.  A 16-position tile that is lost or counted twice
moves an output by about 16 / ctx of |v|, 20 times the bound at ctx 8,000."""
import ctypes

import numpy as np
import pytest

from n550_qwen3_bringup_handover_amd import abi, runtime

pytestmark = pytest.mark.gpu
HD, NKV, LD = 128, 8, 4096
EPS = 1e-6
VP = ctypes.c_void_p
U = 2.0 ** -24


def bits(x):
    return (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)


def norm_rope(x, w, c, s):                    # [n, heads, 128] in float64
    x = x * (1.0 / np.sqrt((x * x).mean(-1, keepdims=True) + EPS)) * w
    c, s = c[:, None], s[:, None]
    a, b = x[..., :64], x[..., 64:]
    return np.concatenate([a * c - b * s, b * c + a * s], -1)


class Case:
    """one layer's inputs, the cache holding pos0 earlier positions"""

    def __init__(self, nt, pos0, max_seq, seed=0):
        r = np.random.default_rng([seed, nt, pos0])
        self.nt, self.pos0, self.max_seq = nt, pos0, max_seq
        self.qkv = r.standard_normal((nt, LD)).astype(np.float32)
        self.qn, self.kn = (bits(1 + 0.1 * r.standard_normal(HD)) for _ in range(2))
        ang = r.uniform(0, 2 * np.pi, (max_seq, HD // 2))
        self.cos, self.sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
        self.k = r.standard_normal((NKV, pos0, HD)).astype(np.float32)
        self.v = r.standard_normal((NKV, pos0, HD)).astype(np.float32)

    def run(self):
        L = runtime.init()
        up = abi.DeviceBuffer.from_array
        kc = np.full((NKV, HD // 4, self.max_seq, 4), np.nan, np.float32)    # unwritten entries must not matter
        vc = np.full((NKV, self.max_seq, HD), np.nan, np.float32)
        kc[:, :, :self.pos0] = self.k.reshape(NKV, self.pos0, HD // 4, 4).transpose(0, 2, 1, 3)
        vc[:, :self.pos0] = self.v
        out = up(np.full(self.nt * 2048, np.nan, np.float32))
        part = abi.DeviceBuffer(8 * 128 * 16 * (HD + 4) * 4)
        b = [up(x) for x in (self.qkv, kc, vc, self.qn, self.kn, self.cos, self.sin,
                             np.array([self.pos0], np.int32))]
        p = [VP(x.ptr) for x in b]
        rc = L.qm_attention(p[0], VP(out.ptr), VP(part.ptr), *p[1:], ctypes.c_int(self.nt),
                            ctypes.c_int(self.max_seq), ctypes.c_int(self.pos0 + self.nt), ctypes.c_float(EPS))
        assert rc == 0
        abi.sync()
        return (out.download(np.float32, self.nt * 2048).reshape(self.nt, 16, HD),
                b[1].download(np.float32, kc.size).reshape(kc.shape), b[2].download(np.float32, vc.size).reshape(vc.shape))

    def exact(self):
        rows = slice(self.pos0, self.pos0 + self.nt)
        c, s = self.cos[rows].astype(np.float64), self.sin[rows].astype(np.float64)
        f = lambda w: (w.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        x = self.qkv.astype(np.float64)
        q = norm_rope(x[:, :2048].reshape(-1, 16, HD), f(self.qn), c, s)
        knew = norm_rope(x[:, 2048:3072].reshape(-1, NKV, HD), f(self.kn), c, s)
        k = np.concatenate([self.k, knew.transpose(1, 0, 2)], 1)
        v = np.concatenate([self.v, x[:, 3072:].reshape(-1, NKV, HD).transpose(1, 0, 2)], 1)
        mask = np.arange(self.pos0 + self.nt)[None] > np.arange(self.pos0, self.pos0 + self.nt)[:, None]
        out = np.empty((self.nt, 16, HD))
        for hd in range(16):
            sc = q[:, hd] @ k[hd // 2].T / np.sqrt(HD)
            sc[mask] = -np.inf
            e = np.exp(sc - sc.max(-1, keepdims=True))
            e /= e.sum(-1, keepdims=True)
            out[:, hd] = np.where(e[..., None] > 0, e[..., None] * v[hd // 2], 0).sum(1) if np.isnan(v).any() or \
                np.isinf(v).any() else e @ v[hd // 2]
        return out, knew


SIZES = [(1, 0, 16), (1, 15, 16), (1, 1900, 1901), (2, 14, 2048), (7, 300, 512), (8, 8, 16), (9, 700, 2048),
         (16, 0, 128), (17, 8000, 8192), (33, 1500, 2048), (127, 1, 128), (128, 0, 2048), (128, 1000, 2048),
         (130, 30, 160), (200, 0, 224), (496, 3, 512), (497, 0, 512), (513, 100, 700), (1030, 0, 1030)]


@pytest.mark.parametrize("nt,pos0,max_seq", SIZES)
def test_chunk_attention(nt, pos0, max_seq):
    print(f"attention nt {nt} pos0 {pos0} max_seq {max_seq}", flush=True)
    x = Case(nt, pos0, max_seq)
    got, kc, vc = x.run()
    want, knew = x.exact()
    ctx = pos0 + nt
    vmax = max(np.abs(x.qkv[:, 3072:]).max(), np.abs(x.v).max() if pos0 else 0)
    tol = (6 * np.sqrt(HD + 16) + 8 + 2 * np.sqrt(ctx)) * U * vmax
    err = np.abs(got - want).max()
    print(f"max err {err:.2e} (bound {tol:.2e})", flush=True)
    assert err <= tol
    # the new cache entries, and nothing past them
    k = kc.transpose(0, 2, 1, 3).reshape(NKV, max_seq, HD)
    assert np.abs(k[:, pos0:ctx] - knew.transpose(1, 0, 2)).max() <= 32 * U * np.abs(knew).max()
    assert np.array_equal(vc[:, pos0:ctx], x.qkv[:, 3072:].reshape(nt, NKV, HD).transpose(1, 0, 2))
    assert np.isnan(k[:, ctx:]).all() and np.isnan(vc[:, ctx:]).all()


@pytest.mark.parametrize("nt,pos0", [(24, 0), (24, 600), (600, 0)])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(nt, pos0):
    """an infinite V entry of token j reaches that dim of tokens j .. only"""
    x = Case(nt, pos0, pos0 + nt)
    j = 13
    clean = x.run()[0]
    x.qkv[j, 3072 + 2 * HD + 5] = np.inf              # kv head 2, dim 5
    got = x.run()[0]
    assert np.array_equal(got[:j], clean[:j])
    assert not np.isfinite(got[j:, 4:6, 5]).any()
    assert np.array_equal(np.delete(got[j], [4, 5], 0), np.delete(clean[j], [4, 5], 0))


@pytest.mark.parametrize("nt,pos0,cached", [(24, 0, ()), (24, 605, (600,)), (600, 0, ()), (600, 5, (3,))])
def test_several_values_that_are_not_finite_in_one_tile(nt, pos0, cached):
    """Two or three positions of one 16-position tile on the diagonal hold an
    entry that is not finite, each in a dim of its own (one of them may lie in
    the cache): every row gets those at and before its own position, and its
    other outputs are those without such entries, bit for bit."""
    x = Case(nt, pos0, pos0 + nt)
    clean = x.run()[0]
    bad = [(p, 7) for p in cached]
    for t in cached:
        x.v[2, t, 7] = np.nan
    first = 0 if pos0 else 13
    for n, j in enumerate((first, first + 1, first + 2)):
        x.qkv[j, 3072 + 2 * HD + 9 + n] = (np.inf, -np.inf, np.nan)[n]
        bad.append((pos0 + j, 9 + n))
    got = x.run()[0]
    rows = pos0 + np.arange(nt)
    for p, d in bad:
        assert np.array_equal(np.isfinite(got[:, 4:6, d]).all(1), rows < p), (p, d)
        got[rows >= p, 4:6, d] = clean[rows >= p, 4:6, d]
    assert np.array_equal(got, clean)


@pytest.mark.parametrize("nt,pos0,splits", [(24, 600, 2), (1, 2047, 8), (24, 16, 1)])
def test_scores_that_are_nan_stay_in_the_sum(nt, pos0, splits):
    """NaN keys at every position of the second key split (of eight waves with
    one split): a range whose maximum is -inf because all its scores are NaN is
    not an empty one."""
    x = Case(nt, pos0, pos0 + nt)
    clean = x.run()[0]
    tile = np.arange(pos0) // 16 % (8 * splits)
    x.k[2, (tile >= 8) & (tile < 16) if splits > 1 else tile == 0] = np.nan
    got = x.run()[0]
    assert np.isnan(got[:, 4:6]).all()
    assert np.array_equal(np.delete(got, [4, 5], 1), np.delete(clean, [4, 5], 1))
