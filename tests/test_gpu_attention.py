"""The batched attention (mhip_attention_batch) against the one-token
attention (mhip_attention, src/model/forward.c:118-165 of the reference) at
every token: outputs and cache rows bit for bit.

From 250 tokens or 1000 positions on (head_dim 128; few heads later) the
scores and the mix run in tiles of 64 x 64 and 32 x 32 (rows x positions; a
row is a token and a head of its key/value group), the softmax sums 128
positions at a time, and batches of long contexts in passes of a bounded
score matrix: the sizes lie around those edges, over groups of 8, 1, 3 and
10 heads. Cache rows past the batch
and the scratch are NaN before the call."""
import ctypes

import numpy as np
import pytest

import motoria_amd as M

pytestmark = pytest.mark.gpu
HD, EPS = 128, 1e-6


def say(*a):
    print(*a, flush=True)


def q8_blocks(rng, rows, cols):
    d = rng.uniform(0.5, 1.5, rows * cols // 32).astype(np.float32) * 1e-3
    q = rng.integers(-127, 128, (rows * cols // 32, 32)).astype(np.int8)
    return np.concatenate([d.view(np.uint8).reshape(-1, 4), q.view(np.uint8)], 1).reshape(-1)


class Layer:
    def __init__(self, torch, dim, nh, nkv, max_seq, seed):
        rng = np.random.default_rng(seed)
        up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
        self.torch, self.g, self.L = torch, M.Gpu(), M.lib()
        self.a = M.AttnDims(dim, nh, nkv, HD, EPS)
        self.dim, self.nh, self.nkv, self.max_seq, self.rng, self.up = dim, nh, nkv, max_seq, rng, up
        qd, kvd = nh * HD, nkv * HD
        self.w = [up(q8_blocks(rng, r, c)) for r, c in ((qd, dim), (kvd, dim), (kvd, dim), (dim, qd))]
        self.norm = up(rng.uniform(0.5, 1.5, dim).astype(np.float32))
        self.qn = up(rng.uniform(0.5, 2.5, HD).astype(np.float32))
        self.kn = up(rng.uniform(0.5, 2.5, HD).astype(np.float32))
        ang = rng.uniform(0, 6.28, (max_seq, HD // 2))
        self.rope = up(np.stack([np.cos(ang), np.sin(ang)], -1))
        self.pack = torch.empty(self.L.mhip_attention_pack_bytes(ctypes.byref(self.a)),
                                dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        self.g.check(self.L.mhip_attention_pack(self.g.h, ctypes.byref(self.a),
                                                *[t.data_ptr() for t in self.w],
                                                self.pack.data_ptr()), "pack")

    def close(self):
        self.g.close()

    def cache(self, pos):
        """Rows 0 .. pos - 1 of a conversation, NaN after them."""
        c = np.full((2, self.max_seq, self.nkv * HD), np.nan, np.float32)
        c[:, :pos] = self.rng.standard_normal((2, pos, self.nkv * HD)).astype(np.float32)
        return self.up(c[0]), self.up(c[1])

    def args(self, kc, vc):
        return ([self.norm.data_ptr()] + [t.data_ptr() for t in self.w] +
                [self.qn.data_ptr(), self.kn.data_ptr(), self.rope.data_ptr(), kc.data_ptr(),
                 vc.data_ptr()])

    def batch(self, x, kc, vc, pos, packed=True, flags=0):
        t, n = self.torch, x.shape[0]
        nb = self.L.mhip_attention_batch_scratch_bytes(ctypes.byref(self.a), n, self.max_seq)
        scratch = t.full((nb,), 255, dtype=t.uint8, device="cuda")
        out = x.clone()
        t.cuda.synchronize()
        self.g.check(self.L.mhip_attention_batch(
            self.g.h, ctypes.byref(self.a), *self.args(kc, vc), pos, n, self.max_seq, out.data_ptr(),
            self.pack.data_ptr() if packed else None, scratch.data_ptr(), flags), "batch")
        t.cuda.synchronize()
        return out

    def token(self, x, kc, vc, pos):
        t = self.torch
        nb = self.L.mhip_attention_scratch_bytes(ctypes.byref(self.a), self.max_seq)
        scratch = t.zeros(nb, dtype=t.uint8, device="cuda")
        out = x.clone()
        t.cuda.synchronize()
        self.g.check(self.L.mhip_attention(self.g.h, ctypes.byref(self.a), *self.args(kc, vc), pos,
                                           self.max_seq, out.data_ptr(), None, scratch.data_ptr(), 0),
                     "token")
        t.cuda.synchronize()
        return out


def bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("nh,nkv", [(32, 4), (2, 2), (6, 2), (30, 3)])
@pytest.mark.parametrize("n,pos", [(1, 999), (2, 997), (2, 998), (16, 984), (17, 1024), (63, 961),
                                   (130, 1023), (249, 3), (250, 0), (257, 1)])
def test_batch_equals_tokens(n, pos, nh, nkv):
    torch = pytest.importorskip("torch")
    say("test_batch_equals_tokens n=%d pos=%d heads %d/%d" % (n, pos, nh, nkv))
    lay = Layer(torch, 256, nh, nkv, pos + n + 5, 7 * n + pos)
    try:
        kc, vc = lay.cache(pos)
        k2, v2 = kc.clone(), vc.clone()
        x = lay.up(lay.rng.standard_normal((n, 256)).astype(np.float32))
        got = lay.batch(x, kc.clone(), vc.clone(), pos, packed=False)
        want = torch.cat([lay.token(x[i:i + 1], k2, v2, pos + i) for i in range(n)])
        assert torch.isfinite(want).all()
        assert np.array_equal(bits(got), bits(want)), "vector rows"
        got = lay.batch(x, kc, vc, pos, flags=M.MHIP_FORCE_SEQ_RMS if n % 2 else 0)
        assert np.array_equal(bits(got), bits(want)), "matrix-core rows"
        assert np.array_equal(bits(kc[:pos + n]), bits(k2[:pos + n]))
        assert np.array_equal(bits(vc[:pos + n]), bits(v2[:pos + n]))
    finally:
        lay.close()


@pytest.mark.parametrize("nh,nkv,n,pos", [
    (4, 4, 64, 1000), (4, 4, 65, 1000), (8, 4, 128, 1000), (8, 4, 129, 1000), (8, 2, 384, 700),
    (8, 2, 385, 700), (1, 1, 1, 4607), (1, 1, 1, 4608), (4, 1, 2, 7486), (4, 1, 2, 7487)])
def test_batch_of_few_heads(n, pos, nh, nkv):
    """Few heads, in groups of one, two and four: a workgroup per token while
    all of them are resident at once, tiles from one token more; the longest
    contexts whose scores fit LDS, and the next."""
    torch = pytest.importorskip("torch")
    say("test_batch_of_few_heads n=%d pos=%d heads %d/%d" % (n, pos, nh, nkv))
    lay = Layer(torch, 256, nh, nkv, pos + n, n + pos)
    try:
        kc, vc = lay.cache(pos)
        k2, v2 = kc.clone(), vc.clone()
        x = lay.up(lay.rng.standard_normal((n, 256)).astype(np.float32))
        want = torch.cat([lay.token(x[i:i + 1], k2, v2, pos + i) for i in range(n)])
        assert torch.isfinite(want).all()
        for packed in (False, True):
            got = lay.batch(x, kc.clone(), vc.clone(), pos, packed=packed)
            assert np.array_equal(bits(got), bits(want)), packed
    finally:
        lay.close()


@pytest.mark.parametrize("n", [1, 15, 33, 64, 100, 511, 512, 577])
def test_batch_rows_on_matrix_cores(n):
    """The weight rows on the matrix cores, 32 (from 512 tokens 64) tokens to
    a workgroup in fragments of 16: dimensions of one and of several 64-row
    tiles, more blocks and fewer than the ring has stages."""
    torch = pytest.importorskip("torch")
    say("test_batch_rows_on_matrix_cores n=%d" % n)
    for dim, nh, nkv in ((64, 2, 1), (320, 8, 2)):
        lay = Layer(torch, dim, nh, nkv, n + 9, n)
        try:
            kc, vc = lay.cache(9)
            k2, v2 = kc.clone(), vc.clone()
            x = lay.up(lay.rng.standard_normal((n, dim)).astype(np.float32))
            got = lay.batch(x, kc, vc, 9)
            want = torch.cat([lay.token(x[i:i + 1], k2, v2, 9 + i) for i in range(n)])
            assert np.array_equal(bits(got), bits(want))
        finally:
            lay.close()


@pytest.mark.parametrize("n", [130, 131])
def test_batch_in_passes(n):
    """A context whose score matrix takes two passes (67 tokens of it fit the
    bounded scratch): of 65 tokens each, and of 66 and 65; every token."""
    torch = pytest.importorskip("torch")
    say("test_batch_in_passes n=%d" % n)
    pos = 60000
    lay = Layer(torch, 256, 32, 4, pos + n, 5)
    try:
        kc, vc = lay.cache(pos)
        x = lay.up(lay.rng.standard_normal((n, 256)).astype(np.float32))
        got = lay.batch(x, kc, vc, pos)
        for i in range(n):
            want = lay.token(x[i:i + 1], kc, vc, pos + i)
            assert np.array_equal(bits(got[i:i + 1]), bits(want)), "token %d" % i
    finally:
        lay.close()


def test_batch_with_infinities():
    """Values that make a token's own softmax or mix infinite or NaN stay
    with the tokens that read them: an infinite value row is read from its
    token on, not by the earlier tokens of the same tile."""
    torch = pytest.importorskip("torch")
    say("test_batch_with_infinities")
    n, pos = 40, 1005
    lay = Layer(torch, 256, 8, 2, pos + n, 21)
    try:
        kc, vc = lay.cache(pos)
        k2, v2 = kc.clone(), vc.clone()
        x = lay.rng.standard_normal((n, 256)).astype(np.float32)
        x[21] = np.inf
        x = lay.up(x)
        got = lay.batch(x, kc, vc, pos)
        want = torch.cat([lay.token(x[i:i + 1], k2, v2, pos + i) for i in range(n)])
        assert torch.isfinite(want[:21]).all()
        assert np.array_equal(bits(got[:21]), bits(want[:21]))
        assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    finally:
        lay.close()


@pytest.mark.parametrize("n,pos", [(5, 30), (40, 1000)])
def test_batch_on_unaligned_buffers(n, pos):
    """x and the value rows at a multiple of 4 bytes, the rotation angles at
    one of 8: what float and double pointers promise."""
    torch = pytest.importorskip("torch")
    say("test_batch_on_unaligned_buffers n=%d pos=%d" % (n, pos))
    lay = Layer(torch, 256, 8, 2, pos + n, n)
    try:
        kc, vc = lay.cache(pos)
        x = lay.up(lay.rng.standard_normal((n, 256)).astype(np.float32))
        k2, v2 = kc.clone(), vc.clone()
        want = lay.batch(x, k2, v2, pos)

        def shifted(t):
            b = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
            b[1:] = t.reshape(-1)
            return b

        xs, vs, rope = shifted(x), shifted(vc), shifted(lay.rope)
        nb = lay.L.mhip_attention_batch_scratch_bytes(ctypes.byref(lay.a), n, pos + n)
        scratch = torch.zeros(nb, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        args = lay.args(kc, vc)
        args[7], args[9] = rope[1:].data_ptr(), vs[1:].data_ptr()
        lay.g.check(lay.L.mhip_attention_batch(
            lay.g.h, ctypes.byref(lay.a), *args, pos, n, pos + n, xs[1:].data_ptr(),
            lay.pack.data_ptr(), scratch.data_ptr(), 0), "batch")
        torch.cuda.synchronize()
        assert np.array_equal(bits(xs[1:].reshape(n, 256)), bits(want))
        assert np.array_equal(bits(kc), bits(k2))
        assert np.array_equal(bits(vs[1:].reshape(vc.shape)), bits(v2))
    finally:
        lay.close()


def test_batch_refuses_null():
    """A missing buffer (the scratch of a failed allocation, say) is an error
    of the call, not a launch."""
    torch = pytest.importorskip("torch")
    say("test_batch_refuses_null")
    lay = Layer(torch, 256, 8, 2, 16, 3)
    try:
        kc, vc = lay.cache(4)
        x = lay.up(np.ones((2, 256), np.float32))
        nb = lay.L.mhip_attention_batch_scratch_bytes(ctypes.byref(lay.a), 2, 16)
        scratch = torch.zeros(nb, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        ptrs = lay.args(kc, vc)
        for miss in range(len(ptrs) + 2):
            p = [None if i == miss else v for i, v in enumerate(ptrs)]
            rc = lay.L.mhip_attention_batch(
                lay.g.h, ctypes.byref(lay.a), *p, 4, 2, 16,
                None if miss == len(ptrs) else x.data_ptr(), lay.pack.data_ptr(),
                None if miss == len(ptrs) + 1 else scratch.data_ptr(), 0)
            assert rc == -1 and b"null" in lay.L.mhip_error(lay.g.h), miss
    finally:
        lay.close()
