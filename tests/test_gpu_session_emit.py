"""ds4hip_session_emit_f32 against the calls it stands for
(ds4hip_compressor_emit_f32 per compressor and the two pushes): arenas,
emitted row and counters bit for bit on a ratio-4 and a ratio-128 layer, from
an empty layer and into the last free row; eager and replayed from a graph.
And the calls it refuses, which change nothing."""
import ctypes as C

import numpy as np
import pytest
import torch

from ds4cuda_amd import Ds4HipError, session, token
from ds4cuda_amd._lib import call
from ds4cuda_amd.ops import _ptr, _stream
from test_gpu_token import arena

pytestmark = pytest.mark.gpu

CTX = 512


def separate(s, il, pos, wc, wi, emit, emit_i):
    L, r = s.layer(il), s.layer(il).compress_ratio
    call("ds4hip_compressor_emit_f32", 1, _ptr(wc), 512, r, pos, il, C.c_void_p(L.attn_state_kv),
         C.c_void_p(L.attn_state_score), _ptr(emit), _stream(None))
    s.push_comp(il, emit)
    if L.has_indexer:
        call("ds4hip_compressor_emit_f32", 0, _ptr(wi), 128, r, pos, il, C.c_void_p(L.index_state_kv),
             C.c_void_p(L.index_state_score), _ptr(emit_i), _stream(None))
        s.push_index_comp(il, emit_i)


def one(s, il, pos, wc, wi, emit):
    call("ds4hip_session_emit_f32", C.byref(s.s), il, pos, _ptr(wc), _ptr(wi), _ptr(emit), _stream(None))


# (layer, tokens of history, position): an empty layer, an ordinary step, the last row that fits
@pytest.mark.parametrize("il,hist,pos", [(2, 0, 3), (42, 383, 383), (2, -1, 2047), (3, 0, 127), (41, 255, 255), (3, -1, 639)])
def test_emit_matches_separate_launches(gpu, il, hist, pos):
    g = torch.Generator(device=gpu).manual_seed(7 + il + pos)
    wc, wi = (1 + 0.1 * torch.randn(n, generator=g, device=gpu) for n in (512, 128))
    ea, ei = torch.empty(512, device=gpu), torch.empty(128, device=gpu)
    sessions = [session.Session(CTX) for _ in range(3)]
    a, b, c = sessions
    try:
        for s in sessions:
            token.fill_history(s, max(hist, 0) or 300)
            L = s.layer(il)
            if hist <= 0:                 # the counters at the ends of the range
                L.n_comp = 0 if hist == 0 else L.cap_comp - 1
                L.n_index_comp = L.n_comp if L.has_indexer else 0
        separate(a, il, pos, wc, wi, ea, ei)
        eb, ec = torch.empty(512, device=gpu), torch.empty(512, device=gpu)
        one(b, il, pos, wc, wi if b.layer(il).has_indexer else None, eb)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            one(c, il, pos, wc, wi, ec)
        graph.replay()
        torch.cuda.synchronize()
        ref = arena(a)
        for s, e in ((b, eb), (c, ec)):
            assert torch.equal(ea.view(torch.int32), e.view(torch.int32)) and torch.isfinite(e).all()
            assert np.array_equal(ref, arena(s))
            assert (s.layer(il).n_comp, s.layer(il).n_index_comp) == (a.layer(il).n_comp, a.layer(il).n_index_comp)
    finally:
        for s in sessions:
            s.close()


def test_emit_refuses(gpu):
    s = session.Session(CTX)
    w, e = torch.ones(512, device=gpu), torch.empty(512, device=gpu)
    try:
        def code(*a):
            with pytest.raises(Ds4HipError) as x:
                one(s, *a)
            return x.value.code

        before = arena(s)
        assert code(0, 3, w, w, e) == -22            # no compressor
        assert code(43, 3, w, w, e) == -22
        assert code(2, 2, w, w, e) == -22            # inside a window
        assert code(2, -1, w, w, e) == -22
        assert code(2, 3, w, None, e) == -22         # the indexer's norm is missing
        assert code(3, 127, w, w, None) == -22
        L = s.layer(2)
        L.n_comp = L.cap_comp
        assert code(2, 3, w, w, e) == -28
        L.n_comp, L.n_index_comp = 0, L.cap_comp
        assert code(2, 3, w, w, e) == -28
        assert (L.n_comp, L.n_index_comp) == (0, L.cap_comp)
        assert np.array_equal(before, arena(s))
    finally:
        s.close()
