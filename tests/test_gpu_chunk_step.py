"""The chunk's Step 12 (ds4hip_session_chunk_step) at the edges of its tiles and
windows, against the token loop: sessions byte-identical (rows, keys, states,
last selection) after chunks of 1 to 128 tokens that start and end inside,
at and across compressor windows, with inputs that are not 16-byte aligned;
and the calls it refuses."""
import ctypes as C

import numpy as np
import pytest
import torch

from ds4cuda_amd import Ds4HipError, session, synth
from ds4cuda_amd._lib import call
from ds4cuda_amd.chunk import forward_chunk_attn
from ds4cuda_amd.ops import _ptr, _stream
from test_gpu_chunk import EMBD, HD, NH, layer_bytes, layer_weights, one_token, token_inputs

pytestmark = pytest.mark.gpu


# (layer, tokens before the chunk, chunk); ratio 4: il 2, ratio 128: il 3
@pytest.mark.parametrize("il,hist,n", [(2, 0, 1), (2, 3, 1), (2, 5, 2), (2, 6, 16), (2, 31, 17), (2, 33, 32),
                                       (2, 40, 33), (2, 9, 128), (3, 0, 128), (3, 100, 128), (3, 127, 1), (3, 126, 5)])
def test_chunk_step_matches_token_loop(gpu, il, hist, n):
    layer = layer_weights(il, gpu)
    sinks = torch.from_numpy(synth.normal(310, il, NH)).to(gpu)
    out1 = torch.empty(NH * HD, device=gpu)
    a, b = session.Session(512), session.Session(512)
    try:
        for pos in range(hist):
            one_token(a, il, pos, layer, sinks, out1, gpu)
            one_token(b, il, pos, layer, sinks, out1, gpu)
        ins = [token_inputs(il, hist + t, gpu) for t in range(n)]

        def stack(k, odd):   # odd: the buffer starts one element into its allocation
            v = torch.stack([x[k] for x in ins])
            if not odd:
                return v
            buf = torch.empty(v.numel() + 1, device=gpu)
            buf[1:] = v.reshape(-1)
            return buf[1:].view(v.shape)

        odd = n % 2 == 1
        out = torch.empty((n, NH, HD), device=gpu)
        forward_chunk_attn(a, il, hist, stack(0, odd), stack(1, odd), stack(2, False).reshape(n, NH, HD), stack(3, False),
                           sinks, out, layer=layer)
        for t in range(n):
            one_token(b, il, hist + t, layer, sinks, out1, gpu)
        torch.cuda.synchronize()
        # the last token's attention: the same rows, another split (test_gpu_chunk's bound)
        ref = out1.cpu().numpy()
        assert np.abs(out[-1].cpu().numpy().reshape(-1) - ref).max() < 1e-4 * np.sqrt(np.mean(ref.astype(np.float64) ** 2))
        (ra, ca), (rb, cb) = layer_bytes(a, il), layer_bytes(b, il)
        assert ca == cb
        for x, y in zip(ra, rb):
            assert np.array_equal(x, y)
    finally:
        a.close()
        b.close()


def test_chunk_step_refuses_what_does_not_fit(gpu):
    il = 2
    layer = layer_weights(il, gpu)
    s = session.Session(256)
    try:
        L = s.layer(il)
        L.n_comp = L.cap_comp          # no room for an emitted row
        before = layer_bytes(s, il)
        x = torch.zeros((8, EMBD), device=gpu)
        args = (torch.zeros((8, 1024), device=gpu), torch.zeros((8, NH, HD), device=gpu), torch.zeros((8, HD), device=gpu),
                torch.zeros(NH, device=gpu), torch.empty((8, NH, HD), device=gpu))
        with pytest.raises(Ds4HipError) as e:
            forward_chunk_attn(s, il, 0, x, *args, layer=layer)
        assert e.value.code == -28
        after = layer_bytes(s, il)
        assert before[1] == after[1] and all(np.array_equal(p, q) for p, q in zip(before[0], after[0]))
    finally:
        s.close()


# 600 keys in a session that could hold more than the 16384 the tokens select
# over together, the limit crossed inside the chunk, and beyond it throughout
@pytest.mark.parametrize("n_keys", [600, 16382, 16400])
def test_chunk_step_in_a_large_session(gpu, n_keys):
    il, hist, n = 2, 2, 24
    layer = layer_weights(il, gpu)
    sinks = torch.from_numpy(synth.normal(310, il, NH)).to(gpu)
    keys = torch.from_numpy(synth.normal(320, n_keys, n_keys * 128)).to(gpu)
    rows = torch.from_numpy(synth.kv_rows(321, n_keys, n_keys)).to(gpu)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    a, b = session.Session(66000), session.Session(66000)
    try:
        for s in (a, b):
            L = s.layer(il)
            assert L.cap_comp > 16400 + hist + n
            call("ds4hip_fp8_kv_quantize_append", _ptr(rows), n_keys, HD, 64, C.c_void_p(s.s.codes),
                 C.c_void_p(s.s.sexp), C.c_void_p(s.s.tail), C.c_longlong(L.row_base), None, _stream(None))
            assert hip.hipMemcpy(L.index_comp_kv, keys.data_ptr(), n_keys * 128 * 4, 3) == 0
            L.n_comp = L.n_index_comp = n_keys
        out1 = torch.empty(NH * HD, device=gpu)
        for pos in range(hist):
            one_token(a, il, pos, layer, sinks, out1, gpu)
            one_token(b, il, pos, layer, sinks, out1, gpu)
        ins = [token_inputs(il, hist + t, gpu) for t in range(n)]
        stack = lambda k: torch.stack([x[k] for x in ins])
        out = torch.empty((n, NH, HD), device=gpu)
        forward_chunk_attn(a, il, hist, stack(0), stack(1), stack(2).reshape(n, NH, HD), stack(3), sinks, out,
                           layer=layer, exact_p=True)
        for t in range(n):
            one_token(b, il, hist + t, layer, sinks, out1, gpu)
            ref = out1.cpu().numpy()   # the same rows, another split (test_gpu_chunk's bound)
            err = np.abs(out[t].cpu().numpy().reshape(-1) - ref).max()
            assert err < 1e-4 * np.sqrt(np.mean(ref.astype(np.float64) ** 2)), t
        (ra, ca), (rb, cb) = layer_bytes(a, il), layer_bytes(b, il)
        assert ca == cb
        for x, y in zip(ra, rb):
            assert np.array_equal(x, y)
    finally:
        a.close()
        b.close()
