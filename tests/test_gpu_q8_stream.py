"""The streamed Q8_0 matvec (rows of 32 and 128 blocks) at the edges of its
waves and workgroups: against the oracle, and bit for bit against the
one-wave-per-row kernel, which weights off a 16-byte boundary take."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from ds4cuda_amd import ops, synth
from oracle import P
from test_oracle_misc import q8_pack

pytestmark = pytest.mark.gpu


def aligned_and_not(a, gpu, shift):
    """a on the GPU at its own address and `shift` bytes past an allocation's start."""
    t = torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).to(gpu)
    buf = torch.empty(t.numel() + shift, dtype=torch.uint8, device=gpu)
    buf[shift:] = t
    return t, buf[shift:]


@pytest.mark.parametrize("n_rows,n_cols", [(16, 1024), (48, 1024), (80, 1024), (17, 1024), (4, 4096), (20, 4096),
                                           (18, 4096), (32, 2048), (6, 8192)])
def test_q8_matvec(gpu, n_rows, n_cols):
    W, _, _ = q8_pack(synth.normal(71, n_rows, n_rows * n_cols).reshape(n_rows, n_cols) * 0.02)
    x = synth.normal(72, n_cols, n_cols)
    x[64:96] = 0.0   # an all-zero block
    ref = np.zeros(n_rows, np.float32)
    O.lib().orc_q8_matvec(P(np.ascontiguousarray(W)), P(x), P(ref), C.c_int(n_rows), C.c_int(n_cols))
    xq = torch.empty(n_cols, dtype=torch.int8, device=gpu)
    xs = torch.empty(n_cols // 32, device=gpu)
    got = []
    for w in aligned_and_not(W, gpu, 4):
        y = torch.full((n_rows,), float("nan"), device=gpu)
        ops.launch_mul_mv_q8_0_q8_0_f32_prealloc(w, torch.from_numpy(x).to(gpu), y, n_rows, n_cols, xq, xs)
        torch.cuda.synchronize()
        got.append(y.cpu().numpy())
    # int32 block dots are exact; the fp32 sums of n_cols / 32 terms differ by their rounding
    assert np.abs(got[0] - ref).max() <= 1e-5 * np.sqrt(np.mean(ref.astype(np.float64) ** 2))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


@pytest.mark.parametrize("rank,out_dim", [(32, 32), (1024, 64)])
def test_attn_out_projections(gpu, rank, out_dim):
    """The grouped projection with its output's quantization, then the dense one."""
    groups, heads, dim = 8, 64, 512
    a, _, _ = q8_pack(synth.normal(73, rank, groups * rank * 4096).reshape(groups * rank, 4096) * 0.02)
    b, _, _ = q8_pack(synth.normal(74, rank, out_dim * groups * rank).reshape(out_dim, groups * rank) * 0.02)
    kqv = torch.from_numpy(synth.normal(75, rank, heads * dim)).to(gpu)
    out = []
    for wa, wb in zip(aligned_and_not(a, gpu, 4), aligned_and_not(b, gpu, 4)):
        y = torch.full((out_dim,), float("nan"), device=gpu)
        ops.attn_out_decode_f32(kqv, wa, wb, y, heads, dim, 64, 77, 2, groups, rank, out_dim)
        torch.cuda.synchronize()
        out.append(y.cpu().numpy())
    assert np.isfinite(out[0]).all() and np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


def test_qkv_weights_off_16_bytes(gpu):
    g = lambda s, r, c, k: q8_pack(synth.normal(76, s, r * c).reshape(r, c) * k)[0]
    ws = {"q_a": g(1, 1024, 4096, 0.02), "kv_a": g(2, 512, 4096, 0.02), "q_b": g(3, 32768, 1024, 0.03)}
    x = torch.from_numpy(synth.normal(77, 1, 4096)).to(gpu)
    n1, n2 = (torch.from_numpy(1 + 0.1 * synth.normal(78, n, n)).to(gpu) for n in (1024, 512))
    pairs = {k: aligned_and_not(v, gpu, 4) for k, v in ws.items()}
    res = []
    for i in range(2):
        o = [torch.full((n,), float("nan"), device=gpu) for n in (1024, 32768, 512)]
        ops.attn_qkv_decode_f32(x, pairs["q_a"][i], n1, pairs["kv_a"][i], n2, pairs["q_b"][i], 4097, 2, *o)
        torch.cuda.synchronize()
        res.append([v.cpu().numpy().view(np.uint32) for v in o])
    for a, b in zip(*res):
        assert np.array_equal(a, b)
