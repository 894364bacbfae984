"""The flat-stage decode on both sides of the rule that drops its copy ring:
row counts whose chunks are one, two, three tiles (no ring) and four, for
direct rows, row lists and pages, bf16 and fp32 queries; and a batch of
problems whose segments share chunks. Against the oracle at the decode tests'
bar (2e-3 x RMS: weights rounded to f16 at 2^-11 each)."""
import numpy as np
import pytest
import torch

import oracle as O
from ds4cuda_amd import ops, synth
from test_gpu_decode import check, make_cache, q_bf16, sinks_for

pytestmark = pytest.mark.gpu


# 256 workgroups of whole tiles: 8192 rows in one-tile chunks, 24576 in three
@pytest.mark.parametrize("n", [1, 33, 8192, 8193, 16385, 24576, 24577])
@pytest.mark.parametrize("form", ["direct", "list", "pages"])
@pytest.mark.parametrize("q_f32", [False, True])
def test_chunk_edges(gpu, n, form, q_f32):
    n_rows = 25600
    cache, (codes, sexp, tail) = make_cache(n_rows, 61, gpu)
    rng = np.random.default_rng(n)
    pt = rng.permutation(n_rows // 256).astype(np.int32)
    idx = np.sort(rng.choice(n_rows, n, replace=False)).astype(np.int32)
    bits, qf = q_bf16(62, 1)
    if q_f32:
        qf = synth.normal(62, 5, 64 * 512).reshape(1, 64, 512) * 2.0
    sinks = sinks_for(63, 1)
    out = torch.full((1, 64, 512), float("nan"), device=gpu)
    q = (torch.from_numpy(qf).to(gpu) if q_f32 else torch.from_numpy(bits.view(np.int16)).to(gpu).view(torch.bfloat16))
    kw = {}
    phys = np.arange(n)
    if form == "list":
        kw, phys = {"row_idx": torch.from_numpy(idx[None]).to(gpu)}, idx
    elif form == "pages":
        kw, phys = {"page_table": torch.from_numpy(pt[None]).to(gpu), "page_rows": 256}, pt[phys // 256] * 256 + phys % 256
    ops.flash_attn_decode_fp8(q, torch.from_numpy(sinks).to(gpu), out, cache, [n], **kw)
    torch.cuda.synchronize()
    check(out[0].cpu().numpy(), O.attn_decode_fp8(qf[0], codes, sexp, tail, phys, sinks[0]))


@pytest.mark.parametrize("counts", [[5, 0, 40, 31, 200] * 20, [200] * 100, [1] * 128])
def test_segments_share_chunks(gpu, counts):
    n = len(counts)
    cache, (codes, sexp, tail) = make_cache(max(sum(counts), 1), 71, gpu)
    base = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int64)
    qf = synth.normal(72, 2, n * 64 * 512).reshape(n, 64, 512) * 2.0
    sinks = sinks_for(73, n)
    out = torch.full((n, 64, 512), float("nan"), device=gpu)
    ops.flash_attn_decode_fp8(torch.from_numpy(qf).to(gpu), torch.from_numpy(sinks).to(gpu), out, cache, counts,
                              row_base=torch.from_numpy(base).to(gpu))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for p in range(0, n, 7):
        if counts[p] == 0:
            assert (got[p] == 0).all()
        else:
            check(got[p], O.attn_decode_fp8(qf[p], codes, sexp, tail, base[p] + np.arange(counts[p]), sinks[p]))


# more than eight chunks a problem (the wide merge) and fewer, on both sides of
# the problem counts from which the slots are read one by one
@pytest.mark.parametrize("n,rows", [(12, 1200), (13, 1200), (31, 300), (32, 300)])
def test_merge_forms(gpu, n, rows):
    cache, (codes, sexp, tail) = make_cache(n * rows, 74, gpu)
    bits, qf = q_bf16(75, n)
    sinks = sinks_for(76, n)
    out = torch.full((n, 64, 512), float("nan"), device=gpu)
    q = torch.from_numpy(bits.view(np.int16)).to(gpu).view(torch.bfloat16)
    ops.flash_attn_decode_fp8(q, torch.from_numpy(sinks).to(gpu), out, cache, [rows] * n, row_base_stride=rows)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for p in (0, n // 2, n - 1):
        check(got[p], O.attn_decode_fp8(qf[p], codes, sexp, tail, p * rows + np.arange(rows), sinks[p]))
