"""Prefill of small chunks (each pair's keys split over workgroups and merged)
and of rows that outgrow the first pass's reference, against the oracle: the
part counts' edges (one part, two, the most, pairs with fewer tiles than
parts), odd query counts, and a row maximum in the last tile."""
import numpy as np
import pytest
import torch

from ds4cuda_amd import synth
from test_gpu_decode import check, make_cache, q_bf16, sinks_for
from test_gpu_prefill import oracle_prefill, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("outlier", [0.0, 0.02])
@pytest.mark.parametrize("exact_p", [False, True])
@pytest.mark.parametrize("n_cached,n_q", [(127, 1), (255, 1), (2100, 3), (8200, 2), (600, 31), (250, 255), (250, 258)])
def test_prefill_split(gpu, n_cached, n_q, exact_p, outlier):
    cache, (codes, sexp, tail) = make_cache(n_cached + n_q, 31 + n_q, gpu, outlier=outlier)
    bits, qf = q_bf16(32, n_q)
    sinks = sinks_for(33, 1)[0]
    got = run(gpu, cache, bits, sinks, n_q, n_cached, exact_p=exact_p)
    ref = oracle_prefill(qf, codes, sexp, tail, n_cached, sinks)
    for t in range(n_q):
        check(got[t], ref[t])


@pytest.mark.parametrize("n_cached,n_q", [(1000, 2), (400, 270)])
def test_prefill_late_maximum(gpu, n_cached, n_q):
    # the last cached row draws all of query 0's attention: its score outgrows
    # every reference by far more than the first pass allows
    from ds4cuda_amd import ops
    bits, qf = q_bf16(35, n_q)
    x = synth.kv_rows(34, 0, n_cached + n_q)
    x[n_cached - 1] = 6.0 * qf[0, 5]
    cache = ops.Fp8KVCache.empty(n_cached + n_q, device=gpu)
    cache.append(torch.from_numpy(x).to(gpu))
    torch.cuda.synchronize()
    codes, sexp = cache.codes.cpu().numpy(), cache.sexp.cpu().numpy()
    tail = cache.tail.cpu().numpy().view(np.uint16)
    sinks = sinks_for(36, 1)[0]
    got = run(gpu, cache, bits, sinks, n_q, n_cached)
    ref = oracle_prefill(qf, codes, sexp, tail, n_cached, sinks)
    for t in range(n_q):
        check(got[t], ref[t])


def test_prefill_workspace_of_another_size(gpu):
    """A workspace sized for a large chunk serves a small one (split), and one
    with room for the flags alone (four bytes a pair) runs it unsplit: the same outputs."""
    import ctypes as C

    from ds4cuda_amd._lib import lib
    from ds4cuda_amd.ops import _ptr, _stream
    n_cached, n_q = 900, 5
    size = lib().ds4hip_flash_attn_prefill_fp8_workspace_size
    assert all(size(a) <= size(b) for a, b in ((1, 2), (5, 300), (300, 511), (511, 513), (513, 4096)))
    cache, (codes, sexp, tail) = make_cache(n_cached + n_q, 41, gpu)
    bits, qf = q_bf16(42, n_q)
    sinks = sinks_for(43, 1)[0]
    ref = oracle_prefill(qf, codes, sexp, tail, n_cached, sinks)
    q = torch.from_numpy(bits.view(np.int16)).to(gpu).view(torch.bfloat16)
    s = torch.from_numpy(np.ascontiguousarray(sinks, np.float32)).to(gpu)
    for nb, rc in ((size(4096), 0), (3 * 516 + 512, 0), (12, 0), (11, -22)):
        out = torch.full((n_q, 64, 512), float("nan"), device=gpu)
        ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
        assert lib().ds4hip_flash_attn_prefill_fp8(
            _ptr(q), _ptr(s), _ptr(out), _ptr(cache.codes), _ptr(cache.sexp), _ptr(cache.tail), n_q, n_cached, 64, 512,
            64, _ptr(ws), C.c_size_t(nb), 0, _stream(None)) == rc
        torch.cuda.synchronize()
        if rc == 0:
            for t in range(n_q):
                check(out[t].cpu().numpy(), ref[t])


@pytest.mark.parametrize("n_cached,n_q", [(1000, 3), (400, 259)])
def test_prefill_late_maximum_with_flags_only(gpu, n_cached, n_q):
    """The smallest workspace holds no row maxima: a pair that the first pass
    gives up is redone all the same, here the first and (odd) last ones."""
    import ctypes as C

    from ds4cuda_amd import ops
    from ds4cuda_amd._lib import lib
    from ds4cuda_amd.ops import _ptr, _stream
    bits, qf = q_bf16(45, n_q)
    x = synth.kv_rows(44, 0, n_cached + n_q)
    x[n_cached - 1] = 6.0 * qf[0, 5]
    x[n_cached - 2] = 6.0 * qf[n_q - 1, 60]
    cache = ops.Fp8KVCache.empty(n_cached + n_q, device=gpu)
    cache.append(torch.from_numpy(x).to(gpu))
    sinks = sinks_for(46, 1)[0]
    q = torch.from_numpy(bits.view(np.int16)).to(gpu).view(torch.bfloat16)
    s = torch.from_numpy(np.ascontiguousarray(sinks, np.float32)).to(gpu)
    out = torch.full((n_q, 64, 512), float("nan"), device=gpu)
    ws = torch.empty(4 * ((n_q + 1) // 2), dtype=torch.uint8, device=gpu)
    assert lib().ds4hip_flash_attn_prefill_fp8(
        _ptr(q), _ptr(s), _ptr(out), _ptr(cache.codes), _ptr(cache.sexp), _ptr(cache.tail), n_q, n_cached, 64, 512, 64,
        _ptr(ws), C.c_size_t(ws.numel()), 0, _stream(None)) == 0
    torch.cuda.synchronize()
    ref = oracle_prefill(qf, cache.codes.cpu().numpy(), cache.sexp.cpu().numpy(),
                         cache.tail.cpu().numpy().view(np.uint16), n_cached, sinks)
    for t in range(n_q):
        check(out[t].cpu().numpy(), ref[t])


# one part and several; the infinite rows: the first tile, and more than a part
@pytest.mark.parametrize("exact_p", [False, True])
@pytest.mark.parametrize("n_cached,n_q,n_inf", [(400, 260, 32), (1000, 2, 32), (1000, 5, 300), (1000, 2, 33)])
def test_prefill_infinite_rows(gpu, n_cached, n_q, n_inf, exact_p):
    """Rows that are +inf in one dim score -inf for the heads whose query is
    negative there: they take no weight, and only that dim of the output, where
    0 * inf is NaN, shows them."""
    cache, (codes, sexp, tail) = make_cache(n_cached + n_q, 51, gpu)
    cache.tail[:n_inf, 7] = 0x7C00
    bits, qf = q_bf16(52, n_q)
    sinks = sinks_for(53, 1)[0]
    got = run(gpu, cache, bits, sinks, n_q, n_cached, exact_p=exact_p)
    ref = oracle_prefill(qf, codes[n_inf:], sexp[n_inf:], tail[n_inf:], n_cached - n_inf, sinks)
    rest = np.arange(512) != 448 + 7
    for t in range(n_q):
        neg = qf[t, :, 448 + 7] < 0
        assert np.isnan(got[t][neg][:, 448 + 7]).all()
        check(got[t][neg][:, rest], ref[t][neg][:, rest])
