"""The fp32-row decode at the edges of its chunks and of the rule that shares a
chunk between workgroups: row counts around one tile and around the last count
that is shared, K and V in one buffer and in two, masked rows that hold NaN,
and workspaces sized for another row count."""
import ctypes as C

import numpy as np
import pytest
import torch

from ds4cuda_amd import ops, synth

pytestmark = pytest.mark.gpu


def reference(q, k, v, sinks):
    """fp64 softmax attention with a sink per head over f16-rounded rows."""
    k, v = (x.astype(np.float16).astype(np.float64) for x in (k, v))
    s = q.astype(np.float64) @ k.T / np.sqrt(512.0)
    m = np.maximum(s.max(1), sinks)
    p = np.exp(s - m[:, None])
    return (p @ v) / (p.sum(1) + np.exp(sinks - m))[:, None]


def check(got, ref):
    # one-f16 P: weights within 2^-11 (the decode tests' bar)
    assert np.abs(got - ref).max() <= 2e-3 * np.sqrt(np.mean(ref ** 2))


def inputs(n, seed):
    return (synth.normal(seed, 1, 64 * 512).reshape(64, 512), synth.normal(seed, 2, n * 512).reshape(n, 512),
            synth.normal(seed, 3, n * 512).reshape(n, 512), synth.normal(seed, 4, 64))


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 200, 4096, 4097, 9001])
def test_raw_rows(gpu, n, two):
    q, k, v, sinks = inputs(n, 80 + n)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    kt = t(k)
    out = torch.full((64, 512), float("nan"), device=gpu)
    ops.launch_flash_attn_decode_raw_f32(t(q), kt, t(v) if two else kt, t(sinks), out, 64, n, 512)
    torch.cuda.synchronize()
    check(out.cpu().numpy(), reference(q, k, v if two else k, sinks.astype(np.float64)))


@pytest.mark.parametrize("n_raw,n_comp", [(0, 40), (5, 27), (128, 1025), (100, 4200)])
def test_masked_rows_hold_nan(gpu, n_raw, n_comp):
    q, k, _, sinks = inputs(n_raw + n_comp, 90 + n_comp)
    allowed = (synth.uniform(91, n_comp, n_comp) < 0.5).astype(np.int32)
    allowed[0] = 1
    dev = k.copy()
    dev[n_raw:][allowed == 0] = np.nan
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    out = torch.full((64, 512), float("nan"), device=gpu)
    ops.launch_flash_attn_decode_mixed_f32(t(q), t(dev[:n_raw]) if n_raw else t(dev[:1]), t(dev[n_raw:]), t(allowed),
                                           t(sinks), out, 64, n_raw, n_comp, 512)
    torch.cuda.synchronize()
    keep = np.concatenate([np.ones(n_raw, bool), allowed.astype(bool)])
    check(out.cpu().numpy(), reference(q, k[keep], k[keep], sinks.astype(np.float64)))


def test_workspace_sized_for_another_row_count(gpu):
    from ds4cuda_amd._lib import lib
    from ds4cuda_amd.ops import _ptr, _stream
    n = 8192
    q, k, _, sinks = inputs(n, 99)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    qt, kt, st = t(q), t(k), t(sinks)
    two_tile = (n // 64) * (64 * 512 * 4 + 2 * 64 * 4) + (n // 64) * 4 + 256 * 4   # 128 chunks of 64 rows
    own = C.c_size_t(0)
    assert lib().ds4hip_flash_attn_decode_f32_workspace_size(C.c_longlong(n), C.byref(own)) == 0
    for nb, rc in ((own.value, 0), (two_tile, 0), (two_tile // 2, -22)):
        out = torch.full((64, 512), float("nan"), device=gpu)
        ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
        assert lib().ds4hip_flash_attn_decode_raw_f32_prealloc(_ptr(qt), _ptr(kt), _ptr(kt), _ptr(st), _ptr(out), 64, n,
                                                              512, _ptr(ws), C.c_size_t(nb), _stream(None)) == rc
        torch.cuda.synchronize()
        if rc == 0:
            check(out.cpu().numpy(), reference(q, k, k, sinks.astype(np.float64)))


def chunked_f16_p(q, k, sinks, rows):
    """The decode's rounding in fp64: chunks of `rows` rows in tiles of 32, P as
    one f16 relative to the chunk's maximum so far, l of the unrounded P."""
    k = k.astype(np.float16).astype(np.float64)
    s = q.astype(np.float64) @ k.T / np.sqrt(512.0) * np.log2(np.e)
    parts = []
    for c in range(0, len(k), rows):
        m, l, o = np.full(64, -np.inf), np.zeros(64), np.zeros((64, 512))
        for t in range(c, min(c + rows, len(k)), 32):
            st = s[:, t:min(t + 32, c + rows)]
            m_new = np.maximum(m, st.max(1))
            p, a = np.exp2(st - m_new[:, None]), np.exp2(m - m_new)
            o = o * a[:, None] + p.astype(np.float16).astype(np.float64) @ k[t:t + st.shape[1]]
            l, m = l * a + p.sum(1), m_new
        parts.append((m, l, o))
    top = np.maximum(np.max([m for m, _, _ in parts], 0), sinks * np.log2(np.e))
    w = [np.exp2(m - top) for m, _, _ in parts]
    den = sum(x * l for x, (_, l, _) in zip(w, parts)) + np.exp2(sinks * np.log2(np.e) - top)
    return sum(x[:, None] * o for x, (_, _, o) in zip(w, parts)) / den[:, None]


@pytest.mark.parametrize("n", [200, 1153, 4000, 8192])
def test_rounding_of_two_tile_chunks(gpu, n):
    """Where the chunks are cut is part of the result: the outputs are those of
    two-tile chunks, not of one-tile ones."""
    q, k, _, sinks = inputs(n, 60 + n)
    q = 2.0 * q
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    kt = t(k)
    out = torch.full((64, 512), float("nan"), device=gpu)
    ops.launch_flash_attn_decode_raw_f32(t(q), kt, kt, t(sinks), out, 64, n, 512)
    torch.cuda.synchronize()
    s64 = sinks.astype(np.float64)
    two, one = chunked_f16_p(q, k, s64, 64), chunked_f16_p(q, k, s64, 32)
    rel = lambda a, b: np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
    # fp32 sums of 512 products move a score by about 1e-6, and with it an output
    # by less than 3e-6, except where a weight crosses an f16 midpoint (2^-11 of
    # that weight): so most heads, not all. The other cut moves half of them or more.
    got = out.cpu().numpy()
    assert np.median(rel(one, two)) > 2e-5
    assert np.percentile(rel(got, two), 40) <= 3e-6


# 4096 rows: the last count whose chunks are shared; tiles without an allowed row
@pytest.mark.parametrize("n_raw,n_comp", [(128, 1025), (128, 3968), (128, 3969), (0, 9000)])
def test_sparse_mask(gpu, n_raw, n_comp):
    q, k, _, sinks = inputs(n_raw + n_comp, 70 + n_comp)
    allowed = (synth.uniform(71, n_comp, n_comp) < 0.01).astype(np.int32)
    allowed[-1] = 1
    dev = k.copy()
    dev[n_raw:][allowed == 0] = np.inf
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    out = torch.full((64, 512), float("nan"), device=gpu)
    ops.launch_flash_attn_decode_mixed_f32(t(q), t(dev[:n_raw]) if n_raw else t(dev[:1]), t(dev[n_raw:]), t(allowed),
                                           t(sinks), out, 64, n_raw, n_comp, 512)
    torch.cuda.synchronize()
    keep = np.concatenate([np.ones(n_raw, bool), allowed.astype(bool)])
    check(out.cpu().numpy(), reference(q, k[keep], k[keep], sinks.astype(np.float64)))
