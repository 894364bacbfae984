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
