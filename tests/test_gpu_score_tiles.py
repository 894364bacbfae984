"""The matrix-core indexer scorer at the edges of its tiles, bit for bit
against the oracle: key counts around the 16-key tile and the one- and
two-tile workgroups, head counts around a wave's 16 and the reference's 32,
every key type, and key / query bases that are not 16-byte aligned."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from ds4cuda_amd import ops, synth
from oracle import P

pytestmark = pytest.mark.gpu

TYPES = [torch.float32, torch.float16, torch.bfloat16]


@pytest.mark.parametrize("n_comp,n_head,kind,shift", [
    (1, 64, 0, 0), (2, 1, 2, 0), (15, 16, 1, 0), (16, 17, 0, 0), (17, 33, 2, 0), (33, 64, 1, 0),
    (500, 64, 0, 1), (513, 48, 2, 1), (514, 31, 1, 1), (16385, 64, 2, 0), (16403, 40, 0, 0), (33000, 64, 1, 0)])
def test_score_tiles_bit_exact(gpu, n_comp, n_head, kind, shift):
    top_k = max(1, n_comp // 3)
    q = synth.normal(61, 1, n_head * 128 + 1)
    w = synth.normal(61, 2, n_head)
    kf = synth.normal(61, 3, n_comp * 128 + 1)
    kf[5::97] = 0.0
    kt = torch.from_numpy(kf).to(TYPES[kind])
    # shift: the buffers start one element into their allocations
    key_dev = kt.to(gpu)[shift:shift + n_comp * 128].view(n_comp, 128)
    q_dev = torch.from_numpy(q).to(gpu)[shift:shift + n_head * 128]
    keys = kt[shift:shift + n_comp * 128].view(torch.float32 if kind == 0 else torch.int16).numpy().copy()
    qh = q[shift:shift + n_head * 128].copy()
    ref = np.zeros(n_comp, np.float32)
    O.lib().orc_indexer_scores(P(qh), P(w), P(keys), C.c_int(kind), C.c_int(n_comp), C.c_int(n_head),
                               C.c_int(128), P(ref))
    ref_pos = np.zeros(top_k, np.int32)
    O.lib().orc_topk_positions(P(ref), C.c_int(n_comp), C.c_int(top_k), C.c_int(0), P(ref_pos))
    # both forms: the positions' own (small or large), and the mask's with the fused histogram
    mask = torch.empty(n_comp, dtype=torch.int32, device=gpu)
    for m in (None, mask):
        pos, _, scores = ops.indexer_topk_positions(q_dev, torch.from_numpy(w).to(gpu), key_dev, top_k, 0, mask=m)
        torch.cuda.synchronize()
        assert np.array_equal(scores.cpu().numpy().view(np.uint32), ref.view(np.uint32))
        assert np.array_equal(pos.cpu().numpy(), ref_pos)
    assert np.array_equal(np.flatnonzero(mask.cpu().numpy()), ref_pos)


# the query, the keys and what they bring out: products and sums below the
# normal range, sums that cancel to a small part of their terms, overflow
SPECIAL = {
    "subnormal products": lambda q, k: (q * 1e-20, k * 1e-20),
    "subnormal keys": lambda q, k: (q, k * 1e-39),
    "subnormal sums": lambda q, k: (q * 1e-19, np.tile(k[:, :64], (1, 2)) * np.where(np.arange(128) < 64, 1e-19, -1e-19)),
    "cancellation": lambda q, k: (np.where(np.arange(128) % 2, 1, -1) * (1e4 + q), 1e4 + k),
    "overflow": lambda q, k: (np.abs(q) * 1e19, np.where(np.arange(len(k))[:, None] % 3 == 0, -1e20, 1e19) * np.abs(k)),
}


@pytest.mark.parametrize("kind", [0, 2])
@pytest.mark.parametrize("name", sorted(SPECIAL))
def test_score_special_values_bit_exact(gpu, name, kind):
    """An fp32 MFMA as a chain of fmas, its subnormals, cancellations and
    infinities included."""
    n_comp, n_head = 300, 64
    q = synth.normal(63, 1, n_head * 128).reshape(n_head, 128).astype(np.float64)
    k = synth.normal(63, 3, n_comp * 128).reshape(n_comp, 128).astype(np.float64)
    w = np.abs(synth.normal(63, 2, n_head))   # (a negative one would make inf - inf of the overflowed heads)
    q, k = (np.ascontiguousarray(v, np.float32) for v in SPECIAL[name](q, k))
    kt = torch.from_numpy(k).to(TYPES[kind])
    keys = kt.view(torch.float32 if kind == 0 else torch.int16).numpy().copy()
    ref = np.zeros(n_comp, np.float32)
    O.lib().orc_indexer_scores(P(q), P(w), P(keys), C.c_int(kind), C.c_int(n_comp), C.c_int(n_head), C.c_int(128), P(ref))
    tiny = np.float32(2.0 ** -126)
    if name.startswith("subnormal"):
        assert ((ref > 0) & (ref < 128 * 64 * tiny)).any()
    if name == "overflow":
        assert np.isinf(ref).any() and np.isfinite(ref).any() and not np.isnan(ref).any()
    _, _, scores = ops.indexer_topk_positions(torch.from_numpy(q).to(gpu), torch.from_numpy(w).to(gpu), kt.to(gpu), 100, 0)
    torch.cuda.synchronize()
    assert np.array_equal(scores.cpu().numpy().view(np.uint32), ref.view(np.uint32))
