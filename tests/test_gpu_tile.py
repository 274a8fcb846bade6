"""The tiled matrix-core decode at the edges of what it takes, against the
float64 oracle, and the same calls with arrays it cannot load (8 bytes off a
16-byte boundary), which the vector kernel answers.

Tolerance.  Both compute in 32 bits: a score is a sum of head_dim products with
a rounding of at most 2^-24 each, so with |q k| sums below 64 here it is good to
~1e-5 absolute in the worst case and ~1e-6 in practice; out is a convex mean of
values below 8, off by the same relative amount.  2e-5 is the reference's own
tolerance for its interpreted kernel.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from kvssd.backends import PackedBatch
from kvssd.backends.hip import HipAttentionBackend
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-5

# bits, qh, kvh, d, g, bt, blocks, dtype: every head size, group counts 1, 2, 3, 4, 6, 8, 12 and 16 per head, one and
# several head chunks with a partial last one, blocks below, at and above a pass of 64 and a workgroup of 256 slots
SHAPES = [
    (4, 1, 1, 64, 64, 16, 1, torch.float16),
    (4, 17, 1, 64, 64, 48, 11, torch.bfloat16),
    (2, 12, 4, 64, 32, 16, 37, torch.float16),
    (4, 18, 2, 64, 32, 128, 5, torch.float32),
    (2, 10, 2, 64, 8, 64, 9, torch.float32),
    (4, 5, 1, 64, 4, 32, 9, torch.float16),
    (4, 16, 2, 96, 96, 80, 7, torch.float16),
    (4, 6, 2, 96, 48, 16, 40, torch.bfloat16),
    (4, 10, 2, 96, 32, 128, 3, torch.float32),
    (4, 3, 1, 96, 16, 32, 21, torch.float16),
    (4, 4, 2, 96, 8, 64, 5, torch.float64),
    (2, 20, 1, 128, 128, 256, 3, torch.float16),
    (4, 36, 4, 128, 64, 272, 3, torch.float32),
    (4, 9, 1, 128, 32, 32, 67, torch.bfloat16),
    (2, 8, 2, 128, 16, 16, 65, torch.float16),
    (4, 24, 12, 128, 8, 96, 4, torch.float16),
    (4, 34, 2, 256, 256, 64, 5, torch.float16),
    (2, 6, 1, 256, 128, 16, 33, torch.float32),
    (4, 6, 1, 256, 64, 512, 2, torch.bfloat16),
    (2, 4, 2, 256, 32, 144, 4, torch.float64),
    (4, 3, 3, 256, 16, 64, 9, torch.float16),
]


def offset_copy(t: torch.Tensor, by: int) -> torch.Tensor:
    """``t`` in memory ``by`` bytes past an allocation's start."""
    raw = torch.empty(t.numel() * t.element_size() + by, dtype=torch.uint8, device=t.device)
    out = raw[by:].view(t.dtype).view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == by
    return out


@pytest.mark.parametrize(("bits", "qh", "kvh", "d", "g", "bt", "nb", "dtype"), SHAPES)
@pytest.mark.parametrize("selected", [False, True])
def test_tile_edges(cuda_device, bits, qh, kvh, d, g, bt, nb, dtype, selected):
    rng = np.random.default_rng(d * 1000 + g * 10 + nb)
    k = rng.standard_normal((nb * bt, kvh, d)).astype(np.float32)
    v = rng.standard_normal((nb * bt, kvh, d)).astype(np.float32)
    # value groups 2^16 apart in size: small weights on large values and the reverse
    v *= np.exp2(rng.integers(-8, 9, (nb * bt, kvh, d // g))).repeat(g, axis=-1) / 64
    q = torch.from_numpy(rng.standard_normal((qh, d)).astype(np.float32)).to(dtype)
    pk, sk, _ = O.quantize_blocks(k, bits, g, bt)
    pv, sv, _ = O.quantize_blocks(v, bits, g, bt)
    # full, partial, empty, oversized and (Python slice) negative counts
    valid = rng.choice([bt, bt, bt - 1, 1, 0, bt + 5, -3, bt // 2], nb).astype(np.int32)
    valid[0] = bt
    table = rng.integers(0, nb, nb + 3).astype(np.int32) if selected else None
    scale = 1 / math.sqrt(d)
    ref_out, ref_lse = O.attention(
        q.double().float().numpy(), pk, pv, sk, sv, valid, bits, g, scale, block_table=table
    )
    arrays = [torch.from_numpy(a).to(cuda_device) for a in (pk, pv, sk, sv)]
    counts = torch.from_numpy(valid).to(cuda_device)
    backend = HipAttentionBackend("general")
    query = q.to(cuda_device)
    size = max(1.0, float(np.abs(ref_out).max()))
    for name, args in (("tile", arrays), ("vector", [offset_copy(a, 8) for a in arrays])):
        batch = PackedBatch(*args, counts, bits, g)
        out, lse = backend.run(query, batch, scale, block_table=None if table is None else table.tolist())
        np.testing.assert_allclose(out.cpu().numpy(), ref_out, atol=TOL * size, rtol=TOL, err_msg=name)
        np.testing.assert_allclose(lse.cpu().numpy(), ref_lse, atol=TOL, rtol=TOL, err_msg=name)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_tile_without_a_valid_token(cuda_device, d):
    pk = torch.randint(0, 256, (5, 32, 2, d // 2), dtype=torch.uint8, device=cuda_device)
    # stale scales of empty blocks: infinities and NaN that must not reach the result
    sk = torch.full((5, 32, 2, d // 64), float("nan"), dtype=torch.float16, device=cuda_device)
    sv = torch.full((5, 32, 2, d // 64), float("inf"), dtype=torch.float16, device=cuda_device)
    batch = PackedBatch(pk, pk, sk, sv, torch.zeros(5, dtype=torch.int32, device=cuda_device), 4, 64)
    query = torch.randn((10, d), device=cuda_device)
    out, lse = HipAttentionBackend("general").run(query, batch, 0.1)
    assert torch.equal(out, torch.zeros_like(out))
    assert bool((lse == -math.inf).all())
