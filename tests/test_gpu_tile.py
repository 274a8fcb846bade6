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

import ctypes
import math

import numpy as np
import pytest
import torch

from kvssd import _native
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
        tiled, _ = split_plan(backend.describe(query, batch, scale, 0 if table is None else len(table)), args)
        assert tiled == (name == "tile")
        out, lse = backend.run(query, batch, scale, block_table=None if table is None else table.tolist())
        np.testing.assert_allclose(out.cpu().numpy(), ref_out, atol=TOL * size, rtol=TOL, err_msg=name)
        np.testing.assert_allclose(lse.cpu().numpy(), ref_lse, atol=TOL, rtol=TOL, err_msg=name)


# bits, query heads, kv heads, head_dim, group size, query dtype: 2, 4, 6, 8 and 16 groups a head
GROUPED = [(4, 8, 2, 128, 64, torch.float32), (4, 8, 2, 64, 16, torch.float16), (4, 6, 2, 96, 16, torch.bfloat16),
           (2, 4, 1, 256, 32, torch.float32), (4, 4, 4, 128, 8, torch.float32), (4, 4, 2, 96, 48, torch.float32)]


def grouped_case(rng, bits, kvh, d, g, spread):
    """Keys or values of 9 blocks of 48 tokens whose first group is 2^spread times the size of the others."""
    x = rng.standard_normal((9 * 48, kvh, d)).astype(np.float32) * np.float32(2.0 ** (-spread / 2))
    x[..., :g] *= np.float32(2.0 ** spread)
    packed, scales, valid = O.quantize_blocks(x, bits, g, 48)
    return packed, scales, valid


@pytest.mark.parametrize(("bits", "qh", "kvh", "d", "g", "dtype"), GROUPED)
@pytest.mark.parametrize("spread", [-22, 22])
def test_value_groups_far_apart(cuda_device, bits, qh, kvh, d, g, dtype, spread):
    # a value group whose scales lie 2^-22 below (or above) the other groups' is as exact as those,
    # compared by itself.  A weight is off by one rounding of p scale_v, one of p (scores below 8:
    # ~2^-21 at most) and 2^-23 of its two parts, some 1e-6 together in the worst case
    rng = np.random.default_rng(d + g)
    pk, sk, valid = grouped_case(rng, bits, kvh, d, g, 0)
    pv, sv, _ = grouped_case(rng, bits, kvh, d, g, spread)
    q = torch.from_numpy(rng.standard_normal((qh, d)).astype(np.float32)).to(dtype)
    ref, _ = O.attention(q.float().numpy(), pk, pv, sk, sv, valid, bits, g, 1 / math.sqrt(d))
    arrays = [torch.from_numpy(a).to(cuda_device) for a in (pk, pv, sk, sv)]
    batch = PackedBatch(*arrays, torch.from_numpy(valid).to(cuda_device), bits, g)
    backend = HipAttentionBackend("auto")
    assert split_plan(backend.describe(q.to(cuda_device), batch, 1.0), arrays)[0] == 1
    out, _ = backend.run(q.to(cuda_device), batch, 1 / math.sqrt(d))
    err = (out.double().cpu().numpy() - ref).reshape(qh, -1, g)
    size = np.asarray(ref, dtype=np.float64).reshape(qh, -1, g)
    assert (np.linalg.norm(err, axis=(0, 2)) < 2e-6 * np.linalg.norm(size, axis=(0, 2))).all()


@pytest.mark.parametrize(("bits", "qh", "kvh", "d", "g", "dtype"), GROUPED)
def test_query_groups_far_apart(cuda_device, bits, qh, kvh, d, g, dtype):
    # a query group 2^-26 below the others counts as much as they do where its keys lie 2^26 above
    # them: a score (below 16 here) is then as exact as any, some ten roundings of 2^-24 of it
    if dtype == torch.float16:
        dtype = torch.bfloat16  # (2^-26 of an fp16 query is zero)
    rng = np.random.default_rng(d + 2 * g)
    pk, sk, valid = grouped_case(rng, bits, kvh, d, g, 26)
    pv, sv, _ = grouped_case(rng, bits, kvh, d, g, 0)
    q = rng.standard_normal((qh, d)).astype(np.float32)
    q[:, :g] *= np.float32(2.0 ** -26)
    q = torch.from_numpy(q).to(dtype)
    scale = 2.0**13 / math.sqrt(d)
    ref, ref_lse = O.attention(q.float().numpy(), pk, pv, sk, sv, valid, bits, g, scale)
    arrays = [torch.from_numpy(a).to(cuda_device) for a in (pk, pv, sk, sv)]
    batch = PackedBatch(*arrays, torch.from_numpy(valid).to(cuda_device), bits, g)
    out, lse = HipAttentionBackend("auto").run(q.to(cuda_device), batch, scale)
    np.testing.assert_allclose(lse.cpu().numpy(), ref_lse, atol=1e-5)
    assert np.linalg.norm(out.double().cpu().numpy() - ref) < 1e-5 * np.linalg.norm(ref)


def split_plan(desc, arrays) -> tuple[int, int]:
    """(1 where the tiled kernel runs and 0 where the vector one does, splits) of a decode of these arrays."""
    kernel, tiled, splits = ctypes.c_int(-1), ctypes.c_int(-1), ctypes.c_int(-1)
    rc = _native.load().kvssd_hip_decode_plan(
        ctypes.byref(desc), *[t.data_ptr() for t in arrays], ctypes.byref(kernel), ctypes.byref(tiled), ctypes.byref(splits)
    )
    assert rc == 0 and kernel.value == _native.KERNEL_GENERAL
    return tiled.value, splits.value


# shapes whose tiled form takes fewer splits than the vector one, and the same number
@pytest.mark.parametrize(("bits", "qh", "kvh", "d", "g", "bt", "nb"), [(4, 4, 1, 128, 32, 16, 67), (4, 32, 2, 256, 16, 64, 150),
                                                                         (2, 12, 2, 64, 32, 32, 40), (4, 16, 8, 128, 64, 128, 9)])
def test_two_phase_calls(cuda_device, bits, qh, kvh, d, g, bt, nb):
    # partials and merge as separate calls, of arrays that the tiled kernel takes and of such that
    # it does not: the merge has no arrays to tell by, and finds the number of splits in the partials
    gen = torch.Generator(device=cuda_device).manual_seed(d + nb)
    packed = [torch.randint(0, 256, (nb, bt, kvh, d * bits // 8), dtype=torch.uint8, generator=gen, device=cuda_device) for _ in "kv"]
    scales = [torch.rand(nb, bt, kvh, d // g, generator=gen, device=cuda_device).half() / 8 for _ in "kv"]
    counts = torch.full((nb,), bt, dtype=torch.int32, device=cuda_device)
    counts[-1] = 3
    query = torch.randn(qh, d, generator=gen, device=cuda_device)
    backend, lib = HipAttentionBackend("auto"), _native.load()
    stream = _native.stream_handle(torch.cuda.current_stream(cuda_device))
    plans = []
    for by in (0, 8):
        arrays = [offset_copy(t, by) for t in (*packed, *scales)]
        batch = PackedBatch(*arrays, counts, bits, g)
        want, want_lse = backend.run(query, batch, 0.1)
        desc = backend.describe(query, batch, 0.1)
        plans.append(split_plan(desc, arrays))
        need = ctypes.c_size_t(0)
        _native.check(lib.kvssd_hip_decode_workspace_bytes(ctypes.byref(desc), ctypes.byref(need)), "workspace")
        work = torch.full((need.value,), 255, dtype=torch.uint8, device=cuda_device)  # NaN where nothing is written
        out, lse = torch.empty_like(want), torch.empty_like(want_lse)
        args = [t.data_ptr() for t in (query, *arrays, counts)]
        _native.check(lib.kvssd_hip_decode_partials(ctypes.byref(desc), *args, None, work.data_ptr(), need.value, stream), "partials")
        _native.check(lib.kvssd_hip_decode_merge(ctypes.byref(desc), work.data_ptr(), need.value, out.data_ptr(), lse.data_ptr(), stream), "merge")
        torch.testing.assert_close(out, want, atol=TOL, rtol=TOL)
        torch.testing.assert_close(lse, want_lse, atol=TOL, rtol=TOL)
    assert [tiled for tiled, _ in plans] == [1, 0] and plans[0][1] <= plans[1][1]


@pytest.mark.parametrize("g", [32, 16, 8])
def test_leftover_shared_memory(cuda_device, g):
    # 3, 6 and 12 groups a head leave rows of the query operand over: what earlier workgroups left in
    # the LDS (here V rows whose dwords are NaN) must not reach their factors
    gen = torch.Generator(device=cuda_device).manual_seed(g)

    def batch(d, group, fill):
        nb, bt, kvh = 64, 64, 8
        packed = [torch.randint(0, 256, (nb, bt, kvh, d // 2), dtype=torch.uint8, generator=gen, device=cuda_device) for _ in "kv"]
        if fill:
            packed[1].fill_(255)
        scales = [torch.rand(nb, bt, kvh, d // group, generator=gen, device=cuda_device).half() / 8 for _ in "kv"]
        return PackedBatch(*packed, *scales, torch.full((nb,), bt, dtype=torch.int32, device=cuda_device), 4, group)

    backend = HipAttentionBackend("auto")
    fills = [(torch.randn(32, d, generator=gen, device=cuda_device), batch(d, 64, True)) for d in (64, 128, 256)]
    query, cases = torch.randn(32, 96, generator=gen, device=cuda_device), batch(96, g, False)
    want, want_lse = backend.run(query, PackedBatch(*[offset_copy(t, 8) for t in (cases.packed_k, cases.packed_v, cases.scales_k,
                                 cases.scales_v)], cases.valid_tokens, 4, g), 0.1)
    for i in range(12):
        backend.run(*fills[i % 3], 0.1)
        out, lse = backend.run(query, cases, 0.1)
        torch.testing.assert_close(out, want, atol=TOL, rtol=TOL)
        torch.testing.assert_close(lse, want_lse, atol=TOL, rtol=TOL)


@pytest.mark.parametrize("g", [96, 48, 32, 24, 16, 12, 8])
def test_infinite_key_scale(cuda_device, g):
    # a token whose last group has an infinite K scale, codes below the middle and a positive query:
    # its score is -inf and its weight 0, whatever the number of groups that share a matrix operand
    # (3, 6 and 12 leave rows over); the vector kernel gives the same
    d, bits, kvh, bt, nb = 96, 4, 2, 16, 5
    rng = np.random.default_rng(g)
    pk, sk, valid = O.quantize_blocks(rng.standard_normal((nb * bt, kvh, d)).astype(np.float32), bits, g, bt)
    pv, sv, _ = O.quantize_blocks(rng.standard_normal((nb * bt, kvh, d)).astype(np.float32), bits, g, bt)
    q = np.abs(rng.standard_normal((6, d))).astype(np.float32)
    keep = np.ones((nb, bt), dtype=bool)
    for b, t in ((0, 3), (2, 0), (4, 15)):
        keep[b, t] = False
        sk[b, t, :, -1] = np.inf
        pk[b, t, :, -g // 2 :] = 0x21  # codes 1 and 2 of the group's values: -7 and -6
    ref, ref_lse = O.attention(q, *(a[keep][None] for a in (pk, pv)), *(a[keep][None] for a in (sk, sv)),
                               np.array([keep.sum()], dtype=np.int32), bits, g, 0.1)
    arrays = [torch.from_numpy(a).to(cuda_device) for a in (pk, pv, sk, sv)]
    counts = torch.from_numpy(valid).to(cuda_device)
    for args in (arrays, [offset_copy(a, 8) for a in arrays]):
        out, lse = HipAttentionBackend("auto").run(torch.from_numpy(q).to(cuda_device), PackedBatch(*args, counts, bits, g), 0.1)
        np.testing.assert_allclose(out.cpu().numpy(), ref, atol=TOL, rtol=TOL)
        np.testing.assert_allclose(lse.cpu().numpy(), ref_lse, atol=TOL, rtol=TOL)


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
