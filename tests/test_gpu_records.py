"""GPU record codec against the CPU oracle, through the C ABI.

Bars: bit-exact bytes for packed codes, fp16 scales, whole records and
CRC-32 values (integer/byte work); the oracle's quantiser and record encoder
are pinned by tests/test_golden.py and tests/test_oracle.py (closed forms,
zlib.crc32 and the check value crc32(b"123456789") == 0xCBF43926).
"""

from __future__ import annotations

import zlib

import numpy as np
import pytest
import torch

from kvssd import records_hip as R
from kvssd.format import CacheSpec
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TORCH_DTYPES = [torch.float16, torch.bfloat16, torch.float32, torch.float64]


def oracle_quantize(x: torch.Tensor, bits: int, g: int) -> tuple[np.ndarray, np.ndarray]:
    # the 1e30 edge row overflows the fp16 scale to inf on purpose (as torch's cast does)
    with np.errstate(over="ignore"):
        codes, scales = O.quantize_np(x.float().cpu().numpy(), bits, g)
    return O.pack_np(codes, bits), scales


def edge_rows(d: int, g: int, dtype: torch.dtype) -> torch.Tensor:
    """Rows that exercise the quantiser's corners: zeros, -0, exact .5 ties,
    tiny groups (scale clamp), the fp16 maximum, single spikes."""
    rows = [
        torch.zeros(d),
        -torch.zeros(d),
        torch.full((d,), 1e-12),
        torch.linspace(-7.0, 7.0, d),            # ties land on x/scale = k + 0.5 for some k
        # max 7 makes the INT4 scale exactly 1: every other value is a .5 tie
        torch.cat([torch.tensor([7.0]), torch.arange(d - 1, dtype=torch.float32) % 8 - 3.5]),
        torch.full((d,), 65504.0 if dtype == torch.float16 else 1e30),
    ]
    spike = torch.zeros(d)
    spike[::g] = 3.0
    rows.append(spike)
    return torch.stack(rows).to(dtype)


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("g", [16, 32])
@pytest.mark.parametrize("dtype", TORCH_DTYPES)
def test_quantize_bit_exact(cuda_device, bits, g, dtype):
    gen = torch.Generator().manual_seed(5 + bits + g)
    x = (torch.randn(513, 128, generator=gen) * 3).to(dtype)
    x = torch.cat([x, edge_rows(128, g, dtype)])
    q = R.quantize(x.to(cuda_device), bits, g)
    packed, scales = oracle_quantize(x, bits, g)
    assert np.array_equal(q.packed.cpu().numpy(), packed)
    assert np.array_equal(q.scales.cpu().numpy().view(np.uint16), scales.view(np.uint16))
    assert q.original_shape == tuple(x.shape)


def test_quantize_matches_product_quantizer(cuda_device):
    # the product's CPU quantize_tensor (itself pinned to the reference's
    # closed form) and the GPU twin agree on a 3-D KV tensor
    from kvssd.quant import quantize_tensor

    gen = torch.Generator().manual_seed(3)
    x = torch.randn(64, 8, 128, generator=gen, dtype=torch.float16)
    cpu = quantize_tensor(x, 4, 32)
    gpu = R.quantize(x.to(cuda_device), 4, 32)
    assert torch.equal(cpu.packed, gpu.packed.cpu())
    assert torch.equal(cpu.scales.view(torch.int16), gpu.scales.cpu().view(torch.int16))


def oracle_records(keys: np.ndarray, values: np.ndarray, spec: CacheSpec, layer: int, first_block: int) -> list[bytes]:
    """Records as KVCacheStore.create writes them (zero-padded last block)."""
    t = keys.shape[0]
    bt = spec.block_tokens
    pk, sk, valid = O.quantize_blocks(keys, spec.bits, spec.group_size, bt)
    pv, sv, _ = O.quantize_blocks(values, spec.bits, spec.group_size, bt)
    out = []
    for b in range(pk.shape[0]):
        out.append(
            O.encode_record(
                layer, first_block + b, int(valid[b]), spec.bits, bt, spec.kv_heads, spec.head_dim, spec.group_size,
                sk[b], sv[b], pk[b], pv[b],
            )
        )
    assert t == sum(int(v) for v in valid)
    return out


SPECS = [
    CacheSpec(layers=1, kv_heads=8, head_dim=128, block_tokens=128, bits=4, group_size=32),
    CacheSpec(layers=1, kv_heads=8, head_dim=128, block_tokens=128, bits=2, group_size=32),
    CacheSpec(layers=1, kv_heads=2, head_dim=64, block_tokens=32, bits=4, group_size=16),
    # payload of 6 * BT * KVH = 18 bytes: not a multiple of 4 (byte paths)
    CacheSpec(layers=1, kv_heads=1, head_dim=4, block_tokens=3, bits=2, group_size=4),
    # 55,296-byte payload: 4 rows of 16-byte chunks behind 10,240 virtual zero bytes
    CacheSpec(layers=1, kv_heads=8, head_dim=128, block_tokens=48, bits=4, group_size=32),
    # 294,912-byte payload: 18 rows of 16-byte chunks, five groups of four rows
    CacheSpec(layers=1, kv_heads=8, head_dim=128, block_tokens=256, bits=4, group_size=32),
]


@pytest.mark.parametrize("spec", SPECS, ids=lambda s: f"b{s.bits}-kvh{s.kv_heads}-d{s.head_dim}-bt{s.block_tokens}")
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_encode_records_bit_exact(cuda_device, spec, dtype):
    gen = torch.Generator().manual_seed(11)
    tokens = 3 * spec.block_tokens - 1  # partial last block
    k = torch.randn(tokens, spec.kv_heads, spec.head_dim, generator=gen).to(dtype)
    v = torch.randn(tokens, spec.kv_heads, spec.head_dim, generator=gen).to(dtype)
    recs, crcs = R.encode_records(k.to(cuda_device), v.to(cuda_device), spec, layer=5, first_block=7)
    want = oracle_records(k.float().numpy(), v.float().numpy(), spec, 5, 7)
    got = recs.cpu().numpy()
    assert got.shape == (len(want), spec.record_bytes)
    for i, w in enumerate(want):
        assert got[i].tobytes() == w, f"record {i} differs"
        assert int(crcs[i]) == int.from_bytes(w[48:52], "little")
        assert int(crcs[i]) == zlib.crc32(w[52 : 52 + int.from_bytes(w[44:48], "little")])


def device_records(recs: list[bytes], device) -> torch.Tensor:
    return torch.from_numpy(np.frombuffer(b"".join(recs), dtype=np.uint8).copy()).to(device)


@pytest.mark.parametrize("spec", SPECS, ids=lambda s: f"b{s.bits}-kvh{s.kv_heads}-d{s.head_dim}-bt{s.block_tokens}")
def test_gather_records_bit_exact(cuda_device, spec):
    rng = np.random.default_rng(2)
    tokens = 4 * spec.block_tokens - 2
    k = rng.standard_normal((tokens, spec.kv_heads, spec.head_dim)).astype(np.float32)
    v = rng.standard_normal((tokens, spec.kv_heads, spec.head_dim)).astype(np.float32)
    recs = oracle_records(k, v, spec, 0, 0)
    raw = device_records(recs, cuda_device)
    pk, pv, sk, sv, valid, status = R.gather_records(raw, spec, len(recs))
    opk, osk, ovalid = O.quantize_blocks(k, spec.bits, spec.group_size, spec.block_tokens)
    opv, osv, _ = O.quantize_blocks(v, spec.bits, spec.group_size, spec.block_tokens)
    assert status.cpu().tolist() == [R.OK] * len(recs)
    assert np.array_equal(valid.cpu().numpy(), ovalid)
    assert np.array_equal(pk.cpu().numpy(), opk)
    assert np.array_equal(pv.cpu().numpy(), opv)
    assert np.array_equal(sk.cpu().numpy().view(np.uint16), osk.view(np.uint16))
    assert np.array_equal(sv.cpu().numpy().view(np.uint16), osv.view(np.uint16))


def test_gather_records_detects_corruption(cuda_device):
    spec = SPECS[0]
    rng = np.random.default_rng(4)
    k = rng.standard_normal((6 * spec.block_tokens, spec.kv_heads, spec.head_dim)).astype(np.float32)
    recs = [bytearray(r) for r in oracle_records(k, k, spec, 2, 10)]
    recs[1][52 + 1000] ^= 0x01                     # payload bit flip -> CRC
    recs[2][0:8] = b"KVSSD002"                     # magic
    recs[3][8:12] = (2).to_bytes(4, "little")      # version
    recs[4][24:28] = (2).to_bytes(4, "little")     # bits: layout differs
    recs[5][44:48] = (1234).to_bytes(4, "little")  # payload length
    raw = device_records([bytes(r) for r in recs], cuda_device)
    *_, status = R.gather_records(raw, spec, len(recs))
    assert status.cpu().tolist() == [R.OK, R.BAD_CRC, R.BAD_HEADER, R.BAD_HEADER, R.BAD_LAYOUT, R.BAD_CRC]
    with pytest.raises(IOError, match="CRC mismatch for layer=2, block=11"):
        R.raise_for_status(status, 2, list(range(10, 16)))
    # without verification a flipped payload byte passes (and is copied as is)
    *_, status = R.gather_records(raw[: 2 * spec.record_bytes], spec, 2, verify_crc=False)
    assert status.cpu().tolist() == [R.OK, R.OK]


def test_gather_then_decode_matches_oracle(cuda_device):
    # records -> GPU gather -> fused decode equals the oracle on the same blocks
    from kvssd.backends import PackedBatch
    from kvssd.backends.hip import HipAttentionBackend

    spec = SPECS[0]
    rng = np.random.default_rng(8)
    tokens = 5 * spec.block_tokens - 17
    k = rng.standard_normal((tokens, spec.kv_heads, spec.head_dim)).astype(np.float32)
    v = rng.standard_normal((tokens, spec.kv_heads, spec.head_dim)).astype(np.float32)
    q = rng.standard_normal((32, spec.head_dim)).astype(np.float32)
    raw = device_records(oracle_records(k, v, spec, 0, 0), cuda_device)
    pk, pv, sk, sv, valid, status = R.gather_records(raw, spec, -(-tokens // spec.block_tokens))
    assert int(status.max()) == R.OK
    out, lse = HipAttentionBackend().run(torch.from_numpy(q).to(cuda_device), PackedBatch(pk, pv, sk, sv, valid, 4, 32), 0.1)
    opk, osk, ovalid = O.quantize_blocks(k, 4, 32, spec.block_tokens)
    opv, osv, _ = O.quantize_blocks(v, 4, 32, spec.block_tokens)
    ref_out, ref_lse = O.attention(q, opk, opv, osk, osv, ovalid, 4, 32, 0.1)
    np.testing.assert_allclose(out.cpu().numpy(), ref_out, atol=2e-3, rtol=1e-2)
    np.testing.assert_allclose(lse.cpu().numpy(), ref_lse, atol=2e-3, rtol=1e-2)


def test_gather_records_unaligned_outputs(cuda_device):
    # outputs that are not 16-byte aligned take the general form; same bytes
    spec = SPECS[0]
    rng = np.random.default_rng(6)
    k = rng.standard_normal((3 * spec.block_tokens, spec.kv_heads, spec.head_dim)).astype(np.float32)
    recs = oracle_records(k, k[::-1].copy(), spec, 0, 0)
    raw = device_records(recs, cuda_device)
    want = R.gather_records(raw, spec, 3)
    n, bt, kvh = 3, spec.block_tokens, spec.kv_heads
    pbytes = n * bt * kvh * spec.packed_dim
    sbytes = n * bt * kvh * (spec.head_dim // spec.group_size) * 2
    buf = torch.zeros(2 * pbytes + 2 * sbytes + 64, dtype=torch.uint8, device=cuda_device)
    pk = buf[4 : 4 + pbytes].view(n, bt, kvh, spec.packed_dim)
    pv = buf[8 + pbytes : 8 + 2 * pbytes].view(n, bt, kvh, spec.packed_dim)
    base = 16 + 2 * pbytes
    sk = buf[base : base + sbytes].view(torch.float16).view(n, bt, kvh, -1)
    sv = buf[base + sbytes + 8 : base + 2 * sbytes + 8].view(torch.float16).view(n, bt, kvh, -1)
    valid = torch.empty(n, dtype=torch.int32, device=cuda_device)
    status = torch.empty(n, dtype=torch.int32, device=cuda_device)
    got = R.gather_records(raw, spec, n, out=(pk, pv, sk, sv, valid, status))
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8) if a.dtype == torch.float16 else a, b.view(torch.uint8) if b.dtype == torch.float16 else b)


@pytest.mark.parametrize("bits", [2, 4])
def test_quantize_unaligned_source_matches(cuda_device, bits):
    # a source that is not 16-byte aligned takes the element-wise form; the
    # word form (aligned) gives the same bytes
    gen = torch.Generator().manual_seed(21)
    x = torch.randn(301, 128, generator=gen).half()
    buf = torch.empty(301 * 128 + 1, dtype=torch.float16, device=cuda_device)
    shifted = buf[1:].view(301, 128)
    shifted.copy_(x.to(cuda_device))
    a = R.quantize(shifted, bits, 32)
    b = R.quantize(x.to(cuda_device), bits, 32)
    packed, scales = oracle_quantize(x, bits, 32)
    assert torch.equal(a.packed, b.packed) and np.array_equal(a.packed.cpu().numpy(), packed)
    assert np.array_equal(a.scales.cpu().numpy().view(np.uint16), scales.view(np.uint16))


@pytest.mark.parametrize("block_tokens", [1, 127, 128, 129, 512, 513, 1300, 2433])
def test_chunked_crc_row_edges(cuda_device, block_tokens):
    # 128 payload bytes a token: part of a row of 1024 16-byte chunks, one row, four (a whole
    # group of rows), one chunk more, and more than 16 rows; CRC values are zlib's, and one
    # flipped bit at either end or in the middle of the payload is seen
    spec = CacheSpec(1, 1, 96, block_tokens, 4, 12)
    gen = torch.Generator().manual_seed(block_tokens)
    k = torch.randn(5 * block_tokens, 1, 96, generator=gen).half().to(cuda_device)
    recs, crcs = R.encode_records(k, k.flip(0), spec, 0)
    n = 128 * block_tokens
    host = recs.cpu().numpy()
    assert crcs.tolist() == [zlib.crc32(r[52 : 52 + n].tobytes()) for r in host]
    for i, (byte, bit) in enumerate([(0, 0), (n // 2, 3), (n - 1, 7), (n // 3, 5)]):
        recs[i, 52 + byte] ^= 1 << bit
    *_, status = R.gather_records(recs.view(-1), spec, 5)
    assert status.tolist() == [R.BAD_CRC] * 4 + [R.OK]


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_quantize_around_ties(cuda_device, bits, dtype):
    # values next to every k + 0.5 of groups with many different largest values, scales whose
    # reciprocal is subnormal among them: where a reciprocal could stand in wrongly for the
    # division; through the quantiser and through whole records, with the oracle's codes
    rng = np.random.default_rng(bits)
    top = (1 << (bits - 1)) - 1
    amax = rng.uniform(1.0, 2.0, 2048) * 2.0 ** rng.integers(-12, 14, 2048)
    if dtype != torch.float16:
        amax[:64] = rng.uniform(1.0, 2.0, 64) * 1.5e38
    amax = torch.from_numpy(amax).to(dtype)
    s32 = amax.float() / top
    ties = (torch.arange(32) % (2 * top) - top + 0.5) * s32[:, None]
    step = torch.tensor([0.0, 1.0, -1.0, 2.0])[torch.arange(32) // 8]
    x = (ties * (1 + step * torch.finfo(dtype).eps)).to(dtype)
    x = torch.minimum(torch.maximum(x, -amax[:, None]), amax[:, None])
    x[:, 31] = amax
    x = x.reshape(-1, 128)  # 512 rows of four groups
    packed, scales = oracle_quantize(x, bits, 32)
    q = R.quantize(x.to(cuda_device), bits, 32)
    assert np.array_equal(q.packed.cpu().numpy(), packed)
    assert np.array_equal(q.scales.cpu().numpy().view(np.uint16), scales.view(np.uint16))
    # one block of 128 tokens x 8 heads: the one-kernel encode
    spec = CacheSpec(1, 8, 128, 128, bits, 32)
    kv = x.repeat(2, 1).reshape(128, 8, 128).to(cuda_device)
    recs, _ = R.encode_records(kv, kv, spec, 0)
    pk, pv, sk, sv, _, status = R.gather_records(recs.view(-1), spec, 1)
    assert status.tolist() == [R.OK]
    for p, s in ((pk, sk), (pv, sv)):
        assert np.array_equal(p.cpu().numpy().reshape(-1, packed.shape[-1]), np.tile(packed, (2, 1)))
        assert np.array_equal(s.cpu().numpy().view(np.uint16).reshape(-1, 4), np.tile(scales.view(np.uint16).reshape(-1, 4), (2, 1)))


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_quantize_nan_and_infinity(cuda_device, bits, dtype):
    # a NaN takes code 0 and leaves its group's scale alone; a group with an infinity has an
    # infinite scale, so finite values take the middle code and the infinity (inf / inf) code 0;
    # the word form as the element-wise one (the same values in a shifted source)
    gen = torch.Generator().manual_seed(17)
    x = torch.randn(64, 128, generator=gen)
    x[3, 5] = x[9, 64] = x[9, 71] = float("nan")
    x[12, 0], x[20, 127], x[31, 40] = float("inf"), float("-inf"), float("inf")
    x[31, 41] = float("nan")
    x[40, 32:64] = float("nan")
    x = x.to(dtype).to(cuda_device)
    buf = torch.empty(64 * 128 + 1, dtype=dtype, device=cuda_device)
    shifted = buf[1:].view(64, 128)
    shifted.copy_(x)
    a, b = R.quantize(x, bits, 32), R.quantize(shifted, bits, 32)
    assert torch.equal(a.packed, b.packed) and torch.equal(a.scales.view(torch.int16), b.scales.view(torch.int16))
    per = 8 // bits
    codes = torch.stack([(a.packed >> (bits * i)) & ((1 << bits) - 1) for i in range(per)], -1).reshape(64, 128).cpu()
    assert codes[3, 5] == 0 and codes[12, 0] == 0 and codes[20, 127] == 0 and (codes[40, 32:64] == 0).all()
    assert (codes[12, 1:32] == 1 << (bits - 1)).all() and torch.isinf(a.scales[12, 0]) and torch.isfinite(a.scales[3]).all()


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_encode_more_records_than_compute_units(cuda_device, bits, dtype):
    # past 256 records the workgroups are of 512 threads; the same bytes and CRC values as the
    # same blocks in smaller calls (which other tests hold to the oracle's), for one and several
    # rows of scales, the last record partly filled
    for kvh in (8, 16):
        spec = CacheSpec(1, kvh, 128, 128, bits, 32)
        gen = torch.Generator(device=cuda_device).manual_seed(bits)
        tokens = 258 * spec.block_tokens - 3
        k = torch.randn(tokens, spec.kv_heads, 128, generator=gen, device=cuda_device).to(dtype)
        v = torch.randn(tokens, spec.kv_heads, 128, generator=gen, device=cuda_device).to(dtype)
        recs, crcs = R.encode_records(k, v, spec, 3)
        at = 0
        for n in (200, 58):
            span = slice(at * spec.block_tokens, (at + n) * spec.block_tokens)
            part, part_crcs = R.encode_records(k[span], v[span], spec, 3, first_block=at)
            assert torch.equal(recs[at : at + n], part) and torch.equal(crcs[at : at + n], part_crcs)
            at += n


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("g", [8, 16, 24, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float64])
def test_word_form_group_sizes(cuda_device, bits, g, dtype):
    # groups of one to 32 lanes of a word each, and sizes that are not (INT2 of 8, 24): rows
    # that end inside a workgroup, a last record partly filled; the oracle's bytes
    d = 2 * g if g >= 64 else 6 * g
    gen = torch.Generator().manual_seed(g)
    x = torch.randn(37, d, generator=gen).to(dtype)
    q = R.quantize(x.to(cuda_device), bits, g)
    packed, scales = oracle_quantize(x, bits, g)
    assert np.array_equal(q.packed.cpu().numpy(), packed)
    assert np.array_equal(q.scales.cpu().numpy().view(np.uint16), scales.view(np.uint16))
    spec = CacheSpec(1, 3, d, 21, bits, g)
    k = torch.randn(50, 3, d, generator=gen).to(dtype)
    v = torch.randn(50, 3, d, generator=gen).to(dtype)
    recs, _ = R.encode_records(k.to(cuda_device), v.to(cuda_device), spec, 2, 4)
    want = oracle_records(k.float().numpy(), v.float().numpy(), spec, 2, 4)
    assert [r.tobytes() for r in recs.cpu().numpy()] == want


def test_encode_more_records_than_a_grid(cuda_device):
    # past 32,767 records the two-pass encode takes several launches: the same bytes and CRC
    # values as two calls of half the records, the last one partly filled, and no slower
    # kernel for them (one record more than a launch holds took ten times as long)
    spec = CacheSpec(1, 4, 64, 16, 4, 32)
    n = 32769
    gen = torch.Generator(device=cuda_device).manual_seed(1)
    k = torch.randn(n * 16 - 5, 4, 64, generator=gen, device=cuda_device).half()
    v = torch.randn(n * 16 - 5, 4, 64, generator=gen, device=cuda_device).half()
    recs, crcs = R.encode_records(k, v, spec, 3)
    at = 0
    for m in (16384, 16385):
        span = slice(at * 16, (at + m) * 16)
        part, part_crcs = R.encode_records(k[span], v[span], spec, 3, first_block=at)
        assert torch.equal(recs[at : at + m], part) and torch.equal(crcs[at : at + m], part_crcs)
        at += m
    del recs, crcs, part

    def fastest(tokens):
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            R.encode_records(k[:tokens], v[:tokens], spec, 3)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert fastest(n * 16 - 5) < 1.5 * fastest(32767 * 16)


@pytest.mark.parametrize(("kvh", "bits", "dtype"), [(24, 4, torch.bfloat16), (32, 4, torch.float16), (32, 4, torch.float32),
                                                    (24, 2, torch.float32), (32, 2, torch.bfloat16)])
def test_encode_wide_layers(cuda_device, kvh, bits, dtype):
    # three and four rows of scales, up to the most LDS a workgroup takes: few records (two passes),
    # more than half a CU's worth each and more than one (16-bit INT4: one kernel); the oracle's
    # bytes for few, and the same bytes in larger calls
    spec = CacheSpec(1, kvh, 128, 128, bits, 32)
    gen = torch.Generator(device=cuda_device).manual_seed(kvh + bits)
    tokens = 258 * 128 - 3
    k = torch.randn(tokens, kvh, 128, generator=gen, device=cuda_device).to(dtype)
    v = torch.randn(tokens, kvh, 128, generator=gen, device=cuda_device).to(dtype)
    parts = [R.encode_records(k[a * 128 : b * 128], v[a * 128 : b * 128], spec, 1, a) for a, b in ((0, 128), (128, 255), (255, 258))]
    want = oracle_records(k[255 * 128 :].float().cpu().numpy(), v[255 * 128 :].float().cpu().numpy(), spec, 1, 255)
    assert [r.tobytes() for r in parts[2][0].cpu().numpy()] == want
    recs, crcs = (torch.cat([p[i] for p in parts]) for i in (0, 1))
    for n in (129, 256, 258):
        got, got_crcs = R.encode_records(k[: n * 128], v[: n * 128], spec, 1)
        assert torch.equal(got, recs[:n]) if n == 258 else torch.equal(got[: n - 1], recs[: n - 1])
        assert torch.equal(got_crcs[: n - 1], crcs[: n - 1])
        host = got[n - 1].cpu().numpy()
        assert int(got_crcs[n - 1]) == zlib.crc32(host[52 : 52 + int.from_bytes(host[44:48].tobytes(), "little")].tobytes())


def test_encode_wide_layers_few_records_keep_their_speed(cuda_device):
    # a layer of 24 kv heads, INT2 of fp32 values, 64 records: one workgroup a record takes about
    # twice the time that the same values take as 24 records' worth of smaller blocks in two passes
    def fastest(spec, dtype):
        k = torch.randn(64 * 128, 24, 128, device=cuda_device).to(dtype)
        times = []
        R.encode_records(k, k, spec, 0)
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                R.encode_records(k, k, spec, 0)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    small = fastest(CacheSpec(1, 24, 128, 64, 2, 32), torch.float32)
    assert fastest(CacheSpec(1, 24, 128, 128, 2, 32), torch.float32) < 1.7 * small


def test_quantize_more_values_than_a_grid(cuda_device):
    # 2^35 INT4 values are 2^32 words of codes, more threads than one launch takes: the rows at the
    # ends and around the seams as in calls of their own
    rows = (1 << 28) + 3
    if torch.cuda.mem_get_info(cuda_device)[0] < 110 << 30:
        pytest.skip("needs 82 GiB of device memory")
    x = torch.empty(rows, 128, dtype=torch.float16, device=cuda_device)
    gen = torch.Generator(device=cuda_device).manual_seed(9)
    spots = [0, (1 << 27) - 2, (1 << 28) - 1]
    for at in spots:
        x[at : at + 4] = torch.randn(4, 128, generator=gen, device=cuda_device).half()
    q = R.quantize(x, 4, 32)
    for at in spots:
        part = R.quantize(x[at : at + 4].clone(), 4, 32)
        assert torch.equal(q.packed[at : at + 4], part.packed) and torch.equal(q.scales[at : at + 4], part.scales)
    del x, q
    torch.cuda.empty_cache()
