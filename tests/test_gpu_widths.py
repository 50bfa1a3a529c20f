"""The kernels for rows of any width at the edges of their tiles, against the oracle (bit-exact)."""

import numpy as np
import pytest
import torch

from helpers import bf16_bits, bf16_tensor, finite_bf16_rows, u8
from kvx import ops
from oracle import kvx_oracle as oracle

pytestmark = pytest.mark.gpu

SCALES = [torch.float32, torch.bfloat16]


def finite_pool(gpu, layers, blocks, bs, heads, hd, seed=0):
    shape = (2, layers, blocks, bs, heads, hd)
    return bf16_tensor(finite_bf16_rows(int(np.prod(shape[:-1])), hd, seed), gpu).view(shape)


# (layers, block tokens, heads, head_dim). A save tile holds at most 768 8-element pieces, cut to whole rows (64 rows
# of 96, 72 of 80, 48 of 112 and of 128); a restore tile 512 pieces. Rows of 8 are one piece, rows of 6144 fill a
# tile, rows of 6152 and of 100 are left to the generic kernels.
WIDTHS = [(2, 63, 1, 96), (2, 64, 1, 96), (1, 65, 1, 96), (1, 256, 3, 96), (2, 73, 1, 80), (1, 49, 2, 112),
          (2, 33, 1, 192), (1, 300, 5, 8), (1, 97, 1, 16), (1, 77, 1, 40), (1, 3, 1, 6144), (1, 2, 1, 6152),
          (1, 5, 3, 100), (2, 49, 1, 128), (1, 17, 1, 256), (1, 200, 1, 64)]
# The launches above are small ones: in one-wave workgroups of 128 pieces to save and 64 to restore where planes have
# more than 256 pieces. Launches of more than 196,608 pieces: planes at and around whole tiles, a last tile spread over
# the others (97 rows of 64, 65 of 96 and 800 of 8 to save, 65 of 64 to restore) and not (81 of 96). 1,040 planes of 192
# pieces (one wave again) and of 200, and 1,000 of 192.
WIDTHS += [(66, 64, 1, 96), (66, 65, 1, 96), (60, 81, 1, 96), (100, 65, 1, 64), (66, 97, 1, 64), (66, 800, 1, 8),
           (260, 24, 1, 64), (260, 25, 1, 64), (260, 16, 1, 96), (250, 16, 1, 96)]
# Rows of 64 around the tiled kernel's 32 rows a plane to save.
WIDTHS += [(2, 32, 1, 64), (2, 33, 1, 64)]
# Rows of 64 above the tiled kernel's 8,192 rows to save. Many planes of a few narrow rows (above 8,192 per 8 elements
# of the row), which one thread per row handles, and the same with a row more.
WIDTHS += [(16, 130, 1, 64), (2060, 8, 1, 8), (2060, 9, 1, 8), (2060, 10, 1, 8), (4110, 2, 1, 16), (4110, 3, 1, 16)]


@pytest.mark.parametrize("shift", [0, 8])  # payloads 16-byte aligned, or only 8
@pytest.mark.parametrize("scale_dtype", SCALES)
@pytest.mark.parametrize("layers,bs,heads,hd", WIDTHS)
def test_fp8_blocks_of_any_row_width(gpu, layers, bs, heads, hd, scale_dtype, shift):
    pool = finite_pool(gpu, layers, 5, bs, heads, hd, seed=hd)
    before = bf16_bits(pool)
    fp32 = scale_dtype == torch.float32
    _, offset, stride = ops.entry_layout(ops.pool_layout(pool, scale_dtype), ops.FORMAT_FP8)
    staging = torch.full((2 * stride + 256,), 0xA5, dtype=torch.uint8, device=gpu)
    entries = [staging.data_ptr() + shift + i * stride for i in range(2)]
    ops.save_blocks(pool, [4, 1], entries, ops.FORMAT_FP8, scale_dtype)
    ops.restore_blocks(pool, [0, 3], entries, ops.FORMAT_FP8, scale_dtype)
    staged, after = u8(staging), bf16_bits(pool)
    expect = np.full(staged.shape, 0xA5, dtype=np.uint8)  # gaps and everything past the entries stay as they were
    for i, (src, dst) in enumerate([(4, 0), (1, 3)]):
        codes, scales = oracle.save_block_fp8(before, src, fp32)
        at = shift + i * stride
        expect[at:at + codes.size] = codes.ravel()
        expect[at + offset:at + offset + scales.nbytes] = scales.view(np.uint8).ravel()
        before[:, :, dst] = oracle.dequantize(codes, scales, fp32)
    assert np.array_equal(staged, expect)
    assert np.array_equal(after, before)


# The linear kernels: rows of 1 to 24 pieces, and payloads on 8 bytes only, in small launches (2 x 96 rows) and in
# launches of more than 196,608 pieces.
@pytest.mark.parametrize("scale_dtype", SCALES)
@pytest.mark.parametrize("hd,shift,rows", [(64, 8, 96), (64, 0, 20100), (96, 0, 96), (96, 0, 10100), (80, 0, 10100),
                                           (112, 0, 10100), (192, 0, 10100), (8, 0, 96), (8, 0, 100100),
                                           (128, 8, 96), (128, 8, 10100)])
def test_fp8_rows_with_nan_or_infinity_of_any_width(gpu, hd, shift, rows, scale_dtype):
    fp32 = scale_dtype == torch.float32
    bits = finite_bf16_rows(2 * rows, hd, seed=hd)
    rng = np.random.default_rng(rows)
    kinds = np.zeros(2 * rows, dtype=np.int32)  # of every third row: 1 a NaN, 2 an infinity, 3 both, 4 the lowest value
    kinds[::3] = rng.integers(1, 5, size=kinds[::3].size)
    at, other = rng.integers(0, hd, size=(2, 2 * rows))
    other = np.where(other == at, (at + 1) % hd, other)
    nans = rng.choice(np.array([0x7FC0, 0xFFC0, 0x7F81, 0xFFFF], dtype=np.uint16), size=2 * rows)
    infinities = rng.choice(np.array([0x7F80, 0xFF80], dtype=np.uint16), size=2 * rows)
    for kind, first, second in ((1, nans, None), (2, infinities, None), (3, infinities, nans),
                                (4, np.full(2 * rows, 0xFF7F, dtype=np.uint16), None)):
        i = np.flatnonzero(kinds == kind)
        bits[i, at[i]] = first[i]
        if second is not None:
            bits[i, other[i]] = second[i]
    pool = bf16_tensor(bits, gpu).view(2, 1, 1, rows, 1, hd)
    _, offset, stride = ops.entry_layout(ops.pool_layout(pool, scale_dtype), ops.FORMAT_FP8)
    staging = torch.zeros(stride + 256, dtype=torch.uint8, device=gpu)
    entry = [staging.data_ptr() + shift]
    ops.save_blocks(pool, [0], entry, ops.FORMAT_FP8, scale_dtype)
    back = torch.zeros_like(pool)
    ops.restore_blocks(back, [0], entry, ops.FORMAT_FP8, scale_dtype)
    staged, back = u8(staging), bf16_bits(back).reshape(2 * rows, hd)
    codes = staged[shift:shift + 2 * rows * hd].reshape(2 * rows, hd)
    scales = staged[shift + offset:shift + offset + 2 * rows * (4 if fp32 else 2)].copy()
    scales = scales.view(np.float32) if fp32 else (scales.view(np.uint16).astype(np.uint32) << 16).view(np.float32)

    finite = (kinds == 0) | (kinds == 4)
    want_codes, want_scales = oracle.quantize(bits[finite], fp32)
    assert np.array_equal(codes[finite], want_codes)
    want_back = oracle.dequantize(want_codes, want_scales, fp32)
    assert np.array_equal(back[finite], want_back)
    want_scales = want_scales.ravel()
    want_scales = want_scales if fp32 else (want_scales.view(np.uint16).astype(np.uint32) << 16).view(np.float32)
    assert np.array_equal(scales[finite], want_scales)
    nan, infinite = (kinds == 1) | (kinds == 3), kinds == 2
    assert np.isnan(scales[nan]).all() and np.isposinf(scales[infinite]).all()
    assert ((codes[nan] & 0x7F) == 0x7F).all()
    # Finite values over an infinite scale are signed zeros; infinity over infinity is NaN.
    is_inf = (bits[infinite] & 0x7FFF) == 0x7F80
    assert ((codes[infinite][is_inf] & 0x7F) == 0x7F).all()
    assert np.array_equal(codes[infinite][~is_inf], (bits[infinite][~is_inf] >> 8 & 0x80).astype(np.uint8))
    assert ((back[~finite] & 0x7FFF) > 0x7F80).all()  # NaN times anything, and zero times infinity


# Token counts whose planes of scales (and, with 3 heads of 40, of codes) are not multiples of 16 bytes.
@pytest.mark.parametrize("scale_dtype", SCALES)
@pytest.mark.parametrize("heads,hd,tokens", [(1, 128, 1), (1, 128, 257), (2, 128, 511), (1, 64, 513), (3, 40, 301),
                                             (1, 256, 255), (3, 96, 512), (1, 112, 299),
                                             # the last block at, above and below whole tiles
                                             (1, 128, 16), (1, 128, 273), (1, 256, 264), (1, 64, 352), (1, 96, 64),
                                             # planes scattered in runs of tiles per XCD
                                             (8, 128, 700), (4, 256, 300),
                                             # rows of 64 above and below the tiled kernel's launches and planes
                                             (8, 64, 600), (1, 64, 32), (1, 64, 33), (4, 64, 257)])
def test_fp8_tokens_of_any_count_and_width(gpu, heads, hd, tokens, scale_dtype):
    pool = finite_pool(gpu, 2, 6, 256, heads, hd, seed=tokens)
    before = bf16_bits(pool)
    fp32 = scale_dtype == torch.float32
    table, dest = [4, 1, 2][:-(-tokens // 256)], [0, 5, 3][:-(-tokens // 256)]
    shape = (2, 2, tokens, heads, hd)
    payload = torch.empty(shape, dtype=torch.float8_e4m3fn, device=gpu)
    scale = torch.empty((*shape[:-1], 1), dtype=scale_dtype, device=gpu)
    ops.gather_tokens_fp8(pool, table, tokens, payload, scale)
    codes, scales = oracle.quantize(oracle.gather_tokens(before, table, tokens), fp32)
    assert np.array_equal(u8(payload), codes)
    assert np.array_equal(u8(scale).ravel(), scales.view(np.uint8).ravel())
    ops.scatter_tokens_fp8(pool, dest, tokens, payload, scale)
    oracle.scatter_tokens(before, dest, oracle.dequantize(codes, scales, fp32))
    assert np.array_equal(bf16_bits(pool), before)


# A tile is 1 KiB of a plane: the last block's share a fraction of one, whole ones, and one row more or less.
@pytest.mark.parametrize("heads,hd,tokens", [(1, 128, 1), (1, 128, 4), (1, 128, 259), (1, 128, 260), (1, 128, 261),
                                             (3, 40, 301), (2, 256, 512), (1, 8, 320), (1, 128, 521)])
def test_raw_tokens_of_any_count_and_width(gpu, heads, hd, tokens):
    pool = finite_pool(gpu, 2, 6, 256, heads, hd, seed=tokens)
    before = bf16_bits(pool)
    table, dest = [4, 1, 2][:-(-tokens // 256)], [0, 5, 3][:-(-tokens // 256)]
    dense = torch.empty((2, 2, tokens, heads, hd), dtype=torch.bfloat16, device=gpu)
    ops.gather_tokens(pool, table, tokens, dense)
    values = oracle.gather_tokens(before, table, tokens)
    assert np.array_equal(bf16_bits(dense), values)
    ops.scatter_tokens(pool, dest, tokens, dense)
    oracle.scatter_tokens(before, dest, values)
    assert np.array_equal(bf16_bits(pool), before)


@pytest.mark.parametrize("scale_dtype", SCALES)
@pytest.mark.parametrize("heads,hd", [(3, 96), (1, 80), (2, 64), (64, 64)])
def test_engine_saves_and_restores_of_other_widths(gpu, heads, hd, scale_dtype):
    # Saves of 1-2 blocks behind a busy caller are written to the host slots by a capped grid of workgroups.
    from kvx.engine.cpu_prefix_cache import _CopyEngine

    pool = finite_pool(gpu, 3, 9, 50, heads, hd, seed=7)
    before = bf16_bits(pool)
    fp32 = scale_dtype == torch.float32
    engine = _CopyEngine(pool, ops.pool_layout(pool, scale_dtype), ops.FORMAT_FP8, split=True)
    try:
        slab = torch.full((6 * engine.entry_stride,), 0xA5, dtype=torch.uint8, pin_memory=True)
        staging = [torch.empty(4 * engine.entry_stride, dtype=torch.uint8, device=gpu) for _ in range(2)]
        engine.add_slab(slab, 6)
        engine.set_staging(*staging, 4)
        compute = torch.cuda.current_stream(gpu).cuda_stream
        for blocks, slots in [([7], [0]), ([2, 5], [1, 2]), ([0, 8, 3], [3, 4, 5])]:
            ops.sleep(1000, device=gpu)
            engine.save(blocks, slots, compute)
        engine.synchronize()
        for slots, blocks, wait in [([0], [4], True), ([1, 2], [6, 1], False), ([3, 4, 5], [7, 2, 5], True)]:
            engine.restore(slots, blocks, wait, compute)
        engine.synchronize()
        entries = slab.numpy().reshape(6, engine.entry_stride)
        for slot, (src, dst) in enumerate(zip([7, 2, 5, 0, 8, 3], [4, 6, 1, 7, 2, 5])):
            codes, scales = oracle.save_block_fp8(before, src, fp32)
            at = engine.scale_offset
            assert np.array_equal(entries[slot, :codes.size], codes.ravel()), slot
            assert np.array_equal(entries[slot, at:at + scales.nbytes], scales.view(np.uint8).ravel()), slot
            assert np.array_equal(bf16_bits(pool[:, :, dst]), oracle.dequantize(codes, scales, fp32)), slot
    finally:
        engine.close()


# Rows of 1 to 512 16-byte pieces: below, at and above a wave, whole waves and not, and one that is not in pieces. The
# token counts put the batch in the small and in the large launch (from 655,360 pieces on), with ragged last workgroups.
@pytest.mark.parametrize("heads,hd,tokens", [(1, 8, 1), (1, 8, 70), (3, 8, 333), (5, 64, 513), (63, 8, 65), (1, 512, 3),
                                             (65, 8, 129), (3, 128, 257), (8, 96, 1000), (32, 128, 33), (6, 100, 50),
                                             (8, 96, 3415), (8, 128, 2561), (1, 504, 5300)])
def test_store_kvcache_of_any_row_width(gpu, heads, hd, tokens):
    g = torch.Generator(device=gpu).manual_seed(tokens)
    slots_total = tokens + 300
    bits = torch.randint(-32768, 32768, (2, tokens + slots_total, heads * hd), generator=g, device=gpu).to(torch.int16)
    key = bits[0, :tokens].view(torch.bfloat16).view(tokens, heads, hd)
    qkv = torch.zeros((tokens, 3 * heads * hd), dtype=torch.bfloat16, device=gpu)
    qkv[:, 2 * heads * hd:] = bits[1, :tokens].view(torch.bfloat16)
    value = qkv[:, 2 * heads * hd:].view(tokens, heads, hd)  # a strided view
    caches = bits[:, tokens:].clone().view(torch.bfloat16).view(2, 1, slots_total, heads, hd)
    slots = torch.randperm(slots_total, generator=g, device=gpu)[:tokens].to(torch.int32)
    slots[torch.rand(tokens, generator=g, device=gpu) < 0.1] = -1
    slots[-1] = slots_total  # outside the cache
    expect = [bf16_bits(c).reshape(slots_total, -1) for c in caches]
    host_slots = slots.cpu().numpy()
    at = (host_slots >= 0) & (host_slots < slots_total)
    for cache, rows in zip(expect, (key, value)):
        cache[host_slots[at]] = bf16_bits(rows).reshape(tokens, -1)[at]
    ops.store_kvcache(key, value, caches[0], caches[1], slots)
    for cache, want in zip(caches, expect):
        assert np.array_equal(bf16_bits(cache).reshape(slots_total, -1), want)


def test_store_kvcache_beyond_one_launch(gpu):
    # More than 2^30 16-byte pieces take several launches. Rows overlap: key's are 8 elements apart and value's 16, so
    # every token has its own, in K and in V; few slots are real.
    tokens = (1 << 22) + 3
    g = torch.Generator(device=gpu).manual_seed(1)
    key, value = (torch.randn(tokens * step + 1024, generator=g, device=gpu, dtype=torch.bfloat16)
                  .as_strided((tokens, 8, 128), (step, 128, 1)) for step in (8, 16))
    slots = torch.full((tokens,), -1, dtype=torch.int32, device=gpu)
    where = [0, (1 << 22) - 1, 1 << 22, tokens - 1]
    slots[torch.tensor(where, device=gpu)] = torch.tensor([5, 0, 7, 3], dtype=torch.int32, device=gpu)
    caches = torch.zeros((2, 1, 8, 8, 128), dtype=torch.bfloat16, device=gpu)
    ops.store_kvcache(key, value, caches[0], caches[1], slots)
    expect = torch.zeros_like(caches)
    for token, slot in zip(where, [5, 0, 7, 3]):
        expect[0, 0, slot], expect[1, 0, slot] = key[token], value[token]
    assert torch.equal(caches.view(torch.int16), expect.view(torch.int16))
