"""The native operator binding: same results and errors as the Python checks behind it, over the forms it accepts."""

import numpy as np
import pytest
import torch

from helpers import bf16_bits, u8
from kvx import _lib, ops

pytestmark = pytest.mark.gpu


class Subclass(torch.Tensor):
    pass


class Declines:
    """Stands in for the binding and takes no call, so the Python checks run."""

    @staticmethod
    def store(*args):
        return None

    codec = blocks = store


VIEWS = {
    "dense": lambda p: p[0, 0],
    "block": lambda p: p[:, :, 2],
    "one_row": lambda p: p[1, 1, 3, 5, 2],
    "rows": lambda p: p[0, 1, 4, ::2, 1],
    "heads": lambda p: p.permute(0, 1, 2, 4, 3, 5)[:, :, 1],  # split into several launches by the Python path
    "size_one": lambda p: p[:, :1, 1:2, :, 1:2],
    "half": lambda p: p[:, :, ::2],
    "expanded": lambda p: p[:, :, 1].unsqueeze(1).expand(2, 3, 2, 6, 3, 96),
}


@pytest.mark.parametrize("scale_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("view", VIEWS)
def test_codec_of_any_view_matches_the_python_checks(gpu, monkeypatch, view, scale_dtype):
    g = torch.Generator(device=gpu).manual_seed(3)
    pool = torch.randn((2, 2, 5, 6, 3, 96), generator=g, device=gpu).to(torch.bfloat16)
    source = VIEWS[view](pool)
    out = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_bind", Declines)  # called: an instance
        payload = torch.empty(source.shape, dtype=torch.float8_e4m3fn, device=gpu)
        scale = torch.empty((*source.shape[:-1], 1), dtype=scale_dtype, device=gpu)
        ops.fp8_quantize(source, payload, scale)
        target = torch.zeros_like(pool)
        if view != "expanded":
            ops.fp8_dequantize(payload, scale, VIEWS[view](target))
        out.append((u8(payload), u8(scale), bf16_bits(target)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_the_binding_takes_the_usual_calls(gpu):
    # One form of each, so that a binding that always declines does not pass unseen.
    pool = torch.zeros((2, 2, 5, 6, 3, 96), dtype=torch.bfloat16, device=gpu)
    staging = torch.zeros(1 << 20, dtype=torch.uint8, device=gpu)
    bind = _lib.bind()
    for ids, entries in (([1], [staging.data_ptr()]), ((1,), (staging.data_ptr(),)), (range(1), [staging.data_ptr()]),
                         ([], [])):
        for fmt, scale in ((ops.FORMAT_FP8, None), (ops.FORMAT_FP8, torch.float32), (ops.FORMAT_RAW, None)):
            assert bind.blocks(True, pool, ids, entries, fmt, scale) == 0
    source = pool[:, :, 1]
    payload = torch.empty(source.shape, dtype=torch.float8_e4m3fn, device=gpu)
    assert bind.codec(True, source, payload, torch.empty((*source.shape[:-1], 1), device=gpu)) == 0
    key = torch.zeros((4, 3, 96), dtype=torch.bfloat16, device=gpu)
    slots = torch.zeros(4, dtype=torch.int32, device=gpu)
    assert bind.store(key, key, pool[0, 0], pool[1, 0], slots) == 0
    # Subclasses, other sequences and other integers are left to Python.
    sub = pool.as_subclass(Subclass)
    assert bind.store(key.as_subclass(Subclass), key, pool[0, 0], pool[1, 0], slots) is None
    assert bind.codec(True, source.as_subclass(Subclass), payload, torch.empty((*source.shape[:-1], 1), device=gpu)) is None
    assert bind.blocks(True, sub, [1], [staging.data_ptr()], ops.FORMAT_RAW, None) is None
    ops.save_blocks(sub, [1], [staging.data_ptr()], ops.FORMAT_RAW)
    assert bind.store(key, key, pool[0, 0], pool[1, 0], slots.long()) is None
    assert bind.store(key[:0], key[:0], pool[0, 0], pool[1, 0], slots[:0]) is None
    assert bind.blocks(True, pool, iter([1]), [staging.data_ptr()], ops.FORMAT_RAW, None) is None
    assert bind.blocks(True, pool, [np.int32(1)], [staging.data_ptr()], ops.FORMAT_RAW, None) is None
    assert bind.blocks(True, pool, [-1], [staging.data_ptr()], ops.FORMAT_RAW, None) is None


def test_errors_are_those_of_the_python_checks(gpu, monkeypatch):
    pool = torch.zeros((2, 2, 5, 6, 3, 96), dtype=torch.bfloat16, device=gpu)
    key = torch.zeros((4, 3, 96), dtype=torch.bfloat16, device=gpu)
    slots = torch.zeros(4, dtype=torch.int32, device=gpu)
    k, v = pool[0, 0], pool[1, 0]
    at = torch.zeros(1 << 20, dtype=torch.uint8, device=gpu).data_ptr()
    source = pool[:, :, 1]
    payload = torch.empty(source.shape, dtype=torch.float8_e4m3fn, device=gpu)
    scale = torch.empty((*source.shape[:-1], 1), device=gpu)
    calls = [
        lambda: ops.store_kvcache(key.transpose(0, 1), key, k, v, slots),
        lambda: ops.store_kvcache(key, key[:3], k, v, slots),
        lambda: ops.store_kvcache(key, key.float(), k, v, slots),
        lambda: ops.store_kvcache(key, key, k, v[:2], slots),
        lambda: ops.store_kvcache(key, key, k, v, slots.long()),
        lambda: ops.store_kvcache(key, key, k, v, slots.cpu()),
        lambda: ops.store_kvcache(key, key, k, v, slots[:3]),
        lambda: ops.store_kvcache(key, key, k.cpu(), v, slots),
        lambda: ops.save_blocks(pool, [5], [at], ops.FORMAT_FP8),
        lambda: ops.save_blocks(pool, [-1], [at], ops.FORMAT_FP8),
        lambda: ops.save_blocks(pool, [1, 2], [at], ops.FORMAT_FP8),
        lambda: ops.save_blocks(pool, [1, 2], [at, at], ops.FORMAT_FP8),
        lambda: ops.save_blocks(pool, [1], [0], ops.FORMAT_RAW),
        lambda: ops.save_blocks(pool, [1], [at + 1], ops.FORMAT_RAW),
        lambda: ops.save_blocks(pool, [1], [at], 7),
        lambda: ops.save_blocks(pool, [1], [at], ops.FORMAT_FP8, torch.float16),
        lambda: ops.save_blocks(pool.float(), [1], [at], ops.FORMAT_FP8),
        lambda: ops.save_blocks(pool.cpu(), [1], [at], ops.FORMAT_FP8),
        lambda: ops.save_blocks(pool.transpose(0, 1), [1], [at], ops.FORMAT_FP8),
        lambda: ops.restore_blocks(pool, [1, 1], [at, at], ops.FORMAT_RAW),
        lambda: ops.fp8_quantize(source.float(), payload, scale),
        lambda: ops.fp8_quantize(source, payload, scale[..., 0]),
        lambda: ops.fp8_quantize(source, payload.transpose(0, 1), scale),
        lambda: ops.fp8_quantize(source.cpu(), payload, scale),
        lambda: ops.fp8_dequantize(payload, scale.double(), source),
    ]
    seen = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_bind", Declines)  # called: an instance
        got = []
        for call in calls:
            with pytest.raises(Exception) as e:
                call()
            got.append((e.type, str(e.value)))
        seen.append(got)
    assert seen[0] == seen[1]
