"""Appending and pooling in one launch (``ChunkedPrefill.step``,
``fpv2_append_pool_kv``): caches, pooled caches and outputs must equal those of
``append`` followed by ``attend`` bit for bit, for chunks that end inside
blocks, start behind unpooled rows, are shorter than a block or a row group,
and for inputs that the launch reads in place or cannot read."""

from __future__ import annotations

import pytest
import torch

from fpv2 import ChunkedPrefill, FPV2Config, _lib

pytestmark = pytest.mark.gpu


def _equal(a, b, n):
    nb = -(-n // a.config.block_k)
    return (torch.equal(a.k[:, :n], b.k[:, :n]) and torch.equal(a.v[:, :n], b.v[:, :n])
            and torch.equal(a.pooled_k[:, :nb], b.pooled_k[:, :nb])
            and torch.equal(a.pooled_v[:, :nb], b.pooled_v[:, :nb])
            and not bool(a.pooled_k[:, nb:].any()) and a.pooled_rows == b.pooled_rows
            and a._complete == b._complete)


@pytest.mark.parametrize(("d", "dtype", "heads", "block"), [
    (128, torch.bfloat16, (8, 2), 128), (64, torch.float16, (4, 4), 128),
    (96, torch.bfloat16, (6, 3), 48), (256, torch.bfloat16, (4, 1), 16)])
@pytest.mark.parametrize("chunks", [(128, 256, 64), (1, 127, 1, 300), (333, 5, 700)])
@pytest.mark.parametrize("layout", ["chunk", "model", "offset"])
def test_step_equals_append_then_attend(cuda, d, dtype, heads, block, chunks, layout):
    hq, hkv = heads
    n = sum(chunks)
    g = torch.Generator().manual_seed(n + d)
    q = torch.randn((hq, n, d), generator=g).to(dtype).to(cuda)
    kv = torch.randn((2, n, hkv, d), generator=g).to(dtype).to(cuda)
    if layout == "model":  # [L, H, D] rows seen as [H, L, D]
        k, v = kv[0].transpose(0, 1), kv[1].transpose(0, 1)
    else:
        k, v = (x.transpose(0, 1).contiguous() for x in kv)
    if layout == "offset":  # off the 16-byte grid: copied by append
        def shift(x):
            flat = torch.empty(x.numel() + 1, dtype=dtype, device=cuda)
            flat[1:] = x.reshape(-1)
            return flat[1:].view(x.shape)
        k, v = shift(k), shift(v)
    a, b = (ChunkedPrefill(hq, hkv, d, n, dtype=dtype, device=cuda, min_tokens=1,
                           config=FPV2Config(block_k=block, sink_tokens=block, window_tokens=block))
            for _ in range(2))
    start = 0
    for i, c in enumerate(chunks):
        s = slice(start, start + c)
        start += c
        if i == 1:  # rows appended earlier and not yet pooled
            a.append(k[:, s], v[:, s])
            b.append(k[:, s], v[:, s])
            continue
        x = a.step(q[:, s], k[:, s], v[:, s])
        b.append(k[:, s], v[:, s])
        y = b.attend(q[:, s])
        torch.cuda.synchronize()
        assert torch.equal(x, y) and _equal(a, b, start), (i, layout)


def test_refusals(cuda):
    """Capacity is checked before anything is written; the entry point refuses
    blocks that are not complete and strides off the grid."""
    cp = ChunkedPrefill(4, 1, 64, 256, device=cuda, min_tokens=1)
    q = torch.zeros((4, 200, 64), dtype=torch.bfloat16, device=cuda)
    k = torch.ones((1, 200, 64), dtype=torch.bfloat16, device=cuda)
    cp.step(q, k, k)
    with pytest.raises(ValueError, match="capacity"):
        cp.step(q, k, k)
    assert cp.length == 200
    lib = _lib.load()

    def call(pooled, row_stride):
        return lib.fpv2_append_pool_kv(
            k.data_ptr(), k.data_ptr(), cp.k.data_ptr(), cp.v.data_ptr(), cp.pooled_k.data_ptr(),
            cp.pooled_v.data_ptr(), _lib.BF16, 1, 8, 200, pooled, 64, 128, k.stride(0),
            row_stride, k.stride(0), k.stride(1), cp.k.stride(0), cp.k.stride(1),
            cp.pooled_k.stride(0), _lib.stream_ptr(cuda))

    assert call(2, 64) == _lib.FPV2_ERR_ARGUMENT
    assert call(1, 60) == _lib.FPV2_ERR_UNSUPPORTED


@pytest.mark.parametrize(("d", "block", "heads", "start", "n", "together"), [
    (256, 1024, 1, 0, 1023, True), (256, 1024, 1, 0, 1024, False), (256, 1024, 1, 900, 2048, False),
    (256, 1024, 8, 0, 2048, True), (256, 2048, 8, 0, 2048, False), (64, 4096, 1, 4000, 200, False),
    (64, 4096, 1, 0, 200, True), (128, 128, 1, 70, 2048, True)])
def test_large_blocks_are_appended_and_pooled_apart(cuda, d, block, heads, start, n, together):
    """Blocks whose rows would pass through one workgroup slower than copies
    and pooling apart; outputs and caches are the same either way."""
    g = torch.Generator().manual_seed(n)
    total = start + n
    q, k, v = (torch.randn((heads, total, d), generator=g).to(torch.bfloat16).to(cuda)
               for _ in range(3))
    a, b = (ChunkedPrefill(heads, heads, d, total, device=cuda, min_tokens=1,
                           config=FPV2Config(block_k=block, tile_q=128)) for _ in range(2))
    calls = []
    fused = a._append_pooled
    a._append_pooled = lambda *args: calls.append(fused(*args)) or calls[-1]
    if start:
        for c in (a, b):
            c.append(k[:, :start], v[:, :start])
            c.attend(q[:, :start])
    x = a.step(q[:, start:], k[:, start:], v[:, start:])
    b.append(k[:, start:], v[:, start:])
    y = b.attend(q[:, start:])
    torch.cuda.synchronize()
    assert calls == [together]
    assert torch.equal(x, y) and _equal(a, b, total)
