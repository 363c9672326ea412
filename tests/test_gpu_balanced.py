"""The balanced walk (``fpv2_sparse_attention_balanced``).

Calls with few query tiles cut the tiles' walks into parts, one workgroup each,
and add the partials of a tile.  On the same inputs and lists the result must equal the whole-tile
kernel's up to float32 summation order: both round the same float32 values
(equal to about 1e-6) to the output type once, so they differ by at most one
unit in the last place, 2^-7 (bfloat16) or 2^-10 (float16) of the value.
Where a part of a row takes the online reference, its P words round against
another reference: half a unit of P per term, 2^-8 of the largest |v| times
the row's weights, which sum to one (1e-2 below covers |v| < 2.5 averages).
"""

from __future__ import annotations

import pytest
import torch

from fpv2 import FPV2Config, _lib, pool_blocks
from fpv2.kernel import _launch_attention, compact_block_indices
from fpv2.selection import block_scores_and_select
from fpv2.synthetic import baseline_qkv, structured_qkv

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def _lists(q, k, config, pk, n, lk):
    off = lk - n
    sel, _ = block_scores_and_select(q, pk, scale=q.shape[-1] ** -0.5, config=config, offset=off,
                                     query_length=n)
    return compact_block_indices(sel, config=config, offset=off, query_length=n, key_length=lk)


def _both(q, k, v, pk, pv, lists, config, n, lk):
    outs = []
    for balanced in (False, True):
        out = torch.full_like(q, float("nan"))
        # (all tiles: whether the call would take the walk by itself depends
        # on its size)
        _launch_attention(q, k, v, pk, pv, *lists, out, device=q.device,
                          scale=q.shape[-1] ** -0.5, config=config, offset=lk - n, query_length=n,
                          key_length=lk, num_blocks=pk.shape[1], padded_query_length=q.shape[1],
                          out_rows=q.shape[1], balanced=balanced,
                          split_tiles=q.shape[1] // config.tile_q if balanced else 0)
        outs.append(out)
    torch.cuda.synchronize()
    return outs


def _close(whole, even, loose=0.0):
    assert bool(torch.isfinite(even).all())
    w, e = whole.float(), even.float()
    bound = ULP[whole.dtype] * torch.maximum(w.abs(), e.abs()) + 1e-5 + loose
    assert bool(((w - e).abs() <= bound).all()), float(((w - e).abs() - bound).max())


def _pad(x, multiple):
    n = -(-x.shape[1] // multiple) * multiple
    out = x.new_zeros((x.shape[0], n, x.shape[2]))
    out[:, :x.shape[1]] = x
    return out


# (queries, keys): one row; one tile; a last tile of one row; a short chunk of
# a long prefix; a whole prompt; a chunk of many tiles
@pytest.mark.parametrize(("n", "lk"), [(1, 5000), (32, 4096), (65, 3001), (300, 16000),
                                       (2048, 2048), (2100, 9000)])
@pytest.mark.parametrize(("d", "dtype", "heads", "corr"), [
    (128, torch.bfloat16, (4, 1), True), (128, torch.bfloat16, (32, 8), False),
    (128, torch.float16, (8, 2), True), (64, torch.float16, (16, 2), False),
    (96, torch.bfloat16, (6, 3), True), (256, torch.bfloat16, (4, 1), True),
    (256, torch.float16, (4, 4), True),
])
def test_equals_whole_tiles(cuda, n, lk, d, dtype, heads, corr):
    hq, hkv = heads
    tq = 128 // (hq // hkv)
    q, k, v = baseline_qkv(lk, query_heads=hq, kv_heads=hkv, head_dim=d, seed=n + d, dtype=dtype,
                           planted=3.0 * d ** 0.5, heavy_fraction=0.1, device=cuda)
    q = _pad(q[:, lk - n:], tq)
    blocks = -(-(lk - n + q.shape[1]) // 128)
    k, v = (_pad(x, 128 * blocks) for x in (k, v))
    config = FPV2Config(alpha=0.1, sink_tokens=128, tile_q=tq, mean_correction=corr)
    pk, pv = pool_blocks(k), pool_blocks(v)
    lists = _lists(q, k, config, pk, n, lk)
    whole, even = _both(q, k, v, pk, pv, lists, config, n, lk)
    # float16 parts after a tile's first walk with the online reference
    _close(whole, even, 2e-3 if dtype == torch.float16 else 0.0)


def test_only_the_last_tiles(cuda):
    """The dense tail of a long sparse call: the other tiles bit for bit."""
    n = 8192
    q, k, v = baseline_qkv(n, planted=3.0 * 128 ** 0.5, seed=7, device=cuda)
    config = FPV2Config(alpha=0.1, sink_tokens=128, tile_q=32)
    pk, pv = pool_blocks(k), pool_blocks(v)
    lists = _lists(q, k, config, pk, n, n)
    outs = []
    for tiles in (0, 2):
        out = torch.empty_like(q)
        _launch_attention(q, k, v, pk, pv, *lists, out, device=q.device, scale=128 ** -0.5,
                          config=config, offset=0, query_length=n, key_length=n, num_blocks=64,
                          padded_query_length=n, out_rows=n, balanced=tiles > 0, split_tiles=tiles)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0][:, :-64], outs[1][:, :-64])
    _close(*outs)


@pytest.mark.parametrize(("d", "tiles"), [
    (64, 300),    # two items for some of the 256 threads that plan, four turns
    (128, 430),
    (64, 1300),   # six items a thread, two past those it keeps
    (256, 1300),  # three items for each of 512 threads
    (96, 3300),   # more turns than parts would be cut for
])
def test_plans_of_many_items(cuda, d, tiles):
    """More (tile, row chunk) items of a head than threads that plan, with
    walks of 1 to 200 sub-tiles, some of them whole and some in parts: each
    item's rows come from its own walk."""
    g = torch.Generator(device=cuda).manual_seed(tiles)
    n = 16 * tiles - 5
    q = torch.randn((8, 16 * tiles, d), generator=g, device=cuda).to(torch.bfloat16)
    q[:, n:] = 0
    blocks = 16 * tiles // 128 + 60
    k, v = (torch.randn((1, 128 * blocks, d), generator=g, device=cuda).to(torch.bfloat16)
            for _ in range(2))
    lk = 128 * blocks
    config = FPV2Config(tile_q=16)
    mask = torch.zeros((1, tiles, blocks), dtype=torch.bool, device=cuda)
    length = torch.randint(1, 50, (tiles,), generator=g, device=cuda)
    length[torch.randint(0, tiles, (tiles // 2,), generator=g, device=cuda)] = 1
    mask[0] = torch.arange(blocks, device=cuda)[None] < length[:, None]
    lists = compact_block_indices(mask, config=config, offset=lk - n, query_length=n, key_length=lk)
    assert torch.equal(lists[1][0], length.to(torch.int32))
    whole, even = _both(q, k, v, pool_blocks(k), pool_blocks(v), lists, config, n, lk)
    _close(whole, even)
    assert not torch.equal(whole, even)


def test_tiles_of_several_row_chunks_and_a_dense_tail(cuda):
    """tile_q 128 at G = 4: four 128-row chunks per tile; the last tile is dense."""
    q, k, v = structured_qkv(length=3072, query_heads=4, kv_heads=1, head_dim=128, seed=5,
                             dtype=torch.bfloat16, device=cuda)
    config = FPV2Config(alpha=0.3, sink_tokens=128, window_tokens=128, last_n_blocks=1)
    pk, pv = pool_blocks(k), pool_blocks(v)
    lists = _lists(q, k, config, pk, 3072, 3072)
    assert int(lists[1].max()) > 2 * int(lists[1][:, -2].max())
    _close(*_both(q, k, v, pk, pv, lists, config, 3072, 3072))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_lists_without_blocks_and_parts_that_overflow(cuda, dtype):
    """Tiles with empty lists come back as zeros; a key far above the rest in
    the middle of the walk sends its part to the online walk."""
    g = torch.Generator().manual_seed(31)
    n, d = 2048, 128
    q, k, v = (torch.randn((h, n, d), generator=g) for h in (4, 1, 1))
    u = torch.randn(d, generator=g)
    u /= u.norm()
    k[:, 1000] = 40.0 * u
    q[:, 1000:] += 40.0 * u
    q, k, v = (x.to(dtype).to(cuda) for x in (q, k, v))
    config = FPV2Config(alpha=0.0, sink_tokens=0, window_tokens=0, last_n_blocks=0, tile_q=32,
                        mean_correction=False)
    pk, pv = pool_blocks(k), pool_blocks(v)
    ids, counts, pids, pcounts = _lists(q, k, config, pk, n, n)
    counts[:, 10:14] = 0
    whole, even = _both(q, k, v, pk, pv, (ids, counts, pids, pcounts), config, n, n)
    assert not bool(even[:, 320:448].any())
    _close(whole, even, 1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("d", "corr"), [(64, True), (128, False), (256, True)])
@pytest.mark.parametrize(("where", "value"), [
    ("q", "nan"), ("q", "inf"), ("k", "nan"), ("k", "inf"), ("v", "nan"),
    ("v", "inf"), ("rows", "nan")])
def test_infinities_and_nan_reach_the_rows_they_reach_whole(cuda, dtype, d, corr, where, value):
    """A NaN or infinite query row, a key row in a middle part, a value row
    that later rows see and the tile's earlier rows only multiply by zero, and
    NaN query rows of whole tiles: the output is NaN and infinite exactly where
    a whole tile's is.  Also through ``out`` of other strides."""
    g = torch.Generator().manual_seed(d)
    n, lk = 200, 5000
    q, k, v = (torch.randn((h, m, d), generator=g) for h, m in ((8, n), (2, lk), (2, lk)))
    x = float(value)
    if where == "q":
        q[3, 70, 2] = x
    elif where == "rows":
        q[:, 60:130] = x
    elif where == "k":
        k[0, 2100, 1] = x
    else:
        v[1, lk - 60, 3] = x
    q, k, v = (t.to(dtype).to(cuda) for t in (q, k, v))
    config = FPV2Config(alpha=0.1, sink_tokens=128, tile_q=32, mean_correction=corr)
    q, blocks = _pad(q, 32), -(-(lk - n + -(-n // 32) * 32) // 128)
    k, v = (_pad(t, 128 * blocks) for t in (k, v))
    # (lists of the finite inputs: every tile keeps some and prunes some)
    mask = torch.ones((2, q.shape[1] // 32, blocks), dtype=torch.bool, device=cuda)
    mask[:, :, 4:9] = False
    lists = compact_block_indices(mask, config=config, offset=lk - n, query_length=n, key_length=lk)
    pk, pv = pool_blocks(k), pool_blocks(v)
    whole, even = (o[:, :n].float() for o in _both(q, k, v, pk, pv, lists, config, n, lk))
    assert torch.equal(whole.isnan(), even.isnan()) and torch.equal(whole.isinf(), even.isinf())
    keep = whole.isfinite()
    assert not bool(keep.all())
    _close(whole[keep].to(dtype), even[keep].to(dtype), 1e-2)
    wide = torch.full((n, 8, d + 8), float("nan"), dtype=dtype, device=cuda)
    _launch_attention(q, k, v, pk, pv, *lists, wide[:, :, :d].transpose(0, 1), device=q.device,
                      scale=d ** -0.5, config=config, offset=lk - n, query_length=n, key_length=lk,
                      num_blocks=blocks, padded_query_length=q.shape[1], out_rows=n, balanced=True,
                      split_tiles=q.shape[1] // 32)
    assert torch.equal(wide[:, :, :d].transpose(0, 1).float().nan_to_num(7.0, 8.0, 9.0),
                       even.nan_to_num(7.0, 8.0, 9.0))
    assert bool(wide[:, :, d:].isnan().all())


def test_workspace_is_checked(cuda):
    """No tiles where whole tiles fill the chip; a short workspace is refused."""
    lib = _lib.load()

    def params(length, hq, hkv):
        nb = length // 128
        return _lib.AttnParams(
            query_heads=hq, kv_heads=hkv, head_dim=64, padded_query_length=length,
            query_length=length, out_rows=length, key_length=length, num_blocks=nb, offset=0,
            block_k=128, tile_q=32, mean_correction=1, scale=0.125, q_head_stride=length * 64,
            q_row_stride=64, k_head_stride=length * 64, k_row_stride=64, v_head_stride=length * 64,
            v_row_stride=64, o_head_stride=length * 64, o_row_stride=64, pooled_head_stride=nb * 64)

    assert lib.fpv2_sparse_attention_balanced_tiles(params(65536, 32, 8)) == 0
    p = params(1024, 4, 1)
    assert lib.fpv2_sparse_attention_balanced_tiles(p) == 32
    assert lib.fpv2_sparse_attention_balanced_workspace_bytes(p, 33) == _lib.FPV2_ERR_ARGUMENT
    need = lib.fpv2_sparse_attention_balanced_workspace_bytes(p, 32)
    assert need > 0
    x = torch.zeros((4, 1024, 64), dtype=torch.bfloat16, device=cuda)
    lists = torch.zeros((32, 8), dtype=torch.int32, device=cuda)
    ws = torch.empty(need - 16, dtype=torch.uint8, device=cuda)
    status = lib.fpv2_sparse_attention_balanced(
        x.data_ptr(), x.data_ptr(), x.data_ptr(), x.data_ptr(), x.data_ptr(), lists.data_ptr(),
        lists.data_ptr(), lists.data_ptr(), lists.data_ptr(), torch.empty_like(x).data_ptr(),
        _lib.BF16, p, 32, ws.data_ptr(), need - 16, _lib.stream_ptr(cuda))
    assert status == _lib.FPV2_ERR_ARGUMENT
    assert b"workspace" in lib.fpv2_last_error()
