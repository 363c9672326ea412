"""The row path of block scoring and selection (raw scores, masks without
lists, non-positive scales, float32), at the edges of its tiles: 32-row
groups that span query heads or end inside one, 32-block chunks, 512-block
windows, against the float64 oracle.

Scores are float32 sums of D products accumulated in some order: each of the
D roundings is at most 2^-24 of the partial sum, so |error| <= D 2^-24
sum_d |q_d k_d| |scale| (and half an ulp for the scale).  Masks must agree
outside the 1e-4 band around alpha.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import to_np
from fpv2 import FPV2Config, block_scores_and_select
from oracle import fpv2_oracle as orc

pytestmark = pytest.mark.gpu

BAND = 1e-4


def _cfg(c):
    return orc.OracleConfig(**{f: getattr(c, f) for f in orc.OracleConfig.__dataclass_fields__})


def _check(cuda, dtype, d, heads, tq, nb, qlen, offset, block, scale_sign=1.0, seed=0):
    hq, hkv = heads
    g = torch.Generator().manual_seed(seed + nb + d)
    lq_pad = -(-qlen // tq) * tq
    q = torch.zeros((hq, lq_pad, d), dtype=dtype)
    q[:, :qlen] = torch.randn((hq, qlen, d), generator=g).to(dtype)
    pk = (0.7 * torch.randn((hkv, nb, d), generator=g)).to(dtype)
    scale = scale_sign * d ** -0.5
    config = FPV2Config(block_k=block, tile_q=tq, alpha=0.2, sink_tokens=block,
                        window_tokens=2 * block, last_n_blocks=1)
    sel, scores = block_scores_and_select(q.to(cuda), pk.to(cuda), scale=scale, config=config,
                                          offset=offset, query_length=qlen)
    alone, none = block_scores_and_select(
        q.to(cuda), pk.to(cuda), scale=scale, offset=offset, query_length=qlen,
        config=FPV2Config(**{**config.__dict__, "score_chunk_tiles": 2}))
    assert none is None and torch.equal(sel, alone)
    qn, kn = to_np(q).astype(np.float64), to_np(pk).astype(np.float64)
    ref, ref_scores, ratio = orc.block_scores_and_select(
        qn, kn, scale=scale, config=_cfg(config), offset=offset, query_length=qlen,
        return_ratio=True)
    near = np.abs(ratio - config.alpha) <= BAND
    assert not ((to_np(sel) != ref) & ~near).any()
    mass = np.einsum("hgnd,hbd->hgnb", np.abs(qn).reshape(hkv, hq // hkv, lq_pad, d), np.abs(kn))
    bound = (d + 2) * 2.0 ** -24 * mass * abs(scale) + 1e-30
    assert (np.abs(to_np(scores) - ref_scores) <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 96, 128, 256])
@pytest.mark.parametrize(("heads", "tq", "nb", "qlen", "offset"), [
    ((1, 1), 1, 1, 3, 0),        # one row, one block
    ((6, 2), 24, 33, 500, 28),   # groups across heads, a chunk of one block
    ((8, 1), 40, 65, 333, 700),  # several groups per wave, ragged last tile
    ((4, 4), 160, 31, 450, 40),  # five groups of one head
])
def test_scores_and_masks_match_oracle(cuda, dtype, d, heads, tq, nb, qlen, offset):
    _check(cuda, dtype, d, heads, tq, nb, qlen, offset, 16 if nb > 1 else 64)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nb", [511, 512, 513, 1100])
def test_windows_of_blocks(cuda, dtype, nb):
    """Blocks past the first 512-block window, seen and unseen."""
    _check(cuda, dtype, 64, (4, 2), 32, nb, 90, nb * 4 - 130, 4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("d", "heads", "tq", "nb", "qlen"), [
    (128, (1, 1), 16, 300, 40),   # one row group, all waves on the chunks
    (64, (1, 1), 33, 300, 70),    # a second row group of one row
    (128, (2, 1), 32, 380, 70),   # 64 rows a wave, all waves on the chunks
    (128, (3, 1), 32, 200, 70),   # two waves on the rows, the second half full
    (64, (4, 1), 48, 390, 100),   # three turns of two waves
    (96, (4, 2), 130, 260, 300),  # five turns of two waves, the last of four rows
    (128, (8, 2), 72, 40, 100),   # five turns of four waves, two chunks
    (128, (8, 1), 72, 1030, 150),  # nine turns, three windows of blocks
])
def test_rows_and_chunks_dealt_to_the_waves(cuda, dtype, d, heads, tq, nb, qlen):
    _check(cuda, dtype, d, heads, tq, nb, qlen, 4 * nb - qlen - 3, 4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("d", "heads", "tq", "nb", "qlen"), [
    (256, (4, 1), 32, 64, 100),  # the mask alone from the owner kernel
    (256, (4, 1), 40, 70, 100),  # its second pass of rows
    (256, (2, 1), 40, 130, 90),  # fewer rows than a pass
])
def test_masks_of_the_owner_kernel(cuda, dtype, d, heads, tq, nb, qlen):
    _check(cuda, dtype, d, heads, tq, nb, qlen, 4 * nb - qlen - 3, 4)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("sign", [-1.0, 0.0])
def test_scales_that_are_not_positive(cuda, dtype, sign):
    _check(cuda, dtype, 128, (4, 2), 32, 40, 600, 0, 16, scale_sign=sign)


def test_infinite_and_nan_queries_leave_other_tiles_alone(cuda):
    """A NaN or infinite query row decides its own tiles only; its scores
    carry it."""
    g = torch.Generator().manual_seed(2)
    q = torch.randn((2, 128, 64), generator=g)
    pk = torch.randn((1, 8, 64), generator=g)
    config = FPV2Config(block_k=16, tile_q=32, alpha=0.2, sink_tokens=16, window_tokens=16)
    clean, _ = block_scores_and_select(q.to(cuda), pk.to(cuda), scale=0.125, config=config)
    q[0, 40, 3] = float("nan")
    q[1, 70, 5] = float("inf")
    sel, scores = block_scores_and_select(q.to(cuda), pk.to(cuda), scale=0.125, config=config)
    assert torch.equal(sel[:, [0, 3]], clean[:, [0, 3]])
    assert bool(scores[0, 0, 40].isnan().all()) and not bool(scores[0, 1, 70].isfinite().any())
    assert bool(scores[0, 0, 39].isfinite().all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 96, 128, 256])
@pytest.mark.parametrize("alpha", [0.0, 0.2])
@pytest.mark.parametrize("poison", ["q inf", "q -inf", "q rows nan", "k nan", "k inf", "k -inf",
                                    "q and k", "large"])
def test_masks_of_infinities_and_nan_do_not_depend_on_the_scores(cuda, dtype, d, alpha, poison):
    """The mask alone (the streaming kernel up to D = 128, the owner kernel for
    the 65 blocks of D = 256) is the mask that comes with the scores (the row
    path) where logits are infinite or NaN, and at 200 times the usual logits."""
    inf = float("inf")
    for heads, tq, bk, nb, qlen, offset in [((4, 1), 32, 16, 65, 333, 700),
                                            ((6, 2), 40, 16, 33, 500, 20),
                                            ((8, 2), 128, 128, 20, 2500, 0)]:
        g = torch.Generator().manual_seed(d + nb)
        q = torch.randn((heads[0], -(-qlen // tq) * tq, d), generator=g)
        q[:, qlen:] = 0
        pk = 0.7 * torch.randn((heads[1], nb, d), generator=g)
        at = qlen // 2 + 3
        if poison in ("q inf", "q and k"):
            q[:, at:at + 40:7, 2] = inf
            q[-1, at + 3, 5] = -inf
        if poison == "q -inf":  # logits of -inf before a wave's first finite one
            pk[:, :, 3] = pk[:, :, 3].abs() + 0.1
            q[:, :qlen:3, 3] = -inf
        if poison == "q rows nan":
            q[:, at:at + 70] = float("nan")
        if poison == "k nan":
            pk[0, nb // 2, 1] = float("nan")
        if poison in ("k inf", "q and k"):
            pk[-1, nb // 2, 2] = inf
        if poison == "k -inf":
            pk[0, nb // 3, 4] = -inf
        if poison == "large":
            q, pk = 200 * q, 200 * pk
        masks = []
        for chunk in (None, 1):
            config = FPV2Config(block_k=bk, tile_q=tq, alpha=alpha, sink_tokens=bk,
                                window_tokens=2 * bk, last_n_blocks=1, score_chunk_tiles=chunk)
            masks.append(block_scores_and_select(q.to(dtype).to(cuda), pk.to(dtype).to(cuda),
                                                 scale=d ** -0.5, config=config, offset=offset,
                                                 query_length=qlen)[0])
        assert torch.equal(*masks), (heads, int((masks[0] != masks[1]).sum()))


def _scored(cuda, q, pk, config, repeat=3):
    """(mask, scores, least milliseconds) of a call with its raw scores."""
    best = float("inf")
    for _ in range(repeat):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        sel, scores = block_scores_and_select(q, pk, scale=q.shape[-1] ** -0.5, config=config)
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end))
    return sel, scores, best


@pytest.mark.parametrize(("dtype", "heads", "tq", "length", "nb"), [
    (torch.bfloat16, 4, 16, 16384, 8192),  # two heads a row group, sixteen windows of blocks
    (torch.float16, 3, 40, 131080, 2049),  # groups that end and begin inside heads
    (torch.float32, 4, 16, 16384, 8192),
])
def test_row_groups_over_2_gib_of_scores(cuda, dtype, heads, tq, length, nb):
    """Row groups whose rows lie 2 GiB of scores and more apart are served by
    the same kernel with 64-bit addresses: scores of rows all over the call
    against float64, mask against the mask alone, and no slower than a call of
    a quarter of the scores by more than twice the work (the kernel that takes
    one thread per block was 250 times slower)."""
    d = 64
    g = torch.Generator(device=cuda).manual_seed(heads)
    q = torch.randn((heads, length, d), generator=g, device=cuda).to(dtype)
    pk = (0.7 * torch.randn((1, nb, d), generator=g, device=cuda)).to(dtype)
    block = -(-length // nb)
    config = FPV2Config(block_k=block, tile_q=tq, alpha=0.2, sink_tokens=block, window_tokens=block)
    assert (32 // tq + 2) * length * nb * 4 >= 2 ** 31
    sel, scores, ms = _scored(cuda, q, pk, config)
    alone, _ = block_scores_and_select(q, pk, scale=d ** -0.5, config=FPV2Config(
        **{**config.__dict__, "score_chunk_tiles": 1}))
    # (energies round to either side of alpha: a few flags of millions)
    assert int((sel != alone).sum()) <= 1e-4 * sel.numel()
    rows = torch.randint(0, length, (200,), generator=g, device=cuda)
    rows[:4] = torch.tensor([0, tq - 1, tq, length - 1])
    want = q[:, rows].double() @ pk[0].double().T * d ** -0.5
    mass = q[:, rows].double().abs() @ pk[0].double().abs().T * d ** -0.5
    assert bool(((scores[0][:, rows].double() - want).abs() <= (d + 2) * 2.0 ** -24 * mass).all())
    del scores, want, mass
    quarter = -(-length // 4 // tq) * tq
    _, _, ms4 = _scored(cuda, q[:, :quarter].contiguous(), pk, config)
    assert ms < 8 * ms4 + 0.2


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("last", [0, 3, 2 ** 31, 2 ** 33, 2 ** 63 - 1])
def test_dense_tails_of_any_length(cuda, d, last):
    """A dense tail past 32 bits covers every tile, in masks with and without
    scores."""
    g = torch.Generator().manual_seed(d)
    q = torch.randn((2, 512, d), generator=g).to(torch.bfloat16).to(cuda)
    pk = torch.randn((1, 130, d), generator=g).to(torch.bfloat16).to(cuda)
    tiles = torch.arange(16)[:, None]
    seen = torch.arange(130)[None] * 4 <= 8 + tiles * 32 + 31
    for chunk in (None, 1):
        # (no energy reaches ten times the largest)
        config = FPV2Config(block_k=4, tile_q=32, alpha=10.0, sink_tokens=0, window_tokens=0,
                            last_n_blocks=last, score_chunk_tiles=chunk)
        sel, _ = block_scores_and_select(q, pk, scale=0.1, config=config, offset=8)
        # (a window of 0 keeps the blocks that reach into the tile's first row on)
        own = torch.arange(130)[None] * 4 + 4 > 8 + tiles * 32
        assert torch.equal(sel[0].cpu(), seen & (own | (tiles >= 16 - last)))
