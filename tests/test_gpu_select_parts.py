"""Selection with a tile's rows shared among workgroups
(``fpv2_score_select_parts``) against one workgroup per tile
(``fpv2_score_select``): the scores are the same bits (each is one row's
products, whichever workgroup holds the row), and so are mask and lists
outside the 1e-4 band around alpha, where the parts' energies, added in
another order, may round to the other side."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import to_np
from fpv2 import FPV2Config, _lib
from fpv2.selection import _select_params
from oracle import fpv2_oracle as orc

pytestmark = pytest.mark.gpu


def _call(q, pk, config, qlen, scale, *, offset=0, parts, scored=True, short=0):
    lib = _lib.load()
    (hq, lq, d), (hkv, nb, _) = q.shape, pk.shape
    nt = lq // config.tile_q
    out = {"selected": torch.empty((hkv, nt, nb), dtype=torch.bool, device=q.device)}
    if scored:
        out["scores"] = torch.empty((hkv, hq // hkv, lq, nb), dtype=torch.float32, device=q.device)
    out["ids"], out["pids"] = (torch.empty((hkv, nt, nb), dtype=torch.int32, device=q.device)
                               for _ in range(2))
    out["counts"], out["pcounts"] = (torch.empty((hkv, nt), dtype=torch.int32, device=q.device)
                                     for _ in range(2))
    params = _select_params(q, nb, kv_heads=hkv, scale=scale, config=config, offset=offset,
                            query_length=qlen, padded_length=lq, key_length=nb * config.block_k)
    args = [q.data_ptr(), pk.data_ptr(), _lib.dtype_code(q.dtype), params,
            out["selected"].data_ptr(), _lib.ptr(out.get("scores")), out["ids"].data_ptr(),
            out["counts"].data_ptr(), out["pids"].data_ptr(), out["pcounts"].data_ptr()]
    need = lib.fpv2_score_select_workspace_bytes(params)
    if parts:
        # (filled with NaN: every pair that is read was written)
        ws = torch.full((need // 4 + 4,), float("nan"), device=q.device)
        args += [ws.data_ptr(), need - short]
    run = lib.fpv2_score_select_parts if parts else lib.fpv2_score_select
    _lib.check(run(*args, _lib.stream_ptr(q.device)), "score_select")
    return out, need


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(("heads", "tq", "nb", "qlen", "offset", "d"), [
    ((2, 1), 64, 5, 60, 20, 64),      # one full part: not shared
    ((2, 1), 65, 33, 129, 0, 96),     # two parts, the second of two rows
    ((8, 2), 128, 40, 500, 100, 128),  # eight parts a tile
    ((5, 1), 72, 513, 200, 8000, 256),  # parts across heads, a second window of blocks
])
def test_parts_equal_whole_tiles(cuda, dtype, heads, tq, nb, qlen, offset, d):
    g = torch.Generator().manual_seed(nb)
    lq = -(-qlen // tq) * tq
    q = torch.randn((heads[0], lq, d), generator=g).to(dtype)
    q[:, qlen:] = 0
    pk = (0.7 * torch.randn((heads[1], nb, d), generator=g)).to(dtype)
    config = FPV2Config(block_k=16, tile_q=tq, alpha=0.2, sink_tokens=16, window_tokens=32,
                        last_n_blocks=1)
    scale = d ** -0.5
    _, _, ratio = orc.block_scores_and_select(
        to_np(q).astype(np.float64), to_np(pk).astype(np.float64), scale=scale,
        config=orc.OracleConfig(**{f: getattr(config, f)
                                   for f in orc.OracleConfig.__dataclass_fields__}),
        offset=offset, query_length=qlen, return_ratio=True)
    near = np.abs(ratio - config.alpha) <= 1e-4
    dq, dk = q.to(cuda), pk.to(cuda)
    whole, need = _call(dq, dk, config, qlen, scale, offset=offset, parts=False)
    assert (need > 0) == (heads[0] // heads[1] * tq > 128)
    got, _ = _call(dq, dk, config, qlen, scale, offset=offset, parts=True)
    assert torch.equal(got["scores"], whole["scores"])
    assert not (to_np(got["selected"] != whole["selected"]) & ~near).any()
    same = ~near.any(axis=-1)
    for name in ("ids", "pids", "counts", "pcounts"):
        assert (to_np(got[name])[same] == to_np(whole[name])[same]).all(), name
    if dtype == torch.float32:
        alone, _ = _call(dq, dk, config, qlen, scale, offset=offset, parts=True, scored=False)
        assert torch.equal(alone["selected"], got["selected"])


def test_a_short_workspace_is_refused(cuda):
    q, pk = torch.zeros((4, 128, 64), device=cuda), torch.zeros((1, 2, 64), device=cuda)
    with pytest.raises(ValueError, match="workspace"):
        _call(q, pk, FPV2Config(), 128, 0.125, parts=True, short=4)
