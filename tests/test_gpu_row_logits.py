"""The head of one position (``fpv2_row_logits``) against float64.

A sum of C products in float32 with one rounding per step is off by at most
C 2^-24 sum |x w|.
"""

from __future__ import annotations

import pytest
import torch

from fpv2.prefill_harness import ChunkedPrefillRunner, DecoderShape, RandomDecoder, _row_logits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("vocab", "cols"), [
    (1, 8),         # one row, one lane
    (15, 512),      # a ragged last workgroup, one whole step of columns
    (17, 520),      # a second workgroup of one row, one lane in the last step
    (1000, 2560),   # an unrolled turn of five steps
    (33, 4104),     # an unrolled turn, whole steps and a remainder
])
def test_row_logits(cuda, dtype, vocab, cols):
    g = torch.Generator().manual_seed(vocab + cols)
    x = torch.randn(cols, generator=g).to(dtype)
    # a wider parent buffer: the row stride differs from cols
    w = (0.02 * torch.randn((vocab, cols + 8), generator=g)).to(dtype)
    got = _row_logits(x.to(cuda), w.to(cuda)[:, :cols]).cpu().double()
    xd, wd = x.double(), w[:, :cols].double()
    bound = cols * 2.0 ** -24 * (wd.abs() @ xd.abs())
    assert got.shape == (vocab,) and bool(((got - wd @ xd).abs() <= bound).all())


def test_refused_forms(cuda):
    x = torch.zeros(24, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(ValueError, match="multiples"):
        _row_logits(x[:12], torch.zeros((3, 12), dtype=torch.bfloat16, device=cuda))
    with pytest.raises(ValueError, match="aligned"):
        _row_logits(x[4:20], torch.zeros((3, 16), dtype=torch.bfloat16, device=cuda))
    with pytest.raises(ValueError, match="dtype"):
        _row_logits(x, torch.zeros((3, 24), dtype=torch.float16, device=cuda))


@pytest.mark.parametrize("layout", ["columns", "odd rows", "off the grid", "gradient"])
def test_prefill_takes_any_layout_of_the_embedding(cuda, layout):
    """An embedding that the kernel cannot read in place still gives the first
    logits (through a library product, rounded to bfloat16: half a unit in the
    last place, 2^-9, and the float32 sums' order)."""
    shape = DecoderShape(layers=1, hidden=256, query_heads=4, kv_heads=1, head_dim=64,
                         intermediate=512, vocab=300)
    model = RandomDecoder(shape, device=cuda, seed=3)
    tokens = torch.arange(200, device=cuda)
    want = ChunkedPrefillRunner(model, 256).prefill(tokens, 128)
    w = model.embed
    if layout == "columns":
        model.embed = w.T.contiguous().T
    elif layout == "odd rows":
        wide = torch.zeros((300, 257), dtype=w.dtype, device=cuda)
        wide[:, :256] = w
        model.embed = wide[:, :256]
    elif layout == "off the grid":
        flat = torch.zeros(w.numel() + 1, dtype=w.dtype, device=cuda)
        flat[1:] = w.reshape(-1)
        model.embed = flat[1:].view(w.shape)
    else:
        model.embed = w.clone().requires_grad_()
    got = ChunkedPrefillRunner(model, 256).prefill(tokens, 128)
    assert got.dtype == torch.float32 and got.requires_grad == (layout == "gradient")
    assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
