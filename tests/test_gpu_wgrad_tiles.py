"""natsl_wgrad with tiles of 192 and of 256 columns: widths around either, last tiles that a few columns fill, weights of a row of tiles and a few rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


# (tokens, columns of x, rows of dY) -> the tiles' columns and the slices of the tokens on 256 compute units (test_kernel_choices.py; None: another kernel
# takes it).  One tile of either width and eight columns more or less; several tiles, last ones partly filled; token slices that end inside a stage
CASES = [(40, 184, (264,), 192, 1), (65, 192, (256, 8), 192, 1), (97, 200, (248,), 192, 1), (130, 248, (136,), 256, 2), (70, 256, (512, 24), 256, 1),
         (1999, 384, (1152, 16), 192, 7), (700, 392, (40,), None, 0), (2011, 512, (768, 768), 256, 5), (3001, 576, (2304, 32), 192, 5),
         (2500, 1536, (1152, 1152, 2304, 2304, 16), 192, 1), (4097, 1024, (768, 768, 1536, 1536, 16), 256, 3),
         (900, 360, (520, 24), 192, 6), (997, 1360, (648,), 192, 3), (700, 392, (264,), 256, 6)]


@pytest.mark.parametrize("T,D,widths", [c[:3] for c in CASES])
def test_weight_grads_by_tile_width(T, D, widths):
    from neuralattentionsearchlinear_amd._front import weight_grads
    torch.manual_seed(T)
    x = torch.randn(T, D, device=DEV).bfloat16()
    dys = [torch.randn(T, n, device=DEV).bfloat16() for n in widths]
    out, again = weight_grads(x, dys), weight_grads(x, dys)
    for dy, a, b in zip(dys, out, again):
        ref = dy.double().t() @ x.double()
        # exact products, fp32 sums (T 2^-24 of the sum of magnitudes, far below), one rounding to bf16
        assert bool(((a.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * T ** 0.5).all()), float((a.double() - ref).abs().max())
        assert torch.equal(a, b)
