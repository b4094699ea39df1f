"""natsl_wgrad with tiles of 192 and of 256 columns: widths around either, last tiles that a few columns fill, weights of a row of tiles and a few rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


# (rows of dY, columns of x): one tile of either width and eight columns more or less; several tiles; token slices that end inside a stage
@pytest.mark.parametrize("T,D,widths", [(40, 184, (264,)), (65, 192, (256, 8)), (97, 200, (248,)), (130, 248, (136,)), (70, 256, (512, 24)), (1999, 384, (1152, 16)),
                                        (700, 392, (40,)), (2011, 512, (768, 768)), (3001, 576, (2304, 32)), (2500, 1536, (1152, 1152, 2304, 2304, 16)),
                                        (4097, 1024, (768, 768, 1536, 1536, 16))])
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
