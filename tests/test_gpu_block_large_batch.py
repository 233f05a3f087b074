"""1D forms of 2-byte inputs hold fewer waves a SIMD from 80 MB (eight waves and more) or 100 MB a
call, and for more than eight repetitions.  The same products in the same order: the bits of
the same problems in small calls, and the plain FP32 product within its rounding."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# m = n, k, waves of the 1D form
FORMS = [(64, 64, 1), (64, 64, 4), (64, 16, 2), (64, 32, 4), (128, 16, 8), (128, 32, 2), (128, 32, 8),
         (128, 128, 4), (192, 16, 12), (192, 32, 4), (256, 32, 8), (224, 224, 14)]


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("form", FORMS, ids=str)
def test_either_side_of_the_limit(form, dt, layout, dev):
    e, k, waves = form
    print(f"\n[case] {form} {dt} {layout}", flush=True)
    problem = 2 * e * k * 2 + e * e * 4
    limit = (80_000_000 if waves >= 8 else 100_000_000) // problem  # the last one below
    g = torch.Generator(device=dev).manual_seed(e + k)
    A = torch.randn((limit + 1, e, k), generator=g, device=dev).to(dt)
    B = torch.randn((limit + 1, e, k) if layout == "nk" else (limit + 1, k, e), generator=g, device=dev).to(dt)
    kw = dict(partition="1d", ranks=waves, b_layout=layout)
    above, below = K.block_gemm(A, B, **kw), K.block_gemm(A[:limit], B[:limit], **kw)
    assert torch.equal(above[:limit], below)
    for s in (0, limit - 15):  # and in small calls
        assert torch.equal(K.block_gemm(A[s:s + 16], B[s:s + 16], **kw), above[s:s + 16])
    Bt = (B.transpose(1, 2) if layout == "nk" else B)[:16].float().contiguous()
    ref = torch.bmm(A[:16].float(), Bt)
    bound = torch.bmm(A[:16].float().abs(), Bt.abs())
    assert torch.all((above[:16] - ref).abs() <= 2 * k * 2.0 ** -24 * bound)
    for iters in (8, 9):
        many, few = (K.block_gemm(A[:n], B[:n], iters=iters, **kw) for n in (limit + 1, 16))
        assert torch.equal(many[:16], few), iters
