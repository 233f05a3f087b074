"""AUTO takes another form for batches of at most 256 problems: the bits are those of the
larger batch's form, on both sides of the line."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("prec,dt,s", [(K.PREC_F64, torch.float64, 64), (K.PREC_F16_F32, torch.float16, 128),
                                       (K.PREC_F16_F32, torch.float16, 256),
                                       (K.PREC_BF16_F32, torch.bfloat16, 128),
                                       (K.PREC_BF16_F32, torch.bfloat16, 256)], ids=str)
def test_small_batches_keep_their_bits(prec, dt, s, layout, dev):
    print(f"\n[case] {prec} {s} {layout}", flush=True)
    g = torch.Generator(device=dev).manual_seed(s)
    A, B = (torch.randn((257, s, s), generator=g, device=dev).to(dt) for _ in range(2))
    C0 = torch.randn((257, s, s), generator=g, device=dev).to(torch.float64 if s == 64 else torch.float32)
    full = K.block_gemm(A, B, C0.clone(), b_layout=layout, alpha=2.0, beta=-1.0)
    for n in (1, 255, 256):
        part = K.block_gemm(A[:n], B[:n], C0[:n].clone(), b_layout=layout, alpha=2.0, beta=-1.0)
        assert torch.equal(part, full[:n]), n
