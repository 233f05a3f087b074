"""Block SpMM over many and over few tiles a row: 16 columns, column groups of one and two atoms,
narrow tiles for a long B, at widths on either side of each rule, exact on integers against
the products of the blocks."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# block rows, block columns, blocks a row, columns of B
CASES = [(513, 7, 1, 16), (512, 7, 1, 16), (300, 9, 2, 32), (300, 9, 3, 32), (1025, 5, 1, 32),
         (700, 20, 2, 48), (700, 20, 2, 64), (600, 20, 3, 80), (400, 20, 6, 112), (257, 20, 1, 128),
         (1100, 30, 8, 144), (800, 40, 16, 272), (900, 2100, 3, 96), (900, 2100, 2, 96), (150, 2100, 4, 208)]


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("dt", [torch.float16, torch.float64], ids=["f16", "f64"])
def test_exact(dt, bs, layout, dev):
    out = torch.float64 if dt == torch.float64 else torch.float32
    g = torch.Generator(device=dev).manual_seed(bs)
    for mb, nb, per, n in CASES:
        print(f"\n[case] {dt} {bs} {layout} {mb} {nb} {per} {n}", flush=True)
        ci = torch.sort(torch.rand((mb, nb), generator=g, device=dev).argsort(1)[:, :per], 1).values
        V = torch.randint(-2, 3, (mb * per, bs, bs), generator=g, device=dev).to(dt)
        B = torch.randint(-2, 3, (nb * bs, n), generator=g, device=dev).to(dt)
        A = K.BsrMatrix(mb, nb, bs, torch.arange(0, mb * per + 1, per, dtype=torch.int32, device=dev),
                        ci.reshape(-1).int(), V)
        wide = torch.full((mb * bs, n + 3), 9.0, dtype=out, device=dev)
        C = wide[:, 1:1 + n]
        C.copy_(torch.randint(-3, 4, (mb * bs, n), generator=g, device=dev))
        ref = -C.double()
        parts = B.float().view(nb, bs, n)
        for p in range(per):  # exact in FP32 too
            ref += 2 * torch.bmm(V.view(mb, per, bs, bs)[:, p].float().contiguous(), parts[ci[:, p]]).view(mb * bs, n).double()
        K.bsr_spmm(A, B if layout == "kn" else B.t().contiguous(), C, b_layout=layout, alpha=2.0, beta=-1.0)
        assert torch.equal(C.double(), ref)
        assert bool((wide[:, :1] == 9.0).all()) and bool((wide[:, 1 + n:] == 9.0).all())
