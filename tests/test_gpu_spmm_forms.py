"""Block SpMM in each of its forms (a row's stages shared by 2, 4, 8 and 16 waves, chosen by
the number of tiles and the rows' length) at ragged widths, in both layouts of B and with C
at any element offset.  Small integers make every sum exact, so C equals the oracle's check
loop bit for bit; the FP64 sums of N(0, 1) values stay within gamma_K |A||B|."""
import numpy as np
import pytest

import kami_amd as K
import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f64": torch.float64}
# (block rows, block columns, blocks per row): few tiles and long rows take 16 or 8 waves
SHAPES = [(3, 70, 66), (40, 40, 24), (300, 12, 3), (2, 5, 1)]


def matrix(rng, mb, nb, per, bs):
    rows = [np.sort(rng.choice(nb, max(0, per - (r % 3)), replace=False)) for r in range(mb)]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return rp, np.concatenate(rows).astype(np.int32), rng.integers(-2, 3, (rp[-1], bs, bs)).astype(np.float64)


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("prec", list(DT))
def test_every_form_exact(prec, bs, layout, dev):
    print(f"\n[case] {prec} {bs} {layout}", flush=True)
    rng = np.random.default_rng(bs)
    out = torch.float64 if prec == "f64" else torch.float32
    for mb, nb, per in SHAPES:
        rp, ci, vals = matrix(rng, mb, nb, per, bs)
        A = K.BsrMatrix(mb, nb, bs, torch.from_numpy(rp).to(dev), torch.from_numpy(ci).to(dev),
                        torch.from_numpy(vals).to(DT[prec]).to(dev))
        for n in (16, 48, 80):
            B = rng.integers(-2, 3, (n, nb * bs)).astype(np.float64)
            Bin = np.ascontiguousarray(B.T) if layout == "kn" else B
            C0 = rng.integers(-3, 4, (mb * bs, n)).astype(np.float64)
            wide = torch.full((mb * bs, n + 5), 9.0, dtype=out, device=dev)
            C = wide[:, 3:3 + n]  # any element offset, odd leading dimension
            C.copy_(torch.from_numpy(C0))
            K.bsr_spmm(A, torch.from_numpy(Bin).to(DT[prec]).to(dev), C, b_layout=layout, alpha=2.0, beta=-1.0)
            ref = 2.0 * oracle.bsr_spmm(mb, nb, bs, rp, ci, vals, Bin, b_kn=layout == "kn") - C0
            np.testing.assert_array_equal(C.double().cpu().numpy(), ref)
            assert bool((wide[:, :3] == 9.0).all()) and bool((wide[:, 3 + n:] == 9.0).all())


@pytest.mark.parametrize("mb,nb,per", SHAPES)
def test_f64_sums_within_bound(mb, nb, per, dev):
    rng = np.random.default_rng(mb)
    bs, n = 32, 48
    rp, ci, vals = matrix(rng, mb, nb, per, bs)
    vals, B = rng.standard_normal(vals.shape), rng.standard_normal((n, nb * bs))
    A = K.BsrMatrix(mb, nb, bs, torch.from_numpy(rp).to(dev), torch.from_numpy(ci).to(dev),
                    torch.from_numpy(vals).to(dev))
    C = K.bsr_spmm(A, torch.from_numpy(B).to(dev)).cpu().numpy()
    ref = oracle.bsr_spmm(mb, nb, bs, rp, ci, vals, B)
    mag = oracle.bsr_spmm(mb, nb, bs, rp, ci, np.abs(vals), np.abs(B))
    k, u = per * bs, 2.0 ** -53
    assert np.all(np.abs(C - ref) <= 2 * k * u / (1 - k * u) * mag * 1.01)  # both sums round
