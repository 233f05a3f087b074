"""SpGEMM on either side of 256 block rows, where the search for an output block's row changes, and of
64 repetitions, where a workgroup becomes one wave: exact on integers against a dense product,
with empty rows at both ends and between."""
import numpy as np
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dt", [torch.float16, torch.float64], ids=["f16", "f64"])
@pytest.mark.parametrize("mb", [1, 63, 64, 65, 255, 256, 257, 1000, 4097])
def test_rows(mb, dt, dev):
    print(f"\n[case] {mb} {dt}", flush=True)
    rng, bs = np.random.default_rng(mb), 16
    nb = min(mb, 40)  # A: mb x nb blocks, B: nb x 3
    a = rng.random((mb, nb)) < 0.1
    a[rng.random(mb) < 0.3] = False
    a[0] = a[-1] = False
    a[mb // 2, 0] = True
    b = rng.random((nb, 3)) < 0.6
    b[0, 1] = True
    mats, vals = [], []
    for p in (a, b):
        rp = np.concatenate([[0], np.cumsum(p.sum(1))]).astype(np.int32)
        ci = np.nonzero(p)[1].astype(np.int32)
        v = rng.integers(-2, 3, (len(ci), bs, bs)).astype(np.float64)
        mats.append(K.BsrMatrix(p.shape[0], p.shape[1], bs, torch.from_numpy(rp).to(dev),
                                torch.from_numpy(ci).to(dev), torch.from_numpy(v).to(dt).to(dev)))
        dense = np.zeros((p.shape[0], p.shape[1], bs, bs))
        dense[p] = v
        vals.append(dense)
    C = K.bsr_spgemm(*mats)
    want = (a.astype(int) @ b.astype(int)) > 0
    assert np.array_equal(C.rowptr.cpu().numpy(), np.concatenate([[0], np.cumsum(want.sum(1))]))
    assert np.array_equal(C.colidx.cpu().numpy(), np.nonzero(want)[1])
    ref = np.einsum("ikxy,kjyz->ijxz", *vals, optimize=True)[want]
    assert np.array_equal(C.vals.double().cpu().numpy(), ref)
    for iters in (2, 63, 64):
        many = K.spgemm_numeric(*mats, C.rowptr, C.colidx, iters=iters)
        assert np.array_equal(many.double().cpu().numpy(), iters * ref), iters
