"""SpGEMM numeric phase at the edges of its searches and staging: output counts that leave
waves of a workgroup idle, block rows found in one, two and three rounds of the 256-way
search, rows of A longer than the 64 entries compared at once, in every precision and
block size.  Small integers make every sum exact; the reference multiplies block pairs in
FP64."""
import numpy as np
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f64": torch.float64}
# (block rows of A, inner blocks, block columns, filled rows, blocks per filled row, blocks per row of B)
SHAPES = [(1, 1, 1, 1, 1, 1), (3, 5, 7, 3, 2, 3), (300, 40, 30, 300, 2, 1), (70000, 9, 4, 40, 3, 2),
          (2, 150, 20, 2, 130, 4)]


def pattern(rng, rows, cols, filled, per):
    at = np.sort(rng.choice(rows, filled, replace=False))
    n = np.zeros(rows, np.int64)
    n[at] = per
    rp = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(cols, per, replace=False)) for _ in at]).astype(np.int32)
    return rp, ci


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("prec", list(DT))
def test_numeric_edges_exact(prec, bs, shape, dev):
    print(f"\n[case] {prec} {bs} {shape}", flush=True)
    mb, kb, nb, filled, pa, pb = shape
    rng = np.random.default_rng(mb + bs)
    rpA, ciA = pattern(rng, mb, kb, filled, pa)
    rpB, ciB = pattern(rng, kb, nb, kb, pb)
    vA = rng.integers(-2, 3, (len(ciA), bs, bs)).astype(np.float64)
    vB = rng.integers(-2, 3, (len(ciB), bs, bs)).astype(np.float64)
    t = lambda x: torch.from_numpy(x).to(dev)  # noqa: E731
    C = K.bsr_spgemm(K.BsrMatrix(mb, kb, bs, t(rpA), t(ciA), t(vA).to(DT[prec])),
                     K.BsrMatrix(kb, nb, bs, t(rpB), t(ciB), t(vB).to(DT[prec])), alpha=2.0)
    ref = {}
    for i in np.nonzero(np.diff(rpA))[0]:
        for a in range(rpA[i], rpA[i + 1]):
            for b in range(rpB[ciA[a]], rpB[ciA[a] + 1]):
                key = (int(i), int(ciB[b]))
                ref[key] = ref.get(key, 0.0) + 2.0 * (vA[a] @ vB[b])
    rp, ci, v = C.rowptr.cpu().numpy(), C.colidx.cpu().numpy(), C.vals.double().cpu().numpy()
    rows = np.repeat(np.arange(mb), np.diff(rp))
    assert [(int(r), int(c)) for r, c in zip(rows, ci)] == sorted(ref)
    np.testing.assert_array_equal(v, np.stack([ref[k] for k in sorted(ref)]))
