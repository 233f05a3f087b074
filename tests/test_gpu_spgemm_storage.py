"""What a sparse C holds: no more than 64 KiB or an eighth of its own size beyond its arrays,
whatever the room its columns were first written to; and its structure where that room is too small
(few long rows) or far too large (many products for a block of C)."""
import numpy as np
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def pattern(name, mb):
    P = np.zeros((mb, mb), bool), np.zeros((mb, mb), bool)
    for i in range(2):
        if name == "diagonal":
            np.fill_diagonal(P[i], True)
        elif name == "arrow":
            np.fill_diagonal(P[i], True)
            P[i][0, :] = P[i][:, 0] = True
    if name == "overlap":  # every block of C takes 64 products
        P[0][:, :64] = True
        P[1][:, :8] = True
    return P


@pytest.mark.parametrize("mb", [100, 256, 512])
@pytest.mark.parametrize("name", ["diagonal", "arrow", "overlap"])
def test_storage_and_structure(name, mb, dev):
    print(f"\n[case] {name} {mb}", flush=True)
    bs, mats, dense = 16, [], pattern(name, mb)
    for p in dense:
        rp = np.concatenate([[0], np.cumsum(p.sum(1))]).astype(np.int32)
        ci = np.nonzero(p)[1].astype(np.int32)
        mats.append(K.BsrMatrix(mb, mb, bs, torch.from_numpy(rp).to(dev), torch.from_numpy(ci).to(dev),
                                torch.ones((len(ci), bs, bs), dtype=torch.float16, device=dev)))
    K.bsr_spgemm(*mats)  # whatever a first call keeps
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    C = K.bsr_spgemm(*mats)
    held = torch.cuda.memory_allocated() - before
    own = sum(t.numel() * t.element_size() for t in (C.rowptr, C.colidx, C.vals))
    assert held <= own + max(64 * 1024, own / 8) + 3 * 512
    count = dense[0].astype(np.float64) @ dense[1].astype(np.float64)
    want = count > 0
    rp = np.concatenate([[0], np.cumsum(want.sum(1))])
    assert np.array_equal(C.rowptr.cpu().numpy(), rp)
    assert np.array_equal(C.colidx.cpu().numpy(), np.nonzero(want)[1])
    assert np.array_equal(C.vals[:, 0, 0].double().cpu().numpy(), bs * count[want])
    assert C.colidx.untyped_storage().nbytes() == C.colidx.numel() * 4
