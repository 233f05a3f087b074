"""Structure of C = A * B through the fused scan and fill: one row and column, words of the
bitmap left over, rows without blocks, an empty product, the most rows it takes and one more,
and more possible blocks than it allocates for; against the pattern's own boolean product."""
import io

import numpy as np
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# (block rows of A, inner blocks, block columns of B, share of blocks held)
SHAPES = [(1, 1, 1, 1.0), (7, 5, 33, 0.3), (300, 60, 257, 0.02), (40, 30, 20, 0.0), (512, 16, 512, 0.2),
          (513, 16, 512, 0.2), (4096, 8, 64, 0.1), (4097, 8, 63, 0.1), (2, 9, 40000, 0.3)]


def bsr(mask, bs, dev):
    rp = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    ci = np.nonzero(mask)[1].astype(np.int32)
    vals = torch.ones((len(ci), bs, bs), dtype=torch.float16, device=dev)
    return K.BsrMatrix(*mask.shape, bs, torch.from_numpy(rp).to(dev), torch.from_numpy(ci).to(dev), vals)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_structure_exact(shape, dev):
    print(f"\n[case] {shape}", flush=True)
    mb, kb, nb, share = shape
    rng = np.random.default_rng(mb)
    ma, mm = rng.random((mb, kb)) < share, rng.random((kb, nb)) < share
    A, B = bsr(ma, 16, dev), bsr(mm, 16, dev)
    ref = ma.astype(np.int64) @ mm.astype(np.int64)
    one = bsr(np.ones((1, 1), bool), 16, dev)
    both = (None, torch.cuda.current_stream())  # the call with both phases in one, and by phase
    for stream, other in (both, both[::-1]):
        K.bsr_spgemm(one, one, stream=other)  # the two ways in turn, with another total
        C = K.bsr_spgemm(A, B, stream=stream)
        rp, ci = C.rowptr.cpu().numpy(), C.colidx.cpu().numpy()
        np.testing.assert_array_equal(np.diff(rp), (ref > 0).sum(1))
        np.testing.assert_array_equal(ci, np.nonzero(ref)[1])
        assert C.colidx.is_contiguous() and C.colidx.dtype == torch.int32 and rp[0] == 0
        np.testing.assert_array_equal(C.vals[:, 0, 0].cpu().numpy(), 16 * ref[ref > 0])
        buf = io.BytesIO()
        torch.save(C.colidx, buf)
        assert buf.getbuffer().nbytes < 4 * len(ci) + 8192
