"""SpMM with more tiles than one dispatch holds: FP64 blocks of 16 take 32-column tiles, so 2^23
block rows and 48 columns are 2^24 workgroups of 256 threads, 2^32 work-items.  Every row of C
is written: those with blocks hold the product, all others beta C = 0."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_every_tile_beyond_one_dispatch(dev):
    mb, n, bs = 1 << 23, 48, 16
    if torch.cuda.mem_get_info()[0] < 60e9:
        pytest.skip("needs 52 GB of device memory")
    print(f"\n[case] {mb} block rows, n {n}", flush=True)
    g = torch.Generator(device=dev)
    g.manual_seed(2)
    rows = [0, 12345, mb // 2 - 1, mb // 2, mb - 1]
    vals = torch.randint(-9, 10, (len(rows), bs, bs), generator=g, device=dev).double()
    B = torch.randint(-9, 10, (n, bs), generator=g, device=dev).double()
    stored = torch.zeros(mb + 1, dtype=torch.int32, device=dev)
    stored[[r + 1 for r in rows]] = 1
    rowptr = stored.cumsum(0, dtype=torch.int32)
    A = K.BsrMatrix(mb, 1, bs, rowptr, torch.zeros(len(rows), dtype=torch.int32, device=dev), vals)
    C = torch.full((mb * bs, n), float("nan"), dtype=torch.float64, device=dev)
    K.bsr_spmm(A, B, C)
    for i, r in enumerate(rows):
        block = C[r * bs:(r + 1) * bs]
        assert torch.equal(block, vals[i] @ B.T)
        block.zero_()
    step = 1 << 23
    for at in range(0, mb * bs, step):
        assert int(torch.count_nonzero(C[at:at + step])) == 0
    del C
    torch.cuda.empty_cache()
