"""FP64 with B stored K x N: what the query reports is what a call runs.  Where nothing is asked
for or measured that is the partition's persistent form of 4 x 4 waves from 64 x 64 up; a measured choice
is taken as it stands; asking for the persistent form stays refused.  CPU only."""
import pytest

import kami_amd as K
from kami_amd import _abi


@pytest.fixture(autouse=True)
def _clean():
    K.lib().kami_tune_clear()
    yield
    K.lib().kami_tune_clear()


@pytest.mark.parametrize("edge,pipe", [(16, 1), (32, 1), (64, 2), (128, 2)])
def test_default_form(edge, pipe):
    assert K.query(edge, edge, edge, K.PREC_F64, b_layout="kn")["pipeline"] == pipe
    assert K.query(edge, edge, edge, K.PREC_F64, b_layout="kn", iters=2)["pipeline"] == 1
    assert K.query(edge, edge, edge, K.PREC_F64, b_layout="kn", pipeline=1)["pipeline"] == 1
    assert K.query(edge, edge, edge, K.PREC_F64, b_layout="kn", partition="1d")["pipeline"] == 1


@pytest.mark.parametrize("ranks", [2, 4])
def test_partition_without_a_form(ranks):
    kn = K.query(64, 64, 64, K.PREC_F64, partition="2d", ranks=ranks, b_layout="kn")
    assert kn == K.query(64, 64, 64, K.PREC_F64, partition="2d", ranks=ranks, pipeline=2 if ranks == 4 else 1)


@pytest.mark.parametrize("prec", [K.PREC_F64, K.PREC_F16_F32, K.PREC_BF16_F32])
def test_asking_for_it_stays_refused(prec):
    with pytest.raises(K.KamiError):
        K.query(64, 64, 64, prec, partition="2d", ranks=4, pipeline=2, b_layout="kn")


@pytest.mark.parametrize("pipe", [1, 2])
def test_measured_choice_is_taken(tmp_path, pipe):
    f = tmp_path / "t.txt"
    f.write_text(f"kami-tune 1\nblock 0 64 64 64 2 2 {pipe}\nblock 1 64 64 64 2 2 {pipe}\n")
    assert K.lib().kami_tune_load(str(f).encode()) == _abi.OK
    got = K.query(64, 64, 64, K.PREC_F64, b_layout="kn")
    assert (got["partition"], got["ranks"], got["pipeline"]) == (2, 2, pipe)
    # 2-byte inputs have no persistent form for K x N
    assert K.query(64, 64, 64, K.PREC_F16_F32, b_layout="kn")["pipeline"] == 1
