"""Other Python threads run while a native call is in the library.  The entry points are replaced
by the C library's usleep (a plan handle, or the address of a descriptor, is the time)."""
import ctypes
import threading
import time

import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture
def sleeping():
    f, real = K._fast(), K._fast_entry_points()
    usleep = ctypes.cast(ctypes.CDLL(None).usleep, ctypes.c_void_p).value
    f.bind(K.check, real[0], real[1], usleep, *real[3:])
    yield f
    f.bind(K.check, *real)


def test_other_threads_run_during_a_call(sleeping, dev):
    steps, stop = [0], threading.Event()

    def count():
        while not stop.is_set():
            steps[0] += 1
            time.sleep(0.001)
    t = threading.Thread(target=count)
    t.start()
    torch.cuda.current_stream()
    before = steps[0]
    assert sleeping.batched_execute(300000) is True  # 0.3 s
    during = steps[0] - before
    stop.set()
    t.join()
    assert during > 20
