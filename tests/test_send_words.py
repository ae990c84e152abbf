"""Words to pinned host memory in either width, with and without the word behind them."""
import ctypes as C

import numpy as np
import pytest

from vkllama_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 3, 4, 255, 256, 1020, 1024, 1028, 4097, 32000])
@pytest.mark.parametrize("from_,to", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("word", [True, False])
def test_words_arrive(dev, rng, n, from_, to, word):
    data = rng.integers(0, 2 ** 32, n + from_ + 1, dtype=np.uint32)
    src, w = dev.upload(data), dev.upload(np.array([77], np.uint32))
    host = C.c_void_p()
    capi.check(capi.lib().vkl_host_malloc_h(C.byref(host), 4 * (n + to + 2)))
    try:
        seen = np.ctypeslib.as_array(C.cast(host, C.POINTER(C.c_uint32)), (n + to + 2,))
        seen[:] = 5
        capi.check(capi.lib().vkl_send_words(src.ptr.value + 4 * from_, n, w.ptr if word else None, host.value + 4 * to,
                                             dev.stream))
        dev.sync()
        assert np.array_equal(seen[to:to + n], data[from_:from_ + n])
        assert seen[to + n] == (77 if word else 5) and seen[to + n + 1] == 5 and np.all(seen[:to] == 5)
    finally:
        capi.check(capi.lib().vkl_host_free_h(host))


def test_arguments_are_checked(dev):
    b, lib = dev.alloc(64), capi.lib()
    assert lib.vkl_send_words(b.ptr, 4, None, None, dev.stream) != 0
    assert lib.vkl_send_words(None, 4, None, b.ptr, dev.stream) != 0
    assert lib.vkl_send_words(b.ptr.value + 2, 4, None, b.ptr, dev.stream) != 0
