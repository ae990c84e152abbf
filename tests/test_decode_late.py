"""A step whose waits gave up leaves nothing that a later step takes for its own: neither what its workgroups have published nor
what one of them publishes that starts after the step has been given up, when the number of the next launch is already valid."""
import numpy as np
import pytest

import decode_util as U
from vkllama_amd import capi

pytestmark = pytest.mark.gpu
LAYERS, STEPS = 3, 5


def lost_step(m):
    m.m.wait_test, m.m.wait_polls = 1, 4
    m.step(7, STEPS, 1)
    m.m.wait_test, m.m.wait_polls = 0, 0


@pytest.mark.parametrize("ffn", [160, 256])             # all layers in one launch; a launch per layer (more than 3 x 64)
def test_words_and_flags_of_a_late_workgroup(dev, ffn):
    m = U.Llama(dev, 64, 1, ffn, 96, LAYERS)
    for pos in range(STEPS):
        m.step(3 + pos, pos, 1)
    assert m.status() == 0
    want = m.step(7, STEPS, 0)
    lost_step(m)
    if ffn <= 192:
        # k, q and v of the lost step's first layer (tag 5 * 3 + 1), as one that reads the advanced counter would write them
        words = m.scratch.read(np.uint32, (m.scratch.nbytes // 4,))
        tag = STEPS * LAYERS + 1
        found = words >> 16 == tag
        assert found.sum() >= 3 * 64
        words[found] = ((tag + LAYERS) << 16) | 0x3C00
        m.scratch.write(words)
    else:
        # every flag of every stage raised for the first launch of the next step
        flags = np.full(4 * 8 * 32, (STEPS + 1) * LAYERS + 1, np.uint32)
        capi.check(capi.lib().vkl_memcpy_h2d(m.m.flags, flags.ctypes.data, flags.nbytes, dev.stream))
        dev.sync()
    assert m.status() != 0
    for _ in range(2):
        got = m.step(7, STEPS, 1)
        assert m.status() == 0
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    m.close()
