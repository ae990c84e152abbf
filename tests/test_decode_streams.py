"""Two models at once, each on a stream of its own: a launch in which workgroups wait for one another takes one of the two
places of a compute unit where rows are narrow, so two of them fit.  Nobody gives up, and results are those of a model alone."""
import threading

import numpy as np
import pytest

import decode_util as U
from vkllama_amd import capi
from vkllama_amd import model as M

pytestmark = pytest.mark.gpu


# one step of all layers each, of every length of row; beside a launch per layer (ffn > 3 dim; 2048 wide)
@pytest.mark.parametrize("a,b", [((256, 4, 704), (256, 4, 704)), ((512, 8, 1376), (1024, 8, 3072)),
                                 ((1024, 16, 2752), (1024, 8, 3072)), ((512, 4, 1376), (512, 8, 1600)),
                                 ((960, 15, 2880), (2048, 16, 5504))])
def test_steps_on_two_streams(dev, a, b):
    models = []
    for i, (dim, heads, ffn) in enumerate((a, b)):
        models.append(U.Llama(dev, dim, heads, ffn, 640, 2, seed=i))
    other = capi.vp()
    capi.check(capi.lib().vkl_stream_create(capi.C.byref(other)))
    want = []
    for m in models:
        for pos in range(4):
            m.step(5, pos, 0)
        want.append(m.step(5, 4, 0))
    models[1].stream = other
    for _ in range(300):
        for m in models:
            m.launch(4, 1)
    for m, w in zip(models, want):
        assert m.status() == 0
        assert np.array_equal(m.logits.read(np.float32, (640,)).view(np.uint32), w.view(np.uint32))
    models[1].stream = dev.stream
    capi.check(capi.lib().vkl_stream_destroy(other))
    for m in models:
        m.close()


@pytest.mark.parametrize("shapes", [((512, 8, 1376, 8), (512, 8, 1376, 8)), ((1024, 16, 2752, 8), (1536, 12, 4096, 8)),
                                    ((1792, 28, 4768, 8), (512, 8, 1376, 1))])
def test_loops_of_two_threads(shapes):
    models, want, got = [], [], [None, None]
    prompt = np.arange(3, 9).astype(np.uint32)
    for i, (dim, heads, ffn, wtype) in enumerate(shapes):
        cfg = dict(dim=dim, n_layers=3, n_heads=heads, ffn=ffn, vocab=32000, maxlen=256, eps=1e-5, wtype=wtype)
        models.append(M.Llama2(cfg, M.synth_weights(cfg, seed=9 + i)))
        models[i].set_option("decode_mode", 1)
        want.append(list(models[i].generate_greedy(prompt, 128)[0]))

    def loop(i):
        got[i] = [list(models[i].generate_greedy(prompt, 128)[0]) for _ in range(6)]
    threads = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m, w, g in zip(models, want, got):
        assert g == [w] * 6
        assert m.decode_recoveries() == 0
        m.close()
