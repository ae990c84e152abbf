"""A small fp16 Llama for the C entry points of the decode step, with its scratch memory in reach."""
import ctypes as C

import numpy as np

from vkllama_amd import capi

vp, i32, f32, u32 = C.c_void_p, C.c_int, C.c_float, C.c_uint32
MATRICES = ("wk", "wq", "wv", "wo", "w_gate", "w_up", "w_down")


class Layer(C.Structure):
    _fields_ = [(n, vp) for n in MATRICES + ("attn_norm", "ffn_norm", "kcache", "vcache")]


class Model(C.Structure):
    _fields_ = [(n, i32) for n in ("dim", "n_layers", "n_heads", "head_dim", "ffn", "vocab", "maxlen", "wtype")] + \
               [("eps", f32), ("final_eps", f32)] + \
               [(n, vp) for n in ("layers", "layers_h", "tok_embd", "output", "output_norm", "freqc", "freqs", "scratch")] + \
               [(n, i32) for n in ("attn_split_min", "separate_attn_wo", "wait_polls", "wait_test")] + [("flags", vp)]


def lib():
    so = capi.lib()
    for name, res, args in (("vkl_decode_scratch_bytes", C.c_size_t, [vp]), ("vkl_decode_flags_acquire", i32, [vp]),
                            ("vkl_decode_flags_release", None, [vp]), ("vkl_decode_status", i32, [vp, vp]),
                            ("vkl_decode_step", i32, [vp, vp, u32, i32, vp, vp, vp]),
                            ("vkl_decode_tail", i32, [vp, vp, vp, vp, vp]), ("vkl_decode_tail_supported", i32, [vp])):
        fn = getattr(so, name)
        fn.restype, fn.argtypes = res, args
    return so


class Llama:
    def __init__(self, dev, dim, heads, ffn, vocab, layers, maxlen=64, seed=1):
        rng = np.random.default_rng(seed)
        self.dev, self.keep, m = dev, [], Model()
        self.stream = dev.stream

        def up(a):
            self.keep.append(dev.upload(a))
            return self.keep[-1].ptr.value

        def matrix(n, k):
            return up((rng.standard_normal((n, k)) * k ** -0.5).astype(np.float16))
        m.dim, m.n_layers, m.n_heads, m.head_dim, m.ffn, m.vocab, m.maxlen = dim, layers, heads, dim // heads, ffn, vocab, maxlen
        m.wtype, m.eps, m.final_eps = 1, 1e-5, 1e-6
        table = (Layer * layers)()
        one, cache = up(np.ones(dim, np.float32)), np.zeros(dim * maxlen, np.float16)
        for t in table:
            for n in MATRICES:
                setattr(t, n, matrix(*{"w_gate": (ffn, dim), "w_up": (ffn, dim), "w_down": (dim, ffn)}.get(n, (dim, dim))))
            t.attn_norm = t.ffn_norm = one
            t.kcache, t.vcache = up(cache), up(cache)
        self.table = table
        m.layers, m.layers_h = up(np.frombuffer(bytes(table), np.uint8)), C.addressof(table)
        m.tok_embd, m.output, m.output_norm = matrix(vocab, dim), matrix(vocab, dim), one
        angle = np.arange(maxlen)[:, None] * 10000.0 ** (-np.arange(m.head_dim // 2) * 2.0 / m.head_dim)
        m.freqc, m.freqs = up(np.cos(angle).astype(np.float32)), up(np.sin(angle).astype(np.float32))
        self.scratch = dev.upload(np.zeros(lib().vkl_decode_scratch_bytes(C.byref(m)), np.uint8))
        m.scratch = self.scratch.ptr
        flags = vp()
        capi.check(lib().vkl_decode_flags_acquire(C.byref(flags)))
        m.flags, self.m = flags, m
        self.tok, self.logits = dev.upload(np.zeros(1, np.uint32)), dev.alloc(vocab * 4)

    def launch(self, pos, mode):
        capi.check(lib().vkl_decode_step(C.byref(self.m), self.tok.ptr, pos, mode, self.logits.ptr, None, self.stream))

    def step(self, tok, pos, mode):
        """logits of one token; (nothing waits for them to be right: see status)"""
        self.tok.write(np.array([tok], np.uint32))
        self.launch(pos, mode)
        return self.logits.read(np.float32, (self.m.vocab,))

    def status(self):
        return lib().vkl_decode_status(C.byref(self.m), self.stream)

    def close(self):
        lib().vkl_decode_flags_release(self.m.flags)
