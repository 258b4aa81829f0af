"""The one-group GEMM tiles (dense layers, LM head) where they can go wrong.

Batches on either side of a 16-row block, of an M tile and of the switch to
these tiles; matrices whose last N tile is moved back; K splits that are not
even; FP32 and BF16-valued activations.  Every output against the layer in
float64: its operands carry at least 16 significand bits (an FP32 value as BF16
hi + lo: 2^-17 relative at most), so an output, a sum of products with
independent roundings, is off by about sqrt(2) * 2^-17 * (its terms' root sum
square), 1.1e-5 of the outputs' 2-norm; twice that for the two GEMMs of a dense
layer, with the FP32 accumulation far below.
"""
import ctypes as C

import numpy as np
import pytest

from hummingflight_amd import capi, synth

pytestmark = pytest.mark.gpu

REL = 2.2e-5


def widen(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def matrix(seed, tensor, rows, cols):
    b = capi.DeviceBuffer(2 * rows * cols)
    synth.fill_bf16(b.ptr, rows * cols, seed, tensor, 0.0, 0.05)
    return b, widen(b.download(np.uint16, rows * cols)).reshape(rows, cols)


def activations(seed, T, d, bf16):
    x = np.random.default_rng(seed).standard_normal((T, d)).astype(np.float32)
    return (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32) if bf16 else x


def configure(hidden, max_tokens):
    shape = synth.LayerShape(hidden=hidden, inter=256, n_experts=32, top_k=4, n_group=4, topk_group=2)
    capi.call("hfmoe_configure", shape.config(max_tokens=max_tokens))


def off(got, want):
    return np.linalg.norm(got - want) / np.linalg.norm(want)


# hidden 576: the down projection's second N tile starts at column 64;
# intermediate 1600: the last gate/up tile starts at 1344.
@pytest.mark.parametrize("d,I,tokens", [(576, 1600, (129, 161, 320, 321)), (1024, 8256, (2, 16, 17, 128, 160)),
                                        (512, 320, (130, 500))])
@pytest.mark.parametrize("bf16", [False, True])
def test_dense(hf, d, I, tokens, bf16):
    configure(d, max(tokens))
    bufs, mats = zip(*[matrix(61, i, *s) for i, s in enumerate([(I, d), (I, d), (d, I)])])
    w = capi.DenseWeights(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, None, I, 0)
    capi.call("hfmoe_register_dense_layer", 0, C.byref(w))
    for T in tokens:
        x = activations(T, T, d, bf16)
        xd, out = capi.DeviceBuffer.of(x), capi.DeviceBuffer(4 * T * d)
        capi.call("hfmoe_dense_mlp_forward", 0, xd.ptr, T, out.ptr, None)
        capi.call("hfmoe_synchronize")
        y = out.download(np.float32, T * d).reshape(T, d)
        g, u = x.astype(np.float64) @ mats[0].T, x.astype(np.float64) @ mats[1].T
        want = (g / (1.0 + np.exp(-g)) * u) @ mats[2].T
        assert off(y, want) <= REL, (d, I, T)
        assert max(off(y[t], want[t]) for t in range(T)) <= 4 * REL, (d, I, T)
        xd.free()
        out.free()
    for b in bufs:
        b.free()


# vocabularies of exactly one tile, of one column more than whole tiles (their
# rows of odd length leave in single floats; K of two stages) and of a short
# table split over K.
@pytest.mark.parametrize("d,vocab,tokens", [(1024, 512, (129,)), (128, 1003, (129, 200)), (1024, 8200, (17, 128, 129)),
                                            (1024, 9601, (31, 64, 321))])
def test_lm_head(hf, d, vocab, tokens):
    configure(d, max(tokens))
    head, wt = matrix(62, 0, vocab, d)
    capi.call("hfmoe_register_lm_head", head.ptr, None, vocab)
    for T in tokens:
        h = activations(T, T, d, False)
        hd, lg, tk = capi.DeviceBuffer.of(h), capi.DeviceBuffer(4 * T * vocab), capi.DeviceBuffer(4 * T)
        capi.call("hfmoe_lm_head", hd.ptr, T, lg.ptr, tk.ptr, None)
        capi.call("hfmoe_synchronize")
        logits = lg.download(np.float32, T * vocab).reshape(T, vocab)
        x = h.astype(np.float64)
        want = (x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5)) @ wt.T
        assert off(logits, want) <= REL, (d, vocab, T)
        assert np.array_equal(tk.download(np.int32, T), logits.argmax(1))
        for b in (hd, lg, tk):
            b.free()
    head.free()
