"""The MLP block of a batch (norm, MoE layer and residual add in the multi-token
path's own kernels) and the x lo-half flag's life from call to call.

The block must be h + forward(norm(h)): the norm in numpy's float32 (its sum of
squares in another order, a few 2^-24), then hfmoe_moe_forward itself, so the
two differ by that and by what it does to the FP32 -> BF16 hi / lo split of x
(16 bits): 2.2e-5 of the layer's part, and far less of h + it.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from hummingflight_amd import capi, synth
from moe_harness import SMALL, Run

pytestmark = pytest.mark.gpu


def forward(r, x, T):
    out = capi.DeviceBuffer(4 * x.size)
    xd = capi.DeviceBuffer.of(x)
    capi.call("hfmoe_moe_forward", r.layer, xd.ptr, T, out.ptr, None)
    capi.call("hfmoe_synchronize")
    y = out.download(np.float32, x.size).reshape(x.shape)
    out.free()
    xd.free()
    return y


def block(r, h, T):
    hd = capi.DeviceBuffer.of(h)
    capi.call("hfmoe_mlp_block", r.layer, hd.ptr, T, None)
    capi.call("hfmoe_synchronize")
    y = hd.download(np.float32, h.size).reshape(h.shape)
    hd.free()
    return y


@pytest.mark.parametrize("dims", [SMALL, dict(hidden=192, inter=64, n_experts=16, top_k=3)], ids=["small", "ragged"])
@pytest.mark.parametrize("n_shared", [1, 0])
def test_block_of_a_batch(hf, dims, n_shared):
    d, most = dims["hidden"], 260
    r = Run(dims, n_group=4, topk_group=2, seed=97, T=most, n_shared=n_shared, with_norm=True)
    w = O.bf16_to_f32(r.dev.norm.download(np.uint16, d))
    rng = np.random.default_rng(97)
    for T in (1, 2, 3, 5, 17, 260):
        h = (3.0 * rng.standard_normal((T, d))).astype(np.float32)
        xn = (h * (1.0 / np.sqrt((h * h).mean(1, dtype=np.float32, keepdims=True) + np.float32(1e-5)))).astype(
            np.float32) * w
        y, moe = block(r, h, T), forward(r, xn, T)
        assert np.linalg.norm(y - h - moe) <= 2.2e-5 * np.linalg.norm(moe) + 2.0 ** -24 * np.linalg.norm(h), T
        assert np.array_equal(y, block(r, h, T)), T  # and again, the same bits
    r.dev.free()


@pytest.mark.parametrize("T", [3, 24, 1024])
def test_bf16_call_with_specials(hf, T):
    # The BF16 call reads x itself; infinities and NaN, whose lo halves in the
    # FP32 call are NaN, must come out as there, and a call after it as before.
    d = SMALL["hidden"]
    r = Run(SMALL, n_group=8, topk_group=4, seed=99, T=T)
    bits = np.random.default_rng(T).standard_normal((T, d)).astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)
    special = bits.copy()
    for t, v in ((0, 0x7F800000), (T // 2, 0xFF800000), (T - 1, 0x7FC00000), (T - 1, 0xFFFF0000)):
        special[t, 7 + t % 5] = v
    special[0, d - 1] = 0x00010000  # a denormal
    for x in (bits, special, bits):
        x = x.view(np.float32)
        xb = capi.DeviceBuffer.of((x.view(np.uint32) >> 16).astype(np.uint16))
        out = capi.DeviceBuffer(4 * x.size)
        capi.call("hfmoe_moe_forward_bf16", r.layer, xb.ptr, T, out.ptr, None)
        capi.call("hfmoe_synchronize")
        got = out.download(np.float32, x.size).reshape(x.shape)
        assert np.array_equal(got, forward(r, x, T), equal_nan=True)
        xb.free()
        out.free()
    r.dev.free()


def test_lo_half_flag_from_call_to_call(hf):
    # An infinite router weight tells whether a BF16-valued x was multiplied
    # with lo halves: 0 * inf makes that expert's logits NaN where inf alone
    # does not.  Such a call gives the same logits first, after a call on FP32
    # activations, after a block, and after a dense layer's and the LM head's
    # calls, whose flag is another.
    T, d = 40, SMALL["hidden"]
    r = Run(SMALL, n_group=8, topk_group=4, seed=98, T=T, with_norm=True)
    capi.call("hfmoe_memcpy_h2d", r.dev.router.ptr + 2 * (3 * d + 5), np.array([0x7F80], np.uint16).ctypes.data, 2)
    r.dev.register()
    table = capi.DeviceBuffer(2 * 3 * d * 512)
    synth.fill_bf16(table.ptr, 3 * d * 512, 98, 1, 0.0, 0.02)
    dense = capi.DenseWeights(table.ptr, table.ptr, table.ptr, None, 512, 0)
    capi.call("hfmoe_register_dense_layer", 7, C.byref(dense))
    capi.call("hfmoe_register_lm_head", table.ptr, None, 3 * 512)
    rng = np.random.default_rng(98)
    xf = rng.standard_normal((T, d)).astype(np.float32)
    xb = (xf.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    xd, xbd, out = capi.DeviceBuffer.of(xf), capi.DeviceBuffer.of(xb), capi.DeviceBuffer(4 * T * max(d, 3 * 512))
    tok = capi.DeviceBuffer(4 * T)
    first = r.forward(xbd)["logits"]
    assert np.isinf(first[:, 3]).all() and np.isfinite(np.delete(first, 3, axis=1)).all()
    assert np.isnan(r.forward(xd)["logits"][:, 3]).any()  # the lo halves do show
    others = [lambda: block(r, xf, T), lambda: forward(r, xf, T),
              lambda: capi.call("hfmoe_dense_mlp_forward", 7, xd.ptr, T, out.ptr, None),
              lambda: capi.call("hfmoe_lm_head", xd.ptr, T, out.ptr, None, None),
              lambda: capi.call("hfmoe_lm_head", xd.ptr, T, out.ptr, tok.ptr, None)]
    for other in others:
        other()
        assert np.array_equal(r.forward(xbd)["logits"], first)
    for b in (table, xd, xbd, out, tok):
        b.free()
    r.dev.free()
