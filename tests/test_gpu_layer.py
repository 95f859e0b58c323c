"""The attention half of a decoder layer on the device (kvl_mla_attention_layer[_q8]_device):
n1 = RMSNorm(h, input_norm); h += attention(n1); n2 = RMSNorm(h, post_attn_norm), as
src/generate.c:34-67 (attention_token) computes it per token.

Bars: bit-identical to the same composition through this library's host API (kvl_rmsnorm_bf16,
the batched decode, an fp32 add); against the oracle's composition, the attention increment and
n2 within max|d|/max|ref| <= 2e-3."""
import ctypes as C

import numpy as np
import pytest

import pyoracle
from helpers import f32, rel_err, u16
from kvl_mla import abi, inputs, lib

pytestmark = pytest.mark.gpu

TOL = 2e-3
ORC = pyoracle.load_oracle()
L = lib.load()
KIMI = dict(inputs.KIMI)

KINDS = {
    "f32": (abi.KvlMlaCompressedState, "mla_compressed_state", "mla_decode_compressed_bf16",
            "mla_decode_compressed_batch_bf16", "mla_attention_layer_device"),
    "q8": (abi.KvlMlaCompressedQ8State, "mla_compressed_q8_state", "mla_decode_compressed_q8_bf16",
           "mla_decode_compressed_q8_batch_bf16", "mla_attention_layer_q8_device"),
}


def prefilled(api, prefix, kind, cfg, w, prompts, cap):
    cls, name, _, _, _ = KINDS[kind]
    out = []
    for p in prompts:
        st = cls()
        assert getattr(api, prefix + name + "_init")(C.byref(st), C.byref(cfg), cap) == 0
        assert getattr(api, prefix + name + "_prefill_bf16")(f32(p), p.shape[0], C.byref(cfg), C.byref(w),
                                                             C.byref(st)) == 0
        out.append(st)
    return out


@pytest.mark.parametrize("kind", ["f32", "q8"])
def test_attention_layer_matches_host_composition_and_oracle(kind):
    print(f"[layer] {kind}", flush=True)
    cfg = inputs.config(**KIMI)
    H = cfg.hidden_size
    layer = inputs.make_layer(cfg, 0xA1)
    w = layer.struct()
    rng = np.random.default_rng(0xA1)
    in_norm = inputs.f32_to_bf16_bits(1.0 + 0.02 * rng.standard_normal(H).astype(np.float32))
    post_norm = inputs.f32_to_bf16_bits(1.0 + 0.02 * rng.standard_normal(H).astype(np.float32))
    lens = [40, 57, 64]
    B = len(lens)
    prompts = [np.ascontiguousarray(inputs.hidden(cfg, 0xA2 + i, n) * np.float32(0.3)) for i, n in enumerate(lens)]
    h0 = np.ascontiguousarray(inputs.hidden(cfg, 0xA3, B))
    cap = max(lens) + 2
    cls, name, single, batch, fused = KINDS[kind]
    P = C.POINTER(cls)

    # device layer
    dev_states = prefilled(L, "kvl_", kind, cfg, w, prompts, cap)
    arr = (P * B)(*[C.pointer(s) for s in dev_states])
    nb = h0.nbytes
    d_h, d_n2 = L.kvl_mla_device_alloc(nb), L.kvl_mla_device_alloc(nb)
    assert d_h and d_n2
    lib.check(L.kvl_mla_copy_to_device(d_h, h0.ctypes.data, nb), "h2d")
    lib.check(getattr(L, "kvl_" + fused)(d_h, d_n2, B, C.byref(cfg), C.byref(w), u16(in_norm), u16(post_norm),
                                         arr, 0), "attention layer")
    h1 = np.zeros_like(h0)
    n2 = np.zeros_like(h0)
    lib.check(L.kvl_mla_copy_to_host(h1.ctypes.data, d_h, nb), "d2h")
    lib.check(L.kvl_mla_copy_to_host(n2.ctypes.data, d_n2, nb), "d2h")
    assert [s.len for s in dev_states] == [n + 1 for n in lens]

    # the same composition through the host API
    host_states = prefilled(L, "kvl_", kind, cfg, w, prompts, cap)
    harr = (P * B)(*[C.pointer(s) for s in host_states])
    n1 = np.zeros_like(h0)
    for b in range(B):
        L.kvl_rmsnorm_bf16(f32(n1[b]), f32(h0[b]), u16(in_norm), H, np.float32(cfg.rms_eps))
    attn = np.zeros_like(h0)
    pos = np.array(lens, np.int32)
    lib.check(getattr(L, "kvl_" + batch)(f32(attn), f32(n1), pos.ctypes.data_as(C.POINTER(C.c_int)), B,
                                         C.byref(cfg), C.byref(w), harr), "host batch decode")
    r1 = (h0 + attn).astype(np.float32)
    n2h = np.zeros_like(h0)
    for b in range(B):
        L.kvl_rmsnorm_bf16(f32(n2h[b]), f32(r1[b]), u16(post_norm), H, np.float32(cfg.rms_eps))
    np.testing.assert_array_equal(h1, r1)
    np.testing.assert_array_equal(n2, n2h)

    # the oracle's composition (src/generate.c:52-64 restated)
    orc_states = prefilled(ORC, "orc_", kind, cfg, w, prompts, cap)
    attn_o = np.zeros_like(h0)
    n2o = np.zeros_like(h0)
    for b in range(B):
        n1o = np.zeros(H, np.float32)
        ORC.orc_rmsnorm_bf16(f32(n1o), f32(h0[b]), u16(in_norm), H, C.c_float(cfg.rms_eps))
        assert getattr(ORC, "orc_" + single)(f32(attn_o[b]), f32(n1o), lens[b], C.byref(cfg), C.byref(w),
                                             C.byref(orc_states[b])) == 0
        r1o = (h0[b] + attn_o[b]).astype(np.float32)
        ORC.orc_rmsnorm_bf16(f32(n2o[b]), f32(r1o), u16(post_norm), H, C.c_float(cfg.rms_eps))
    e_attn, e_n2 = rel_err(h1 - h0, attn_o), rel_err(n2, n2o)
    print(f"[layer]   attention increment {e_attn:.3e}, n2 {e_n2:.3e}", flush=True)
    assert e_attn <= TOL and e_n2 <= TOL

    L.kvl_mla_device_free(d_h)
    L.kvl_mla_device_free(d_n2)
    for sts, api, pre in ((dev_states, L, "kvl_"), (host_states, L, "kvl_"), (orc_states, ORC, "orc_")):
        for s in sts:
            getattr(api, pre + name + "_free")(C.byref(s))


def test_attention_layer_rejects_bad_arguments():
    cfg = inputs.config(**KIMI)
    layer = inputs.make_layer(cfg, 0xA4)
    w = layer.struct()
    norm = inputs.f32_to_bf16_bits(np.ones(cfg.hidden_size, np.float32))
    st = abi.KvlMlaCompressedQ8State()
    assert L.kvl_mla_compressed_q8_state_init(C.byref(st), C.byref(cfg), 4) == 0
    arr = (C.POINTER(abi.KvlMlaCompressedQ8State) * 1)(C.pointer(st))
    d, e = L.kvl_mla_device_alloc(cfg.hidden_size * 4), L.kvl_mla_device_alloc(cfg.hidden_size * 4)
    fn = L.kvl_mla_attention_layer_q8_device
    assert fn(d, d, 1, C.byref(cfg), C.byref(w), u16(norm), u16(norm), arr, 0) == -1      # n2 aliases h
    assert fn(d, e, 1, C.byref(cfg), C.byref(w), u16(norm), u16(norm), arr, lib.RESIDUAL) == -1  # flag
    assert fn(d, e, 0, C.byref(cfg), C.byref(w), u16(norm), u16(norm), arr, 0) == -1      # empty batch
    assert st.len == 0
    L.kvl_mla_device_free(d)
    L.kvl_mla_device_free(e)
    L.kvl_mla_compressed_q8_state_free(C.byref(st))


@pytest.mark.parametrize("lens", [[6000] * 8, [5950, 6000, 6010, 6050, 6090, 6120, 6130, 6150], [8300], [7000, 5100, 9000]],
                         ids=["8", "8-lengths", "1", "3"])
def test_layer_norm_inside_the_projection_equals_its_launch(lens):
    """Eight sequences with equal split counts (24 of 256 rows here, also for the eight different lengths)
    have their projection and their combine inside the attention launch, which then normalises its input
    too; with the projection in its own launch the norm is a launch. Same sums in the same order: h and n2
    are equal bit for bit, from hidden states of very different scale per sequence. One and three sequences
    keep the norm's launch in both forms."""
    cfg = inputs.config(**KIMI)
    H, B = cfg.hidden_size, len(lens)
    layer = inputs.make_layer(cfg, 0xA7)
    w = layer.struct()
    lib.check(L.kvl_mla_bind_weights(C.byref(cfg), C.byref(w)), "bind")
    rng = np.random.default_rng(0xA7)
    norms = [inputs.f32_to_bf16_bits(1.0 + 0.1 * rng.standard_normal(H).astype(np.float32)) for _ in range(2)]
    h0 = np.ascontiguousarray(inputs.hidden(cfg, 0xA8, B) * (10.0 ** (np.arange(B) % 5 - 2))[:, None].astype(np.float32))
    states = []
    for i, n in enumerate(lens):
        st = abi.KvlMlaCompressedQ8State()
        lib.check(L.kvl_mla_compressed_q8_state_init(C.byref(st), C.byref(cfg), n + 1), "init")
        lib.check(L.kvl_mla_compressed_q8_state_fill_synthetic(C.byref(st), 0, n, 0xA70 + i), "fill")
        states.append(st)
    arr = (C.POINTER(abi.KvlMlaCompressedQ8State) * B)(*[C.pointer(s) for s in states])
    nb = h0.nbytes
    d_h, d_n2 = L.kvl_mla_device_alloc(nb), L.kvl_mla_device_alloc(nb)
    got = {}
    for on in (1, 0):
        prev = L.kvl_mla_set_fused_projection(on)
        try:
            lib.check(L.kvl_mla_copy_to_device(d_h, h0.ctypes.data, nb), "h2d")
            lib.check(L.kvl_mla_attention_layer_q8_device(d_h, d_n2, B, C.byref(cfg), C.byref(w), u16(norms[0]),
                                                          u16(norms[1]), arr, lib.NO_ADVANCE), "layer")
            h, n2 = np.zeros_like(h0), np.zeros_like(h0)
            lib.check(L.kvl_mla_copy_to_host(h.ctypes.data, d_h, nb), "d2h")
            lib.check(L.kvl_mla_copy_to_host(n2.ctypes.data, d_n2, nb), "d2h")
            got[on] = (h, n2)
        finally:
            L.kvl_mla_set_fused_projection(prev)
    for a, b in zip(got[1], got[0]):
        assert np.all(np.isfinite(a))
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    L.kvl_mla_device_free(d_h)
    L.kvl_mla_device_free(d_n2)
    for s in states:
        L.kvl_mla_compressed_q8_state_free(C.byref(s))
    lib.check(L.kvl_mla_release_weights(C.byref(w)), "release")


@pytest.mark.parametrize("lens", [[8300], [6000] * 8, [7000, 5100, 9000]], ids=["1", "8", "3"])
def test_layer_from_an_unaligned_buffer_keeps_the_fused_launch(lens):
    """The projection inside the attention launch reads 16-byte vectors. Hidden states at a 4-byte
    boundary go through the norm's launch into the library's aligned buffer and keep that form: no launch
    of the projection (stage 0) is timed, and h and n2 equal those of an aligned buffer bit for bit."""
    cfg = inputs.config(**KIMI)
    H, B = cfg.hidden_size, len(lens)
    layer = inputs.make_layer(cfg, 0xAB)
    w = layer.struct()
    lib.check(L.kvl_mla_bind_weights(C.byref(cfg), C.byref(w)), "bind")
    norms = [inputs.normal_bf16(0xAB, n, (H,), mean=1.0, std=0.1) for n in ("n1", "n2")]
    h0 = np.ascontiguousarray(inputs.hidden(cfg, 0xAC, B))
    states = []
    for i, n in enumerate(lens):
        st = abi.KvlMlaCompressedQ8State()
        lib.check(L.kvl_mla_compressed_q8_state_init(C.byref(st), C.byref(cfg), n + 1), "init")
        lib.check(L.kvl_mla_compressed_q8_state_fill_synthetic(C.byref(st), 0, n, 0xAC0 + i), "fill")
        states.append(st)
    arr = (C.POINTER(abi.KvlMlaCompressedQ8State) * B)(*[C.pointer(s) for s in states])
    nb = h0.nbytes
    base, d_n2 = L.kvl_mla_device_alloc(nb + 16), L.kvl_mla_device_alloc(nb)
    got = []
    for off in (0, 4):
        d_h = base + off
        lib.check(L.kvl_mla_copy_to_device(d_h, h0.ctypes.data, nb), "h2d")
        ms, count = (C.c_double * 6)(), (C.c_int * 6)()
        lib.check(L.kvl_mla_timing_enable(1), "timing on")
        try:
            lib.check(L.kvl_mla_attention_layer_q8_device(d_h, d_n2, B, C.byref(cfg), C.byref(w), u16(norms[0]),
                                                          u16(norms[1]), arr, lib.NO_ADVANCE), "layer")
            lib.check(L.kvl_mla_timing_read(ms, count), "timing read")
        finally:
            lib.check(L.kvl_mla_timing_enable(0), "timing off")
        h, n2 = np.zeros_like(h0), np.zeros_like(h0)
        lib.check(L.kvl_mla_copy_to_host(h.ctypes.data, d_h, nb), "d2h")
        lib.check(L.kvl_mla_copy_to_host(n2.ctypes.data, d_n2, nb), "d2h")
        got.append((h, n2))
        print(f"[layer] offset {off}: launches per stage {list(count)}", flush=True)
        assert count[0] == 0 and count[3] == 1, (off, list(count))
    for a, b in zip(*got):
        assert np.all(np.isfinite(a)) and np.any(a)
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    L.kvl_mla_device_free(base)
    L.kvl_mla_device_free(d_n2)
    for s in states:
        L.kvl_mla_compressed_q8_state_free(C.byref(s))
    lib.check(L.kvl_mla_release_weights(C.byref(w)), "release")
