"""Prefill with the state fill of the same tokens (kvl_mla_prefill_compressed[_q8]_state_*),
the call sequence of src/generate.c:208-210 (kvl_mla_prefill_bf16, then the state prefill of
src/mla_compressed_state.c:52-84 / src/mla_compressed_q8_state.c:129-159) as one call.

Bars: output and state rows bit-identical to the two separate calls of this library; against
the oracle, outputs max|got - ref| / max|ref| <= 2e-3 and state rows within the rounding of
the kv_a projection (the Q8 codes of a row move by at most one step)."""
import ctypes as C

import numpy as np
import pytest

import pyoracle
from helpers import Api, decode_seq, f32, rel_err, snapshot
from kvl_mla import abi, inputs, lib

pytestmark = pytest.mark.gpu

TOL = 2e-3
ORC = pyoracle.load_oracle()
O = Api(ORC, "orc_")
L = lib.load()
G = Api(L, "kvl_")

STREAM = dict(hidden_size=16, num_heads=2, qk_nope_dim=4, qk_rope_dim=4, v_head_dim=8,
              kv_lora_rank=6, rms_eps=1e-5, rope_theta=800000.0)  # src/mla_streaming_probe.c:39,46
KIMI = dict(inputs.KIMI)

STATE = {"f32": (abi.KvlMlaCompressedState, "mla_compressed_state"),
         "bf16": (abi.KvlMlaCompressedBF16State, "mla_compressed_bf16_state"),
         "q8": (abi.KvlMlaCompressedQ8State, "mla_compressed_q8_state")}
FUSED = {"f32": "mla_prefill_compressed_state", "bf16": "mla_prefill_compressed_bf16_state",
         "q8": "mla_prefill_compressed_q8_state"}


def new_state(api, kind, cfg, cap):
    cls, name = STATE[kind]
    st = cls()
    assert getattr(api, name + "_init")(C.byref(st), C.byref(cfg), cap) == 0
    return st


def free_state(api, kind, st):
    getattr(api, STATE[kind][1] + "_free")(C.byref(st))


def separate(kind, cfg, w, x, cap):
    S, H = x.shape
    out = np.zeros((S, H), np.float32)
    lib.check(L.kvl_mla_prefill_bf16(f32(out), f32(x), S, C.byref(cfg), C.byref(w)), "prefill")
    st = new_state(G, kind, cfg, cap)
    lib.check(getattr(G, STATE[kind][1] + "_prefill_bf16")(f32(x), S, C.byref(cfg), C.byref(w), C.byref(st)),
              "state prefill")
    return out, st


def fused(kind, cfg, w, x, cap):
    S, H = x.shape
    out = np.zeros((S, H), np.float32)
    st = new_state(G, kind, cfg, cap)
    lib.check(getattr(G, FUSED[kind] + "_bf16")(f32(out), f32(x), S, C.byref(cfg), C.byref(w), C.byref(st)),
              "fused prefill")
    return out, st


def assert_snap_equal(a, b):
    assert a.keys() == b.keys()
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


CASES = [("stream", STREAM, 37, 0.2, False), ("kimi", KIMI, 130, 0.02, False), ("kimi", KIMI, 300, 0.02, True)]


@pytest.mark.parametrize("name,dims,S,std,bf16_x", CASES, ids=[f"{c[0]}-{c[2]}" for c in CASES])
@pytest.mark.parametrize("kind", ["f32", "q8"])
def test_fused_equals_prefill_then_state_prefill(name, dims, S, std, bf16_x, kind):
    """State bit-identical to the state prefill's. Generic route (stream-probe shapes, the fill
    computes its own kv_a): output bit-identical too. Kimi-VL MFMA route (one kv_a for the
    attention and the state, in the decode's summation order): output within 5e-4 of the plain
    prefill's (a last-bit change of kv_a can move the bf8 rounding of a score correction
    operand, 2^-14 of |K||Q|; each output is within 2e-3 of the oracle's). S not a multiple of
    the tiles."""
    print(f"[fused] {kind} {name} S={S}", flush=True)
    cfg = inputs.config(**dims)
    layer = inputs.make_layer(cfg, 0xF0 + S, std=std)
    w = layer.struct()
    x = inputs.hidden(cfg, 0xF0 + S, S, bf16_exact=bf16_x)
    oa, sa = separate(kind, cfg, w, x, S + 3)
    ob, sb = fused(kind, cfg, w, x, S + 3)
    assert sa.len == sb.len == S
    if name == "stream":
        np.testing.assert_array_equal(ob, oa)
    else:
        print(f"[fused]   vs plain prefill max|d|/max|ref| = {rel_err(ob, oa):.3e}", flush=True)
        assert rel_err(ob, oa) <= 5e-4
    assert_snap_equal(snapshot(kind, sb, cfg), snapshot(kind, sa, cfg))
    free_state(G, kind, sa)
    free_state(G, kind, sb)


@pytest.mark.parametrize("kind", ["f32", "q8"])
def test_fused_then_decode_matches_oracle(kind):
    """Prompt of 200 tokens through the fused call, then 3 decode tokens, against the oracle's
    prefill, state prefill and decode."""
    print(f"[fused] {kind} prompt 200 + decode 3 vs oracle", flush=True)
    cfg = inputs.config(**KIMI)
    layer = inputs.make_layer(cfg, 0xF7)
    w = layer.struct()
    P, T = 200, 3
    x = inputs.hidden(cfg, 0xF7, P + T)
    xp = np.ascontiguousarray(x[:P])
    out, st = fused(kind, cfg, w, xp, P + T + 1)
    ref = np.zeros_like(out)
    assert ORC.orc_mla_prefill_streaming(f32(ref), f32(xp), P, C.byref(cfg), C.byref(w)) == 0
    assert rel_err(out, ref) <= TOL, rel_err(out, ref)
    # state rows against the oracle's state prefill of the same tokens
    ost = new_state(O, kind, cfg, P + T + 1)
    assert getattr(O, STATE[kind][1] + "_prefill_bf16")(f32(xp), P, C.byref(cfg), C.byref(w), C.byref(ost)) == 0
    got, exp = snapshot(kind, st, cfg), snapshot(kind, ost, cfg)
    if kind == "f32":
        assert rel_err(got["latent"], exp["latent"]) <= 1e-5
    else:
        dc = np.abs(got["codes"].astype(np.int32) - exp["codes"].astype(np.int32))
        assert dc.max() <= 1 and np.mean(dc) <= 1e-2, (dc.max(), np.mean(dc))
        np.testing.assert_allclose(got["scale"], exp["scale"], rtol=1e-5)
    if kind == "q8":  # BF16 keys: one rounding step of 2^-8 at most
        assert rel_err(inputs.bf16_bits_to_f32(got["rope"]), inputs.bf16_bits_to_f32(exp["rope"])) <= 1e-2
    else:
        assert rel_err(got["rope"], exp["rope"]) <= 1e-5
    free_state(O, kind, ost)
    # decode continues from the fused state; the oracle from its own
    dec = getattr(G, "mla_decode_compressed_bf16" if kind == "f32" else "mla_decode_compressed_q8_bf16")
    outs = np.zeros((T, cfg.hidden_size), np.float32)
    for t in range(T):
        assert dec(f32(outs[t]), f32(np.ascontiguousarray(x[P + t])), P + t, C.byref(cfg), C.byref(w),
                   C.byref(st)) == 0
    refs, _ = decode_seq(O, kind, cfg, w, x, prefix=P)
    print(f"[fused]   decode max|d|/max|ref| = {rel_err(outs, refs):.3e}", flush=True)
    assert rel_err(outs, refs) <= TOL
    # and equals this library's own separate calls followed by the same decode
    mine, _ = decode_seq(G, kind, cfg, w, x, prefix=P)
    np.testing.assert_array_equal(outs, mine)
    free_state(G, kind, st)


@pytest.mark.parametrize("kind", ["f32", "q8"])
def test_fused_device_variant_matches_host_variant(kind):
    print(f"[fused] {kind} device variant S=257", flush=True)
    cfg = inputs.config(**KIMI)
    layer = inputs.make_layer(cfg, 0xF9)
    w = layer.struct()
    S = 257
    x = np.ascontiguousarray(inputs.hidden(cfg, 0xF9, S))
    oh, sh = fused(kind, cfg, w, x, S)
    sd = new_state(G, kind, cfg, S)
    nbytes = x.nbytes
    dx, dout = L.kvl_mla_device_alloc(nbytes), L.kvl_mla_device_alloc(nbytes)
    assert dx and dout
    lib.check(L.kvl_mla_copy_to_device(dx, x.ctypes.data, nbytes), "h2d")
    lib.check(getattr(G, FUSED[kind] + "_device")(dout, dx, S, C.byref(cfg), C.byref(w), C.byref(sd)),
              "fused device")
    od = np.zeros_like(x)
    lib.check(L.kvl_mla_copy_to_host(od.ctypes.data, dout, nbytes), "d2h")
    assert sd.len == S
    pull = L.kvl_mla_compressed_state_pull if kind == "f32" else L.kvl_mla_compressed_q8_state_pull
    lib.check(pull(C.byref(sd), 0, S), "pull")
    np.testing.assert_array_equal(od, oh)
    assert_snap_equal(snapshot(kind, sd, cfg), snapshot(kind, sh, cfg))
    L.kvl_mla_device_free(dx)
    L.kvl_mla_device_free(dout)
    free_state(G, kind, sh)
    free_state(G, kind, sd)


def test_fused_rejects_bad_arguments():
    """The state prefill's checks (empty state, seq_len within capacity); nothing written."""
    cfg = inputs.config(**KIMI)
    layer = inputs.make_layer(cfg, 0xFA)
    w = layer.struct()
    x = inputs.hidden(cfg, 0xFA, 8)
    out = np.full((8, cfg.hidden_size), 7.0, np.float32)
    st = new_state(G, "q8", cfg, 4)
    assert L.kvl_mla_prefill_compressed_q8_state_bf16(f32(out), f32(x), 8, C.byref(cfg), C.byref(w), C.byref(st)) == -1
    assert st.len == 0 and np.all(out == 7.0)
    lib.check(L.kvl_mla_prefill_compressed_q8_state_bf16(f32(out), f32(x), 2, C.byref(cfg), C.byref(w),
                                                         C.byref(st)), "fused")
    assert st.len == 2
    assert L.kvl_mla_prefill_compressed_q8_state_bf16(f32(out), f32(x), 2, C.byref(cfg), C.byref(w), C.byref(st)) == -1
    assert st.len == 2
    free_state(G, "q8", st)


_long_rows = {}


def f32_rows(S):
    """FP32 state rows of the first S tokens of one 2000-token input (bit patterns)."""
    cfg = inputs.config(**inputs.KIMI)
    layer = inputs.make_layer(cfg, 0xD7)
    w = layer.struct()
    x = np.ascontiguousarray(inputs.hidden(cfg, 0xD7, 2000)[:S])
    st = abi.KvlMlaCompressedState()
    lib.check(L.kvl_mla_compressed_state_init(C.byref(st), C.byref(cfg), S), "init")
    lib.check(L.kvl_mla_compressed_state_prefill_bf16(f32(x), S, C.byref(cfg), C.byref(w), C.byref(st)), "prefill")
    lat = np.ctypeslib.as_array(st.latent, (S, 512)).copy().view(np.uint32)
    key = np.ctypeslib.as_array(st.rope, (S, 64)).copy().view(np.uint32)
    L.kvl_mla_compressed_state_free(C.byref(st))
    return lat, key


@pytest.mark.parametrize("S", [1, 33, 96, 97, 224, 225, 448, 449, 896, 897, 1344, 1345])
def test_rows_do_not_depend_on_the_prompt_length(S):
    """A row depends on its token alone, in one summation order: the rows of a shorter prompt equal
    those of a longer one bit for bit at the edges of the tile shapes of the kv_a projection (96, 224,
    448, 896 and 1344 tokens)."""
    if 2000 not in _long_rows:
        _long_rows[2000] = f32_rows(2000)
    for got, full in zip(f32_rows(S), _long_rows[2000]):
        np.testing.assert_array_equal(got, full[:S])


@pytest.mark.parametrize("kind", ["f32", "q8"])
def test_prefilled_special_rows_equal_decoded_rows(kind):
    """The rows kernel of a state prefill against the append of a decode, on tokens whose rows meet the
    quantiser's special cases: all zero, overflowing, NaN, subnormal products (NaN compares equal)."""
    cfg = inputs.config(**inputs.KIMI)
    layer = inputs.make_layer(cfg, 0xD9)
    w = layer.struct()
    x = np.ascontiguousarray(inputs.hidden(cfg, 0xD9, 7))
    x[1] = 0.0
    x[2] *= np.float32(1e38)
    x[3, 100] = np.nan
    x[4] *= np.float32(1e-30)
    x[5, 0] = np.inf
    _, dec = decode_seq(G, kind, cfg, w, x)
    st = new_state(G, kind, cfg, 7)
    lib.check(getattr(G, STATE[kind][1] + "_prefill_bf16")(f32(x), 7, C.byref(cfg), C.byref(w), C.byref(st)),
              "state prefill")
    pre = snapshot(kind, st, cfg)
    free_state(G, kind, st)
    for name in dec:
        a, b = pre[name], dec[name]
        if name == "rope" and kind == "q8":
            a, b = (inputs.bf16_bits_to_f32(v) for v in (a, b))
        np.testing.assert_array_equal(a, b, err_msg=f"{kind} {name}")


def rows_of(kind, st, cfg):
    """The host rows [0, len), bit patterns."""
    n = st.len
    if kind != "bf16":
        return snapshot(kind, st, cfg)
    return {"latent": np.ctypeslib.as_array(st.latent, (n, cfg.kv_lora_rank)).copy(),
            "rope": np.ctypeslib.as_array(st.rope, (n, cfg.qk_rope_dim)).copy()}


def fused_device(kind, cfg, w, x):
    """Output and pulled rows of the device call."""
    S, nbytes = x.shape[0], x.nbytes
    st = new_state(G, kind, cfg, S)
    dx, do = L.kvl_mla_device_alloc(nbytes), L.kvl_mla_device_alloc(nbytes)
    lib.check(L.kvl_mla_copy_to_device(dx, x.ctypes.data, nbytes), "h2d")
    lib.check(getattr(G, FUSED[kind] + "_device")(do, dx, S, C.byref(cfg), C.byref(w), C.byref(st)), "fused device")
    out = np.zeros_like(x)
    lib.check(L.kvl_mla_copy_to_host(out.ctypes.data, do, nbytes), "d2h")
    lib.check(getattr(G, STATE[kind][1] + "_pull")(C.byref(st), 0, S), "pull")
    rows = rows_of(kind, st, cfg)
    free_state(G, kind, st)
    L.kvl_mla_device_free(dx)
    L.kvl_mla_device_free(do)
    return out, rows


def state_rows(kind, cfg, w, x):
    """Rows of the state prefill alone."""
    st = new_state(G, kind, cfg, x.shape[0])
    lib.check(getattr(G, STATE[kind][1] + "_prefill_bf16")(f32(x), x.shape[0], C.byref(cfg), C.byref(w), C.byref(st)),
              "state prefill")
    rows = rows_of(kind, st, cfg)
    free_state(G, kind, st)
    return rows


_long_fill = {}


def long_fill():
    """Layer, input, output and FP32 rows of a 4500-token prefill with state fill, computed once: its output
    against the plain prefill's (see test_fused_equals_prefill_then_state_prefill), its rows against the
    state prefill's."""
    if not _long_fill:
        cfg = inputs.config(**KIMI)
        layer = inputs.make_layer(cfg, 0xDB)
        w = layer.struct()
        x = inputs.hidden(cfg, 0xDB, 4500)
        out, rows = fused_device("f32", cfg, w, x)
        plain = np.zeros_like(x)
        lib.check(L.kvl_mla_prefill_bf16(f32(plain), f32(x), 4500, C.byref(cfg), C.byref(w)), "prefill")
        assert np.all(np.isfinite(out)) and rel_err(out, plain) <= 5e-4, rel_err(out, plain)
        assert_snap_equal(rows, state_rows("f32", cfg, w, x))
        _long_fill.update(layer=layer, x=x, out=out, rows=rows)
    return _long_fill


@pytest.mark.parametrize("S", [1, 37, 64, 65, 128, 160, 161, 321, 650, 705, 1000, 1025, 1281, 1921, 2600, 4097])
def test_fill_is_a_prefix_of_a_longer_one(S):
    """The projection without kv_a, whose tile shapes change at other sizes than the plain prefill's (64, 160,
    320, 640, 704, 1280, 1920, 2560 and 4096 tokens): outputs and rows of S tokens are the first S of 4500
    bit for bit, through the device call and through the host call, which is staged through pinned memory
    up to 1024 tokens."""
    ref = long_fill()
    cfg = inputs.config(**KIMI)
    w = ref["layer"].struct()
    x = np.ascontiguousarray(ref["x"][:S])
    out, rows = fused_device("f32", cfg, w, x)
    host, st = fused("f32", cfg, w, x, S)
    for o, r in ((out, rows), (host, snapshot("f32", st, cfg))):
        np.testing.assert_array_equal(o, ref["out"][:S])
        for k in r:
            np.testing.assert_array_equal(r[k], ref["rows"][k][:S], err_msg=k)
    free_state(G, "f32", st)


@pytest.mark.parametrize("kind", ["bf16", "q8"])
@pytest.mark.parametrize("S", [1000, 1100])
def test_fused_host_call_on_both_sides_of_the_staging_limit(kind, S):
    """1000 tokens go through pinned memory, 1100 do not: outputs and rows equal the device call's."""
    ref = long_fill()
    cfg = inputs.config(**KIMI)
    w = ref["layer"].struct()
    x = np.ascontiguousarray(ref["x"][:S])
    host, st = fused(kind, cfg, w, x, S)
    out, rows = fused_device(kind, cfg, w, x)
    np.testing.assert_array_equal(host, out)
    assert_snap_equal(rows_of(kind, st, cfg), rows)
    free_state(G, kind, st)


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_long_fill_rows(kind):
    """8197 rows: four to a block, so more than the 2048 blocks that the rows kernel launches."""
    cfg = inputs.config(**KIMI)
    layer = inputs.make_layer(cfg, 0xDC)
    w = layer.struct()
    x = inputs.hidden(cfg, 0xDC, 8197)
    out, rows = fused_device(kind, cfg, w, x)
    assert np.all(np.isfinite(out))
    assert_snap_equal(rows, state_rows(kind, cfg, w, x))


@pytest.mark.parametrize("S", [256, 1100])
def test_fused_host_call_beyond_the_operand_range(S):
    """kv_b x 3000 raises the range flag (row-max logits of about 4400): the host call, staged through pinned
    memory (256) or not (1100), computes the output again on the fp32 route and keeps the rows, which do
    not depend on the attention."""
    cfg = inputs.config(**KIMI)
    layer = inputs.make_layer(cfg, 0xDD)
    layer.kv_b_proj[...] = inputs.f32_to_bf16_bits(inputs.bf16_bits_to_f32(layer.kv_b_proj) * np.float32(3000.0))
    w = layer.struct()
    x = inputs.hidden(cfg, 0xDD, S, bf16_exact=True)
    out, st = fused("q8", cfg, w, x, S)
    idx = np.ascontiguousarray(sorted({0, 1, S // 2, S - 2, S - 1}), dtype=np.int32)
    ref = np.zeros((len(idx), cfg.hidden_size), np.float32)
    assert ORC.orc_mla_prefill_streaming_rows(f32(ref), f32(x), S, idx.ctypes.data_as(C.POINTER(C.c_int)), len(idx),
                                              C.byref(cfg), C.byref(w)) == 0
    e = rel_err(out[idx], ref)
    print(f"[fused] range S={S}: {e:.3e}", flush=True)
    assert np.all(np.isfinite(out)) and e <= TOL, e
    assert L.kvl_mla_prefill_range_status() == 0
    assert st.len == S
    assert_snap_equal(rows_of("q8", st, cfg), state_rows("q8", cfg, w, x))
    dx, do = L.kvl_mla_device_alloc(x.nbytes), L.kvl_mla_device_alloc(x.nbytes)
    lib.check(L.kvl_mla_copy_to_device(dx, x.ctypes.data, x.nbytes), "h2d")
    lib.check(L.kvl_mla_prefill_device(do, dx, S, C.byref(cfg), C.byref(w)), "device prefill")
    assert L.kvl_mla_prefill_range_status() == 1  # the flag was up
    L.kvl_mla_device_free(dx)
    L.kvl_mla_device_free(do)
    free_state(G, "q8", st)
