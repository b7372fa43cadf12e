"""The split-D pipeline's tile kernels against the oracle: edges of both tile
sizes, odd and even stage counts, head sizes that are no whole number of
vectors, misaligned bases, encodings per side, every softmax row form, and the
in-kernel encoding that remains where the scratch holds no encoded copies."""
import ctypes

import numpy as np
import pytest

import helpers as H
import oracle

pytestmark = pytest.mark.gpu


def _desc(am, pe):
    return {"none": None, "rope": am.make_pe("rope"), "half": am.make_pe("rope", "half"),
            "rope_q": am.make_pe("rope", apply_k=False), "half_k": am.make_pe("rope", "half", apply_q=False),
            "sin": am.make_pe("sinusoidal")}[pe]


def _ref(pe, Q, K, V):
    L, D = max(Q.shape[2], K.shape[2]), Q.shape[3]
    if pe == "none":
        return oracle.attention(Q, K, V, nthreads=16)
    if pe == "sin":
        return oracle.attention_sinusoidal(Q, K, V, *oracle.sinusoidal_table(L, D), nthreads=16)
    c, s = oracle.rope_cache(L, D)
    return oracle.attention_rope(Q, K, V, c, s, pairing="half" if pe.startswith("half") else "interleaved",
                                 rotate_q=pe != "half_k", rotate_k=pe != "rope_q", nthreads=16)


def _check(got, Q, K, V, pe):
    n, mabs, _ = H.check_f32(got, _ref(pe, Q, K, V))
    assert n == 0, mabs


@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("shape,pe", [
    ((1, 1, 65, 129, 260), "none"),      # one past a tile, 9 stages
    ((2, 1, 128, 128, 320), "none"),     # whole tiles, 10 stages
    ((1, 2, 127, 255, 288), "rope"),
    ((1, 1, 193, 131, 261), "none"),     # head_d % 4 == 1
    ((1, 1, 129, 200, 330), "half"),     # head_d % 4 == 2
    ((1, 2, 130, 190, 263), "sin"),      # head_d % 4 == 3
    ((1, 1, 140, 150, 1028), "rope_q"),
    ((1, 1, 150, 140, 512), "half_k"),
], ids=str)
def test_tile_edges(am, dev, tuner, tile, shape, pe):
    import hip_rt
    B, Hh, Lq, Lk, D = shape
    print(f"[case] tile {tile} {shape} {pe}", flush=True)
    assert am.path(0, B, Hh, Lq, Lk, D, _desc(am, pe)) == am.ATN_PATH_SPLIT_D
    tuner.set(splitd_tile=tile)
    sigma = 0.5 if pe == "sin" else 1.0
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 900 + Lq + D, "f32", sigma)
    out = H.empty(Q.shape)
    am.attention_ex(q, k, v, out, pe=_desc(am, pe))
    hip_rt.synchronize()
    _check(out.numpy(), Q, K, V, pe)


@pytest.mark.parametrize("Lq,Lk", [(70, 257), (5000, 40), (3, 1025), (4100, 513), (4100, 1030),
                                   (2, 4097), (2, 8190), (2, 8193)], ids=str)
def test_softmax_row_forms(am, dev, Lq, Lk):
    import hip_rt
    D = 264
    print(f"[case] softmax rows {Lq} x {Lk}", flush=True)
    (q, k, v), (Q, K, V) = H.device_inputs((1, 1, Lq, D), (1, 1, Lk, D), 950 + Lk)
    out = H.empty(Q.shape)
    am.attention_ex(q, k, v, out)
    hip_rt.synchronize()
    _check(out.numpy(), Q, K, V, "none")


@pytest.mark.parametrize("D", [264, 267], ids=str)
def test_misaligned_bases(am, dev, D):
    """Tensors 4 bytes off a 16-byte boundary."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 2, 100, 140
    print(f"[case] misaligned {D}", flush=True)
    Q, K, V = H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), seed=960)
    dev_t = [H.upload(np.concatenate([[0.0], x.ravel()]).astype(np.float32)) for x in (Q, K, V)]
    out = H.empty((Q.size + 1,))
    st = am.lib().atn_attention_fwd_ex(0, *[t.ptr + 4 for t in dev_t], out.ptr + 4, B, Hh, Lq, Lk, D,
                                       ctypes.POINTER(am.PeDesc)(), None, 0, None)
    assert st == 0
    hip_rt.synchronize()
    _check(out.numpy()[1:].reshape(Q.shape), Q, K, V, "none")


# Inputs far from magnitude 1 (exponents of 2 on Q, K and V), and one large
# element among ordinary ones.
RANGES = {"v-20": (0, 0, -20), "v-30": (0, 0, -30), "v-90": (0, 0, -90), "v+60": (0, 0, 60), "v+120": (0, 0, 120),
          "q-13": (-13, 13, 0), "q+13": (13, -13, 0), "q-60": (-60, 60, 0), "outliers": (0, 0, 0)}


def _ranged(rng_case, dims, seed):
    B, Hh, Lq, Lk, D = dims
    Q, K, V = H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), seed=seed)
    eq, ek, ev = RANGES[rng_case]
    Q, K, V = (np.ldexp(x, e).astype(np.float32) for x, e in ((Q, eq), (K, ek), (V, ev)))
    if rng_case == "outliers":
        V[:, :, Lk // 2, 5] = 1e9     # one column; the others keep their bits
        Q[:, :, 7] *= np.float32(1e-6)
        K[:, :, 3] *= np.float32(1e-6)
        K[:, :, 40, 11] = 1e6         # a key that some rows see alone
    return Q, K, V


def _offset_call(am, Q, K, V, es=4):
    """The call on tensors `es` bytes off a 16-byte boundary."""
    import hip_rt
    B, Hh, Lq, D = Q.shape
    dev_t = [H.upload(np.concatenate([[0.0], x.ravel()]).astype(np.float32)) for x in (Q, K, V)]
    out = H.empty((Q.size + 1,))
    st = am.lib().atn_attention_fwd_ex(0, *[t.ptr + es for t in dev_t], out.ptr + es, B, Hh, Lq, K.shape[2], D,
                                       None, None, 0, None)
    assert st == 0
    hip_rt.synchronize()
    return out.numpy()[1:].reshape(Q.shape)


def _check64(got, Q, K, V, skip=()):
    """Normwise against float64, column by column of the output (an outlier's
    column says nothing about the others).  fp32 sums keep 2^-24 of their
    terms; with the exponential's and the softmax's roundings the worst column
    of these sizes shows 1e-6, the bar is 4e-6."""
    ref = H.sdpa64(Q, K, V)
    keep = [d for d in range(Q.shape[-1]) if d not in skip]
    g, r = (x[..., keep].reshape(-1, len(keep)).astype(np.float64) for x in (got, ref))
    assert np.isfinite(g).all()
    err = np.linalg.norm(g - r, axis=0) / np.linalg.norm(r, axis=0)
    assert err.max() < 4e-6, (float(err.max()), int(err.argmax()))


@pytest.mark.parametrize("rng_case", list(RANGES))
@pytest.mark.parametrize("D,off", [(258, 0), (261, 0), (263, 0), (264, 4), (1030, 0)], ids=str)
def test_fp32_magnitudes_of_odd_rows(am, dev, D, off, rng_case):
    """fp32 with head_d % 4 != 0 or misaligned bases keeps fp32's accuracy
    wherever the values lie."""
    print(f"[case] magnitudes {D} +{off} {rng_case}", flush=True)
    Q, K, V = _ranged(rng_case, (1, 2, 150, 140, D), 980 + D)
    if off:
        got = _offset_call(am, Q, K, V, off)
    else:
        import hip_rt
        out = H.empty(Q.shape)
        am.attention_ex(*(H.upload(x) for x in (Q, K, V)), out)
        hip_rt.synchronize()
        got = out.numpy()
    _check64(got, Q, K, V)


@pytest.mark.parametrize("tile", [64, 128])
def test_fp32_infinities_of_odd_rows(am, dev, tuner, tile):
    """Infinite operands: a key whose scores are -inf weighs nothing, an
    infinite value stays in its column, as the same products in float64."""
    import hip_rt
    tuner.set(splitd_tile=tile)
    B, Hh, Lq, Lk, D = 1, 1, 140, 150, 261
    print(f"[case] infinities, tile {tile}", flush=True)
    Q, K, V = H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), seed=991)
    K[0, 0, 20, 9] = -np.inf
    Q[..., 9] = np.abs(Q[..., 9])      # every score of key 20 is -inf
    V[0, 0, 77, 130] = np.inf
    V[0, 0, 78, 200] = np.float32(3.4e38)
    out = H.empty(Q.shape)
    am.attention_ex(*(H.upload(x) for x in (Q, K, V)), out)
    hip_rt.synchronize()
    got = out.numpy()
    assert np.isposinf(got[..., 130]).all()
    _check64(got, Q, K, V, skip=(130,))


def test_fp32_sums_of_one_sign(am, dev):
    """Sinusoidal rows make long sums of one sign: compensated, the call is no
    further from float64 than the kernels that cut D into more chunks (6.8e-7
    normwise at this head size; plain sums 7.6e-7)."""
    import hip_rt
    B, Hh, Lq, Lk, D = 4, 4, 567, 279, 904
    print("[case] sums of one sign", flush=True)
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 993)
    out = H.empty(Q.shape)
    am.attention_ex(q, k, v, out, pe=_desc(am, "sin"))
    hip_rt.synchronize()
    st, ct = (np.asarray(t, np.float64).reshape(-1, D) for t in oracle.sinusoidal_table(max(Lq, Lk), D))
    pe = np.where(np.arange(D) % 2 == 0, st, ct)
    ref = H.sdpa64(Q + pe[:Lq], K + pe[:Lk], V)
    err = np.linalg.norm(out.numpy() - ref) / np.linalg.norm(ref)
    print(f"normwise {err:.3g}", flush=True)
    assert err < 6.5e-7


@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("D,Lk", [(260, 150), (288, 31), (320, 129)], ids=str)  # odd, one and even stage counts
@pytest.mark.parametrize("where", ["first", "late", "all"])
def test_values_beyond_fp16_range(am, dev, tuner, tile, D, Lk, where):
    """fp32 values of 65504 and more, in the first stage of Q K^T and P V (seen
    before the pass), in the last (after it) and everywhere."""
    import hip_rt
    tuner.set(splitd_tile=tile)
    B, Hh, Lq = 1, 2, 140
    print(f"[case] beyond fp16 {tile} {D} {Lk} {where}", flush=True)
    Q, K, V = H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), seed=992)
    if where == "all":
        Q, K, V = np.ldexp(Q, -20), np.ldexp(K, 20), np.ldexp(V, 18)
    else:
        d, j = (3, 2) if where == "first" else (D - 2, Lk - 1)
        Q[:, :, :, d] *= np.float32(2.0 ** -17)
        K[:, :, :, d] *= np.float32(2.0 ** 17)
        V[:, :, j, 7] = 1e6
    out = H.empty(Q.shape)
    am.attention_ex(*(H.upload(x) for x in (Q, K, V)), out)
    hip_rt.synchronize()
    scale = np.float32(2.0 ** 18 if where == "all" else 1.0)
    n, mabs, _ = H.check_f32(out.numpy() / scale, _ref("none", Q, K, V) / scale)
    assert n == 0, mabs


@pytest.mark.parametrize("dt,D,pe,off", [
    ("f32", 1024, "rope", 0), ("f32", 1024, "half", 0), ("f32", 1024, "sin", 0), ("f32", 1024, "half_k", 0),
    ("f32", 1026, "rope", 0), ("f32", 1026, "half", 0), ("f32", 1025, "sin", 0), ("f32", 1024, "half", 1),
    ("bf16", 1004, "none", 0), ("bf16", 1004, "rope", 0), ("bf16", 1002, "half", 0), ("bf16", 1001, "sin", 0),
    ("bf16", 1001, "none", 0), ("bf16", 1008, "none", 1), ("bf16", 1008, "rope", 1)], ids=str)
def test_scratch_without_copies(am, dev, dt, D, pe, off):
    """What K's encoded copy, or K's and V's padded ones, would need exceeds the
    scratch: the kernels that need none, in chunks of rows (positions and
    pointers at an offset), for every row alignment; `off`: tensors one element
    off a 16-byte boundary."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 2, 70, 400  # 1.6 MB of copies
    print(f"[case] lean {dt} {D} {pe} +{off}", flush=True)
    desc, (code, es) = _desc(am, pe), {"f32": (0, 4), "bf16": (1, 2)}[dt]
    if not off:
        plan = am.call_plan(code, B, Hh, Lq, Lk, D, desc, 1 << 20)
        assert (plan["path"], plan["tiles"]) == (am.ATN_PATH_SPLIT_D, 0) and plan["chunk_rows"] < Lq
    sigma = 0.5 if pe == "sin" else 1.0
    Q, K, V = H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 970, sigma)
    if dt == "bf16":
        Q, K, V = (oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(x)) for x in (Q, K, V))
    dev_t = [H.upload(np.concatenate([[0.0] * off, x.ravel()]).astype(np.float32), dt) for x in (Q, K, V)]
    ws = hip_rt.DeviceArray(((1 << 20) // 4,), "f32", fill=0)
    out = H.empty((Q.size + off,), dt)
    st = am.lib().atn_attention_fwd_ex(code, *[t.ptr + off * es for t in dev_t], out.ptr + off * es, B, Hh, Lq,
                                       Lk, D, ctypes.byref(desc) if desc else None, ws.ptr, 1 << 20, None)
    assert st == 0
    hip_rt.synchronize()
    got = out.numpy()[off:].reshape(Q.shape)
    n, a, b = (H.check_f32 if dt == "f32" else H.check_bf16)(got, _ref(pe, Q, K, V))
    assert n == 0, (a, b)


@pytest.mark.parametrize("D", [264, 263], ids=str)
def test_scratch_for_scores_alone(am, dev, D):
    """fp32 without an encoding needs no copies: a scratch that holds one row of
    scores but not P beside them."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 1, 3, 90001
    nb = 40960 + 256 + 4 * Lk + 4096
    print(f"[case] scores alone {D}", flush=True)
    plan = am.call_plan(0, B, Hh, Lq, Lk, D, None, nb)
    assert (plan["tiles"], plan["chunk_rows"]) == (0, 1)
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 971)
    ws, out = hip_rt.DeviceArray((nb // 4,), "f32", fill=0), H.empty(Q.shape)
    am.attention_ex(q, k, v, out, workspace=ws)
    hip_rt.synchronize()
    _check(out.numpy(), Q, K, V, "none")


@pytest.mark.parametrize("dt,D,pe,kib", [("f32", 1024, "rope", 1160), ("bf16", 1004, "none", 1200)], ids=str)
def test_scratch_that_copies_nearly_fill(am, dev, dt, D, pe, kib):
    """K's copy (and V's) would leave the scratch a few rows a chunk: the
    kernels without copies."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 1, 300, 260
    print(f"[case] copies nearly fill the scratch {dt} {D} {pe}", flush=True)
    desc, code = _desc(am, pe), {"f32": 0, "bf16": 1}[dt]
    assert am.call_plan(code, B, Hh, Lq, Lk, D, desc, kib << 10)["tiles"] == 0
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 975, dt)
    ws = hip_rt.DeviceArray(((kib << 10) // 4,), "f32", fill=0)
    out = H.empty(Q.shape, dt)
    am.attention_ex(q, k, v, out, pe=desc, workspace=ws)
    hip_rt.synchronize()
    n, a, b = (H.check_f32 if dt == "f32" else H.check_bf16)(out.numpy(), _ref(pe, Q, K, V))
    assert n == 0, (a, b)


@pytest.mark.parametrize("tile", [0, 64, 128])
@pytest.mark.parametrize("shape,pe", [
    ((1, 2, 68, 68, 624), "none"),       # a small grid of the GEMM path's
    ((1, 1, 129, 200, 264), "none"),     # 4 full 64-deep stages and one of 8 dims
    ((1, 2, 130, 140, 328), "half"),
    ((1, 1, 65, 257, 1000), "rope_q"),   # K only widened
    ((2, 1, 200, 70, 512), "half_k"),
    ((1, 1, 70, 65, 2056), "sin"),
    ((1, 1, 131, 129, 261), "none"),     # head_d % 8 == 1: padded copies
    ((1, 2, 66, 200, 262), "none"),
    ((1, 1, 128, 128, 516), "rope"),
    ((1, 1, 90, 150, 269), "sin"),
    ((1, 1, 150, 90, 18), "half"),
], ids=str)
def test_tile_edges_bf16(am, dev, tuner, tile, shape, pe):
    import hip_rt
    B, Hh, Lq, Lk, D = shape
    print(f"[case] bf16 tile {tile} {shape} {pe}", flush=True)
    if tile:
        tuner.set(splitd_tile=tile)
    sigma = 0.5 if pe == "sin" else 1.0
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 800 + Lq + D, "bf16", sigma)
    out = H.empty(Q.shape, "bf16")
    am.attention_ex(q, k, v, out, pe=_desc(am, pe))
    hip_rt.synchronize()
    n, nrel, mabs = H.check_bf16(out.numpy(), _ref(pe, Q, K, V))
    assert n == 0, (nrel, mabs)
    # one rounding of the output (2^-9 at most), P to 16 bits or more, exact products
    assert nrel < 2.0 ** -9


@pytest.mark.parametrize("eq,ek", [(-60, 60), (60, -60), (-14, 14), (18, -18)], ids=str)
@pytest.mark.parametrize("D,pe", [(272, "half"), (262, "rope"), (272, "half_k")], ids=str)
def test_bf16_encoded_magnitudes(am, dev, D, pe, eq, ek):
    """Encoded bf16 Q and K at any magnitude (16 bits of them, 24 where head_d
    % 8 != 0): the output's own rounding is the error."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 2, 130, 140
    print(f"[case] bf16 encoded magnitudes {D} {pe} {eq} {ek}", flush=True)
    assert am.call_plan(1, B, Hh, Lq, Lk, D, _desc(am, pe))["tiles"] == 1
    (_, _, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 815, "bf16")
    q, k = H.upload(np.ldexp(Q, eq), "bf16"), H.upload(np.ldexp(K, ek), "bf16")
    out = H.empty(Q.shape, "bf16")
    am.attention_ex(q, k, v, out, pe=_desc(am, pe))
    hip_rt.synchronize()
    n, nrel, mabs = H.check_bf16(out.numpy(), _ref(pe, Q, K, V))
    assert n == 0, (nrel, mabs)
    assert nrel < 2.0 ** -9


@pytest.mark.parametrize("D", [264, 267, 40], ids=str)
def test_misaligned_bases_bf16(am, dev, D):
    """bf16 tensors 2 bytes off: copied into aligned rows first."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 2, 100, 140
    print(f"[case] misaligned bf16 {D}", flush=True)
    Q, K, V = (oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(x))
               for x in H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), seed=961))
    dev_t = [H.upload(np.concatenate([[0.0], x.ravel()]).astype(np.float32), "bf16")
             for x in (Q, K, V)]
    out = H.empty((Q.size + 1,), "bf16")
    st = am.lib().atn_attention_fwd_ex(1, *[t.ptr + 2 for t in dev_t], out.ptr + 2, B, Hh, Lq, Lk, D,
                                       None, None, 0, None)
    assert st == 0
    hip_rt.synchronize()
    n, nrel, mabs = H.check_bf16(out.numpy()[1:].reshape(Q.shape), _ref("none", Q, K, V))
    assert n == 0, (nrel, mabs)


@pytest.mark.parametrize("dt,D,pe", [("bf16", 264, "none"), ("bf16", 264, "half"), ("bf16", 40, "none"),
                                     ("f32", 264, "none"), ("f32", 40, "none")], ids=str)
def test_misaligned_output(am, dev, dt, D, pe):
    """The output alone off a 16-byte boundary."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 2, 100, 140
    code, es = (1, 2) if dt == "bf16" else (0, 4)
    print(f"[case] misaligned output {dt} {D} {pe}", flush=True)
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 964, dt)
    out = H.empty((Q.size + 1,), dt)
    desc = _desc(am, pe)
    st = am.lib().atn_attention_fwd_ex(code, q.ptr, k.ptr, v.ptr, out.ptr + es, B, Hh, Lq, Lk, D,
                                       ctypes.byref(desc) if desc else None, None, 0, None)
    assert st == 0
    hip_rt.synchronize()
    n, a, b = (H.check_f32 if dt == "f32" else H.check_bf16)(out.numpy()[1:].reshape(Q.shape),
                                                             _ref(pe, Q, K, V))
    assert n == 0, (a, b)


@pytest.mark.parametrize("dt,D", [("bf16", 264), ("bf16", 40), ("bf16", 267), ("f32", 264), ("f32", 64)], ids=str)
def test_misaligned_bases_in_the_reported_workspace(am, dev, dt, D):
    """atn_attention_workspace_bytes covers tensors off a 16-byte boundary."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 2, 100, 140
    code, es = (1, 2) if dt == "bf16" else (0, 4)
    print(f"[case] misaligned in the reported workspace {dt} {D}", flush=True)
    (Q, K, V) = H.rng_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), seed=963)
    if dt == "bf16":
        Q, K, V = (oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(x)) for x in (Q, K, V))
    dev_t = [H.upload(np.concatenate([[0.0], x.ravel()]).astype(np.float32), dt) for x in (Q, K, V)]
    out = H.empty((Q.size + 1,), dt)
    nb = am.workspace_bytes(code, B, Hh, Lq, Lk, D)
    ws = hip_rt.DeviceArray((nb // 4,), "f32", fill=0)
    st = am.lib().atn_attention_fwd_ex(code, *[t.ptr + es for t in dev_t], out.ptr + es, B, Hh, Lq, Lk, D,
                                       None, ws.ptr, nb // 4 * 4, None)
    assert st == 0
    hip_rt.synchronize()
    n, a, b = (H.check_f32 if dt == "f32" else H.check_bf16)(out.numpy()[1:].reshape(Q.shape),
                                                             _ref("none", Q, K, V))
    assert n == 0, (a, b)


@pytest.mark.parametrize("scale", [2.0 ** 40, 2.0 ** -40, 2.0 ** 123], ids=str)
@pytest.mark.parametrize("D", [272, 261], ids=str)
def test_bf16_range(am, dev, scale, D):
    """bf16 keeps fp32's exponents: V far outside fp16's range, up to its
    largest values."""
    import hip_rt
    B, Hh, Lq, Lk = 1, 1, 70, 90
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 811, "bf16")
    v = H.upload(V * np.float32(scale), "bf16")
    out = H.empty(Q.shape, "bf16")
    am.attention_ex(q, k, v, out)
    hip_rt.synchronize()
    n, nrel, mabs = H.check_bf16(out.numpy() / np.float32(scale), _ref("none", Q, K, V))
    assert n == 0, (nrel, mabs)


def test_chunked_tiles(am, dev):
    """A bf16 call of the tiles in chunks of heads and rows: the same bits (a
    head size that the GEMM path, which needs less scratch, does not take)."""
    import hip_rt
    B, Hh, Lq, Lk, D = 1, 3, 300, 260, 1004
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 812, "bf16")
    full, out = H.empty(Q.shape, "bf16"), H.empty(Q.shape, "bf16")
    am.attention_ex(q, k, v, full)
    hip_rt.synchronize()
    plan = am.call_plan(1, B, Hh, Lq, Lk, D, None, 2 << 20)
    assert plan["tiles"] == 1 and (plan["chunk_heads"], plan["chunk_rows"]) == (1, 75)
    ws = hip_rt.DeviceArray(((2 << 20) // 4,), "f32", fill=0)
    am.attention_ex(q, k, v, out, workspace=ws)
    hip_rt.synchronize()
    assert np.array_equal(out.bits(), full.bits())
    n, nrel, mabs = H.check_bf16(out.numpy(), _ref("none", Q, K, V))
    assert n == 0, (nrel, mabs)


@pytest.mark.parametrize("dt,shape", [
    ("f32", (1, 4, 300, 300, 256)), ("f32", (1, 8, 130, 130, 200)), ("f32", (1, 16, 100, 100, 256)),
    ("f32", (2, 3, 65, 129, 248)), ("bf16", (1, 4, 417, 417, 256)), ("bf16", (1, 8, 130, 130, 200)),
    ("bf16", (2, 3, 65, 129, 248))], ids=str)
def test_small_grids_of_the_flash_kernel(am, dev, tuner, dt, shape):
    """head_d 129-256 on small grids runs on the tiles, and on the flash kernel
    where the scratch is too small for them: both against the oracle, and a
    forced flash form agrees with the small-scratch call bit for bit."""
    import hip_rt
    B, Hh, Lq, Lk, D = shape
    code = {"f32": 0, "bf16": 1}[dt]
    print(f"[case] flash or tiles {dt} {shape}", flush=True)
    assert am.path(code, B, Hh, Lq, Lk, D) == am.ATN_PATH_FLASH
    assert am.call_plan(code, B, Hh, Lq, Lk, D)["tiles"] == 1
    assert am.call_plan(code, B, Hh, Lq, Lk, D, None, 64 << 10)["path"] == am.ATN_PATH_FLASH
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 820 + Lq, dt)
    out, small, flash = (H.empty(Q.shape, dt) for _ in range(3))
    am.attention_ex(q, k, v, out)
    ws = hip_rt.DeviceArray(((64 << 10) // 4,), "f32", fill=0)
    am.attention_ex(q, k, v, small, workspace=ws)
    tuner.set(flash_split=1)
    am.attention_ex(q, k, v, flash)
    hip_rt.synchronize()
    ref = _ref("none", Q, K, V)
    for got in (out, small):
        n, nrel, mabs = H.check_f32(got.numpy(), ref) if dt == "f32" else H.check_bf16(got.numpy(), ref)
        assert n == 0, (nrel, mabs)
    assert np.array_equal(small.numpy(), flash.numpy())
    assert not np.array_equal(out.numpy(), flash.numpy())  # the tiles' sums


@pytest.mark.parametrize("rng_case", list(RANGES))
def test_fp32_magnitudes_of_small_flash_grids(am, dev, rng_case):
    """fp32 of head_d 129-256 moved to the tiles keeps its accuracy wherever
    the values lie."""
    import hip_rt
    dims = (1, 2, 150, 140, 256)
    print(f"[case] magnitudes, small flash grid {rng_case}", flush=True)
    assert am.call_plan(0, *dims)["tiles"] == 1
    Q, K, V = _ranged(rng_case, dims, 985)
    out = H.empty(Q.shape)
    am.attention_ex(*(H.upload(x) for x in (Q, K, V)), out)
    hip_rt.synchronize()
    _check64(out.numpy(), Q, K, V)
