"""The split-D pipeline's tile kernels against the oracle: edges of both tile
sizes, odd and even stage counts, head sizes that are no whole number of
vectors, misaligned bases, encodings per side, every softmax row form, and the
in-kernel encoding that remains where the scratch holds no encoded copies."""
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
    import ctypes

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


@pytest.mark.parametrize("pe", ["rope", "half", "sin"])
def test_scratch_without_encoded_copies(am, dev, tuner, pe):
    """K's encoded copy alone exceeds the scratch: encoded in the QK^T kernel."""
    import hip_rt
    B, Hh, Lq, Lk, D = 1, 1, 70, 400, 1024  # 1.6 MB of encoded K
    print(f"[case] lean {pe}", flush=True)
    desc = _desc(am, pe)
    tuner.set(workspace_cap_mib=1)
    assert am.workspace_bytes(0, B, Hh, Lq, Lk, D, desc) <= 1 << 20
    sigma = 0.5 if pe == "sin" else 1.0
    (q, k, v), (Q, K, V) = H.device_inputs((B, Hh, Lq, D), (B, Hh, Lk, D), 970, "f32", sigma)
    ws = hip_rt.DeviceArray(((1 << 20) // 4,), "f32", fill=0)
    out = H.empty(Q.shape)
    am.attention_ex(q, k, v, out, pe=desc, workspace=ws)
    hip_rt.synchronize()
    _check(out.numpy(), Q, K, V, pe)
