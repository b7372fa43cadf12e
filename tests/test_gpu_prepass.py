"""The positional-encoding pre-pass against the oracle, bit for bit: row and
group counts around the kernel's blocks, position wrap-around, both table
layouts, partial rotary widths, in-place calls, both dtypes, and the kernel
for head sizes and tables that are no whole vectors."""
import numpy as np
import pytest

import helpers as H
import oracle

pytestmark = pytest.mark.gpu


def _tables(kind, L, D, rot):
    return oracle.sinusoidal_table(L, D) if kind == "sinusoidal" else oracle.rope_cache(L, rot)


def _want(x, kind, L, D, rot, pairing, dup):
    a, b = _tables(kind, L, D, rot)
    rows = x.reshape(-1, D)
    n = -(-rows.shape[0] // L) * L  # whole slabs of L positions
    pad = np.zeros((n, D), np.float32)
    pad[:rows.shape[0]] = rows
    slabs = pad.reshape(-1, L, D)
    y = (oracle.add_sinusoidal(slabs, a, b) if kind == "sinusoidal" else
         oracle.apply_rope(slabs, a, b, rotary_dim=rot, pairing=pairing))
    return y.reshape(-1, D)[:rows.shape[0]]


@pytest.mark.parametrize("rows,L,D,rot,kind,pairing,dup,dtype,inplace", [
    (1, 1, 4, 4, "rope", "interleaved", False, "f32", False),        # one group
    (1025, 1, 4, 4, "rope", "interleaved", True, "f32", False),      # one past a block
    (3000, 7, 8, 8, "rope", "half", False, "f32", False),
    (257, 1500, 100, 100, "rope", "interleaved", True, "f32", False),
    (500, 33, 100, 40, "rope", "half", False, "f32", True),          # in place, pairs apart
    (500, 33, 256, 256, "rope", "half", True, "f32", True),
    (64, 64, 2048, 128, "rope", "interleaved", True, "f32", False),
    (40, 3, 8192, 8192, "rope", "half", False, "bf16", True),
    (700, 129, 72, 72, "sinusoidal", "interleaved", False, "bf16", False),
    (700, 129, 72, 72, "sinusoidal", "interleaved", True, "f32", True),
    (5, 40000, 36, 36, "rope", "interleaved", False, "f32", False),  # positions past 2^15
    (3, 2, 140000, 140000, "sinusoidal", "interleaved", False, "f32", False),  # groups past 2^15
    (100, 20, 98, 50, "rope", "half", False, "f32", False),          # a workgroup per row
    (100, 20, 96, 50, "rope", "interleaved", True, "bf16", False),
    (100, 20, 77, 77, "sinusoidal", "interleaved", False, "bf16", False),
], ids=str)
def test_prepass_bit_exact(am, dev, rows, L, D, rot, kind, pairing, dup, dtype, inplace):
    import hip_rt
    print(f"[case] prepass {rows}x{D} L={L} rot={rot} {kind} {pairing} dup={dup} {dtype}",
          flush=True)
    rng = np.random.default_rng(rows + D)
    x = H.upload(rng.standard_normal((rows, D), dtype=np.float32), dtype)
    host = x.numpy()
    tabs = [H.upload(t) for t in _tables(kind, L, D, rot)] if dup else [None, None]
    pe = am.make_pe(kind, pairing, rot if kind == "rope" else 0, table_a=tabs[0], table_b=tabs[1])
    out = x if inplace else H.empty((rows, D), dtype)
    am.pe_apply_ex(x, out, L, pe)
    hip_rt.synchronize()
    want = _want(host, kind, L, D, rot, pairing, dup)
    if dtype == "bf16":
        want = oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(want))
    assert np.array_equal(out.numpy(), want)


def test_prepass_misaligned_tables(am, dev):
    """Caller tables off a 16-byte boundary."""
    import hip_rt
    L, D = 50, 64
    c, s = oracle.rope_cache(L, D)
    off = [np.concatenate([[0.0], t.ravel()]).astype(np.float32) for t in (c, s)]
    dc, ds = (H.upload(t) for t in off)
    pe = am.make_pe("rope", "interleaved", D)
    pe.table_a, pe.table_b = dc.ptr + 4, ds.ptr + 4
    x = np.random.default_rng(3).standard_normal((2, L, D), dtype=np.float32)
    dx, out = H.upload(x), H.empty(x.shape)
    am.pe_apply_ex(dx, out, L, pe)
    hip_rt.synchronize()
    assert np.array_equal(out.numpy(), oracle.apply_rope(x, c, s))


def test_separate_rope_reusing_q_memory(am, dev):
    """K's rotated copy written over Q once Q has been rotated."""
    import hip_rt
    B, Hh, L, D = 1, 2, 96, 64
    Q, K, V = H.rng_inputs((B, Hh, L, D), (B, Hh, L, D), seed=77)
    c, s = oracle.rope_cache(L, D)
    q, k, v, tc, ts = (H.upload(t) for t in (Q, K, V, c, s))
    qr, out = H.empty(Q.shape), H.empty(Q.shape)
    am.attention_forward_separate_rope(q, k, v, qr, q, out, tc, ts, D)
    hip_rt.synchronize()
    assert np.array_equal(qr.numpy(), oracle.apply_rope(Q, c, s))
    assert np.array_equal(q.numpy(), oracle.apply_rope(K, c, s))
    n, mabs, _ = H.check_f32(out.numpy(), oracle.attention_rope(Q, K, V, c, s, nthreads=8))
    assert n == 0, mabs
