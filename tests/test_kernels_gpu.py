"""GPU parity of every single-kernel hook against the oracle's float64 closed forms.

Mirrors the reference's tests/test_kernels.py:43-229 (same seeds, shapes, grids and tolerances),
then widens it: every Llama-3.2-1B projection shape the reference benchmarks, the generic-width
matvec path, context lengths up to 8192 (its long-context attention case), and the GPU quantisers bit-exact.
"""
import numpy as np
import pytest

from cudallm_amd import engine as E
from cudallm_amd import quantize as GQ
from oracle import kernels as K
from oracle import quantize as Q

pytestmark = pytest.mark.gpu

NH, NKV, HD, MAX_SEQ = 32, 8, 64, 4096


@pytest.fixture(autouse=True)
def _gpu(gpu):
    return gpu


def _operands(wtype: str, rows: int, cols: int, seed: int, bf16_master: bool = False):
    """(stored weight, scales or None, exact dequantised weight in float64)."""
    w = np.random.default_rng(seed).normal(0, 0.02, size=(rows, cols)).astype(np.float32)
    if bf16_master:
        w = Q.bf16_bits_to_f32(Q.bf16_round_bits(w))
    if wtype == "bf16":
        bits = Q.bf16_round_bits(w)
        return bits, None, Q.bf16_bits_to_f32(bits).astype(np.float64)
    if wtype == "int8":
        q, s = Q.quantize_int8_rows(w)
        return q, s, Q.dequantize_int8_rows(q, s).astype(np.float64)
    p, s = Q.quantize_int4_groups(w, 128)
    return p, s, Q.dequantize_int4_groups(p, s).astype(np.float64)


# ---- matvec (reference tests/test_kernels.py:43-96) ----------------------------------------

def test_matvec_naive_bf16_store():
    rows, cols = 1024, 2048
    rng = np.random.default_rng(10)
    bits = Q.bf16_round_bits(rng.normal(0, 0.02, size=(rows, cols)))
    x = rng.standard_normal(cols).astype(np.float32)
    y = E.kernel_matvec("naive", "bf16", "store", 0, 0, bits, None, x, None, 1e-5, None, rows, cols)
    ref = Q.bf16_bits_to_f32(bits).astype(np.float64) @ x.astype(np.float64)
    assert np.allclose(y, ref, rtol=1e-4, atol=1e-4)


def _check_matvec(wtype, epilogue, fuse_norm, rpb, rows, cols, seed, bf16_master=False):
    eps = 1e-5
    w, s, w64 = _operands(wtype, rows, cols, seed, bf16_master)
    rng = np.random.default_rng(seed + 1)
    x = rng.standard_normal(cols).astype(np.float32)
    norm_w = rng.uniform(0.5, 1.5, cols).astype(np.float32)
    out_rows = rows // 2 if epilogue == "swiglu" else rows
    y_init = rng.standard_normal(out_rows).astype(np.float32) if epilogue == "add" else None
    print(f"[matvec] {wtype} {epilogue} norm={fuse_norm} rpb={rpb} {rows}x{cols}", flush=True)
    y = E.kernel_matvec("opt", wtype, epilogue, fuse_norm, rpb, w, s, x, norm_w if fuse_norm else None, eps, y_init,
                        rows, cols)
    ref = K.matvec(w64, x, epilogue, norm_w if fuse_norm else None, eps, y_init)
    err = np.abs(y - ref) - (1e-4 + 1e-4 * np.abs(ref))
    assert np.all(err <= 0), f"max excess {err.max():.3e} at row {int(np.argmax(err))}"


@pytest.mark.parametrize("shape", [(1024, 2048), (2048, 8192)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("rpb", [1, 2, 4, 8])
@pytest.mark.parametrize("fuse_norm", [0, 1])
@pytest.mark.parametrize("epilogue", ["store", "add", "swiglu"])
@pytest.mark.parametrize("wtype", ["bf16", "int8", "int4"])
def test_matvec_opt(wtype, epilogue, fuse_norm, rpb, shape):
    rows, cols = shape
    _check_matvec(wtype, epilogue, fuse_norm, rpb, rows, cols, seed=20 + rows + cols)


# Every projection shape the reference benchmarks, with the engine epilogues (norm fused on the input side
# of q/k/v/gate/up/lm_head, residual add on o/down), bf16-rounded N(0, 0.02) master weights.
MODEL_SHAPES = [("q", 2048, 2048, "store", 1), ("k", 512, 2048, "store", 1), ("v", 512, 2048, "store", 1),
                ("o", 2048, 2048, "add", 0), ("gate", 8192, 2048, "store", 1), ("up", 8192, 2048, "store", 1),
                ("down", 2048, 8192, "add", 0), ("wqkv", 3072, 2048, "store", 1),
                ("gate_up", 16384, 2048, "swiglu", 1), ("lm_head", 128256, 2048, "store", 1)]


@pytest.mark.parametrize("wtype", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("name,rows,cols,epilogue,norm", MODEL_SHAPES, ids=[s[0] for s in MODEL_SHAPES])
def test_matvec_model_shapes(wtype, name, rows, cols, epilogue, norm):
    _check_matvec(wtype, epilogue, norm, 0, rows, cols, seed=rows * 7 + cols, bf16_master=True)


@pytest.mark.parametrize("wtype", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("rows,cols", [(1000, 1024), (37, 3072), (130, 12288), (6, 2048), (10, 8192), (20483, 2048)])
@pytest.mark.parametrize("epilogue", ["store", "add", "swiglu"])
def test_matvec_generic_and_ragged(wtype, rows, cols, epilogue):
    """Widths other than 2048/8192 (LDS-staged path) and row counts that leave partial blocks; 20483 rows of 2048
    give the waves uneven row ranges of several passes each."""
    if epilogue == "swiglu" and rows % 2:
        rows += 1
    _check_matvec(wtype, epilogue, 1, 4, rows, cols, seed=rows + 3 * cols)


@pytest.mark.parametrize("wtype", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("rows,cols,epilogue", [(1, 1024, "store"), (3, 5120, "add"), (2, 11264, "swiglu"),
                                                (8191, 1024, "store"), (8194, 7168, "swiglu"), (600000, 1024, "store"),
                                                (4094, 8192, "swiglu"), (4098, 8192, "swiglu"), (513, 2048, "store"),
                                                (1025, 2048, "add"), (1025, 8192, "add")])
def test_matvec_wide_rows(wtype, rows, cols, epilogue):
    """The any-width kernel where its division of the rows changes: one row, an odd last row, widths that end inside a
    line, waves without rows, waves with as many rows as they take (600000 rows); and both sides of the row counts at
    which the choice of kernel or of rows per wave changes.  The error against 64 bits stays
    under cols roundings of 2^-24 of the inputs, in the root mean square about sqrt(cols) of them: 1e-5 is ten times."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + cols)
    n = rows // 2 if epilogue == "swiglu" else rows
    q = torch.randint(-8 if wtype == "int4" else -127, 8 if wtype == "int4" else 128, (rows, cols), generator=g,
                      device="cuda", dtype=torch.int8)
    scales = None
    if wtype == "bf16":
        w = q.to(torch.bfloat16)
    elif wtype == "int8":
        w, scales = q, torch.rand(rows, generator=g, device="cuda") + 0.5
    else:
        u = (q + 8).view(rows, cols // 2, 2).to(torch.uint8)
        w, scales = u[..., 0] | (u[..., 1] << 4), (torch.rand(rows, cols // 128, generator=g, device="cuda") + 0.5).half()
    x, norm = torch.randn(cols, generator=g, device="cuda"), torch.rand(cols, generator=g, device="cuda") + 0.5
    y0 = torch.randn(n, generator=g, device="cuda")
    y = torch.cat([y0, torch.full((8,), 3.0, device="cuda")])
    E.launch_matvec(wtype, epilogue, 0, w.data_ptr(), None if scales is None else scales.data_ptr(), x.data_ptr(),
                    norm.data_ptr(), 1e-5, y.data_ptr(), rows, cols, torch.cuda.current_stream().cuda_stream)
    xn = x.double()
    xn = xn * torch.rsqrt((xn * xn).mean() + 1e-5) * norm.double()
    d = torch.empty(rows, dtype=torch.float64, device="cuda")
    for r in range(0, rows, 50000):
        m = q[r:r + 50000].double()
        if wtype == "int8":
            m *= scales[r:r + 50000, None].double()
        elif wtype == "int4":
            m = (m.view(len(m), -1, 128) * scales[r:r + 50000, :, None].double()).view(len(m), cols)
        d[r:r + 50000] = m @ xn
    ref = torch.nn.functional.silu(d[:n]) * d[n:] if epilogue == "swiglu" else d + y0.double() if epilogue == "add" else d
    assert (y[:n].double() - ref).norm() <= 1e-5 * ref.norm()
    assert bool((y[n:] == 3.0).all())  # nothing past the outputs


@pytest.mark.parametrize("wtype", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_matvec_wide_non_finite_input(wtype, norm, value):
    """An infinite or NaN input does not come out as a number: with a norm, and for the quantised types, every output is
    NaN; plain bf16 outputs are the infinity with the weight's sign."""
    import torch
    rows, cols = 40, 3072
    w, s, w64 = _operands(wtype, rows, cols, 5)
    x = np.random.default_rng(6).standard_normal(cols).astype(np.float32)
    x[1000] = value
    y = E.kernel_matvec("opt", wtype, "store", int(norm), 0, w, s, x, np.ones(cols, np.float32), 1e-5, None, rows, cols)
    if wtype == "bf16" and not norm:
        want = w64[:, 1000] * value
        np.testing.assert_array_equal(y, want.astype(np.float32))
    else:
        assert np.isnan(y).all()


@pytest.mark.parametrize("wtype", ["int8", "int4"])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("outlier", [1e3, 1e6])
@pytest.mark.parametrize("rows,cols,epilogue", [(1001, 1024, "store"), (700, 2048, "store"), (500, 5120, "add"),
                                                (300, 12288, "store"), (4096, 8192, "swiglu")])
def test_matvec_outlier_input(wtype, norm, outlier, rows, cols, epilogue):
    """One input far above the others that meets zero weights: it may cost the 16 (int8) or 32 (int4) inputs of its own
    chunk bits, and no others.  A chunk's fixed-point words have a step of at most 2 m / 7829350 for its largest input m,
    which leaves a row an error of sigma = that step / sqrt(12) times the 2-norm of the row's weights in the chunk.  Bound
    for every row: 8 sigma, and 1e-6 (16 roundings) of the 2-norms of the row and of the other inputs.  One scale for all
    columns leaves 8 (1024 columns) to 28 sigma in the root mean square over the rows, and more than three times that in
    the worst of them."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + cols)
    n, col, chunk = rows // 2 if epilogue == "swiglu" else rows, cols // 2 + 37, 32 if wtype == "int4" else 16
    top = 7 if wtype == "int4" else 127
    q = torch.randint(-top, top + 1, (rows, cols), generator=g, device="cuda", dtype=torch.int8)
    q[:, col] = 0
    if wtype == "int8":
        w, scales = q, torch.ones(rows, device="cuda")
    else:
        u = (q + 8).view(rows, cols // 2, 2).to(torch.uint8)
        w, scales = u[..., 0] | (u[..., 1] << 4), torch.ones(rows, cols // 128, device="cuda").half()
    x, nw = torch.randn(cols, generator=g, device="cuda"), torch.rand(cols, generator=g, device="cuda") + 0.5
    x[col] = outlier
    y0 = torch.randn(n, generator=g, device="cuda")
    y = y0.clone()
    E.launch_matvec(wtype, epilogue, 0, w.data_ptr(), scales.data_ptr(), x.data_ptr(), nw.data_ptr() if norm else None, 1e-5,
                    y.data_ptr(), rows, cols, torch.cuda.current_stream().cuda_stream)
    xn = x.double()
    if norm:
        xn = xn * torch.rsqrt((xn * xn).mean() + 1e-5) * nw.double()
    m = q.double()
    d = m @ xn
    c0 = col // chunk * chunk
    sigma = 2 * xn[col].abs() / 7829350 / 12 ** 0.5 * m[:, c0:c0 + chunk].norm(dim=1)
    rest = xn.clone()
    rest[col] = 0.0
    bound = 8 * sigma + 1e-6 * m.norm(dim=1) * rest.norm()
    if epilogue == "swiglu":  # silu's slope is at most 1.1
        act = torch.nn.functional.silu(d[:n])
        ref, bound = act * d[n:], 1.1 * bound[:n] * (d[n:].abs() + bound[n:]) + act.abs() * bound[n:] + 1e-6 * (act * d[n:]).abs()
    else:
        ref = d + y0.double() if epilogue == "add" else d
        bound = bound + 1e-6 * ref.abs()
    excess = ((y.double() - ref).abs() / bound).max().item()
    assert excess <= 1, f"{excess} times the bound"


@pytest.mark.parametrize("wtype", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("cols", [2048, 3072])
@pytest.mark.parametrize("size,weight", [(1e15, 1e25), (1e-18, 1e-24), (1e-18, 1e24), (0.0, 1.0)])
def test_matvec_norm_weight_range(wtype, cols, size, weight):
    """Inputs whose products with the norm weights leave the floats' range although the normalised inputs do not."""
    rows, rng = 40, np.random.default_rng(cols)
    w, s, w64 = _operands(wtype, rows, cols, 7)
    x = (size * rng.standard_normal(cols)).astype(np.float32)
    norm_w = (weight * rng.uniform(0.5, 1.5, cols)).astype(np.float32)
    eps = 1e-5 if size == 0 else 0.0
    y = E.kernel_matvec("opt", wtype, "store", 1, 0, w, s, x, norm_w, eps, None, rows, cols)
    x64 = x.astype(np.float64)
    ref = w64 @ (x64 / np.sqrt((x64 * x64).mean() + eps) * norm_w)
    assert np.linalg.norm(y - ref) <= 1e-5 * np.linalg.norm(ref)


def test_stream_read_timed_hook():
    """The bandwidth kernel on a device buffer through its timed hook: every launch shape records both events, and the
    sink (written only for one XOR-folded word that a zero buffer never gives) stays untouched."""
    import torch
    buf = torch.zeros(8 << 20, dtype=torch.uint8, device="cuda")
    sink = torch.zeros(16 * 1024, dtype=torch.int32, device="cuda")
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    stream = torch.cuda.current_stream()
    a.record(stream)
    b.record(stream)
    for bpc in (4, 8, 16):
        E.launch_stream_read_timed(buf.data_ptr(), buf.numel(), bpc, sink.data_ptr(), sink.numel(), stream.cuda_stream,
                                   a.cuda_event, b.cuda_event)
        b.synchronize()
        assert 0 < a.elapsed_time(b) < 100
    assert int(sink.abs().sum()) == 0


def test_matvec_config1_int8_known_case():
    """The reference's int8 8192x2048 matvec case: bf16 master N(0, 0.02), x bf16 N(0, 1), checked in float64."""
    rng = np.random.default_rng(1)
    w = Q.bf16_bits_to_f32(Q.bf16_round_bits(rng.normal(0, 0.02, size=(8192, 2048)).astype(np.float32)))
    x = Q.bf16_bits_to_f32(Q.bf16_round_bits(rng.standard_normal(2048).astype(np.float32)))
    q, s = Q.quantize_int8_rows(w)
    y = E.kernel_matvec("opt", "int8", "store", 0, 0, q, s, x, None, 1e-5, None, 8192, 2048)
    ref = (q.astype(np.float64) * s.astype(np.float64)[:, None]) @ x.astype(np.float64)
    assert np.allclose(y, ref, rtol=1e-4, atol=1e-4)
    assert np.max(np.abs(y - ref) / np.maximum(np.abs(ref), 1e-3)) < 1e-2


# ---- rmsnorm, rope, attention, silu, argmax (reference tests/test_kernels.py:101-229) -------

def test_rmsnorm():
    n, eps = 2048, 1e-5
    rng = np.random.default_rng(11)
    x = rng.standard_normal(n).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    assert np.allclose(E.kernel_rmsnorm(x, w, eps), K.rms_normalize(x, w, eps), rtol=1e-5, atol=1e-5)


SENTINEL = np.float16(-7.25)


def _ulp_diff(a, b):
    def ordered(v):
        u = v.astype(np.float16).view(np.uint16).astype(np.int32)
        return np.where(u & 0x8000, 0x8000 - u, u)
    return np.abs(ordered(a) - ordered(b))


@pytest.mark.parametrize("pos", [0, 1, 777, 4095])
@pytest.mark.parametrize("fused", [0, 1])
def test_rope_kv(fused, pos):
    rng = np.random.default_rng(12 + pos)
    inv = K.llama3_inv_freq()
    qkv = rng.standard_normal((NH + 2 * NKV) * HD).astype(np.float32)
    kc = np.full((NKV, MAX_SEQ, HD), SENTINEL, dtype=np.float16)
    vc = np.full((NKV, MAX_SEQ, HD), SENTINEL, dtype=np.float16)
    out, k_out, v_out = E.kernel_rope_kv(fused, qkv, inv, pos, kc, vc, NH, NKV, HD, MAX_SEQ)
    k_out, v_out = k_out.reshape(NKV, MAX_SEQ, HD), v_out.reshape(NKV, MAX_SEQ, HD)
    q_ref, k_ref, _, vc_ref = K.rope_kv(qkv, inv, pos, kc, vc, NH, NKV, HD)
    assert np.allclose(out[:NH * HD].reshape(NH, HD), q_ref, rtol=0, atol=1e-5)
    if not fused:
        assert np.allclose(out[NH * HD:(NH + NKV) * HD].reshape(NKV, HD), k_ref, rtol=0, atol=1e-5)
        np.testing.assert_array_equal(out[(NH + NKV) * HD:], qkv[(NH + NKV) * HD:])
    else:
        np.testing.assert_array_equal(out[NH * HD:], qkv[NH * HD:])  # k and v slices untouched
    assert np.all(_ulp_diff(k_out[:, pos, :], k_ref.astype(np.float16)) <= 1)
    np.testing.assert_array_equal(v_out, vc_ref)  # v row bit-exact, every other slot untouched
    others = np.ones(MAX_SEQ, dtype=bool)
    others[pos] = False
    assert np.all(k_out[:, others, :] == SENTINEL)


@pytest.fixture(scope="module")
def attn_data():
    rng = np.random.default_rng(13)
    return (rng.standard_normal(NH * HD).astype(np.float32),
            rng.standard_normal((NKV, MAX_SEQ, HD)).astype(np.float16),
            rng.standard_normal((NKV, MAX_SEQ, HD)).astype(np.float16))


@pytest.mark.parametrize("ctx", [1, 7, 128, 129, 1000, 4096])
@pytest.mark.parametrize("impl", ["naive", "opt"])
def test_attention(impl, ctx, attn_data):
    q, k, v = attn_data
    out = E.kernel_attention(impl, q, k, v, ctx, NH, NKV, HD, MAX_SEQ)
    assert np.allclose(out, K.attention(q, k, v, ctx, NH, NKV, HD), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("ctx", [128, 512, 2048, 4096, 8192, 8191])
def test_attention_config4_long_context(ctx):
    """The reference's long-context attention case: max_seq 8192 (grid 8 x 64 splits), chunk 128, LSE merge."""
    rng = np.random.default_rng(40 + ctx)
    q = rng.standard_normal(NH * HD).astype(np.float32)
    k = rng.standard_normal((NKV, 8192, HD)).astype(np.float16)
    v = rng.standard_normal((NKV, 8192, HD)).astype(np.float16)
    out = E.kernel_attention("opt", q, k, v, ctx, NH, NKV, HD, 8192)
    assert np.allclose(out, K.attention(q, k, v, ctx, NH, NKV, HD), rtol=1e-4, atol=1e-4)


def test_attention_large_scores_are_stable():
    """Scores up to ~+-200: the split-local max and the LSE merge must not overflow."""
    rng = np.random.default_rng(14)
    q = (rng.standard_normal(NH * HD) * 12).astype(np.float32)
    k = (rng.standard_normal((NKV, 1024, HD)) * 2).astype(np.float16)
    v = rng.standard_normal((NKV, 1024, HD)).astype(np.float16)
    out = E.kernel_attention("opt", q, k, v, 1000, NH, NKV, HD, 1024)
    assert np.all(np.isfinite(out))
    assert np.allclose(out, K.attention(q, k, v, 1000, NH, NKV, HD), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("nkv,max_seq", [(8, 4096), (1, 640), (2, 128), (64, 1024), (300, 512)])
@pytest.mark.parametrize("shift", [0, 1])
def test_attention_launch_splits(nkv, max_seq, shift):
    """The device-pointer launch where its division of the tokens changes: one tile or split more or less, contexts
    that leave waves without tokens, more kv heads than workgroups; scratch whose words start off 8-byte alignment.
    One tolerance: the 64-bit result within 2^-24 of each of the 64 products, the weight and the sums over splits,
    about 1e-5 relative to the largest |v|."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(nkv + max_seq)
    nh, slots = 4 * nkv, 4 * nkv * (max_seq // 128)
    q = torch.randn(nh * 64, generator=g, device="cuda")
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    part_o = torch.full((slots * 64 + 1,), 7.0, device="cuda")[shift:]
    part_ml = torch.full((slots * 2 + 1,), 7.0, device="cuda")[shift:]
    out = torch.empty(nh * 64, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for ctx in (1, 2, 31, 32, 33, 100, 255, 256, 257, 288, 289, 511, 513, 640, 1000, 2049, 3969, 4095, 4096):
        if ctx > max_seq:
            continue
        pos = torch.tensor([ctx - 1], dtype=torch.int32, device="cuda")
        E.launch_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), part_o.data_ptr(), part_ml.data_ptr(),
                           out.data_ptr(), nh, nkv, 64, max_seq, stream)
        s = torch.matmul(q.double().view(nkv, 4, 64).cpu(), k[:, :ctx].double().cpu().transpose(1, 2)) * 0.125
        ref = torch.matmul(torch.softmax(s, dim=-1), v[:, :ctx].double().cpu()).view(-1)
        err = (out.double().cpu() - ref).abs().max().item()
        assert err <= 1e-5 * v.abs().max().item(), f"ctx {ctx}: {err}"


@pytest.mark.parametrize("fill", [0xFFC00000, 0xFFFFFFFF, 0x7FC00000, 0x3F800000, 0])
def test_attention_scratch_content(fill):
    """The caller's scratch may hold anything before a call, also before each replay of a captured one: NaNs, fills, and
    what another shape's call left.  Bit for bit, since the splits are merged in their order whichever comes last."""
    import torch
    nkv, max_seq, ctx = 3, 4096, 4000
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    q = torch.randn(nkv * 256, generator=g, device="cuda")
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    pos = torch.tensor([ctx - 1], dtype=torch.int32, device="cuda")
    slots = 4 * nkv * (max_seq // 128)
    part_o, part_ml = (torch.empty(slots * n, dtype=torch.int32, device="cuda") for n in (64, 2))
    out, want = (torch.full((nkv * 256,), 9.0, device="cuda") for _ in range(2))
    value = fill - (1 << 32) if fill >> 31 else fill

    def launch(dst, kv_heads, seq):
        E.launch_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), part_o.data_ptr(), part_ml.data_ptr(),
                           dst.data_ptr(), 4 * kv_heads, kv_heads, 64, seq, torch.cuda.current_stream().cuda_stream)

    part_o.fill_(value), part_ml.fill_(value)
    launch(want, nkv, max_seq)
    s = torch.matmul(q.double().view(nkv, 4, 64).cpu(), k[:, :ctx].double().cpu().transpose(1, 2)) * 0.125
    ref = torch.matmul(torch.softmax(s, dim=-1), v[:, :ctx].double().cpu()).view(-1)
    assert (want.double().cpu() - ref).abs().max().item() <= 1e-5 * v.abs().max().item()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch(out, nkv, max_seq)
    for i in range(4):
        out.fill_(9.0)
        if i == 1:
            part_o.fill_(value), part_ml.fill_(value)
        elif i == 2:  # the other shape's words lie elsewhere
            pos.fill_(2047), launch(out, 2, 2048), pos.fill_(ctx - 1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"replay {i}"


@pytest.mark.parametrize("nkv", [3, 100])
def test_attention_overlapping_calls(nkv):
    """Calls on four streams at once, each stream with scratch of its own, give what they give one at a time."""
    import torch
    max_seq, n = 4096, 12
    g = torch.Generator(device="cuda")
    g.manual_seed(nkv)
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    q = torch.randn(4 * n, nkv * 256, generator=g, device="cuda")
    pos = torch.randint(0, max_seq, (4 * n,), generator=g, device="cuda", dtype=torch.int32)
    slots = 4 * nkv * (max_seq // 128)
    scratch = [(torch.empty(slots * 64, device="cuda"), torch.empty(slots * 2, device="cuda")) for _ in range(4)]
    got, want = torch.zeros_like(q), torch.zeros_like(q)

    def launch(i, out, stream):
        part_o, part_ml = scratch[i % 4]
        E.launch_attention(q[i].data_ptr(), k.data_ptr(), v.data_ptr(), pos[i].data_ptr(), part_o.data_ptr(),
                           part_ml.data_ptr(), out[i].data_ptr(), 4 * nkv, nkv, 64, max_seq, stream.cuda_stream)

    for i in range(4 * n):
        launch(i, want, torch.cuda.current_stream())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]
    for i in range(4 * n):
        launch(i, got, streams[i % 4])
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("pos", [-1, -2, -300])
def test_attention_without_tokens(pos):
    """A position before the first token: no token weighs anything, and every output is the sums' 0 / 0."""
    import torch
    nkv, max_seq = 2, 1024
    q, out = torch.ones(nkv * 256, device="cuda"), torch.ones(nkv * 256, device="cuda")
    k, v = (torch.ones(nkv, max_seq, 64, device="cuda").half() for _ in range(2))
    d_pos = torch.tensor([pos], dtype=torch.int32, device="cuda")
    E.launch_attention_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), d_pos.data_ptr(), out.data_ptr(), 4 * nkv, nkv, 64,
                              max_seq, torch.cuda.current_stream().cuda_stream)
    assert bool(out.isnan().all())


def test_attention_replayed_launch():
    """A captured launch replayed over changing contexts (its split words are its own each time), against eager calls."""
    import torch
    nkv, max_seq = 8, 4096
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    q = torch.randn(nkv * 256, generator=g, device="cuda")
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    pos = torch.zeros(1, dtype=torch.int32, device="cuda")
    out, want = (torch.empty(nkv * 256, device="cuda") for _ in range(2))

    def launch(dst):
        E.launch_attention_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), dst.data_ptr(), 4 * nkv, nkv, 64,
                                  max_seq, torch.cuda.current_stream().cuda_stream)

    launch(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch(out)
    for i, ctx in enumerate((4096, 3000, 4096, 1, 257, 4000, 256, 513)):
        pos.fill_(ctx - 1)
        q.mul_(-1.01)  # the words of the replay before would give another result
        graph.replay()
        if i % 2:
            torch.cuda.synchronize()
        launch(want)
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"ctx {ctx}"


@pytest.mark.parametrize("case", ["small weights", "small query", "tiny query", "large query", "large keys"])
def test_attention_dynamic_range(case):
    """Terms far below the largest keep their bits: tokens whose weights are 2^-31 of one that adds nothing, query
    columns 2^-30 of one that meets zeros, queries near the ends of the floats, keys at the end of fp16.  Against 64
    bits within 1e-4 of the result (a weight's exponent carries the rounding of a score of up to 1e3 or so: 6e-5)."""
    import torch
    nkv, max_seq, ctx = 2, 2048, 1900
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    q = torch.randn(nkv, 4, 64, generator=g, device="cuda")
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    if case == "small weights":
        q[..., 0], q[..., 1:] = 16.0, 0.01
        k[..., 0] = 0.0
        k[:, 700, 0], v[:, 700] = 0.125 ** -1 * 21.5 / 16, 0.0  # e^21.5 = 2^31
    elif case == "small query":
        q[..., 0] = 2.0 ** 30
        k[..., 0] = 0.0
    elif case == "tiny query":
        q *= 1e-38
    elif case == "large query":
        q *= 1e37
        k[:] = k[:, :1] * 1e-3  # equal scores: a uniform average
    else:
        k.mul_(15000.0).clamp_(-65504.0, 65504.0)
        q *= 1e-4
    pos = torch.tensor([ctx - 1], dtype=torch.int32, device="cuda")
    out = torch.empty(nkv * 256, device="cuda")
    E.launch_attention_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), out.data_ptr(), 4 * nkv, nkv, 64,
                              max_seq, torch.cuda.current_stream().cuda_stream)
    s = torch.matmul(q.double().cpu(), k[:, :ctx].double().cpu().transpose(1, 2)) * 0.125
    p = torch.softmax(torch.zeros_like(s) if case == "large query" else s, dim=-1)
    ref = torch.matmul(p, v[:, :ctx].double().cpu()).view(-1)
    assert (out.double().cpu() - ref).norm() <= 1e-4 * ref.norm()


@pytest.mark.parametrize("case", ["top of the floats", "one column far above", "far apart"])
def test_attention_query_range(case):
    """Finite queries at the top of the floats with finite scores; query columns so far apart that the small ones fall
    below what the fp16 parts of a head hold, beside zero keys under the large ones.  The bound of the test above; the
    first case's scores differ by far more than their rounding, so its softmax picks one token."""
    import torch
    nkv, max_seq, ctx = 2, 2048, 1900
    g = torch.Generator(device="cuda")
    g.manual_seed(23)
    q = torch.randn(nkv, 4, 64, generator=g, device="cuda")
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    if case == "top of the floats":
        q = (torch.rand(nkv, 4, 64, generator=g, device="cuda") + 0.1) * 3e38 * q.sign()
        k *= 1e-4
    elif case == "one column far above":
        q[..., 5] = 2.0 ** 70
        k[..., 5] = 0.0
    else:
        q[..., ::2] *= 2.0 ** 100
        k[..., ::2] = 0.0
    pos = torch.tensor([ctx - 1], dtype=torch.int32, device="cuda")
    out = torch.empty(nkv * 256, device="cuda")
    E.launch_attention_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), out.data_ptr(), 4 * nkv, nkv, 64,
                              max_seq, torch.cuda.current_stream().cuda_stream)
    s = torch.matmul(q.double().cpu(), k[:, :ctx].double().cpu().transpose(1, 2)) * 0.125
    ref = torch.matmul(torch.softmax(s, dim=-1), v[:, :ctx].double().cpu()).view(-1)
    assert (out.double().cpu() - ref).norm() <= 1e-4 * ref.norm()


@pytest.mark.parametrize("where", ["k", "v", "q"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_attention_non_finite(where, value):
    """One infinity or NaN in the inputs: the outputs are the closed form's, term by term (a score of -inf weighs 0)."""
    import torch
    nkv, max_seq, ctx, t, d = 2, 1024, 700, 333, 5
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    q = torch.rand(nkv * 256, generator=g, device="cuda") + 0.5
    k, v = (torch.randn(nkv, max_seq, 64, generator=g, device="cuda").half() for _ in range(2))
    k[:, ctx:] = float("nan")  # past the context: read in whole tiles, but of no weight
    v[:, ctx:] = float("inf")
    if where == "q":
        q[d] = value
    else:
        (k if where == "k" else v)[0, t, d] = value
    pos = torch.tensor([ctx - 1], dtype=torch.int32, device="cuda")
    out = torch.empty(nkv * 256, device="cuda")
    E.launch_attention_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), out.data_ptr(), 4 * nkv, nkv, 64,
                              max_seq, torch.cuda.current_stream().cuda_stream)
    s = torch.matmul(q.double().view(nkv, 4, 64).cpu(), k[:, :ctx].double().cpu().transpose(1, 2)) * 0.125
    p = torch.exp(s - s.amax(-1, keepdim=True))
    ref = (torch.matmul(p, v[:, :ctx].double().cpu()) / p.sum(-1, keepdim=True)).view(-1)
    np.testing.assert_allclose(out.double().cpu().numpy(), ref.numpy(), rtol=1e-5, atol=1e-5)


def test_silu_mul():
    gu = (np.random.default_rng(14).standard_normal(2 * 8192) * 2).astype(np.float32)
    assert np.allclose(E.kernel_silu_mul(gu), K.silu_mul(gu), rtol=1e-5)
    # the whole range where e^-g is a finite float, and past it (silu -> 0 below, -> g above)
    g = np.concatenate([np.linspace(-87, 87, 8192), np.array([-200.0, -100.0, -88.5, 88.5, 100.0, 200.0] + [0.0] * 8186)])
    gu = np.concatenate([g, np.ones_like(g)]).astype(np.float32)
    got, want = E.kernel_silu_mul(gu), K.silu_mul(gu)
    assert np.allclose(got, want, rtol=1e-5, atol=1e-30)


VOCAB = 128256


def test_argmax_random():
    lg = np.random.default_rng(15).standard_normal(VOCAB).astype(np.float32)
    assert E.kernel_argmax(lg) == K.argmax_lowest(lg)


def test_argmax_tie_lowest_index():
    lg = np.random.default_rng(16).standard_normal(VOCAB).astype(np.float32)
    lg[5] = lg[100000] = 50.0
    assert E.kernel_argmax(lg) == 5


def test_argmax_last_index():
    lg = np.random.default_rng(17).standard_normal(VOCAB).astype(np.float32)
    lg[-1] = 50.0
    assert E.kernel_argmax(lg) == VOCAB - 1


@pytest.mark.parametrize("n", [1, 255, 256, 65537])
def test_argmax_sizes_and_all_equal(n):
    assert E.kernel_argmax(np.zeros(n, np.float32)) == 0
    lg = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    assert E.kernel_argmax(lg) == K.argmax_lowest(lg)


# ---- quantisers: bit-exact against the oracle (reference python/cudallm/quantize.py) ----------

@pytest.mark.parametrize("rows,cols", [(64, 256), (8192, 2048), (3, 128)])
def test_quantize_int8_bit_exact(rows, cols):
    w = np.random.default_rng(rows + cols).normal(0, 0.02, size=(rows, cols)).astype(np.float32)
    w[0, :4] = [1.27, -1.27, 0.005, 0.015]  # exact .5 ties under s = 0.01
    w[-1] = 0.0  # zero row -> scale 1
    q, s = GQ.quantize_int8_rows(w)
    q_ref, s_ref = Q.quantize_int8_rows(w)
    np.testing.assert_array_equal(s, s_ref)
    np.testing.assert_array_equal(q, q_ref)


@pytest.mark.parametrize("rows,cols", [(32, 512), (8192, 2048), (1, 128)])
def test_quantize_int4_bit_exact(rows, cols):
    w = np.random.default_rng(rows * cols).normal(0, 0.02, size=(rows, cols)).astype(np.float32)
    w[0, :4] = [7.0, -7.0, 0.0, 1.0]
    if rows > 1:
        w[1, :128] = 0.0  # zero group -> scale fp16(1)
    p, s = GQ.quantize_int4_groups(w, 128)
    p_ref, s_ref = Q.quantize_int4_groups(w, 128)
    np.testing.assert_array_equal(s.view(np.uint16), s_ref.view(np.uint16))
    np.testing.assert_array_equal(p, p_ref)
    np.testing.assert_array_equal(GQ.unpack_int4(p), Q.unpack_int4(p_ref))


def test_unpack_roundtrip_and_known_answer():
    np.testing.assert_array_equal(GQ.unpack_int4(np.array([[0x0F, 0x98]], dtype=np.uint8)), [[7, -8, 0, 1]])
    q = np.random.default_rng(3).integers(-8, 8, size=(16, 256), dtype=np.int8)
    u = (q + 8).astype(np.uint8)
    np.testing.assert_array_equal(GQ.unpack_int4((u[:, 0::2] | (u[:, 1::2] << 4)).astype(np.uint8)), q)
