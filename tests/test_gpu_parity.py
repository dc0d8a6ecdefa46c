"""GPU parity: the HIP kernels (through ops -> ctypes -> C ABI) against the CPU oracle.

Bar: bit-exact for the embedding gather; rtol 1.6e-2 / atol 1e-2 against the fp32-upcast
oracle for every bf16 output. Inputs are the seeded synthetic tensors of the benchmark
configurations plus edge cases (ragged rows, wrap-around positions, clamps, odd sizes).
"""
import sys
import threading
from itertools import chain, repeat, starmap

import pytest
import torch

import tritonllm_amd as T
from oracle import layers as O
from tritonllm_amd import _lib, ops, scratch_pool
from tritonllm_amd._lib import host

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1.6e-2, 1e-2


def close(out, ref, rtol=RTOL, atol=ATOL):
    torch.testing.assert_close(out.float().cpu(), ref.float(), rtol=rtol, atol=atol)


@pytest.fixture(scope="module")
def yarn():
    return T.gpt_oss_yarn()


# ----------------------------------------------------------------------------------- RMSNorm
@pytest.mark.parametrize("rows", [1, 8, 32, 513, 2048, 8192])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
def test_rmsnorm_parity(gpu, rows, scale_dtype):
    d = O.make_inputs(rows, seed=rows, norm_scale_dtype=scale_dtype)
    out = T.rmsnorm_forward(d["x"].to(gpu), d["norm_scale"].to(gpu), 1e-5)
    assert out.dtype == torch.bfloat16 and out.shape == (rows, 2880)
    close(out, O.rmsnorm_ref(d["x"], d["norm_scale"], 1e-5))


def test_rmsnorm_in_place_leading_dims_and_pool(gpu):
    d = O.make_inputs(24, seed=3)
    x = d["x"].view(2, 12, 2880).to(gpu)
    s = d["norm_scale"].float().to(gpu)
    ref = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).view(2, 12, 2880)
    a = T.rmsnorm_forward(x, s, 1e-5)
    b = T.rmsnorm_forward(x, s, 1e-5)
    assert a.data_ptr() == b.data_ptr()            # borrowed pool buffer, as the reference's scratch pool
    close(a, ref)
    r = T.rmsnorm_forward(x, s, 1e-5, out=x)       # final-norm style aliasing
    assert r.data_ptr() == x.data_ptr()
    close(x, ref)


@pytest.mark.parametrize("hidden", [8, 40, 2881, 4096, 8192, 20000])
def test_rmsnorm_other_hidden_sizes(gpu, hidden):
    g = torch.Generator().manual_seed(hidden)
    x = torch.randn(5, hidden, generator=g).bfloat16()
    s = (1 + 0.1 * torch.randn(hidden, generator=g))
    close(T.rmsnorm_forward(x.to(gpu), s.to(gpu), 1e-5), O.rmsnorm_ref(x, s, 1e-5))
    many = torch.randn(700, hidden if hidden < 9000 else 512, generator=g).bfloat16()   # wave-per-row path
    s2 = torch.ones(many.shape[1])
    close(T.rmsnorm_forward(many.to(gpu), s2.to(gpu), 1e-5), O.rmsnorm_ref(many, s2, 1e-5))


def test_rmsnorm_invariants_on_gpu(gpu):
    x = torch.zeros(4, 2880, dtype=torch.bfloat16)
    x[1] = 3.0
    x[2] = -0.5
    s = torch.linspace(0.5, 1.5, 2880)
    out = T.rmsnorm_forward(x.to(gpu), s.to(gpu), 1e-5).float().cpu()
    assert torch.all(out[0] == 0) and torch.all(out[3] == 0)
    close(out[1], s / (1 + 1e-5 / 9.0) ** 0.5)
    close(out[2], -s / (1 + 1e-5 / 0.25) ** 0.5)


# ----------------------------------------------------------------------------------- embedding
@pytest.mark.parametrize("id_dtype", [torch.int32, torch.int64])
def test_embedding_bit_exact_full_table(gpu, id_dtype):
    g = torch.Generator().manual_seed(0)
    table = torch.empty(O.VOCAB, O.HIDDEN, dtype=torch.bfloat16)
    for lo in range(0, O.VOCAB, 25136):                      # chunked draw keeps host memory modest
        table[lo:lo + 25136] = (0.02 * torch.randn(min(25136, O.VOCAB - lo), O.HIDDEN, generator=g)).bfloat16()
    ids = torch.randint(0, O.VOCAB, (1, 2048), generator=g).to(id_dtype)
    ids[0, 0], ids[0, 1], ids[0, 2], ids[0, 3] = 0, O.VOCAB - 1, 7, 7
    out = T.embedding_forward(ids.to(gpu), table.to(gpu))
    assert out.shape == (1, 2048, O.HIDDEN)
    assert torch.equal(out.cpu(), O.embedding_ref(table, ids))


def test_embedding_edges(gpu):
    g = torch.Generator().manual_seed(1)
    for hidden in (2880, 24, 7):                               # vector path, small vector path, scalar path
        table = torch.randn(50, hidden, generator=g).bfloat16()
        tg = table.to(gpu)
        ids = torch.tensor([[0, 49], [3, 3]], dtype=torch.int64)
        assert torch.equal(T.embedding_forward(ids.to(gpu), tg).cpu(), O.embedding_ref(table, ids))
        empty = T.embedding_forward(torch.zeros((0,), dtype=torch.int32, device=gpu), tg)
        assert empty.shape == (0, hidden)
        flag = torch.zeros((), dtype=torch.int32, device=gpu)
        bad = torch.tensor([1, 50, -1, 2], dtype=torch.int64)
        out = T.embedding_forward(bad.to(gpu), tg, oob_flag=flag).cpu()
        assert int(flag.item()) == 1
        assert torch.equal(out[0], table[1]) and torch.equal(out[3], table[2])
        assert torch.all(out[1] == 0) and torch.all(out[2] == 0)
    emb = T.Embedding(50, 24, device=gpu)
    with torch.no_grad():
        emb.weight.copy_(torch.randn(50, 24, generator=g).bfloat16())
    ids = torch.tensor([[4, 9]], dtype=torch.int32, device=gpu)
    assert torch.equal(emb(ids).cpu(), emb.weight.detach().cpu()[[4, 9]][None])
    emb.check_ids()
    emb(torch.tensor([77], device=gpu))
    with pytest.raises(IndexError):
        emb.check_ids()


# ----------------------------------------------------------------------------------- SwiGLU
@pytest.mark.parametrize("rows", [4, 32, 128, 4096, 32768])
def test_swiglu_parity(gpu, rows):
    g = torch.Generator().manual_seed(rows)
    x = (2.0 * torch.randn(rows, 5760, generator=g)).bfloat16()
    out = T.swiglu(x.to(gpu))
    assert out.shape == (rows, 2880)
    close(out, O.swiglu_ref(x))


def test_swiglu_edges_and_variants(gpu):
    gs = [-30.0, -7.0, 0.0, 6.99, 7.0, 7.01, 30.0, -100.0]
    ls = [-30.0, -7.01, -7.0, -1.0, 0.0, 7.0, 30.0, 1.0]
    x = torch.tensor([[v for l in ls for v in (gv, l)] for gv in gs]).bfloat16()        # [8, 16] interleaved
    out = T.swiglu(x.to(gpu))
    close(out, O.swiglu_ref(x), rtol=1e-2, atol=1e-6)
    assert torch.all(out.cpu()[:, ls.index(-1.0)] == 0)                                  # l = -1 => exact zero
    g = torch.Generator().manual_seed(5)
    y = (2.0 * torch.randn(3, 7, 48, generator=g)).bfloat16()
    close(T.swiglu(y.to(gpu), interleaved=False), O.swiglu_ref(y, interleaved=False))
    close(T.swiglu(y.to(gpu), alpha=1.0, limit=None), O.swiglu_ref(y, alpha=1.0, limit=None))
    perm = torch.cat((y[..., ::2], y[..., 1::2]), dim=-1)
    assert torch.equal(T.swiglu(y.to(gpu)).cpu(), T.swiglu(perm.to(gpu), interleaved=False).cpu())
    odd = (2.0 * torch.randn(5, 2 * 13, generator=g)).bfloat16()                         # scalar path
    close(T.swiglu(odd.to(gpu)), O.swiglu_ref(odd))
    wide = (2.0 * torch.randn(6, 96, generator=g)).bfloat16().to(gpu)
    close(T.swiglu(wide[:, :64]), O.swiglu_ref(wide.cpu()[:, :64]))                      # row stride > row length
    from tritonllm_amd.swiglu_compat import PrecisionConfig, swiglu as swiglu_pc
    close(swiglu_pc(y.to(gpu), 1.702, PrecisionConfig(limit=7.0)), O.swiglu_ref(y))
    nanrow = torch.tensor([[float("nan"), 1.0, 1.0, float("nan")]]).bfloat16()
    assert torch.isnan(T.swiglu(nanrow.to(gpu))).all()


# ----------------------------------------------------------------------------------- rotary
def _qk(batch, tokens, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(batch, tokens, 64, 64, generator=g).bfloat16()
    k = torch.randn(batch, tokens, 8, 64, generator=g).bfloat16()
    return q, k


@pytest.mark.parametrize("batch,tokens,offset", [(1, 1, 0), (8, 1, 4095), (2, 70, 4000), (1, 2048, 0), (1, 8192, 0), (1, 5, 131070)])
def test_rope_parity_yarn_and_tables(gpu, yarn, batch, tokens, offset):
    q, k = _qk(batch, tokens, seed=tokens + offset)
    pos = O.token_positions(batch, tokens, offset)
    cos, sin = O.yarn_cos_sin(pos)
    q_ref = O.rope_rotate_ref(q.view(-1, 64, 64), cos, sin).view(q.shape)
    k_ref = O.rope_rotate_ref(k.view(-1, 8, 64), cos, sin).view(k.shape)
    off = torch.tensor([offset], dtype=torch.int64, device=gpu)
    # in-register cos/sin
    qg, kg = q.to(gpu), k.to(gpu)
    T.rope_forward(qg, kg, None, None, O.MAX_CTX, off, yarn=yarn)
    close(qg, q_ref)
    close(kg, k_ref)
    # table-driven, with the oracle's own tables (the reference's calling convention)
    cos_t, sin_t = O.yarn_cos_sin(torch.arange(O.MAX_CTX))
    qt, kt = q.to(gpu), k.to(gpu)
    T.rope_forward(qt, kt, sin_t.to(gpu), cos_t.to(gpu), O.MAX_CTX, off)
    close(qt, q_ref)
    close(kt, k_ref)


def test_rope_module_tables_and_per_row_positions(gpu, yarn):
    rope = T.RotaryEmbedding(64, 150000, torch.float32, initial_context_length=4096, scaling_factor=32.0, ntk_alpha=1.0,
                             ntk_beta=32.0, device=gpu)
    assert rope.cos.shape == (O.MAX_CTX, 32) and rope.cos.dtype == torch.float32
    rows = torch.tensor([0, 1, 4095, 4096, 8191, 65537, 131071])
    cos_ref, sin_ref = O.yarn_cos_sin(rows)
    torch.testing.assert_close(rope.cos[rows.to(gpu)].cpu(), cos_ref, rtol=0, atol=1e-6)
    torch.testing.assert_close(rope.sin[rows.to(gpu)].cpu(), sin_ref, rtol=0, atol=1e-6)
    q, k = _qk(1, 33, seed=11)
    off = torch.tensor([8000], dtype=torch.int64, device=gpu)
    q1, k1 = q.to(gpu), k.to(gpu)
    rope(q1, k1, off)                                      # tables carry YaRN parameters -> register path
    q2, k2 = q.to(gpu), k.to(gpu)
    T.rope_forward(q2, k2, rope.sin.clone(), rope.cos.clone(), O.MAX_CTX, off)   # plain tables -> table path
    assert torch.equal(q1, q2) and torch.equal(k1, k2)     # same device routine either way
    pos = torch.tensor([5, 8191, 0, 77777], dtype=torch.int64)
    q, k = _qk(4, 1, seed=12)
    cos, sin = O.yarn_cos_sin(pos)
    qg, kg = q.to(gpu), k.to(gpu)
    T.rope_forward(qg, kg, None, None, O.MAX_CTX, None, yarn=yarn, positions=pos.to(gpu))
    close(qg, O.rope_rotate_ref(q.view(-1, 64, 64), cos, sin).view(q.shape))
    close(kg, O.rope_rotate_ref(k.view(-1, 8, 64), cos, sin).view(k.shape))


@pytest.mark.parametrize("scaling_factor", [32.0, 1.0])
def test_yarn_table_whole_context(gpu, scaling_factor):
    """The device's sin/cos routine (the one every rotary kernel uses in registers) over ALL 131072 positions x 32
    frequencies, in fp32, against the oracle's tables (model.py:307-313 restated): absolute error within
    4e-7 x concentration, i.e. a few units in the last place of values of magnitude ~1. YaRN and plain RoPE."""
    yp = T.YarnParams(head_dim=64, base=150000.0, initial_context_length=4096, scaling_factor=scaling_factor, ntk_alpha=1.0, ntk_beta=32.0)
    cos = torch.empty(O.MAX_CTX, 32, dtype=torch.float32, device=gpu)
    sin = torch.empty(O.MAX_CTX, 32, dtype=torch.float32, device=gpu)
    import ctypes
    from tritonllm_amd import _lib
    rc = _lib.lib().tllm_yarn_table_f32(cos.data_ptr(), sin.data_ptr(), 0, O.MAX_CTX, ctypes.byref(yp.c_struct()),
                                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    cos_ref, sin_ref = O.yarn_cos_sin(torch.arange(O.MAX_CTX), scaling_factor=scaling_factor)
    conc = 0.1 * __import__("math").log(scaling_factor) + 1.0 if scaling_factor > 1 else 1.0
    assert abs(yp.concentration - conc) < 1e-12
    torch.testing.assert_close(cos.cpu(), cos_ref, rtol=0, atol=4e-7 * conc)
    torch.testing.assert_close(sin.cpu(), sin_ref, rtol=0, atol=4e-7 * conc)
    # a table requested from the middle of the context is the same numbers
    c2 = torch.empty(1000, 32, dtype=torch.float32, device=gpu)
    s2 = torch.empty(1000, 32, dtype=torch.float32, device=gpu)
    rc = _lib.lib().tllm_yarn_table_f32(c2.data_ptr(), s2.data_ptr(), 130000, 1000, ctypes.byref(yp.c_struct()), torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(c2, cos[130000:131000]) and torch.equal(s2, sin[130000:131000])


def test_rope_positions_must_cover_every_row(gpu, yarn):
    """The kernels read positions[row] for every row; a shorter tensor is refused on the host."""
    q, k = _qk(4, 1, seed=14)
    with pytest.raises(ValueError, match="3 entries for 4 rows"):
        T.rope_forward(q.to(gpu), k.to(gpu), None, None, O.MAX_CTX, None, yarn=yarn, positions=torch.zeros(3, dtype=torch.int64, device=gpu))
    d = O.make_inputs(8, seed=15)
    with pytest.raises(ValueError, match="7 entries for 8 rows"):
        T.qkv_rope_forward(d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"][:7].to(gpu))
    with pytest.raises((ValueError, RuntimeError)):
        T.qkv_rope_forward(d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"])   # CPU positions


def test_rope_norm_property_full_size(gpu, yarn):
    q, k = _qk(1, 8192, seed=13)
    qg, kg = q.to(gpu), k.to(gpu)
    T.rope_forward(qg, kg, None, None, O.MAX_CTX, torch.zeros(1, dtype=torch.int64, device=gpu), yarn=yarn)
    n_in = q.float()[..., :32] ** 2 + q.float()[..., 32:] ** 2
    n_out = qg.float().cpu()[..., :32] ** 2 + qg.float().cpu()[..., 32:] ** 2
    torch.testing.assert_close(n_out, yarn.concentration ** 2 * n_in, rtol=3e-2, atol=3e-2)


# ----------------------------------------------------------------------------------- fused QKV
def _check_qkv(gpu, yarn, rows, mode, seed, prefill_positions=False, max_pos=8192):
    d = O.make_inputs(rows, seed=seed, prefill=prefill_positions, max_pos=max_pos)
    q, k, v = T.qkv_rope_forward(d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn,
                                 positions=d["positions"].to(gpu), mode=mode)
    qr, kr, vr = O.qkv_rope_ref(d["x"], d["w"], d["b"], d["positions"])
    assert q.shape == (rows, 4096) and k.shape == (rows, 512) and v.shape == (rows, 512)
    close(q, qr)
    close(k, kr)
    close(v, vr)


@pytest.mark.parametrize("rows", [1, 8, 15, 16, 17, 32, 33, 50, 64, 65, 96, 100, 192, 450])
def test_qkv_rope_decode_parity(gpu, yarn, rows):
    """Up to 8 / 32 rows the two streaming kernels; from 33 rows the kernel that holds the weight and streams the rows
    past it (33: a one-row last block; 64 / 65 and 96: whole and ragged blocks; 450: more blocks than ring slots)."""
    _check_qkv(gpu, yarn, rows, "decode", seed=rows)


@pytest.mark.parametrize("rows", [64, 65, 448, 449])
def test_qkv_rope_auto_mode_either_side_of_the_row_threshold(gpu, yarn, rows):
    """``mode="auto"``: the weight-streaming kernels up to 448 rows at the gpt-oss shape, the MFMA GEMM above."""
    _check_qkv(gpu, yarn, rows, "auto", seed=40 + rows)


def test_qkv_rope_auto_mode_follows_the_row_threshold(gpu, yarn, monkeypatch):
    """One place holds the number of rows: an fp8 weight has decode kernels only, so its refusal shows the mode that was chosen."""
    d = O.make_inputs(8, seed=41)
    w8, ws = T.quantize_fp8_rows(d["w"].to(gpu))
    args, kw = (d["x"].to(gpu), w8, d["b"].to(gpu), 64, 8, 64), dict(yarn=yarn, positions=d["positions"].to(gpu), weight_scale=ws)
    T.qkv_rope_forward(*args, **kw)
    monkeypatch.setattr(ops, "DECODE_MAX_ROWS_2880", 7)
    with pytest.raises(NotImplementedError):
        T.qkv_rope_forward(*args, **kw)


@pytest.mark.parametrize("rows", [1, 100, 128, 200, 2048])
def test_qkv_rope_prefill_parity(gpu, yarn, rows):
    _check_qkv(gpu, yarn, rows, "prefill", seed=100 + rows, prefill_positions=rows >= 128)


@pytest.mark.parametrize("rows", [1, 5, 8, 16, 17, 32, 50])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
def test_norm_qkv_fused_decode_parity(gpu, yarn, rows, scale_dtype):
    """RMSNorm inside the decode kernel == oracle rmsnorm (rounded to bf16, as the layer boundary does) -> oracle QKV.
    Rows carry different magnitudes so that a per-row statistic applied to the wrong row would show."""
    d = O.make_inputs(rows, seed=300 + rows, norm_scale_dtype=scale_dtype)
    x = (d["x"].float() * (2.0 ** (torch.arange(rows) % 7 - 3))[:, None]).bfloat16()
    q, k, v = T.qkv_rope_forward(x.to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu),
                                 mode="decode", norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
    t_ref = O.rmsnorm_ref(x, d["norm_scale"].float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], d["positions"])
    close(q, qr)
    close(k, kr)
    close(v, vr)
    # and against the two-launch form on the GPU
    q, k, v = q.clone(), k.clone(), v.clone()
    t = T.rmsnorm_forward(x.to(gpu), d["norm_scale"].to(gpu), 1e-5)
    q2, k2, v2 = T.qkv_rope_forward(t, d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu), mode="decode")
    close(q, q2.float().cpu())
    close(k, k2.float().cpu())
    close(v, v2.float().cpu())


@pytest.mark.parametrize("rows", [1, 5, 8, 9, 16, 20])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("id_dtype", [torch.int32, torch.int64])
def test_embed_norm_qkv_one_launch(gpu, yarn, rows, scale_dtype, id_dtype):
    """The first layer of a decode step in one launch: gathered rows bit-exact, q / k / v identical to what the
    separate gather + fused norm/QKV kernel gives (same arithmetic on the same rows) and within tolerance of the oracle.
    20 rows exercises the composed path behind the same call."""
    d = O.make_inputs(rows, seed=500 + rows, norm_scale_dtype=scale_dtype)
    g = torch.Generator().manual_seed(rows)
    vocab = 1000
    table = (torch.randn(vocab, 2880, generator=g) * (2.0 ** (torch.arange(vocab) % 7 - 3))[:, None]).bfloat16()
    ids = torch.randint(0, vocab, (rows,), generator=g, dtype=id_dtype)
    ids[0] = vocab - 1
    if rows > 1:
        ids[-1] = 0
    flag = torch.zeros(1, dtype=torch.int32, device=gpu)
    x, q, k, v = T.embed_qkv_rope_forward(ids.to(gpu), table.to(gpu), d["norm_scale"].to(gpu), 1e-5, d["w"].to(gpu), d["b"].to(gpu),
                                          64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu), oob_flag=flag)
    x_ref = O.embedding_ref(table, ids)
    assert torch.equal(x.cpu(), x_ref)
    assert flag.item() == 0
    q, k, v = q.clone(), k.clone(), v.clone()
    t_ref = O.rmsnorm_ref(x_ref, d["norm_scale"].float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], d["positions"])
    close(q, qr)
    close(k, kr)
    close(v, vr)
    q2, k2, v2 = T.qkv_rope_forward(x_ref.to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu),
                                    mode="decode", norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
    assert torch.equal(q, q2) and torch.equal(k, k2) and torch.equal(v, v2)


def test_embed_norm_qkv_fp8_weight_and_bad_ids(gpu, yarn):
    d = O.make_inputs(8, seed=77)
    g = torch.Generator().manual_seed(3)
    table = torch.randn(64, 2880, generator=g).bfloat16()
    ids = torch.randint(0, 64, (8,), generator=g, dtype=torch.int64)
    w8, ws = T.quantize_fp8_rows(d["w"].to(gpu))
    x, q, k, v = T.embed_qkv_rope_forward(ids.to(gpu), table.to(gpu), d["norm_scale"].to(gpu), 1e-5, w8, d["b"].to(gpu), 64, 8, 64,
                                          yarn=yarn, positions=d["positions"].to(gpu), weight_scale=ws)
    assert torch.equal(x.cpu(), table[ids])
    q, k, v = q.clone(), k.clone(), v.clone()
    q2, k2, v2 = T.qkv_rope_forward(x, w8, d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu), mode="decode",
                                    norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5, weight_scale=ws)
    assert torch.equal(q, q2) and torch.equal(k, k2) and torch.equal(v, v2)
    # ids outside the table: a zero row (as the stand-alone gather gives), flag raised, no fault
    bad = ids.clone()
    bad[2], bad[5] = -7, 64
    flag = torch.zeros(1, dtype=torch.int32, device=gpu)
    x, q, k, v = T.embed_qkv_rope_forward(bad.to(gpu), table.to(gpu), d["norm_scale"].to(gpu), 1e-5, d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64,
                                          yarn=yarn, positions=d["positions"].to(gpu), oob_flag=flag)
    assert flag.item() == 1
    want = table[bad.clamp(0, 63)]
    want[2] = 0
    want[5] = 0
    assert torch.equal(x.cpu(), want)
    # pooled outputs and a caller-provided x_out
    xo = torch.empty(8, 2880, dtype=torch.bfloat16, device=gpu)
    x, *_ = T.embed_qkv_rope_forward(ids.to(gpu), table.to(gpu), d["norm_scale"].to(gpu), 1e-5, d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64,
                                     yarn=yarn, positions=d["positions"].to(gpu), x_out=xo)
    assert x.data_ptr() == xo.data_ptr() and torch.equal(xo.cpu(), table[ids])


def test_embed_qkv_refuses_a_table_beyond_32_bit_offsets(gpu):
    """The fused gather addresses table rows with 32-bit byte offsets: a table of 4 GiB or more is refused before
    anything is launched (the pointers below are never dereferenced)."""
    from tritonllm_amd import _lib
    L = _lib.lib()
    t = torch.zeros(8 * 5120, dtype=torch.bfloat16, device=gpu)
    ids = torch.zeros(8, dtype=torch.int32, device=gpu)
    scale = torch.ones(2880, dtype=torch.float32, device=gpu)
    p = t.data_ptr()
    rc = L.tllm_embed_norm_qkv_rope_decode_bf16(ids.data_ptr(), 0, p, 745655, p, None, scale.data_ptr(), 0, 1e-5, p, None, None, p, p, p,
                                                4096, 512, 512, 0, 8, 2880, 64, 8, 64, None, None)
    assert rc == -2 and b"too large for the fused gather" in L.tllm_last_error()


@pytest.mark.parametrize("id_dtype", [torch.int32, torch.int64])
def test_embed_qkv_bad_ids_same_policy_either_side_of_16_rows(gpu, yarn, id_dtype):
    """One launch (<= 16 rows) and gather + QKV (> 16 rows) behind the same call treat an id outside the table alike: a
    zero row of x, the q / k / v that follow from a zero row (the rotated bias), the flag raised -- and every other row
    untouched by it."""
    g = torch.Generator().manual_seed(41)
    vocab = 300
    table = torch.randn(vocab, 2880, generator=g).bfloat16()
    for rows in (16, 17):
        d = O.make_inputs(rows, seed=500 + rows)
        ids = torch.randint(0, vocab, (rows,), generator=g, dtype=id_dtype)
        ids[0], ids[rows // 2], ids[rows - 1] = -1, vocab, vocab + 12345
        flag = torch.zeros(1, dtype=torch.int32, device=gpu)
        x, q, k, v = T.embed_qkv_rope_forward(ids.to(gpu), table.to(gpu), d["norm_scale"].to(gpu), 1e-5, d["w"].to(gpu), d["b"].to(gpu),
                                              64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu), oob_flag=flag)
        assert flag.item() == 1
        ok = (ids >= 0) & (ids < vocab)
        want_x = torch.where(ok[:, None], table[ids.long().clamp(0, vocab - 1)], torch.zeros((), dtype=torch.bfloat16))
        assert torch.equal(x.cpu(), want_x), rows
        t_ref = O.rmsnorm_ref(want_x, d["norm_scale"].float(), 1e-5).bfloat16()
        assert (t_ref[~ok] == 0).all()
        qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], d["positions"])
        close(q, qr)
        close(k, kr)
        close(v, vr)
        # no bad id: the flag stays down
        flag.zero_()
        T.embed_qkv_rope_forward(ids.clamp(0, vocab - 1).to(gpu), table.to(gpu), d["norm_scale"].to(gpu), 1e-5, d["w"].to(gpu), d["b"].to(gpu),
                                 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu), oob_flag=flag)
        assert flag.item() == 0


@pytest.mark.parametrize("rows", [17, 50])
def test_norm_qkv_fused_entry_point_refuses_more_than_16_rows(gpu, yarn, rows, monkeypatch):
    """Beyond 16 rows the norm is a launch of its own: the host composes the two, the C entry point says so."""
    from tritonllm_amd import ops
    d = O.make_inputs(rows, seed=400 + rows)
    args = (d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64)
    kw = dict(yarn=yarn, positions=d["positions"].to(gpu), mode="decode", norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
    q, k, v = T.qkv_rope_forward(*args, **kw)                     # two launches
    t_ref = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], d["positions"])
    close(q, qr)
    close(k, kr)
    close(v, vr)
    monkeypatch.setattr(ops, "_norm_fusable", lambda kind, r, hidden, hd: kind == "decode" and hidden == 2880 and hd == 64)
    with pytest.raises(RuntimeError, match="up to 16 rows"):
        T.qkv_rope_forward(*args, **kw)


@pytest.mark.parametrize("rows", [1, 8, 13, 16, 32, 40])
@pytest.mark.parametrize("with_norm", [False, True])
def test_qkv_fp8_weight_decode_parity(gpu, yarn, rows, with_norm):
    """fp8 e4m3 weight + per-row scale (triton_kernels.py:261-268, 927-965): the kernel must equal the oracle's
    projection with the dequantised weight fp32(W8) * scale; the quantiser must equal the oracle's bit for bit."""
    d = O.make_inputs(rows, seed=500 + rows)
    w8_ref, s_ref = O.quantize_fp8_rows_ref(d["w"])
    w8, s = T.quantize_fp8_rows(d["w"].to(gpu))
    # the quantiser is torch arithmetic on the GPU: same scales to the last bits, same codes except where the GPU's
    # division rounds a quotient to the other side of an fp8 tie
    torch.testing.assert_close(s.cpu(), s_ref, rtol=1e-6, atol=0)
    assert (w8.cpu().view(torch.uint8) != w8_ref.view(torch.uint8)).float().mean().item() < 1e-3
    w8_ref, s_ref = w8.cpu(), s.cpu()          # the kernel is checked on exactly the bytes it was given
    kw = dict(norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5) if with_norm else {}
    q, k, v = T.qkv_rope_forward(d["x"].to(gpu), w8, d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu),
                                 mode="decode", weight_scale=s, **kw)
    xin = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16() if with_norm else d["x"]
    qr, kr, vr = O.qkv_rope_ref(xin, O.dequant_fp8_ref(w8_ref, s_ref), d["b"], d["positions"])
    close(q, qr)
    close(k, kr)
    close(v, vr)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 31])
def test_streaming_decode_kernels_every_row_count(gpu, yarn, rows):
    """The kernels that stream their operands straight into LDS fetch only the rows that exist (the LDS of the others
    keeps what the launch before left there). Every row count of one workgroup, QKV and out-projection, bf16 and fp8
    weight, with and without the fused norm (9 to 16 rows with the norm: the 16-row form of the 8-row kernel); each run
    is preceded by one of the same kernel on NaN activations of its full 8 / 16 / 32 rows so that whatever is left
    behind in LDS would show, and the rows behind the last one in memory are NaN as well."""
    full = 8 if rows <= 8 else 32
    d = O.make_inputs(rows, seed=900 + rows)
    w, b = d["w"].to(gpu), d["b"].to(gpu)
    w8, ws = T.quantize_fp8_rows(w)
    w8_deq = O.dequant_fp8_ref(w8.cpu(), ws.cpu())
    xbuf = torch.full((full + 1, 2880), float("nan"), dtype=torch.bfloat16, device=gpu)
    xbuf[:rows] = d["x"].to(gpu)
    x = xbuf[:rows]
    nan_x = torch.full((full, 2880), float("nan"), dtype=torch.bfloat16, device=gpu)
    nan_pos = torch.zeros(full, dtype=torch.int64, device=gpu)
    pos = d["positions"].to(gpu)
    scale = d["norm_scale"].to(gpu)
    normed = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16()
    for weight, wscale, wref in ((w, None, d["w"]), (w8, ws, w8_deq)):
        for with_norm in (False, True):
            if with_norm and rows > 16 and wscale is None:
                continue                                    # composed of two launches above 16 rows: covered elsewhere
            kw = dict(weight_scale=wscale) if wscale is not None else {}
            if with_norm:
                kw.update(norm_scale=scale, norm_eps=1e-5)
            nfull = min(full, 16) if with_norm else full
            T.qkv_rope_forward(nan_x[:nfull], weight, b, 64, 8, 64, yarn=yarn, positions=nan_pos[:nfull], mode="decode", **kw)
            q, k, v = T.qkv_rope_forward(x, weight, b, 64, 8, 64, yarn=yarn, positions=pos, mode="decode", **kw)
            qr, kr, vr = O.qkv_rope_ref(normed if with_norm else d["x"], wref, d["b"], d["positions"])
            close(q, qr)
            close(k, kr)
            close(v, vr)
    o = _out_inputs(rows, 950 + rows)
    ow, ob = o["w"].to(gpu), o["b"].to(gpu)
    ow8, ows = T.quantize_fp8_rows(ow)
    oxbuf = torch.full((full + 1, 4096), float("nan"), dtype=torch.bfloat16, device=gpu)
    oxbuf[:rows] = o["x"].to(gpu)
    nan_ox = torch.full((full, 1, 4096), float("nan"), dtype=torch.bfloat16, device=gpu)
    for weight, wscale, wref in ((ow, None, o["w"]), (ow8, ows, O.dequant_fp8_ref(ow8.cpu(), ows.cpu()))):
        T.out_residual_decode_forward(nan_ox, weight, ob, torch.zeros(full, 1, 2880, dtype=torch.bfloat16, device=gpu), weight_scale=wscale)
        out = T.out_residual_decode_forward(oxbuf[:rows].view(rows, 1, 4096), weight, ob, o["r"].view(rows, 1, 2880).to(gpu), weight_scale=wscale)
        close(out.view(rows, 2880), O.out_residual_ref(o["x"], wref, o["b"], o["r"]))


@pytest.mark.parametrize("rows", [33, 47, 81])
def test_rows_streaming_kernel_ragged_last_block(gpu, yarn, rows):
    """Above 32 rows one kernel holds the weight and streams the activations past it in blocks of 16 rows; the last
    block re-reads the last row instead of reading past it. The memory behind the last row is NaN, the launch before
    ran on NaN activations (whatever it left in LDS would show), bf16 and fp8 weight, and the norm composed in front."""
    d = O.make_inputs(rows, seed=1300 + rows)
    w, b = d["w"].to(gpu), d["b"].to(gpu)
    w8, ws = T.quantize_fp8_rows(w)
    xbuf = torch.full((rows + 16, 2880), float("nan"), dtype=torch.bfloat16, device=gpu)
    xbuf[:rows] = d["x"].to(gpu)
    x, pos = xbuf[:rows], d["positions"].to(gpu)
    nan_x = torch.full((96, 2880), float("nan"), dtype=torch.bfloat16, device=gpu)
    nan_pos = torch.zeros(96, dtype=torch.int64, device=gpu)
    for weight, wscale, wref in ((w, None, d["w"]), (w8, ws, O.dequant_fp8_ref(w8.cpu(), ws.cpu()))):
        kw = dict(weight_scale=wscale) if wscale is not None else {}
        T.qkv_rope_forward(nan_x, weight, b, 64, 8, 64, yarn=yarn, positions=nan_pos, mode="decode", **kw)
        q, k, v = T.qkv_rope_forward(x, weight, b, 64, 8, 64, yarn=yarn, positions=pos, mode="decode", **kw)
        qr, kr, vr = O.qkv_rope_ref(d["x"], wref, d["b"], d["positions"])
        close(q, qr)
        close(k, kr)
        close(v, vr)
    q, k, v = T.qkv_rope_forward(x, w, b, 64, 8, 64, yarn=yarn, positions=pos, mode="decode", norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
    qr, kr, vr = O.qkv_rope_ref(O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16(), d["w"], d["b"], d["positions"])
    close(q, qr)
    close(k, kr)
    close(v, vr)


def test_fused_norm_wait_for_the_other_wavefronts_never_expires(gpu, yarn):
    """Inside the fused-norm decode kernels a wavefront waits for the others' partial sums with a bounded poll; a wait
    that runs out is recorded in a device word. After the row-count cases above (and a few more here) it must be 0."""
    import ctypes
    from tritonllm_amd import _lib
    for rows in (1, 5, 8, 11, 16):
        d = O.make_inputs(rows, seed=1200 + rows)
        for _ in range(20):
            T.qkv_rope_forward(d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu),
                               mode="decode", norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
    expired = ctypes.c_int32(-1)
    assert _lib.lib().tllm_qkv_decode_wait_expired(ctypes.byref(expired)) == 0, _lib.lib().tllm_last_error()
    assert expired.value == 0
    assert _lib.lib().tllm_qkv_decode_wait_expired(None) == -1


def test_qkv_fp8_weight_cache_form_module_and_refusals(gpu, yarn, monkeypatch):
    d = O.make_inputs(8, seed=51)
    monkeypatch.setenv("ATTN_FP8", "1")
    qkv = T.QKV(2880, 5120, device=gpu)
    with torch.no_grad():
        qkv.weight.copy_(d["w"])
        qkv.bias.copy_(d["b"])
    w8, ws = qkv._fp8_weight
    assert w8.dtype == torch.float8_e4m3fn and ws.shape == (5120,) and qkv._fp8_weight[0] is w8      # quantised once
    rope = T.RotaryEmbedding(64, 150000, torch.float32, initial_context_length=4096, scaling_factor=32.0, device=gpu)
    slot = 5
    cache_k = torch.zeros(8, 16, 8, 64, dtype=torch.bfloat16, device=gpu)
    cache_v = torch.zeros_like(cache_k)
    q = T.qkv_rope_cache_decode_forward(d["x"].view(8, 1, 2880).to(gpu), w8, qkv.bias, rope.sin, rope.cos, rope.max_context_length,
                                        cache_k, cache_v, torch.tensor([slot], device=gpu), 64, 8, 64, ws)
    qr, kr, vr = O.qkv_rope_ref(d["x"], O.dequant_fp8_ref(w8.cpu(), ws.cpu()), d["b"], torch.full((8,), slot, dtype=torch.int64))
    close(q.view(8, 4096), qr)
    close(cache_k[:, slot].reshape(8, 512), kr)
    close(cache_v[:, slot].reshape(8, 512), vr)
    monkeypatch.delenv("ATTN_FP8")
    assert T.QKV(2880, 5120, device=gpu)._fp8_weight == (None, None)
    with pytest.raises(AssertionError):      # an fp8 weight without its scales
        T.qkv_rope_forward(d["x"].to(gpu), w8, d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu))
    with pytest.raises(NotImplementedError): # prefill sizes keep the bf16 weight
        T.qkv_rope_forward(d["x"].to(gpu), w8, d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=d["positions"].to(gpu), mode="prefill",
                           weight_scale=ws)
    with pytest.raises(AssertionError):
        T.qkv_decode_forward(d["x"].view(8, 1, 2880).to(gpu), w8, d["b"].to(gpu), 4096, 512)


def test_norm_qkv_composed_when_not_fusable_and_cache_form(gpu, yarn):
    """norm_scale on shapes the decode kernel does not fuse (prefill rows, other hidden sizes) runs rmsnorm first;
    the cache-writing decode call takes it too."""
    d = O.make_inputs(100, seed=41, norm_scale_dtype=torch.float32)
    t_ref = O.rmsnorm_ref(d["x"], d["norm_scale"], 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], d["positions"])
    q, k, v = T.qkv_rope_forward(d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn,
                                 positions=d["positions"].to(gpu), mode="prefill", norm_scale=d["norm_scale"].to(gpu))
    close(q, qr)
    close(k, kr)
    close(v, vr)
    g = O.make_inputs(6, seed=42, hidden=256, n_q_heads=4, n_kv_heads=2, head_dim=32)
    t_ref = O.rmsnorm_ref(g["x"], g["norm_scale"].float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, g["w"], g["b"], g["positions"], 4, 2, 32, base=10000.0, scaling_factor=1.0)
    q, k, v = T.qkv_rope_forward(g["x"].to(gpu), g["w"].to(gpu), g["b"].to(gpu), 4, 2, 32, yarn=T.YarnParams(head_dim=32, base=10000.0),
                                 positions=g["positions"].to(gpu), norm_scale=g["norm_scale"].to(gpu))
    close(q, qr)
    close(k, kr)
    close(v, vr)
    d = O.make_inputs(8, seed=43)
    slot = 11
    cache_k = torch.zeros(8, 16, 8, 64, dtype=torch.bfloat16, device=gpu)
    cache_v = torch.zeros_like(cache_k)
    rope = T.RotaryEmbedding(64, 150000, torch.float32, initial_context_length=4096, scaling_factor=32.0, device=gpu)
    q = T.qkv_rope_cache_decode_forward(d["x"].view(8, 1, 2880).to(gpu), d["w"].to(gpu), d["b"].to(gpu), rope.sin, rope.cos,
                                        rope.max_context_length, cache_k, cache_v, torch.tensor([slot], device=gpu), 64, 8, 64,
                                        norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
    t_ref = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], torch.full((8,), slot, dtype=torch.int64))
    close(q.view(8, 4096), qr)
    close(cache_k[:, slot].reshape(8, 512), kr)
    close(cache_v[:, slot].reshape(8, 512), vr)


def test_qkv_rope_prefill_long_context(gpu, yarn):
    _check_qkv(gpu, yarn, 8192, "prefill", seed=4, prefill_positions=True)


@pytest.mark.parametrize("rows", [2049, 2304, 2817, 3333, 3841, 4000, 4096, 5000])
def test_qkv_rope_prefill_256_token_tiles(gpu, yarn, rows):
    """Row counts that would need a second round of 128-token tiles run on 256-token tiles instead (two-pass epilogue,
    table built after the K loop; 8192 rows in the long-context test too): ragged last tiles, the XCD-swizzled and the
    plain tile order, arbitrary positions. 5000 rows fall back on 128-token tiles in three rounds, and 2049 and 2304, a little
    more than one round of those, on the smaller GEMM tiles."""
    _check_qkv(gpu, yarn, rows, "prefill", seed=rows, prefill_positions=rows % 2 == 0, max_pos=131072)


@pytest.mark.parametrize("rows", [300, 2304, 2000, 3000])
def test_qkv_rope_prefill_cos_sin_tables(gpu, rows):
    """The prefill kernels' table variants (cos / sin loaded, as the reference passes them, triton_kernels.py:90) at both
    tile heights, arbitrary positions, against the oracle; plain tensors, which the host side cannot trace back to YaRN
    parameters."""
    d = O.make_inputs(rows, seed=7000 + rows, prefill=False, max_pos=131072)
    cos_t, sin_t = O.yarn_cos_sin(torch.arange(O.MAX_CTX))
    q, k, v = T.qkv_rope_forward(d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, cos=cos_t.to(gpu), sin=sin_t.to(gpu),
                                 positions=d["positions"].to(gpu), mode="prefill")
    qr, kr, vr = O.qkv_rope_ref(d["x"], d["w"], d["b"], d["positions"])
    close(q, qr)
    close(k, kr)
    close(v, vr)


def test_qkv_decode_and_prefill_agree(gpu, yarn):
    d = O.make_inputs(40, seed=21)
    args = (d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64)
    kw = dict(yarn=yarn, positions=d["positions"].to(gpu))
    qd, kd, vd = [t.clone() for t in T.qkv_rope_forward(*args, mode="decode", **kw)]
    qp, kp, vp = T.qkv_rope_forward(*args, mode="prefill", **kw)
    close(qd, qp.float().cpu())
    close(kd, kp.float().cpu())
    close(vd, vp.float().cpu())


def test_qkv_offset_form_tables_and_no_rope(gpu, yarn):
    d = O.make_inputs(12, seed=22)
    xg, wg, bg = d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu)
    off = torch.tensor([131070], dtype=torch.int64, device=gpu)
    pos = O.token_positions(2, 6, 131070)
    qr, kr, vr = O.qkv_rope_ref(d["x"], d["w"], d["b"], pos)
    cos_t, sin_t = O.yarn_cos_sin(torch.arange(O.MAX_CTX))
    for mode in ("decode", "prefill"):
        q, k, v = T.qkv_rope_forward(xg, wg, bg, 64, 8, 64, yarn=yarn, offset=off, tokens_per_batch=6, mode=mode)
        close(q, qr)
        close(k, kr)
        q, k, v = T.qkv_rope_forward(xg, wg, bg, 64, 8, 64, cos=cos_t.to(gpu), sin=sin_t.to(gpu), offset=off,
                                     tokens_per_batch=6, mode=mode)
        close(q, qr)
        close(k, kr)
        close(v, vr)
        q, k, v = T.qkv_rope_forward(xg, wg, None, 64, 8, 64, rotate=False, mode=mode)
        plain = O.linear_ref(d["x"], d["w"], None)
        close(q, plain[:, :4096])
        close(k, plain[:, 4096:4608])
        close(v, plain[:, 4608:])


@pytest.mark.parametrize("hd,nq,nkv", [(128, 4, 2), (32, 5, 1), (16, 3, 3)])
@pytest.mark.parametrize("rows", [5, 20])
def test_qkv_decode_other_head_dims(gpu, hd, nq, nkv, rows):
    """The general MFMA decode kernel at head dims other than 64 (rotation partners head_dim / 2 apart, head_dim / 16
    workgroups per head), hidden a multiple of 32 with a K tail; 20 rows = two row chunks, the second ragged."""
    g = torch.Generator().manual_seed(1000 + hd + rows)
    hidden = 608
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * hd, hidden, generator=g)).bfloat16()
    b = (0.05 * torch.randn((nq + 2 * nkv) * hd, generator=g)).bfloat16()
    y = T.YarnParams(head_dim=hd, base=10000.0)
    pos = torch.randint(0, 8192, (rows,), generator=g)
    qr, kr, vr = O.qkv_rope_ref(x, w, b, pos, nq, nkv, hd, base=10000.0, scaling_factor=1.0)
    q, k, v = T.qkv_rope_forward(x.to(gpu), w.to(gpu), b.to(gpu), nq, nkv, hd, yarn=y, positions=pos.to(gpu), mode="decode")
    close(q, qr)
    close(k, kr)
    close(v, vr)


@pytest.mark.parametrize("hd,nq,nkv", [(128, 4, 2), (64, 6, 1), (32, 5, 1)])
@pytest.mark.parametrize("rows", [5, 20])
def test_qkv_decode_fp8_weight_other_shapes(gpu, hd, nq, nkv, rows):
    """fp8 weight with per-row scales at shapes other than gpt-oss's (the reference's fp8 branch is generic,
    triton_kernels.py:927-940): the general MFMA decode kernel, against the oracle on the dequantised weight; with a
    norm requested the host side runs the RMSNorm launch first."""
    g = torch.Generator().manual_seed(2000 + hd + rows)
    hidden = 608
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * hd, hidden, generator=g)).bfloat16()
    b = (0.05 * torch.randn((nq + 2 * nkv) * hd, generator=g)).bfloat16()
    sc = (1 + 0.1 * torch.randn(hidden, generator=g)).bfloat16()
    y = T.YarnParams(head_dim=hd, base=10000.0)
    pos = torch.randint(0, 8192, (rows,), generator=g)
    w8, ws = T.quantize_fp8_rows(w.to(gpu))
    wd = O.dequant_fp8_ref(w8.cpu(), ws.cpu())
    qr, kr, vr = O.qkv_rope_ref(x, wd, b, pos, nq, nkv, hd, base=10000.0, scaling_factor=1.0)
    q, k, v = T.qkv_rope_forward(x.to(gpu), w8, b.to(gpu), nq, nkv, hd, yarn=y, positions=pos.to(gpu), mode="decode", weight_scale=ws)
    close(q, qr)
    close(k, kr)
    close(v, vr)
    t_ref = O.rmsnorm_ref(x, sc.float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, wd, b, pos, nq, nkv, hd, base=10000.0, scaling_factor=1.0)
    q, k, v = T.qkv_rope_forward(x.to(gpu), w8, b.to(gpu), nq, nkv, hd, yarn=y, positions=pos.to(gpu), mode="decode", weight_scale=ws,
                                 norm_scale=sc.to(gpu), norm_eps=1e-5)
    close(q, qr)
    close(k, kr)
    close(v, vr)


@pytest.mark.parametrize("fp8,rows,k,nq,nkv,streams", [
    (True, 5, 96, 6, 2, 1), (True, 9, 288, 6, 2, 2), (True, 20, 544, 6, 2, 4), (True, 20, 1312, 6, 2, 4),                      # by K
    (True, 45, 1056, 40, 5, 2), (True, 45, 4096, 40, 5, 2), (True, 200, 608, 64, 8, 1), (True, 200, 4096, 64, 8, 1), (True, 200, 256, 64, 8, 1),   # by workgroups
    (False, 5, 96, 6, 2, 1), (False, 9, 160, 6, 2, 2), (False, 20, 288, 6, 2, 4), (False, 40, 1056, 52, 6, 2), (False, 40, 2048, 52, 6, 2),
    (False, 200, 416, 64, 8, 1), (False, 200, 2048, 64, 8, 1)])
def test_decode_general_streaming_wavefronts(gpu, fp8, rows, k, nq, nkv, streams):
    """One, two and four wavefronts that stream the weight of a general-shape decode projection, as K and the number of
    workgroups have it: one phase each and several, a last phase that is cut short or missing, rows of a pitch of 4 KB."""
    n = (nq + 2 * nkv) * 32
    assert _lib.lib().tllm_decode_general_streams(rows, k, n, fp8) == _lib.lib().tllm_decode_general_streams(rows, k, n - 3, fp8) == streams
    g = torch.Generator().manual_seed(rows + k)
    x, w, b, r = (f * torch.randn(*s, generator=g) for f, s in ((1, (rows, k)), (0.05, (n, k)), (0.05, (n,)), (1, (rows, n))))
    x, w, b, r = x.bfloat16(), w.bfloat16(), b.bfloat16(), r.bfloat16()
    wg, ws = T.quantize_fp8_rows(w.to(gpu)) if fp8 else (w.to(gpu), None)
    want = O.linear_ref(x, O.dequant_fp8_ref(wg.cpu(), ws.cpu()) if fp8 else w, b)
    got = T.qkv_rope_forward(x.to(gpu), wg, b.to(gpu), nq, nkv, 32, rotate=False, mode="decode", weight_scale=ws)
    for have, part in zip(got, torch.split(want, (nq * 32, nkv * 32, nkv * 32), dim=1)):
        close(have, part)
    m = n - 3
    y = T.out_residual_decode_forward(x.view(rows, 1, k).to(gpu), wg[:m], b[:m].to(gpu), r[:, :m].contiguous().view(rows, 1, m).to(gpu), None if ws is None else ws[:m])
    close(y.view(rows, m), want[:, :m] + r[:, :m].float())


@pytest.mark.parametrize("rows,hidden,nq,nkv", [(1, 64, 3, 1), (65, 128, 2, 1), (97, 2880, 64, 8), (130, 192, 40, 8), (200, 320, 64, 8),
                                                (333, 640, 64, 8), (450, 2880, 64, 8), (600, 704, 64, 8), (999, 448, 64, 8),
                                                (1100, 576, 64, 8), (1400, 512, 64, 8), (1500, 1024, 64, 8)])
@pytest.mark.parametrize("how", ["positions", "offset", "wrap", "table", "plain"])
def test_qkv_tile_gemm(gpu, rows, hidden, nq, nkv, how):
    """GEMM tiles at widths up to 2880: fewer K slices than ring stages and more, odd and even slice counts (tiles that split a
    stage's two slices between their wavefronts), ragged last row and column tiles, and every source of the rotary
    positions: a tensor, one sequence behind an offset, several sequences with wrap-around, a cos / sin table, no rotation."""
    assert _lib.lib().tllm_qkv_gemm_tile(1, rows, hidden, nq, nkv, 64) != 0
    g = torch.Generator().manual_seed(40 + rows)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * 64, hidden, generator=g)).bfloat16()
    b = (0.05 * torch.randn((nq + 2 * nkv) * 64, generator=g)).bfloat16()
    kw, pos = {}, torch.randint(0, 8192, (rows,), generator=g)
    if how == "positions":
        kw = dict(yarn=T.gpt_oss_yarn(), positions=pos.to(gpu))
    elif how == "offset":
        pos = 37 + torch.arange(rows)
        kw = dict(yarn=T.gpt_oss_yarn(), offset=torch.tensor([37], device=gpu))
    elif how == "wrap":
        pos = (90 + torch.arange(rows) % 100) % 150
        kw = dict(yarn=T.gpt_oss_yarn(), offset=torch.tensor([90], device=gpu), tokens_per_batch=100, max_context_length=150)
    elif how == "table":
        cos, sin = O.yarn_cos_sin(torch.arange(8192))
        kw = dict(cos=cos.to(gpu), sin=sin.to(gpu), positions=pos.to(gpu), max_context_length=8192)
    else:
        kw = dict(rotate=False)
    q, k, v = T.qkv_rope_forward(x.to(gpu), w.to(gpu), b.to(gpu), nq, nkv, 64, mode="prefill", **kw)
    if how == "plain":
        want = O.linear_ref(x, w, b)
        qr, kr, vr = want[:, :nq * 64], want[:, nq * 64:(nq + nkv) * 64], want[:, (nq + nkv) * 64:]
    else:
        qr, kr, vr = O.qkv_rope_ref(x, w, b, pos, nq, nkv, 64)
    close(q, qr)
    close(k, kr)
    close(v, vr)


def _qkv_position_sources(gpu, rows, g):
    """(name, arguments, positions): every source of the rotary positions; two of them wrap around and hold several sequences."""
    pos, seqs = torch.randint(0, 8192, (rows,), generator=g), (90 + torch.arange(rows) % 100) % 150
    cos, sin = (t.to(gpu) for t in O.yarn_cos_sin(torch.arange(8192)))
    wrap = dict(offset=torch.tensor([90], device=gpu), tokens_per_batch=100, max_context_length=150)
    return [("positions", dict(yarn=T.gpt_oss_yarn(), positions=pos.to(gpu)), pos),
            ("offset", dict(yarn=T.gpt_oss_yarn(), offset=torch.tensor([37], device=gpu)), 37 + torch.arange(rows)),
            ("wrap", dict(yarn=T.gpt_oss_yarn(), **wrap), seqs),
            ("table", dict(cos=cos, sin=sin, positions=pos.to(gpu), max_context_length=8192), pos),
            ("table, wrap", dict(cos=cos, sin=sin, **wrap), seqs),
            ("plain", dict(rotate=False), None)]


def _check_qkv_position_sources(gpu, rows, hidden, nq, nkv, mode, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * 64, hidden, generator=g)).bfloat16()
    b = (0.05 * torch.randn((nq + 2 * nkv) * 64, generator=g)).bfloat16()
    plain = O.linear_ref(x, w, b)
    xg, wg, bg = x.to(gpu), w.to(gpu), b.to(gpu)
    for name, kw, pos in _qkv_position_sources(gpu, rows, g):
        want = plain.clone()
        if pos is not None:
            n = (nq + nkv) * 64
            want[:, :n] = O.rope_rotate_ref(plain[:, :n].reshape(rows, nq + nkv, 64), *O.yarn_cos_sin(pos)).reshape(rows, n)
        got = T.qkv_rope_forward(xg, wg, bg, nq, nkv, 64, mode=mode, **kw)
        try:
            for have, part in zip(got, torch.split(want, (nq * 64, nkv * 64, nkv * 64), dim=1)):
                close(have, part)
        except AssertionError as e:
            raise AssertionError(f"{name}: {e}") from None


@pytest.mark.parametrize("bm,bn,rows,nq,nkv", [(64, 32, 33, 1, 1), (64, 48, 67, 64, 8), (64, 64, 131, 64, 8), (64, 80, 771, 10, 5), (64, 96, 2307, 6, 1),
                                              (64, 128, 1155, 10, 5), (64, 160, 701, 32, 8), (64, 192, 515, 64, 8), (128, 96, 771, 32, 8),
                                              (128, 128, 2307, 10, 5), (128, 160, 771, 64, 8), (128, 192, 1411, 40, 8), (128, 224, 1155, 64, 8),
                                              (128, 256, 2307, 32, 8)])
@pytest.mark.parametrize("hidden", [64, 192])
def test_qkv_every_gemm_tile(gpu, bm, bn, rows, nq, nkv, hidden):
    """Each tile that is compiled, with every source of the rotary positions: a K of one slice and of three (tiles that take
    two slices to a stage: the last stage is half empty), ragged last row tiles."""
    assert _lib.lib().tllm_qkv_gemm_tile(1, rows, hidden, nq, nkv, 64) == bm << 16 | bn
    _check_qkv_position_sources(gpu, rows, hidden, nq, nkv, "prefill", seed=bm + bn + hidden)


@pytest.mark.parametrize("rows", [2011, 4000])
def test_qkv_large_tiles_every_position_source(gpu, rows):
    """The 128- and 256-token tiles of long prompts."""
    assert _lib.lib().tllm_qkv_gemm_tile(1, rows, 2880, 64, 8, 64) == 0
    _check_qkv_position_sources(gpu, rows, 2880, 64, 8, "prefill", seed=rows)


@pytest.mark.parametrize("rows,hidden,tile", [(65, 192, True), (333, 64, True), (2011, 2880, False), (4000, 2880, False)])
@pytest.mark.parametrize("length", [1, 2, 7, 64, 65, 100, 10000])
def test_qkv_positions_of_several_sequences(gpu, rows, hidden, tile, length):
    """Sequences of every length beside what a wavefront counts through (8 or 16 rows), without a positions tensor, up to the last position
    there is; then one step further, where the last row of a whole sequence wraps around."""
    nq, nkv = (8, 2) if tile else (64, 8)
    assert bool(_lib.lib().tllm_qkv_gemm_tile(1, rows, hidden, nq, nkv, 64)) == tile
    g = torch.Generator().manual_seed(rows + length)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * 64, hidden, generator=g)).bfloat16()
    plain = O.linear_ref(x, w, torch.zeros(w.shape[0]).bfloat16())
    used, n = min(length, rows), (nq + nkv) * 64
    for first in (4096 - used, 4097 - used):
        want = plain.clone()
        pos = (first + torch.arange(rows) % length) % 4096
        want[:, :n] = O.rope_rotate_ref(plain[:, :n].reshape(rows, nq + nkv, 64), *O.yarn_cos_sin(pos)).reshape(rows, n)
        got = T.qkv_rope_forward(x.to(gpu), w.to(gpu), torch.zeros(w.shape[0], dtype=torch.bfloat16, device=gpu), nq, nkv, 64, mode="prefill",
                                 yarn=T.gpt_oss_yarn(), offset=torch.tensor([first], device=gpu), tokens_per_batch=length, max_context_length=4096)
        for have, part in zip(got, torch.split(want, (nq * 64, nkv * 64, nkv * 64), dim=1)):
            close(have, part)


@pytest.mark.parametrize("rows,hidden,tile", [(97, 192, True), (2011, 2880, False)])
def test_qkv_positions_out_of_range(gpu, rows, hidden, tile):
    """Positions that wrap around -- one step too far, negative, wide of 32 bits -- at the first row, inside and in the last run of rows that
    a wavefront reads, beside rows that do not; and offsets like that."""
    nq, nkv = (8, 2) if tile else (64, 8)
    assert bool(_lib.lib().tllm_qkv_gemm_tile(1, rows, hidden, nq, nkv, 64)) == tile
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * 64, hidden, generator=g)).bfloat16()
    plain, n = O.linear_ref(x, w, torch.zeros(w.shape[0]).bfloat16()), (nq + nkv) * 64
    sources = []
    for odd in (4096, -1, (1 << 32) + 7, (1 << 62) + 5, -(1 << 31)):
        pos = torch.arange(rows) % 300
        pos[[0, rows // 2, rows - 1]] = odd
        sources.append((dict(positions=pos.to(gpu)), pos % 4096))
    for first in (-3, (1 << 32) - 2, 1 << 40):
        sources.append((dict(offset=torch.tensor([first], device=gpu)), (first + torch.arange(rows)) % 4096))
    for source, pos in sources:
        want = plain.clone()
        want[:, :n] = O.rope_rotate_ref(plain[:, :n].reshape(rows, nq + nkv, 64), *O.yarn_cos_sin(pos)).reshape(rows, n)
        got = T.qkv_rope_forward(x.to(gpu), w.to(gpu), torch.zeros(w.shape[0], dtype=torch.bfloat16, device=gpu), nq, nkv, 64, mode="prefill",
                                 yarn=T.gpt_oss_yarn(), max_context_length=4096, **source)
        for have, part in zip(got, torch.split(want, (nq * 64, nkv * 64, nkv * 64), dim=1)):
            close(have, part)


@pytest.mark.parametrize("batch,hidden,nq,nkv,tiles", [(100, 2880, 64, 8, False), (131, 2880, 64, 8, True), (41, 4096, 64, 8, True), (40, 512, 8, 2, False)])
@pytest.mark.parametrize("how", ["offset", "positions"])
def test_qkv_cache_form_of_large_batches(gpu, batch, hidden, nq, nkv, tiles, how):
    """Batches above 32 rows write k and v into their slot of the cache and touch no other, by the kernel that streams the rows,
    by GEMM tiles and by the general kernel; all rows at the slot's position, or each at its own."""
    assert bool(_lib.lib().tllm_qkv_gemm_tile(0, batch, hidden, nq, nkv, 64)) == tiles
    g = torch.Generator().manual_seed(batch + hidden)
    x = torch.randn(batch, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * 64, hidden, generator=g)).bfloat16()
    b = (0.05 * torch.randn((nq + 2 * nkv) * 64, generator=g)).bfloat16()
    scale = 1 + 0.1 * torch.randn(hidden, generator=g)
    slots, slot = 7, 5
    ck, cv = (torch.full((batch, slots, nkv, 64), 3.0, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    pos = torch.randint(0, 8192, (batch,), generator=g) if how == "positions" else torch.full((batch,), slot)
    q = T.qkv_rope_cache_decode_forward(x.view(batch, 1, hidden).to(gpu), w.to(gpu), b.to(gpu), None, None, 131072, ck, cv,
                                        torch.tensor([slot], device=gpu), nq, nkv, 64, yarn=T.gpt_oss_yarn(),
                                        positions=pos.to(gpu) if how == "positions" else None, norm_scale=scale.to(gpu), norm_eps=1e-5)
    qr, kr, vr = O.qkv_rope_ref(O.rmsnorm_ref(x, scale, 1e-5).bfloat16(), w, b, pos, nq, nkv, 64)
    close(q.view(batch, -1), qr)
    close(ck[:, slot].reshape(batch, -1), kr)
    close(cv[:, slot].reshape(batch, -1), vr)
    others = [s for s in range(slots) if s != slot]
    assert (ck[:, others] == 3.0).all() and (cv[:, others] == 3.0).all()


@pytest.mark.parametrize("bm,bn,rows,n", [(64, 32, 1, 16), (64, 48, 67, 5120), (64, 64, 131, 4096), (64, 80, 2307, 400), (64, 96, 2307, 512), (64, 128, 333, 4096),
                                         (64, 160, 2051, 1024), (64, 192, 515, 5120), (128, 96, 2307, 1024), (128, 128, 1501, 2048), (128, 160, 771, 5120),
                                         (128, 192, 1155, 4096), (128, 224, 1411, 4096), (128, 256, 1411, 5120)])
@pytest.mark.parametrize("k", [64, 192])
def test_linear_every_gemm_tile(gpu, bm, bn, rows, n, k):
    """Each tile that is compiled, through the entry point: the columns behind the last row's end are left alone."""
    L = _lib.lib()
    assert L.tllm_linear_gemm_tile(rows, k, n) == bm << 16 | bn
    g = torch.Generator().manual_seed(rows + n + k)
    x, w, b = torch.randn(rows, k, generator=g).bfloat16(), (0.05 * torch.randn(n, k, generator=g)).bfloat16(), (0.05 * torch.randn(n, generator=g)).bfloat16()
    xg, wg, bg, out = x.to(gpu), w.to(gpu), b.to(gpu), torch.full((rows, n + 8), 7.0, dtype=torch.bfloat16, device=gpu)
    rc = L.tllm_linear_bf16(xg.data_ptr(), wg.data_ptr(), bg.data_ptr(), out.data_ptr(), n + 8, rows, k, n, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, L.tllm_last_error()
    close(out[:, :n], O.linear_ref(x, w, b))
    assert (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("bm,bn,rows,n,k", [(64, 32, 113, 2880, 4096), (64, 32, 128, 2880, 4160), (64, 48, 128, 5120, 2880), (64, 64, 152, 5120, 2880),
                                            (64, 80, 221, 5120, 2880), (64, 96, 450, 2880, 4096), (64, 128, 300, 5120, 2880), (64, 160, 500, 5120, 2880),
                                            (64, 192, 513, 5120, 2880), (128, 96, 600, 4096, 2880), (128, 128, 595, 5120, 2880)])
def test_linear_walks_spread_over_k(gpu, bm, bn, rows, n, k):
    """Tiles whose row tiles begin at different places in K: an odd number of slices where a stage has two, so that the stage without
    a second one is met in the middle of a walk, and what is infinite in the last slice stays infinite."""
    L = _lib.lib()
    assert L.tllm_linear_gemm_tile(rows, k, n) == bm << 16 | bn and L.tllm_gemm_tile_spread(rows, k, n) == 1
    g = torch.Generator().manual_seed(rows + n + k)
    x, w, b = torch.randn(rows, k, generator=g).bfloat16(), (0.02 * torch.randn(n, k, generator=g)).bfloat16(), (0.05 * torch.randn(n, generator=g)).bfloat16()
    x[rows - 1, k - 1] = float("inf")
    xg, wg, bg, out = x.to(gpu), w.to(gpu), b.to(gpu), torch.empty(rows, n, dtype=torch.bfloat16, device=gpu)
    assert L.tllm_linear_bf16(xg.data_ptr(), wg.data_ptr(), bg.data_ptr(), out.data_ptr(), n, rows, k, n, torch.cuda.current_stream().cuda_stream) == 0
    close(out[:rows - 1], O.linear_ref(x[:rows - 1], w, b))
    assert torch.equal(out[rows - 1].float().cpu()[w[:, k - 1] != 0], (w[:, k - 1].float() * float("inf"))[w[:, k - 1] != 0])


@pytest.mark.parametrize("rows,n,k", [(200, 5120, 2880), (333, 5120, 2880), (640, 4096, 2880)])
def test_linear_equal_rows(gpu, rows, n, k):
    """Equal rows have equal results where row tiles walk K in step, and always within a row tile; between tiles whose walks are spread the fp32
    sums differ in their order, by up to 2 k u of the sum of the products' magnitudes, which can move a bf16 result by that and one place."""
    L = _lib.lib()
    spread = L.tllm_gemm_tile_spread(rows, k, n)
    assert spread == (rows != 200)
    g = torch.Generator().manual_seed(rows)
    x, w = torch.randn(1, k, generator=g).bfloat16(), (0.02 * torch.randn(n, k, generator=g)).bfloat16()
    xg, wg, out = x.expand(rows, k).contiguous().to(gpu), w.to(gpu), torch.empty(rows, n, dtype=torch.bfloat16, device=gpu)
    assert L.tllm_linear_bf16(xg.data_ptr(), wg.data_ptr(), None, out.data_ptr(), n, rows, k, n, torch.cuda.current_stream().cuda_stream) == 0
    out, bm = out.cpu(), L.tllm_linear_gemm_tile(rows, k, n) >> 16
    tiles = out[::bm]
    assert torch.equal(out, tiles.repeat_interleave(bm, 0)[:rows])
    if not spread:
        assert torch.equal(tiles, tiles[:1].expand_as(tiles))
    sums = 2 * k * 2.0 ** -24 * (x.float().abs() @ w.float().abs().T)
    assert ((tiles.float() - tiles[:1].float()).abs() <= sums + 2.0 ** -7 * tiles[:1].float().abs()).all()


@pytest.mark.parametrize("rows,n,k,tiles_m,group", [(1024, 1040, 2048, 16, 16), (1025, 1040, 2048, 17, 8), (1536, 1040, 2048, 24, 8), (1551, 1040, 2048, 25, 8),
                                                    (2048, 1024, 64, 32, 32), (2049, 1024, 64, 33, 8), (2177, 2064, 1088, 18, 8)])
def test_linear_row_tiles_in_groups(gpu, rows, n, k, tiles_m, group):
    """Either side of the rules, a last group of one row tile, of two and of all eight, a ragged last column."""
    L = _lib.lib()
    assert -(-rows // (L.tllm_linear_gemm_tile(rows, k, n) >> 16)) == tiles_m and L.tllm_gemm_tile_group(rows, k, n) == group
    g = torch.Generator().manual_seed(rows + n + k)
    x, w, b = torch.randn(rows, k, generator=g).bfloat16(), (0.05 * torch.randn(n, k, generator=g)).bfloat16(), (0.05 * torch.randn(n, generator=g)).bfloat16()
    xg, wg, bg, out = x.to(gpu), w.to(gpu), b.to(gpu), torch.full((rows, n), 7.0, dtype=torch.bfloat16, device=gpu)
    assert L.tllm_linear_bf16(xg.data_ptr(), wg.data_ptr(), bg.data_ptr(), out.data_ptr(), n, rows, k, n, torch.cuda.current_stream().cuda_stream) == 0
    close(out, O.linear_ref(x, w, b))


@pytest.mark.parametrize("rows", [128, 192, 333, 513, 640])
def test_qkv_walks_spread_over_k(gpu, rows):
    assert _lib.lib().tllm_gemm_tile_spread(rows, 2880, 5120) == 1
    _check_qkv_position_sources(gpu, rows, 2880, 64, 8, "prefill", seed=rows)


@pytest.mark.parametrize("rows,k,n", [(1, 64, 16), (3, 4096, 2880), (97, 4096, 2880), (200, 448, 2880), (333, 576, 2880), (512, 640, 2880),
                                      (999, 320, 2880), (1400, 256, 2880), (2048, 192, 2880), (70, 128, 48)])
def test_linear_tile_gemm(gpu, rows, k, n):
    """OUT.forward of a prompt against the oracle, through the module, and where it hands over to the library: a gradient
    wanted, and more rows than one round of tiles."""
    g = torch.Generator().manual_seed(900 + rows)
    x = torch.randn(1, rows, k, generator=g).bfloat16()
    mod = T.OUT(k, n, device=gpu).requires_grad_(False)
    mod.weight.copy_((0.05 * torch.randn(n, k, generator=g)).bfloat16())
    mod.bias.copy_((0.05 * torch.randn(n, generator=g)).bfloat16())
    want = O.linear_ref(x[0], mod.weight.cpu(), mod.bias.cpu())
    assert host().linear(x.to(gpu), mod.weight, mod.bias) is not None
    out = mod(x.to(gpu))
    assert out.shape == (1, rows, n)
    close(out[0], want)
    assert host().linear(torch.empty(128 * 256 + 1, k, dtype=torch.bfloat16, device=gpu), mod.weight, mod.bias) is None
    mod.weight.requires_grad_(True)
    assert host().linear(x.to(gpu), mod.weight, mod.bias) is None
    y = mod(x.to(gpu))
    assert y.requires_grad
    close(y.detach()[0], want)


@pytest.mark.parametrize("k,n,tiles,library", [(4096, 2880, (1, 24, 65, 97, 640, 2048, 2432), (32, 64, 2600)), (2048, 512, (), (1, 16, 48, 128)),
                                               (8192, 1024, (), (1, 48, 128, 2048)), (5120, 2880, (200,), (8, 64)), (1024, 1024, (1, 32, 128, 2048), (2, 24, 3000)),
                                               (128, 2880, (1, 24, 64, 2000), (3000,))])
def test_linear_hands_over_to_the_library_where_that_is_ahead(gpu, k, n, tiles, library):
    w, b = torch.zeros(n, k, dtype=torch.bfloat16, device=gpu), torch.zeros(n, dtype=torch.bfloat16, device=gpu)
    took = lambda rows: host().linear(torch.zeros(rows, k, dtype=torch.bfloat16, device=gpu), w, b) is not None
    assert [took(rows) for rows in tiles] == [True] * len(tiles) and [took(rows) for rows in library] == [False] * len(library)


@pytest.mark.parametrize("rows,k,n,tiles", [(2433, 192, 2880, True), (2560, 192, 2880, True), (2561, 192, 2880, False), (1920, 128, 4080, True),
                                            (1921, 128, 4080, True), (2049, 128, 4080, False), (2433, 128, 3072, False)])
def test_linear_one_round_of_the_widest_tiles(gpu, rows, k, n, tiles):
    """Outputs that are no multiple of 128 stay on GEMM tiles while 128 x 256 ones cover them in one round."""
    g = torch.Generator().manual_seed(rows + n)
    x, w = torch.randn(rows, k, generator=g).bfloat16(), (0.05 * torch.randn(n, k, generator=g)).bfloat16()
    b = (0.05 * torch.randn(n, generator=g)).bfloat16()
    got = host().linear(x.to(gpu), w.to(gpu), b.to(gpu))
    assert (got is not None) == tiles
    if tiles:
        close(got, O.linear_ref(x, w, b))


def test_linear_leaves_torch_its_hooks(gpu):
    """OUT.forward under what F.linear takes part in: vmap, forward-mode derivatives, autocast, tracing, symbolic tracing, a
    dispatch mode, a tensor subclass; a strided operand and one that is not 16-byte aligned."""
    from torch.utils._python_dispatch import TorchDispatchMode

    g = torch.Generator().manual_seed(77)
    x, dx = (torch.randn(3, 40, 128, generator=g).bfloat16().to(gpu) for _ in range(2))
    mod = T.OUT(128, 48, device=gpu).requires_grad_(False)
    mod.weight.copy_((0.05 * torch.randn(48, 128, generator=g)).bfloat16())
    mod.bias.copy_((0.05 * torch.randn(48, generator=g)).bfloat16())
    w, b = mod.weight, mod.bias
    want = O.linear_ref(x.cpu().view(120, 128), w.cpu(), b.cpu()).view(3, 40, 48)
    close(mod(x), want)
    close(torch.vmap(mod)(x), want)
    y, dy = torch.func.jvp(mod, (x,), (dx,))
    close(y, want)
    close(dy, O.linear_ref(dx.cpu().view(120, 128), w.cpu(), torch.zeros(48)).view(3, 40, 48))
    with torch.autocast("cuda", dtype=torch.float16):
        assert mod(x).dtype == torch.float16
    traced = torch.jit.trace(mod, (x,))
    close(traced(dx), mod(dx).cpu())
    close(torch.fx.symbolic_trace(mod)(x), want)

    class Seen(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops += 1
            return func(*args, **(kwargs or {}))

    with Seen() as seen:
        close(mod(x), want)
    assert seen.ops > 0

    class Sub(torch.Tensor):
        pass

    assert type(mod(x.as_subclass(Sub))) is Sub
    close(mod(x.transpose(0, 1)), want.transpose(0, 1))
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=gpu)[1:].view(x.shape)
    flat.copy_(x)
    close(mod(flat), want)


def test_a_launch_error_is_raised_and_the_op_not_repeated(gpu):
    """The runtime reports the error an earlier call has left at the next launch, which has gone out by then: the op raises
    it, and the residual, updated in place, has the projection added once."""
    g = torch.Generator().manual_seed(90)
    h, w, b, res = (torch.randn(*s, generator=g).bfloat16().to(gpu) for s in ((3, 1, 128), (64, 128), (64,), (3, 1, 64)))
    scale = torch.ones(128, device=gpu)
    once = T.out_residual_decode_forward(h, w, b, res.clone())
    calls = [lambda r: T.out_residual_decode_forward(h, w, b, r), lambda r: T.rmsnorm_forward(h, scale, 1e-5),
             lambda r: T.swiglu(h), lambda r: T.qkv_rope_forward(h.view(3, 128), w, b, 2, 1, 16, rotate=False)]
    for i, call in enumerate(calls):
        r = res.clone()
        call(res.clone())
        assert _lib.lib().hipSetDevice(1 << 20) != 0            # an error that nothing has looked at yet
        with pytest.raises(RuntimeError, match="launch failed"):
            call(r)
        torch.cuda.synchronize()
        call(res.clone())                                       # it has been reported: the next call is an ordinary one
        if i == 0:
            assert torch.equal(r, once)


def test_launches_give_up_the_interpreter_lock(gpu):
    """(as test_allocation_gives_up_the_interpreter_lock)"""
    n, stop = [0], threading.Event()

    def count():
        while not stop.is_set():
            n[0] += 1

    x, s, w, b = (torch.randn(*shape, device=gpu).bfloat16() for shape in ((4, 128), (128,), (64, 128), (64,)))
    out = torch.empty_like(x)
    calls = {"rmsnorm": (x, s, 1e-5, out), "swiglu": (x, 1.7, 7.0, True, out[:, :64].contiguous()), "linear": (x, w, b),
             "out_residual": (x.view(4, 1, 128), w, b, torch.zeros(4, 1, 64, device=gpu).bfloat16(), None)}
    interval, thread = sys.getswitchinterval(), threading.Thread(target=count)
    sys.setswitchinterval(1e-6)                      # the waiting thread asks for the lock at once
    thread.start()
    try:
        seen = {}
        for name, args in calls.items():
            op = getattr(host(), name)
            assert op(*args) is not None
            got = list(chain(map(n.__getitem__, [0]), starmap(op, repeat(args, 200)), map(n.__getitem__, [0])))
            seen[name] = got[-1] - got[0]
    finally:
        stop.set()
        thread.join()
        sys.setswitchinterval(interval)
    assert all(d > 0 for d in seen.values()), seen


def test_two_threads_on_two_streams(gpu):
    g = torch.Generator().manual_seed(91)
    sets = []
    for rows in (5, 37):
        x, s, w, b, r = (torch.randn(*shape, generator=g).bfloat16().to(gpu) for shape in ((rows, 256), (256,), (256, 256), (256,), (rows, 1, 256)))
        mod = T.OUT(256, 256, device=gpu).requires_grad_(False)
        mod.weight.copy_(w)
        mod.bias.copy_(b)
        sets.append((x, s.float(), mod, r))

    def step(x, s, mod, r):
        t = T.rmsnorm_forward(x, s, 1e-5, out=torch.empty_like(x))
        y = mod(t)
        y = T.out_residual_decode_forward(y.view(-1, 1, 256), mod.weight, mod.bias, r.clone())
        return T.swiglu(y.view(-1, 256))

    want = [step(*s) for s in sets]
    torch.cuda.synchronize()
    got, errors = [[], []], []

    def run(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(200):
                    got[i].append(step(*sets[i]))
                torch.cuda.current_stream().synchronize()
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert all(torch.equal(y, want[i]) for i in range(2) for y in got[i])


@pytest.mark.parametrize("rotate", [True, False])
@pytest.mark.parametrize("name", ["cos", "sin", "positions", "offset"])
def test_qkv_rope_refuses_tensors_that_are_not_on_the_gpu(gpu, name, rotate):
    rope = T.RotaryEmbedding(64, 150000, torch.float32, initial_context_length=4096, scaling_factor=32.0, device=gpu)   # (its tables carry their parameters)
    x, w, b = (torch.zeros(*s, dtype=torch.bfloat16, device=gpu) for s in ((4, 64), (192, 64), (192,)))
    kw = dict(cos=rope.cos, sin=rope.sin, positions=torch.arange(4, device=gpu), offset=torch.zeros(1, dtype=torch.int64, device=gpu), rotate=rotate)
    T.qkv_rope_forward(x, w, b, 1, 1, 64, **kw)
    away = kw[name].cpu()
    if hasattr(kw[name], "_tllm_yarn"):
        away._tllm_yarn = kw[name]._tllm_yarn
    with pytest.raises(RuntimeError, match="GPU only"):
        T.qkv_rope_forward(x, w, b, 1, 1, 64, **{**kw, name: away})


def test_scratch_pool_shapes_on_the_gpu(gpu):
    deep = (1,) * 17 + (2,)
    assert scratch_pool.get(deep, torch.float32, gpu).data_ptr() == scratch_pool.get(deep, torch.float32, gpu).data_ptr()
    with pytest.raises(torch.OutOfMemoryError):                  # what a caller that frees memory and tries again looks for
        scratch_pool.get((1 << 45,), torch.float32, gpu)
    with pytest.raises((TypeError, OverflowError)):              # torch's own error: no such size
        scratch_pool.get((1 << 70,), torch.float32, gpu)


def test_qkv_generic_shapes(gpu):
    g = torch.Generator().manual_seed(23)
    hidden, nq, nkv, hd = 100, 3, 1, 32                     # hidden % 32 != 0, head_dim != 64 -> generic kernel
    x = torch.randn(5, hidden, generator=g).bfloat16()
    w = (0.1 * torch.randn((nq + 2 * nkv) * hd, hidden, generator=g)).bfloat16()
    b = (0.1 * torch.randn((nq + 2 * nkv) * hd, generator=g)).bfloat16()
    y = T.YarnParams(head_dim=hd, base=10000.0)
    pos = torch.tensor([0, 3, 17, 100, 4000], dtype=torch.int64)
    qr, kr, vr = O.qkv_rope_ref(x, w, b, pos, nq, nkv, hd, base=10000.0, scaling_factor=1.0)
    for mode in ("decode", "prefill"):
        q, k, v = T.qkv_rope_forward(x.to(gpu), w.to(gpu), b.to(gpu), nq, nkv, hd, yarn=y, positions=pos.to(gpu), mode=mode)
        close(q, qr)
        close(k, kr)
        close(v, vr)
    # MFMA kernels at another K and head count (ragged last head tile, K loop with a tail)
    hidden, nq, nkv, hd = 320, 6, 1, 64
    x = torch.randn(150, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn((nq + 2 * nkv) * hd, hidden, generator=g)).bfloat16()
    b = (0.05 * torch.randn((nq + 2 * nkv) * hd, generator=g)).bfloat16()
    pos = torch.randint(0, 8192, (150,), generator=g)
    yy = T.gpt_oss_yarn()
    qr, kr, vr = O.qkv_rope_ref(x, w, b, pos, nq, nkv, hd)
    for mode, n in (("decode", 20), ("prefill", 150)):
        q, k, v = T.qkv_rope_forward(x[:n].to(gpu), w.to(gpu), b.to(gpu), nq, nkv, hd, yarn=yy, positions=pos[:n].to(gpu), mode=mode)
        close(q, qr[:n])
        close(k, kr[:n])
        close(v, vr[:n])


def test_reference_signatures_decode_with_cache(gpu):
    """qkv_rope_cache_decode_forward / qkv_decode_forward / QKV / RMSNorm modules as model.py calls them."""
    scratch_pool.clear()
    d = O.make_inputs(8, seed=31)
    norm = T.RMSNorm(2880, device=gpu)
    qkv = T.QKV(2880, 5120, device=gpu)
    rope = T.RotaryEmbedding(64, 150000, torch.float32, initial_context_length=4096, scaling_factor=32.0, device=gpu)
    with torch.no_grad():
        norm.scale.copy_(d["norm_scale"].float())
        qkv.weight.copy_(d["w"])
        qkv.bias.copy_(d["b"])
    x = d["x"].view(8, 1, 2880).to(gpu)
    t = norm(x)
    t_ref = O.rmsnorm_ref(d["x"], d["norm_scale"].float()).bfloat16()
    n_ctx, slot = 64, 37
    cache_k = torch.zeros(8, n_ctx, 8, 64, dtype=torch.bfloat16, device=gpu)
    cache_v = torch.zeros_like(cache_k)
    offset = torch.tensor([slot], dtype=torch.int64, device=gpu)
    q = T.qkv_rope_cache_decode_forward(t, qkv.weight, qkv.bias, rope.sin, rope.cos, rope.max_context_length, cache_k, cache_v,
                                        offset, 64, 8, 64)
    assert q.shape == (8, 1, 4096)
    pos = torch.full((8,), slot, dtype=torch.int64)
    qr, kr, vr = O.qkv_rope_ref(t.cpu().view(8, 2880), d["w"], d["b"], pos)
    close(q.view(8, 4096), qr)
    close(cache_k[:, slot].reshape(8, 512), kr)
    close(cache_v[:, slot].reshape(8, 512), vr)
    mask = torch.ones(n_ctx, dtype=torch.bool)
    mask[slot] = False
    assert torch.all(cache_k.cpu()[:, mask] == 0) and torch.all(cache_v.cpu()[:, mask] == 0)   # nothing else touched
    close(t.view(8, 2880), t_ref.float())
    # unfused decode + F.linear-style forward
    qd, kd, vd = qkv.decode(t, 4096, 512)
    assert qd.shape == (8, 1, 4096) and kd.shape == (8, 1, 512)
    plain = O.linear_ref(t.cpu().view(8, 2880), d["w"], d["b"])
    close(qd.view(8, 4096), plain[:, :4096])
    close(kd.view(8, 512), plain[:, 4096:4608])
    close(vd.view(8, 512), plain[:, 4608:])
    full = qkv(t)
    assert full.shape == (8, 1, 5120)
    close(full.view(8, 5120), plain)
    seq = O.make_inputs(300, seed=32)["x"].view(1, 300, 2880)
    close(qkv(seq.to(gpu)).view(300, 5120), O.linear_ref(seq.view(300, 2880), d["w"], d["b"]))
    # fused prefill through the module
    qf, kf, vf = qkv.forward_rope(seq.to(gpu), rope, 64, 8, offset=torch.tensor([10], dtype=torch.int64, device=gpu))
    qr, kr, vr = O.qkv_rope_ref(seq.view(300, 2880), d["w"], d["b"], O.token_positions(1, 300, 10))
    close(qf.reshape(300, 4096), qr)
    close(kf.reshape(300, 512), kr)
    close(vf.reshape(300, 512), vr)
    with pytest.raises(AssertionError):      # a scale without an fp8 weight
        T.qkv_rope_cache_decode_forward(t, qkv.weight, qkv.bias, rope.sin, rope.cos, rope.max_context_length, cache_k, cache_v,
                                        offset, 64, 8, 64, weight_scale=torch.ones(5120, device=gpu))
    with pytest.raises(AssertionError):
        T.qkv_decode_forward(torch.zeros(8, 2, 2880, dtype=torch.bfloat16, device=gpu), qkv.weight, qkv.bias, 4096, 512)


def test_qkv_linearity_full_size(gpu):
    """Size-independent property at T=8192 without the oracle: the projection is linear in x."""
    g = torch.Generator().manual_seed(41)
    x1 = torch.randn(8192, 2880, generator=g).bfloat16().to(gpu)
    w = (0.02 * torch.randn(5120, 2880, generator=g)).bfloat16().to(gpu)
    y1 = [t.float() for t in T.qkv_rope_forward(x1, w, None, 64, 8, 64, rotate=False, mode="prefill")]
    y2 = [t.float() for t in T.qkv_rope_forward((2 * x1), w, None, 64, 8, 64, rotate=False, mode="prefill")]
    for a, b in zip(y1, y2):
        torch.testing.assert_close(b, 2 * a, rtol=1.6e-2, atol=1e-2)


def test_graph_replay_reads_positions_from_device(gpu, yarn):
    """Capture the decode chain once, replay with new positions: results must follow the device-side offset."""
    d = O.make_inputs(8, seed=51)
    xg, wg, bg, sg = d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), d["norm_scale"].to(gpu)
    offset = torch.zeros(1, dtype=torch.int64, device=gpu)
    outs = {}

    def chain():
        t = T.rmsnorm_forward(xg, sg, 1e-5)
        outs["q"], outs["k"], outs["v"] = T.qkv_rope_forward(t, wg, bg, 64, 8, 64, yarn=yarn, offset=offset, tokens_per_batch=1,
                                                              mode="decode")

    chain()                                       # warm up (allocates pool buffers)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        chain()
    t_ref = O.rmsnorm_ref(d["x"], d["norm_scale"]).bfloat16()
    for p in (0, 4097, 8191):
        offset.fill_(p)
        graph.replay()
        torch.cuda.synchronize()
        qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], torch.full((8,), p, dtype=torch.int64))
        close(outs["q"], qr, rtol=3e-2, atol=2e-2)   # t_ref is the oracle's rounding of the norm, the GPU's may differ by one bf16 ulp
        close(outs["k"], kr, rtol=3e-2, atol=2e-2)


# ----------------------------------------------------------------------------------- out-projection (decode)
def _out_inputs(rows, seed, in_dim=4096, out_dim=2880):
    g = torch.Generator().manual_seed(seed)
    return dict(x=torch.randn(rows, in_dim, generator=g).bfloat16(), w=(0.02 * torch.randn(out_dim, in_dim, generator=g)).bfloat16(),
                b=(0.02 * torch.randn(out_dim, generator=g)).bfloat16(), r=torch.randn(rows, out_dim, generator=g).bfloat16())


@pytest.mark.parametrize("rows", [1, 8, 9, 11, 12, 13, 16, 17, 20, 21, 24, 25, 28, 29, 32, 33, 41, 45, 49, 52, 53, 56, 57, 64, 65, 70, 73, 80, 96, 97, 113, 128, 129, 161, 300])
@pytest.mark.parametrize("fp8", [False, True])
def test_out_residual_decode_parity(gpu, rows, fp8):
    d = _out_inputs(rows, 600 + rows)
    res = d["r"].view(rows, 1, 2880).to(gpu)
    res_before = res.clone()
    if fp8:
        w8, ws = T.quantize_fp8_rows(d["w"].to(gpu))
        out = T.out_residual_decode_forward(d["x"].view(rows, 1, 4096).to(gpu), w8, d["b"].to(gpu), res, weight_scale=ws)
        want = O.out_residual_ref(d["x"], O.dequant_fp8_ref(w8.cpu(), ws.cpu()), d["b"], d["r"])
    else:
        out = T.out_residual_decode_forward(d["x"].view(rows, 1, 4096).to(gpu), d["w"].to(gpu), d["b"].to(gpu), res)
        want = O.out_residual_ref(d["x"], d["w"], d["b"], d["r"])
    assert out.shape == (rows, 1, 2880) and out.data_ptr() == res.data_ptr()          # written into the residual, as the reference does
    assert not torch.equal(res, res_before)
    close(out.view(rows, 2880), want)


@pytest.mark.parametrize("rows,out_dim", [(49, 1536), (65, 1536), (97, 1536), (113, 2304), (128, 1536), (128, 2304)])
@pytest.mark.parametrize("fp8", [False, True])
def test_out_residual_narrow_outputs(gpu, rows, out_dim, fp8):
    """Two to four chunks of 24, 28 and 32 rows beside one pass over the weight: with a bf16 weight only narrower outputs than 2880 have
    four, and with fp8 the walks over K are spread over its phases from 2048 outputs on."""
    assert _lib.lib().tllm_out_gemm_tile(rows, 4096, out_dim) == 0
    d = _out_inputs(rows, 900 + rows, out_dim=out_dim)
    w, ws = T.quantize_fp8_rows(d["w"].to(gpu)) if fp8 else (d["w"].to(gpu), None)
    out = T.out_residual_decode_forward(d["x"].view(rows, 1, 4096).to(gpu), w, d["b"].to(gpu), d["r"].view(rows, 1, out_dim).to(gpu), weight_scale=ws)
    want = O.dequant_fp8_ref(w.cpu(), ws.cpu()) if fp8 else d["w"]
    close(out.view(rows, out_dim), O.out_residual_ref(d["x"], want, d["b"], d["r"]))


@pytest.mark.parametrize("rows", [1, 5, 8, 13, 32, 37])
@pytest.mark.parametrize("fp8", [False, True])
def test_out_residual_decode_strides_alignment_and_absent_operands(gpu, rows, fp8):
    """The C entry point with what the host wrapper never passes: a separate output buffer, row strides that rule
    out 8-byte accesses (2882) and ones that allow them (2884), an output that starts 2 bytes off an 8-byte boundary,
    no bias, no residual; bf16 weight and fp8 weight with row scales. Untouched padding columns must stay untouched."""
    from tritonllm_amd import _lib
    L = _lib.lib()
    d = _out_inputs(rows, 650 + rows)
    x, w, b = d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu)
    w_ref, ws = d["w"], None
    if fp8:
        w, ws = T.quantize_fp8_rows(w)
        w_ref = O.dequant_fp8_ref(w.cpu(), ws.cpu())
    for stride, shift, with_bias, with_res in ((2884, 0, True, True), (2882, 0, True, True), (2884, 1, True, True),
                                               (2880, 0, False, True), (2880, 0, True, False), (2880, 0, False, False)):
        res = torch.zeros(rows, stride, dtype=torch.bfloat16, device=gpu)
        res[:, :2880] = d["r"].to(gpu)
        buf = torch.full((rows * stride + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
        out = buf[shift:shift + rows * stride].view(rows, stride)
        rc = L.tllm_out_residual_decode_bf16(x.data_ptr(), w.data_ptr(), ws.data_ptr() if fp8 else None, b.data_ptr() if with_bias else None,
                                             res.data_ptr() if with_res else None, out.data_ptr(), stride, stride, rows, 4096, 2880, None)
        assert rc == 0, L.tllm_last_error()
        torch.cuda.synchronize()
        want = O.out_residual_ref(d["x"], w_ref, d["b"] if with_bias else torch.zeros_like(d["b"]),
                                  d["r"] if with_res else torch.zeros_like(d["r"]))
        close(out[:, :2880], want)
        assert torch.all(out[:, 2880:] == 7.0) and torch.all(buf[:shift] == 7.0) and torch.all(buf[shift + rows * stride:] == 7.0)


@pytest.mark.parametrize("in_dim,out_dim", [(32, 1), (608, 17), (1056, 100), (4096, 4096), (100, 30)])
@pytest.mark.parametrize("rows", [1, 8, 9, 33])
@pytest.mark.parametrize("fp8", [False, True])
def test_out_residual_general_stream(gpu, in_dim, out_dim, rows, fp8):
    """The general out-projection stream at its edges: one k32 step, K that ends inside a wavefront's phase, fewer output
    features than a tile and ragged last tiles, both activation-row forms and a ragged last chunk; in_dim 100 is the
    plain kernel behind it."""
    d = _out_inputs(rows, 7000 + in_dim + rows, in_dim=in_dim, out_dim=out_dim)
    w, ws, ref = d["w"].to(gpu), None, d["w"]
    if fp8:
        w, ws = T.quantize_fp8_rows(w)
        ref = O.dequant_fp8_ref(w.cpu(), ws.cpu())
    out = T.out_residual_decode_forward(d["x"].view(rows, 1, in_dim).to(gpu), w, d["b"].to(gpu), d["r"].view(rows, 1, out_dim).to(gpu), weight_scale=ws)
    close(out.view(rows, out_dim), O.out_residual_ref(d["x"], ref, d["b"], d["r"]))


@pytest.mark.parametrize("bm,bn,spread,rows,in_dim,out_dim", [
    (64, 32, 0, 129, 4096, 48), (64, 32, 1, 113, 2880, 2880), (64, 48, 0, 113, 192, 5120), (64, 48, 1, 113, 2048, 5120), (64, 64, 0, 129, 192, 5120),
    (64, 64, 1, 113, 1088, 8192), (64, 80, 0, 2307, 192, 400), (64, 80, 1, 221, 2048, 5120), (64, 96, 0, 1411, 64, 1024), (64, 96, 1, 273, 2112, 4096),
    (64, 128, 0, 193, 64, 8192), (64, 128, 1, 153, 1088, 8192), (64, 160, 0, 515, 64, 4032), (64, 160, 1, 515, 2112, 4032), (64, 192, 0, 257, 64, 8192),
    (64, 192, 1, 273, 1600, 8192), (128, 96, 0, 2307, 64, 1024), (128, 96, 1, 640, 2112, 4032), (128, 128, 0, 333, 64, 8192), (128, 128, 1, 640, 2048, 5120),
    (128, 160, 0, 771, 64, 5120), (128, 192, 0, 515, 64, 8192), (128, 224, 0, 1411, 64, 4096), (128, 256, 0, 771, 64, 8192), (64, 32, 0, 81, 4096, 2880),
    (64, 32, 1, 128, 4096, 2880), (64, 32, 0, 33, 4096, 4032)])
def test_out_residual_in_gemm_tiles(gpu, bm, bn, spread, rows, in_dim, out_dim):
    """Every tile the projection takes for many rows, walks in step and spread: in place with strides that allow 16-byte accesses; a
    residual and an output of their own, two bytes off and with odd strides; no bias; no residual. Padding columns stay untouched."""
    L = _lib.lib()
    assert L.tllm_out_gemm_tile(rows, in_dim, out_dim) == bm << 16 | bn
    assert L.tllm_gemm_tile_spread(rows, in_dim, out_dim) == spread
    d = _out_inputs(rows, 7300 + in_dim + rows, in_dim=in_dim, out_dim=out_dim)
    x, w, b = d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu)
    product = d["x"].float() @ d["w"].float().T
    for pad, shift, with_bias, with_res in ((8, 0, True, True), (3, 1, False, True), (0, 0, True, False)):
        stride = out_dim + pad
        buf = torch.full((rows * stride + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
        out = buf[shift:shift + rows * stride].view(rows, stride)
        res = out if with_res and not shift else torch.zeros(rows * stride + 8, dtype=torch.bfloat16, device=gpu)[shift:shift + rows * stride].view(rows, stride)
        if with_res:
            res[:, :out_dim] = d["r"].to(gpu)
        rc = L.tllm_out_residual_decode_bf16(x.data_ptr(), w.data_ptr(), None, b.data_ptr() if with_bias else None, res.data_ptr() if with_res else None,
                                             out.data_ptr(), stride, stride, rows, in_dim, out_dim, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, L.tllm_last_error()
        close(out[:, :out_dim], product + (d["b"].float() if with_bias else 0) + (d["r"].float() if with_res else 0))
        assert (out[:, out_dim:] == 7.0).all() and (buf[:shift] == 7.0).all() and (buf[shift + rows * stride:] == 7.0).all()


def test_out_residual_other_shapes_module_and_errors(gpu, monkeypatch):
    # a shape the streaming kernel does not serve (in_dim != 4096): the plain kernel, bf16 and fp8
    d = _out_inputs(5, 61, in_dim=320, out_dim=100)
    res = d["r"].view(5, 1, 100).to(gpu)
    out = T.out_residual_decode_forward(d["x"].view(5, 1, 320).to(gpu), d["w"].to(gpu), d["b"].to(gpu), res)
    close(out.view(5, 100), O.out_residual_ref(d["x"], d["w"], d["b"], d["r"]))
    w8, ws = T.quantize_fp8_rows(d["w"].to(gpu))
    out = T.out_residual_decode_forward(d["x"].view(5, 1, 320).to(gpu), w8, d["b"].to(gpu), d["r"].view(5, 1, 100).to(gpu), weight_scale=ws)
    close(out.view(5, 100), O.out_residual_ref(d["x"], O.dequant_fp8_ref(w8.cpu(), ws.cpu()), d["b"], d["r"]))
    # the module, plain and under ATTN_FP8 (model.py:170-216)
    d = _out_inputs(8, 62)
    for env in ("0", "1"):
        monkeypatch.setenv("ATTN_FP8", env)
        mod = T.OUT(4096, 2880, device=gpu)
        with torch.no_grad():
            mod.weight.copy_(d["w"])
            mod.bias.copy_(d["b"])
        y = mod.decode_residual(d["x"].view(8, 1, 4096).to(gpu), d["r"].view(8, 1, 2880).to(gpu))
        w_used = O.dequant_fp8_ref(*[t.cpu() for t in mod._fp8_weight]) if env == "1" else d["w"]
        close(y.view(8, 2880), O.out_residual_ref(d["x"], w_used, d["b"], d["r"]))
    with pytest.raises(AssertionError):
        T.out_residual_decode_forward(torch.zeros(8, 2, 4096, dtype=torch.bfloat16, device=gpu), mod.weight, mod.bias,
                                      torch.zeros(8, 1, 2880, dtype=torch.bfloat16, device=gpu))
    with pytest.raises(AssertionError):
        T.out_residual_decode_forward(torch.zeros(8, 1, 4096, dtype=torch.bfloat16, device=gpu), mod.weight, mod.bias,
                                      torch.zeros(8, 1, 2881, dtype=torch.bfloat16, device=gpu))


# ----------------------------------------------------------------------------------- unembedding (decode)
def _argmax_ok(ids, logits_ref):
    """The chosen token must be an argmax of the fp32 oracle logits up to summation noise: its oracle logit within
    1e-3 of the oracle maximum; and where the oracle's winner is clear (margin > 1e-2) it must be that very token."""
    ids = ids.cpu().long()
    top2 = logits_ref.topk(2, dim=-1)
    chosen = logits_ref.gather(1, ids[:, None])[:, 0]
    assert torch.all(chosen >= top2.values[:, 0] - 1e-3), (chosen, top2.values[:, 0])
    clear = (top2.values[:, 0] - top2.values[:, 1]) > 1e-2
    assert torch.equal(ids[clear], top2.indices[clear, 0])


def test_unembedding_fp8_logits_rows_that_allow_2_byte_stores_only(gpu):
    """The fp8 kernel for an even vocabulary stores the logits of two neighbouring vocabulary rows as one 4-byte pair
    where the logits buffer allows it; here it does not (odd row stride, first element 2 bytes into a word)."""
    from tritonllm_amd._lib import lib
    g = torch.Generator().manual_seed(8642)
    rows, vocab = 5, 3000
    x = torch.randn(rows, 2880, generator=g).bfloat16()
    w = (0.02 * torch.randn(vocab, 2880, generator=g)).bfloat16()
    w8, ws = T.quantize_fp8_rows(w.to(gpu))
    want = O.linear_ref(x, O.dequant_fp8_ref(w8.cpu(), ws.cpu()), None)
    ld = vocab + 3
    buf = torch.full((rows * ld + 8,), float("nan"), dtype=torch.bfloat16, device=gpu)
    xg = x.to(gpu)
    rc = lib().tllm_unembedding_decode_bf16(xg.data_ptr(), w8.data_ptr(), ws.data_ptr(), buf.data_ptr() + 2, ld, rows, 2880, vocab,
                                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    got = buf[1:1 + rows * ld].view(rows, ld)
    close(got[:, :vocab], want)
    assert torch.isnan(got[:, vocab:].float()).all() and torch.isnan(buf[0].float())   # nothing outside the rows was written


def test_unembedding_argmax_ties_negative_maxima_and_zeros(gpu):
    """The winner among the per-wavefront candidates is picked through one sortable key per candidate: exact ties (the
    same vocabulary row planted in tiles that different wavefronts and workgroups own) must go to the lowest index, a
    row whose logits are all negative must still find its maximum, and a row of zeros (every logit +-0) must return
    token 0."""
    g = torch.Generator().manual_seed(4242)
    vocab = 140000                                            # 4375 tiles: more than one per wavefront
    x = torch.randn(4, 2880, generator=g).bfloat16()
    x[1] = -x[0]
    x[2] = 0
    w = (0.02 * torch.randn(vocab, 2880, generator=g)).bfloat16()
    planted = [131071, 777, 65536, 40000]
    for i in planted:
        w[i] = x[0]                                           # logit |x0|^2 for row 0, the most negative one for row 1
    x[3] = x[3].abs()
    ids = T.unembedding_decode_argmax_forward(x.view(4, 1, 2880).to(gpu), w.to(gpu)).cpu().long()
    want = O.linear_ref(x, w, None)
    assert ids[0].item() == min(planted)
    assert ids[2].item() == 0
    _argmax_ok(ids[[1, 3]], want[[1, 3]])
    # all logits of a row negative: w = -|w|, x >= 0
    wn = -w.abs()
    idn = T.unembedding_decode_argmax_forward(x[3:4].view(1, 1, 2880).to(gpu), wn.to(gpu))
    wantn = O.linear_ref(x[3:4], wn, None)
    assert wantn.max() < 0
    _argmax_ok(idn, wantn)


@pytest.mark.parametrize("rows,vocab", [(1, 4096), (8, 5000), (13, 4097), (16, 20000), (20, 3001)])
@pytest.mark.parametrize("fp8", [False, True])
def test_unembedding_decode_parity_small_vocab(gpu, rows, vocab, fp8):
    g = torch.Generator().manual_seed(700 + rows)
    x = torch.randn(rows, 2880, generator=g).bfloat16()
    w = (0.02 * torch.randn(vocab, 2880, generator=g)).bfloat16()
    xg = x.view(rows, 1, 2880).to(gpu)
    if fp8:
        w8, ws = T.quantize_fp8_rows(w.to(gpu))
        want = O.linear_ref(x, O.dequant_fp8_ref(w8.cpu(), ws.cpu()), None)
        logits = T.unembedding_decode_fp8_forward(xg, w8, ws).clone()
        ids = T.unembedding_decode_fp8_argmax_forward(xg, w8, ws)
    else:
        want = O.linear_ref(x, w, None)
        logits = T.unembedding_decode_forward(xg, w.to(gpu)).clone()
        ids = T.unembedding_decode_argmax_forward(xg, w.to(gpu))
    assert logits.shape == (rows, 1, vocab) and ids.shape == (rows,) and ids.dtype == torch.int32
    close(logits.view(rows, vocab), want)
    _argmax_ok(ids, want)


@pytest.mark.parametrize("rows", [5, 11, 16, 19])
@pytest.mark.parametrize("hidden", [64, 4096])
def test_unembedding_other_hidden_sizes(gpu, rows, hidden):
    """Hidden sizes other than gpt-oss's: above eight rows the kernel keeps sixteen activation rows in LDS where they
    fit (2880 wide) and falls back to chunks of eight where they do not (4096 wide), logits and argmax alike."""
    g = torch.Generator().manual_seed(880 + rows + hidden)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = (0.05 * torch.randn(3001, hidden, generator=g)).bfloat16()
    xg = x.view(rows, 1, hidden).to(gpu)
    want = O.linear_ref(x, w, None)
    close(T.unembedding_decode_forward(xg, w.to(gpu)).view(rows, 3001), want)
    _argmax_ok(T.unembedding_decode_argmax_forward(xg, w.to(gpu)), want)
    w8, ws = T.quantize_fp8_rows(w.to(gpu))
    want8 = O.linear_ref(x, O.dequant_fp8_ref(w8.cpu(), ws.cpu()), None)
    close(T.unembedding_decode_fp8_forward(xg, w8, ws).view(rows, 3001), want8)
    _argmax_ok(T.unembedding_decode_fp8_argmax_forward(xg, w8, ws), want8)


@pytest.mark.parametrize("hidden", [2048, 4096, 6144, 8192])
def test_rows_of_a_power_of_two_pitch(gpu, hidden):
    """Weights whose rows begin on the same memory channels: every workgroup begins its walk over K somewhere else -- logits
    (tiles for some wavefronts only, several each, a ragged last one; fp8 in pairs of rows and one by one) and projections."""
    g = torch.Generator().manual_seed(hidden)
    for rows, vocab in ((1, 3001), (8, 100002 if hidden == 2048 else 9001)) if hidden <= 4096 else ():   # (wider: not built for logits)
        x = torch.randn(rows, hidden, generator=g).bfloat16()
        w = (0.02 * torch.randn(vocab, hidden, generator=g)).bfloat16()
        w[vocab // 3], w[5] = w[vocab - 1], w[vocab - 1]       # equal rows: the argmax of a tie is the lowest
        x[0] = w[5] * 50
        xg = x.view(rows, 1, hidden).to(gpu)
        want = O.linear_ref(x, w, None)
        close(T.unembedding_decode_forward(xg, w.to(gpu)).view(rows, vocab), want)
        ids = T.unembedding_decode_argmax_forward(xg, w.to(gpu))
        assert int(ids[0]) == 5
        _argmax_ok(ids, want)
        w8, ws = T.quantize_fp8_rows(w.to(gpu))
        close(T.unembedding_decode_fp8_forward(xg, w8, ws).view(rows, vocab), O.linear_ref(x, O.dequant_fp8_ref(w8.cpu(), ws.cpu()), None))
    for rows in (1, 7, 16, 19):
        x = torch.randn(rows, 1, hidden, generator=g).bfloat16()
        w, b = (0.02 * torch.randn(1040, hidden, generator=g)).bfloat16(), torch.randn(1040, generator=g).bfloat16()
        def zero():
            return torch.zeros(rows, 1, 1040, dtype=torch.bfloat16, device=gpu)

        close(T.out_residual_decode_forward(x.to(gpu), w.to(gpu), b.to(gpu), zero()).view(rows, 1040), O.linear_ref(x[:, 0], w, b))
        w8, ws = T.quantize_fp8_rows(w.to(gpu))
        close(T.out_residual_decode_forward(x.to(gpu), w8, b.to(gpu), zero(), ws).view(rows, 1040), O.linear_ref(x[:, 0], O.dequant_fp8_ref(w8.cpu(), ws.cpu()), b))


@pytest.mark.parametrize("hidden,rows,vocab,fp8", [(4096, 8, 32000, False), (2048, 1, 200000, False), (2048, 8, 32000, True),
                                                   (4096, 8, 32000, True), (4096, 12, 32000, False), (2880, 8, 32000, False),
                                                   (4096, 7, 60002, True), (2048, 8, 60002, True), (2048, 12, 60002, True), (4096, 7, 49152, True), (4096, 7, 49154, True),
                                                   (4096, 8, 12288, False), (4096, 8, 12290, False)])
def test_equal_rows_have_equal_logits(gpu, hidden, rows, vocab, fp8):
    """Two equal rows of the weight give the same number whichever workgroups they fall to (a pitch of a multiple of 4 KB: where
    the walk over K does not begin at 0 everywhere, from a vocabulary of about 12000, 24000 or 49000 on) and whether they are the
    first or the second of a pair (fp8), so that a caller's argmax over the logits sees a tie, as the argmax op does."""
    g = torch.Generator(device=gpu).manual_seed(hidden + rows)
    x = torch.randn(rows, 1, hidden, device=gpu, generator=g).bfloat16()
    w = (0.02 * torch.randn(vocab // 2, hidden, device=gpu, generator=g)).bfloat16()
    w, ws = ops.quantize_fp8_rows(w) if fp8 else (w, None)
    w = torch.cat((w.view(torch.uint8), w.view(torch.uint8))).view(w.dtype)
    ws = torch.cat((ws, ws)) if fp8 else None
    logits = T.unembedding_decode_forward(x, w, ws)[:, 0]
    assert torch.equal(logits[:, :vocab // 2], logits[:, vocab // 2:])
    one = w[:vocab // 2].cpu()
    close(logits[:, :vocab // 2], O.linear_ref(x[:, 0].cpu(), O.dequant_fp8_ref(one, ws[:vocab // 2].cpu()) if fp8 else one, None))
    assert (T.unembedding_decode_argmax_forward(x, w, ws) < vocab // 2).all()


@pytest.mark.parametrize("rows,vocab,hidden", [(17, 3001, 2880), (32, 140000, 2880), (33, 70001, 2880), (50, 4096, 2880), (64, 9000, 2880),
                                                (24, 5000, 128), (32, 5000, 192), (29, 5000, 1024), (20, 270000, 128)])
def test_unembedding_more_than_16_rows_one_pass_over_the_weight(gpu, rows, vocab, hidden):
    """Above sixteen rows a workgroup takes 32 batch rows and keeps one K half of them in LDS at a time; a wavefront's
    tiles wait in registers between the halves. Vocabularies that give a wavefront 0, 1, 2, 3 and 4 tiles (2048
    wavefronts) and one that would give it five (which goes back to chunks of sixteen rows), ragged last tiles, ragged
    last chunks of rows, K halves of equal and unequal length (hidden / 64 odd), logits and argmax."""
    g = torch.Generator().manual_seed(990 + rows + hidden)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = ((0.02 if hidden == 2880 else 0.05) * torch.randn(vocab, hidden, generator=g)).bfloat16()
    planted = torch.randint(0, vocab, (rows,), generator=g)
    planted[0], planted[-1] = vocab - 1, 0
    for r in range(rows):                                      # row r of x points at weight row planted[r] ...
        w[planted[r]] = (x[r].float() * 0.05).bfloat16()
    xg = x.view(rows, 1, hidden).to(gpu)
    logits = T.unembedding_decode_forward(xg, w.to(gpu))
    want = O.linear_ref(x, w, None)
    close(logits.view(rows, vocab), want)
    ids = T.unembedding_decode_argmax_forward(xg, w.to(gpu))
    _argmax_ok(ids, want)
    # the fp8 weight takes the same path above sixteen rows
    w8, ws = T.quantize_fp8_rows(w.to(gpu))
    want8 = O.linear_ref(x, O.dequant_fp8_ref(w8.cpu(), ws.cpu()), None)
    close(T.unembedding_decode_fp8_forward(xg, w8, ws).view(rows, vocab), want8)
    _argmax_ok(T.unembedding_decode_fp8_argmax_forward(xg, w8, ws), want8)


@pytest.mark.parametrize("rows,vocab,hidden", [(9, 40, 4096), (24, 3001, 4096), (33, 20, 2880), (48, 70003, 2880), (65, 40000, 2880), (96, 5001, 64),
                                                (97, 33001, 2880), (128, 9000, 2880), (128, 3001, 128), (131, 5000, 2880), (300, 2050, 192), (17, 40, 4096),
                                                (65, 20, 2880), (20, 70001, 3200), (40, 65000, 128), (50, 81000, 192), (70, 100003, 64), (128, 75000, 128),
                                                (90, 114000, 128), (128, 201088, 64), (97, 151936, 64), (128, 70000, 128), (96, 234000, 64),
                                                (66, 8193, 128)])
def test_unembedding_logits_in_tiles(gpu, rows, vocab, hidden):
    """More rows than the kernels that keep them in LDS take: tiles of the vocabulary with the activations streamed next to
    the weight. One to four row blocks per wavefront, several chunks of rows, workgroups with no vocabulary, one unit, many
    and a last tile narrower than the others, every width of tile that has a kernel of its own, vocabularies that are no multiple
    of 16 (and odd: no 8-byte stores), K of one slice up (fewer stages than the ring), and neighbouring rows of the output left alone."""
    from tritonllm_amd._lib import lib
    g = torch.Generator().manual_seed(1300 + rows + hidden)
    x = torch.randn(rows, hidden, generator=g).bfloat16()
    w = ((0.02 if hidden == 2880 else 0.05) * torch.randn(vocab, hidden, generator=g)).bfloat16()
    xg = x.view(rows, 1, hidden).to(gpu)
    close(T.unembedding_decode_forward(xg, w.to(gpu)).view(rows, vocab), O.linear_ref(x, w, None))
    w8, ws = T.quantize_fp8_rows(w.to(gpu))
    want8 = O.linear_ref(x, O.dequant_fp8_ref(w8.cpu(), ws.cpu()), None)
    close(T.unembedding_decode_fp8_forward(xg, w8, ws).view(rows, vocab), want8)
    ld = vocab + 5                                             # a row stride of its own: the gap between rows is not written
    buf = torch.full((rows, ld), 7.0, dtype=torch.bfloat16, device=gpu)
    rc = lib().tllm_unembedding_decode_bf16(xg.data_ptr(), w8.data_ptr(), ws.data_ptr(), buf.data_ptr(), ld, rows, hidden, vocab,
                                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    close(buf[:, :vocab], want8)
    assert (buf[:, vocab:] == 7.0).all()


def test_unembedding_32_rows_full_vocabulary(gpu):
    """[201088, 2880] at 32 rows: three or four tiles per wavefront. Logits against the oracle on a sample of columns,
    argmax against planted winners."""
    vocab, rows = 201088, 32
    gg = torch.Generator(device=gpu).manual_seed(5)
    w = torch.empty(vocab, 2880, dtype=torch.bfloat16, device=gpu).normal_(0, 0.02, generator=gg)
    g = torch.Generator().manual_seed(72)
    x = torch.randn(rows, 2880, generator=g).bfloat16()
    planted = torch.randint(0, vocab, (rows,), generator=g)
    planted[:6] = torch.tensor([0, 31, 32, 201087, 201056, 65535])
    for r in range(rows):
        w[planted[r]] = (x[r].float() * 0.05).bfloat16().to(gpu)
    xg = x.view(rows, 1, 2880).to(gpu)
    logits = T.unembedding_decode_forward(xg, w).view(rows, vocab)
    cols = torch.cat([torch.arange(0, 64), torch.arange(100000, 100064), torch.arange(vocab - 64, vocab), planted])
    close(logits[:, cols.to(gpu)], O.linear_ref(x, w[cols.to(gpu)].cpu(), None))
    assert torch.equal(logits.float().argmax(dim=-1).cpu(), planted)
    assert torch.equal(T.unembedding_decode_argmax_forward(xg, w).cpu().long(), planted)


def test_unembedding_full_vocabulary_and_module(gpu, monkeypatch):
    """The real size: [201088, 2880]. Logits against the oracle on a sample of columns (the full fp32 product on
    the CPU would take minutes), argmax against a planted winner, and the module's dispatch."""
    monkeypatch.delenv("UNEMBED_FP8", raising=False)
    vocab, rows = 201088, 8
    gg = torch.Generator(device=gpu).manual_seed(3)
    mod = T.UnEmbedding(2880, vocab, device=gpu)
    with torch.no_grad():
        mod.weight.normal_(0, 0.02, generator=gg)
    g = torch.Generator().manual_seed(71)
    x = torch.randn(rows, 2880, generator=g).bfloat16()
    planted = torch.tensor([0, 31, 32, 100000, 201087, 77777, 12345, 201056])
    with torch.no_grad():
        for r in range(rows):                                  # row r of x points at weight row planted[r]
            mod.weight[planted[r]] = (x[r].float() * 0.05).bfloat16().to(gpu)
    xg = x.view(rows, 1, 2880).to(gpu)
    logits = mod(xg).clone()
    assert logits.shape == (rows, 1, vocab)
    cols = torch.cat([torch.arange(0, 64), torch.arange(100000, 100064), torch.arange(vocab - 64, vocab), planted])
    close(logits.view(rows, vocab)[:, cols.to(gpu)], O.linear_ref(x, mod.weight.detach()[cols.to(gpu)].cpu(), None))
    ids = mod.forward_argmax(xg)
    assert torch.equal(ids.cpu().long(), planted)
    assert torch.equal(logits.view(rows, vocab).float().argmax(dim=-1).cpu(), planted)
    # prefill-shaped input goes to the library GEMM like the reference's module
    y = mod(torch.zeros(1, 3, 2880, dtype=torch.bfloat16, device=gpu))
    assert y.shape == (1, 3, vocab)
    # fp8 copy under UNEMBED_FP8
    monkeypatch.setenv("UNEMBED_FP8", "1")
    mod8 = T.UnEmbedding(2880, vocab, device=gpu)
    with torch.no_grad():
        mod8.weight.copy_(mod.weight)
    assert torch.equal(mod8.forward_argmax(xg).cpu().long(), planted)
    w8, ws = mod8._fp8()
    l8 = mod8(xg)
    close(l8.view(rows, vocab)[:, cols.to(gpu)], O.linear_ref(x, O.dequant_fp8_ref(w8[cols.to(gpu)].cpu(), ws[cols.to(gpu)].cpu()), None))
    with pytest.raises(AssertionError):
        T.unembedding_decode_forward(torch.zeros(2, 2, 2880, dtype=torch.bfloat16, device=gpu), mod.weight)


# ----------------------------------------------------------------------------------- decode attention
def _attn_case(gpu, batch_size, num_keys, sliding_window, start_q, start_dtype=torch.int32, seed=0, with_sinks=True, groups=8, kv_heads=8):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(batch_size, 1, kv_heads, groups, 64, generator=g).bfloat16()
    k = torch.randn(batch_size, num_keys, kv_heads, 64, generator=g).bfloat16()
    v = torch.randn(batch_size, num_keys, kv_heads, 64, generator=g).bfloat16()
    sinks = torch.randn(kv_heads * groups, generator=g).bfloat16() if with_sinks else None
    o1 = T.attention_decode(q.to(gpu), k.to(gpu), v.to(gpu), sinks.to(gpu) if with_sinks else None, 0.125, sliding_window,
                            torch.tensor([start_q], dtype=start_dtype, device=gpu))
    o2 = O.attention_decode_ref(q, k, v, sinks, 0.125, sliding_window, start_q)
    assert o1.shape == (batch_size, 1, kv_heads * groups * 64) and o1.dtype == torch.bfloat16
    # the reference's own bar (attention_tt_decode.py:429, 454) ...
    torch.testing.assert_close(o1.float().cpu(), o2.bfloat16().float(), atol=1e-2, rtol=1e-1)
    # ... and the tolerance of the other bf16 outputs of this library
    close(o1, o2)


@pytest.mark.parametrize("batch_size", [1, 2])
@pytest.mark.parametrize("num_keys", [128, 1024])
@pytest.mark.parametrize("sliding_window", [None, 128])
@pytest.mark.parametrize("start_q", [0, 5, 63])
def test_attention_decode_eq(gpu, batch_size, num_keys, sliding_window, start_q):
    """The reference's test_decode_eq (attention_tt_decode.py:413-429), same parameter grid."""
    _attn_case(gpu, batch_size, num_keys, sliding_window, start_q, seed=start_q + num_keys)


@pytest.mark.parametrize("batch_size", [1, 2])
@pytest.mark.parametrize("num_keys", [2048, 4096])
@pytest.mark.parametrize("sliding_window", [None, 2048])
@pytest.mark.parametrize("start_q", [0, 1023, 2047])
def test_attention_decode_splitk(gpu, batch_size, num_keys, sliding_window, start_q):
    """The reference's test_decode_splitk (attention_tt_decode.py:432-454): long contexts, split over workgroups."""
    _attn_case(gpu, batch_size, num_keys, sliding_window, start_q, seed=start_q + num_keys)


def test_attention_decode_edges(gpu):
    _attn_case(gpu, 8, 4096, None, 4095, start_dtype=torch.int64, seed=1)       # full cache, int64 offset as the model passes it
    _attn_case(gpu, 3, 4096, 128, 3000, start_dtype=torch.int64, seed=2)        # sliding window deep into a long cache
    _attn_case(gpu, 1, 777, None, 776, seed=3)                                  # ragged last block
    _attn_case(gpu, 2, 300, 128, 299, seed=4, with_sinks=False)                 # sinks=None -> logit 0 (attention_tt_decode.py:55-58)
    _attn_case(gpu, 2, 256, None, 10000, seed=5)                                # start_q beyond the cache: every key is visible
    _attn_case(gpu, 2, 200, None, 150, seed=6, groups=4)                        # another group size
    # strided cache views (a cache allocated for more tokens than are handed over)
    g = torch.Generator().manual_seed(7)
    q = torch.randn(2, 1, 8, 8, 64, generator=g).bfloat16()
    kc = torch.randn(2, 512, 8, 64, generator=g).bfloat16()
    vc = torch.randn(2, 512, 8, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    o1 = T.attention_decode(q.to(gpu), kc.to(gpu)[:, :300], vc.to(gpu)[:, :300], sinks.to(gpu), 0.125, None, torch.tensor([299], device=gpu))
    close(o1, O.attention_decode_ref(q, kc[:, :300], vc[:, :300], sinks, 0.125, None, 299))
    with pytest.raises(AssertionError):
        T.attention_decode(q.to(gpu).expand(-1, 2, -1, -1, -1), kc.to(gpu), vc.to(gpu), sinks.to(gpu), 0.125, None, torch.tensor([1], device=gpu))


@pytest.mark.parametrize("case", [
    dict(batch_size=8, num_keys=32768, sliding_window=None, start_q=32767, hpw=4),        # 16 splits of 2048 keys, four heads per workgroup
    dict(batch_size=256, num_keys=4128, sliding_window=None, start_q=4127, groups=1, hpw=8),   # eight heads per workgroup, two splits
    dict(batch_size=8, num_keys=8192, sliding_window=None, start_q=8191, hpw=4),          # four heads per workgroup, 16 splits
    dict(batch_size=8, num_keys=8192, sliding_window=None, start_q=8000, start_dtype=torch.int64, hpw=4),   # ragged last split
    dict(batch_size=8, num_keys=8192, sliding_window=None, start_q=100, hpw=4),           # most splits hold no key at all
    dict(batch_size=8, num_keys=8192, sliding_window=None, start_q=0, hpw=4),             # one key
    dict(batch_size=16, num_keys=8192, sliding_window=4096, start_q=7000, hpw=4),         # window under the split planning
    dict(batch_size=256, num_keys=600, sliding_window=None, start_q=599, hpw=8),          # one split: written straight to the output
    dict(batch_size=256, num_keys=600, sliding_window=None, start_q=580, with_sinks=False, hpw=8),
    dict(batch_size=64, num_keys=2048, sliding_window=None, start_q=2047, kv_heads=4, groups=2, hpw=4),    # a model with four KV heads
    dict(batch_size=32, num_keys=4096, sliding_window=None, start_q=4000, kv_heads=16, groups=4, hpw=4),   # sixteen KV heads: four groups of four
], ids=lambda c: "-".join(f"{k[0]}{v}" for k, v in c.items() if not isinstance(v, torch.dtype)))
def test_attention_decode_row_workgroups(gpu, case):
    """Large batch x context: the workgroup shape with one wavefront per KV head over groups of eight or four heads
    (chosen inside the library from batch, heads and context; each case states the grouping it expects)."""
    from tritonllm_amd._lib import lib
    c = dict(case)
    hpw = c.pop("hpw")
    assert lib().tllm_attention_decode_heads_per_workgroup(c["batch_size"], c.get("kv_heads", 8), c["num_keys"], c["sliding_window"] or 0) == hpw
    _attn_case(gpu, seed=11 + c["start_q"], **c)


@pytest.mark.parametrize("batch_size,num_keys,start_q,hpw", [
    (1, 129, 128, 0), (1, 512, 511, 0), (3, 200, 37, 0), (8, 640, 639, 0), (8, 800, 799, 0), (12, 800, 799, 0),        # eight wavefronts per KV head; less than a block each
    (33, 256, 255, 2), (64, 1280, 1279, 2), (49, 1111, 1110, 2), (43, 4096, 30, 2),   # two heads, two wavefronts each: ragged, nearly empty
    (8, 3000, 2999, 2), (16, 1111, 700, 2),                                           # ... with context splits
    (65, 100, 99, 4), (97, 333, 332, 4), (111, 515, 31, 4), (128, 511, 0, 4),         # four heads, two wavefronts each
])
@pytest.mark.parametrize("kv", [dict(), dict(groups=5, with_sinks=False)], ids=["g8", "g5"])
def test_attention_decode_wavefronts_per_head(gpu, batch_size, num_keys, start_q, hpw, kv):
    """Workgroup shapes with several wavefronts per KV head, at the edges of the ranges that take them."""
    from tritonllm_amd._lib import lib
    assert lib().tllm_attention_decode_heads_per_workgroup(batch_size, 8, num_keys, 0) == hpw
    _attn_case(gpu, batch_size, num_keys, None, start_q, seed=batch_size + num_keys, **kv)


@pytest.mark.parametrize("batch_size,window", [(65, 128), (40, 300), (6, 200)])
def test_attention_decode_window_wavefronts_per_head(gpu, batch_size, window):
    """... and under a sliding window, whose first block is ragged too."""
    _attn_case(gpu, batch_size, 700, window, 613, seed=window)


@pytest.mark.parametrize("batch_size,num_keys", [(2, 600), (8, 8192)])
def test_attention_decode_strided_cache_views(gpu, batch_size, num_keys):
    """K / V handed over as views of a larger allocation: more tokens and more heads per token than are used, so both
    the batch stride and the token stride differ from the dense ones (small case: one KV head per workgroup; large
    case: the row-shaped workgroups, whose wavefronts then read 8 of every 10 heads' worth of each cache row)."""
    g = torch.Generator().manual_seed(batch_size + num_keys)
    q = torch.randn(batch_size, 1, 8, 8, 64, generator=g).bfloat16()
    kc = torch.randn(batch_size, num_keys + 100, 10, 64, generator=g).bfloat16()
    vc = torch.randn(batch_size, num_keys + 100, 10, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    kg, vg = kc.to(gpu)[:, :num_keys, 1:9], vc.to(gpu)[:, :num_keys, 1:9]
    assert kg.stride(1) == 640 and not kg.is_contiguous()
    o1 = T.attention_decode(q.to(gpu), kg, vg, sinks.to(gpu), 0.125, None, torch.tensor([num_keys - 1], device=gpu))
    close(o1, O.attention_decode_ref(q, kc[:, :num_keys, 1:9], vc[:, :num_keys, 1:9], sinks, 0.125, None, num_keys - 1))


@pytest.mark.parametrize("batch_size,cache,start_q", [(8, 32768, 4095), (8, 32768, 1000), (8, 32768, 31), (1, 32768, 4095),
                                                      (2, 16384, 8000), (16, 8192, 2500)])
@pytest.mark.parametrize("hint", [None, "exact", "small", "large"])
def test_attention_decode_short_context_in_a_large_cache(gpu, batch_size, cache, start_q, hint):
    """K / V are the whole preallocated cache and the context is a fraction of it: the launch is planned for the cache
    (or for the hint), the kernels use the splits the context needs. The result does not depend on the hint, whether
    it is right, far too small or too large."""
    g = torch.Generator().manual_seed(batch_size + start_q)
    q = torch.randn(batch_size, 1, 8, 8, 64, generator=g).bfloat16()
    k = torch.randn(batch_size, start_q + 1, 8, 64, generator=g).bfloat16()
    v = torch.randn(batch_size, start_q + 1, 8, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    kc = torch.full((batch_size, cache, 8, 64), float("nan"), dtype=torch.bfloat16, device=gpu)   # unused slots must never be read into a result
    vc = torch.full((batch_size, cache, 8, 64), float("nan"), dtype=torch.bfloat16, device=gpu)
    kc[:, :start_q + 1] = k.to(gpu)
    vc[:, :start_q + 1] = v.to(gpu)
    h = {None: None, "exact": start_q + 1, "small": 100, "large": 10 * cache}[hint]
    o1 = T.attention_decode(q.to(gpu), kc, vc, sinks.to(gpu), 0.125, None, torch.tensor([start_q], dtype=torch.int64, device=gpu),
                            kv_len_hint=h)
    close(o1, O.attention_decode_ref(q, k, v, sinks, 0.125, None, start_q))


def _attn_prefill_case(gpu, batch_size, num_queries, num_keys, sliding_window, start_q, start_dtype=torch.int32, seed=0, with_sinks=True,
                       groups=8, kv_heads=8):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(batch_size, num_queries, kv_heads, groups, 64, generator=g).bfloat16()
    k = torch.randn(batch_size, num_keys, kv_heads, 64, generator=g).bfloat16()
    v = torch.randn(batch_size, num_keys, kv_heads, 64, generator=g).bfloat16()
    sinks = torch.randn(kv_heads * groups, generator=g).bfloat16() if with_sinks else None
    o1 = T.attention(q.to(gpu), k.to(gpu), v.to(gpu), sinks.to(gpu) if with_sinks else None, 0.125, sliding_window,
                     torch.tensor([start_q], dtype=start_dtype, device=gpu))
    o2 = O.attention_ref(q, k, v, sinks, 0.125, sliding_window, start_q)
    assert o1.shape == (batch_size, num_queries, kv_heads * groups * 64) and o1.dtype == torch.bfloat16
    # the reference's own bar (attention_tt.py:268) and the tolerance of the other bf16 outputs of this library
    torch.testing.assert_close(o1.float().cpu(), o2.bfloat16().float(), atol=1e-2, rtol=1e-1)
    close(o1, o2)


@pytest.mark.parametrize("batch_size", [1, 2])
@pytest.mark.parametrize("num_queries", [1, 16])
@pytest.mark.parametrize("num_keys", [128, 32])
@pytest.mark.parametrize("sliding_window", [None, 128])
@pytest.mark.parametrize("start_q", [0, 5])
def test_attention_prefill_eq(gpu, batch_size, num_queries, num_keys, sliding_window, start_q):
    """The reference's test_eq (attention_tt.py:245-268), same parameter grid."""
    _attn_prefill_case(gpu, batch_size, num_queries, num_keys, sliding_window, start_q, seed=start_q + num_keys + num_queries)


@pytest.mark.parametrize("case", [
    dict(batch_size=1, num_queries=300, num_keys=300, sliding_window=None, start_q=0),            # ragged last tile and block
    dict(batch_size=2, num_queries=257, num_keys=257, sliding_window=128, start_q=0),             # the model's sliding layers
    dict(batch_size=1, num_queries=1024, num_keys=1024, sliding_window=128, start_q=0),
    dict(batch_size=1, num_queries=200, num_keys=1000, sliding_window=None, start_q=800, start_dtype=torch.int64),   # a later chunk of a long prompt
    dict(batch_size=1, num_queries=200, num_keys=1000, sliding_window=100, start_q=800),
    dict(batch_size=2, num_queries=130, num_keys=400, sliding_window=None, start_q=100),          # keys beyond the last query are never visible
    dict(batch_size=1, num_queries=100, num_keys=60, sliding_window=None, start_q=0),             # fewer keys than positions
    dict(batch_size=1, num_queries=100, num_keys=60, sliding_window=16, start_q=30),              # the last queries see no key at all: zeros
    dict(batch_size=2, num_queries=150, num_keys=150, sliding_window=None, start_q=0, with_sinks=False),
    dict(batch_size=2, num_queries=150, num_keys=150, sliding_window=64, start_q=0, groups=3),    # odd group: one head per wavefront
    dict(batch_size=1, num_queries=150, num_keys=150, sliding_window=None, start_q=0, groups=1, kv_heads=4),
    dict(batch_size=3, num_queries=129, num_keys=140, sliding_window=None, start_q=11, groups=4, kv_heads=2),
], ids=lambda c: "-".join(f"{k[0]}{v}" for k, v in c.items() if not isinstance(v, torch.dtype)))
def test_attention_prefill_shapes(gpu, case):
    _attn_prefill_case(gpu, seed=3 + case["num_queries"] + case["start_q"], **case)


@pytest.mark.parametrize("batch_size,num_queries,num_keys,start_q,window", [
    (1, 1, 193, 192, None), (1, 33, 260, 200, None), (1, 97, 1597, 1500, None), (2, 128, 448, 320, None), (4, 64, 700, 1, None),   # four key groups
    (1, 97, 1597, 1500, 128), (1, 200, 1000, 800, 1), (2, 100, 800, 333, 300),
    (1, 64, 192, 128, None), (1, 65, 65, 0, None), (1, 257, 300, 40, None), (8, 64, 100, 9, None), (3, 129, 1200, 1071, 200),      # two
], ids=str)
@pytest.mark.parametrize("kv", [dict(), dict(groups=3, kv_heads=4, with_sinks=False)], ids=["g8", "g3"])
def test_attention_prefill_key_groups(gpu, batch_size, num_queries, num_keys, start_q, window, kv):
    """Launches of at most two workgroups of 64 queries x 1 head per CU: the key blocks are shared out between wavefronts,
    from fewer blocks than groups to many of them, the last round ragged, a group with nothing visible among them."""
    _attn_prefill_case(gpu, batch_size, num_queries, num_keys, window, start_q, seed=num_queries + num_keys, **kv)


@pytest.mark.parametrize("window", [None, 128])
def test_attention_prefill_odd_group_large_launch(gpu, window):
    """Three query heads per KV head, more than two workgroups of 64 queries x 1 head per CU: 128 queries of one head each."""
    assert _lib.lib().tllm_attention_prefill_key_groups(1, 1500, 1500, 8, 3, window or 0) == 1
    _attn_prefill_case(gpu, 1, 1500, 1500, window, 0, groups=3, seed=15)


@pytest.mark.parametrize("batch_size,num_keys,kv_heads,plan", [(33, 1400, 16, (4, 2)), (19, 1400, 32, (8, 3))])
def test_attention_decode_more_than_eight_kv_heads(gpu, batch_size, num_keys, kv_heads, plan):
    L = _lib.lib()
    assert (L.tllm_attention_decode_heads_per_workgroup(batch_size, kv_heads, num_keys, 0), L.tllm_attention_decode_splits(batch_size, kv_heads, num_keys, 0)) == plan
    _attn_case(gpu, batch_size, num_keys, None, num_keys - 1, groups=2, kv_heads=kv_heads, seed=batch_size)


def test_attention_prefill_views_of_the_qkv_buffer_and_the_cache(gpu):
    """q as a slice of the fused projection output, k / v as slices of a larger cache whose other slots hold NaN: the
    kernel reads them in place (batch and token strides) and never touches a key no query can see."""
    g = torch.Generator().manual_seed(21)
    bs, n_tok, start = 2, 200, 40
    qkv = torch.randn(bs, n_tok, 5120, generator=g).bfloat16()
    kc = torch.full((bs, 512, 10, 64), float("nan")).bfloat16()
    vc = torch.full((bs, 512, 10, 64), float("nan")).bfloat16()
    kc[:, : start + n_tok, 1:9] = torch.randn(bs, start + n_tok, 8, 64, generator=g).bfloat16()
    vc[:, : start + n_tok, 1:9] = torch.randn(bs, start + n_tok, 8, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    q = qkv[:, :, :4096].view(bs, n_tok, 8, 8, 64)
    qg = qkv.to(gpu)[:, :, :4096].view(bs, n_tok, 8, 8, 64)
    assert not qg.is_contiguous()
    kg, vg = kc.to(gpu)[:, :, 1:9], vc.to(gpu)[:, :, 1:9]
    for window in (None, 128):
        o1 = T.attention(qg, kg, vg, sinks.to(gpu), 0.125, window, torch.tensor([start], device=gpu))
        o2 = O.attention_ref(q, kc[:, : start + n_tok, 1:9], vc[:, : start + n_tok, 1:9], sinks, 0.125, window, start)
        close(o1, o2)


def test_attention_prefill_full_prompt(gpu):
    """The benchmark shape: one prompt of 2048 tokens, 64 query heads over 8 KV heads, both kinds of layer."""
    _attn_prefill_case(gpu, 1, 2048, 2048, None, 0, seed=31)
    _attn_prefill_case(gpu, 1, 2048, 2048, 128, 0, seed=32)


@pytest.mark.parametrize("sliding_window", [None, 128])
def test_attention_prefill_large_launch_ragged(gpu, sliding_window):
    """Enough workgroups for 64 queries x four heads, two per wavefront (the library picks the workgroup shape from
    the size of the launch), with a ragged last tile, a later chunk of the prompt and keys beyond the last query."""
    _attn_prefill_case(gpu, 4, 600, 700, sliding_window, 77, start_dtype=torch.int64, seed=41)


def _prefill_shape(*sizes):
    shape = _lib.lib().tllm_attention_prefill_shape(*sizes)
    return shape >> 24, shape >> 16 & 255, shape >> 8 & 255, shape & 255          # in chunks, queries, query heads, key groups


@pytest.mark.parametrize("batch_size,num_queries,num_keys,start_q,window,kv,shape", [
    (1, 777, 777, 0, None, dict(), (64, 2)),                                   # one head per wavefront
    (1, 833, 1200, 310, 322, dict(), (64, 2)),                                 # the window's edge inside blocks; keys beyond the last query
    (2, 450, 1100, 520, 400, dict(), (64, 2)),
    (1, 600, 448, 0, None, dict(with_sinks=False), (64, 2)),                   # as short as walks in chunks get; queries past the keys
    (8, 128, 2048, 0, None, dict(), (64, 2)), (5, 60, 1500, 700, None, dict(kv_heads=16), (64, 2)),       # a cache larger than what is walked
    (4, 600, 700, 77, 400, dict(), (64, 4)),                                   # two per wavefront
    (3, 449, 640, 191, 333, dict(groups=4, kv_heads=16), (64, 4)),
    (9, 650, 700, 49, None, dict(groups=2), (128, 2)), (6, 700, 777, 40, 350, dict(groups=6, kv_heads=4), (128, 2)),
    (2, 1000, 1100, 100, 400, dict(groups=5), (128, 1)), (1, 777, 900, 123, None, dict(groups=7), (128, 1)),
], ids=str)
def test_attention_prefill_chunks(gpu, batch_size, num_queries, num_keys, start_q, window, kv, shape):
    """Keys of more than six blocks and no narrower window: in chunks of 32 keys x one head, in every shape of workgroup."""
    assert _prefill_shape(batch_size, num_queries, num_keys, kv.get("kv_heads", 8), kv.get("groups", 8), window or 0) == (1, *shape, 1)
    _attn_prefill_case(gpu, batch_size, num_queries, num_keys, window, start_q, seed=num_queries + num_keys, **kv)


@pytest.mark.parametrize("batch_size,num_queries,num_keys,start_q,window,kv,shape", [
    (1, 833, 1200, 310, 257, dict(), (64, 2)), (3, 449, 640, 191, 321, dict(groups=4, kv_heads=16), (64, 4)),
    (4, 600, 700, 77, 128, dict(), (64, 4)),
    (8, 650, 700, 49, 128, dict(groups=2), (128, 2)), (8, 380, 384, 4, None, dict(groups=2, kv_heads=16), (128, 2)),
    (6, 700, 777, 40, 130, dict(groups=6, kv_heads=4), (128, 2)),
    (2, 1000, 1100, 100, 300, dict(groups=5), (128, 1)),
], ids=str)
def test_attention_prefill_short_walks(gpu, batch_size, num_queries, num_keys, start_q, window, kv, shape):
    """Up to six blocks of keys, or a window of up to 321, in every shape of workgroup."""
    assert _prefill_shape(batch_size, num_queries, num_keys, kv.get("kv_heads", 8), kv.get("groups", 8), window or 0) == (0, *shape, 1)
    _attn_prefill_case(gpu, batch_size, num_queries, num_keys, window, start_q, seed=num_queries + num_keys, **kv)


@pytest.mark.parametrize("batch_size,num_queries", [(1, 777), (4, 600)])
def test_attention_prefill_growing_logits(gpu, batch_size, num_queries):
    """Keys that grow along the context, so that block after block tops what the weights are taken relative to by far more than
    2^8; and one query of nan, which stays alone."""
    g = torch.Generator().manual_seed(77)
    q = torch.randn(batch_size, num_queries, 8, 8, 64, generator=g).bfloat16()
    k = (torch.randn(batch_size, num_queries, 8, 64, generator=g) * torch.linspace(0.1, 60.0, num_queries)[None, :, None, None]).bfloat16()
    v = torch.randn(batch_size, num_queries, 8, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    q[0, 40] = float("nan")
    o1 = T.attention(q.to(gpu), k.to(gpu), v.to(gpu), sinks.to(gpu), 0.125, None, torch.tensor([0], device=gpu)).float().cpu()
    o2 = O.attention_ref(q, k, v, sinks, 0.125, None, 0).float()
    assert o1[0, 40].isnan().all()
    o1[0, 40] = o2[0, 40] = 0.0
    close(o1, o2)


def test_attention_graph_replay_follows_device_start(gpu):
    """Both attention kernels read start_q on the device: a graph captured once follows the tensor's new value on every
    replay (decode: the growing context; prefill: the next chunk of a prompt), with eager work between the replays."""
    g = torch.Generator().manual_seed(61)
    bs, n_ctx, chunk = 2, 700, 150
    k = torch.randn(bs, n_ctx, 8, 64, generator=g).bfloat16()
    v = torch.randn(bs, n_ctx, 8, 64, generator=g).bfloat16()
    q1 = torch.randn(bs, 1, 8, 8, 64, generator=g).bfloat16()
    qn = torch.randn(bs, chunk, 8, 8, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    kg, vg, q1g, qng, sg = k.to(gpu), v.to(gpu), q1.to(gpu), qn.to(gpu), sinks.to(gpu)
    start = torch.zeros(1, dtype=torch.int64, device=gpu)
    outs = {}

    def both():
        outs["dec"] = T.attention_decode(q1g, kg, vg, sg, 0.125, None, start)
        outs["pre"] = T.attention(qng, kg, vg, sg, 0.125, 128, start)

    both()                                        # warm up (allocates pool buffers)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        both()
    for p in (0, 37, 300, 549, 37):
        start.fill_(p)
        graph.replay()
        torch.cuda.synchronize()
        close(outs["dec"], O.attention_decode_ref(q1, k, v, sinks, 0.125, None, p))
        close(outs["pre"], O.attention_ref(qn, k, v, sinks, 0.125, 128, p))
        T.rmsnorm_forward(qng.view(-1, 4096)[:4], torch.ones(4096, device=gpu), 1e-5)   # eager work between the replays


def test_attention_prefill_argument_errors(gpu):
    q = torch.zeros(1, 16, 8, 8, 64, dtype=torch.bfloat16, device=gpu)
    k = torch.zeros(1, 16, 8, 64, dtype=torch.bfloat16, device=gpu)
    s = torch.zeros(64, dtype=torch.bfloat16, device=gpu)
    st = torch.tensor([0], device=gpu)
    with pytest.raises(AssertionError):
        T.attention(q, k, k[:, :8], s, 0.125, None, st)                       # k and v disagree
    with pytest.raises(AssertionError):
        T.attention(q, k, k, s[:32], 0.125, None, st)                         # one sink per query head
    with pytest.raises((AssertionError, RuntimeError)):
        T.attention(q, k, k, s, -0.125, None, st)                             # the kernel folds the scale into exp2: positive only
    assert T.attention(q[:, :0], k, k, s, 0.125, None, st).shape == (1, 0, 4096)


def test_attention_block_decode_chain(gpu):
    """The whole attention block of a decode step as model.py:471-573 strings it together -- RMSNorm, QKV + bias + RoPE
    with the new k/v written into the cache at `offset`, attention over the cache with sinks (full and windowed),
    out-projection + bias + residual -- every stage on the HIP kernels, against the oracle chain."""
    bs, n_ctx, slot = 4, 300, 207
    d = O.make_inputs(bs, seed=81)
    g = torch.Generator().manual_seed(82)
    cache_k = torch.randn(bs, n_ctx, 8, 64, generator=g).bfloat16()
    cache_v = torch.randn(bs, n_ctx, 8, 64, generator=g).bfloat16()
    sinks = torch.randn(64, generator=g).bfloat16()
    w_out = (0.02 * torch.randn(2880, 4096, generator=g)).bfloat16()
    b_out = (0.02 * torch.randn(2880, generator=g)).bfloat16()
    rope = T.RotaryEmbedding(64, 150000, torch.float32, initial_context_length=4096, scaling_factor=32.0, device=gpu)
    offset = torch.tensor([slot], dtype=torch.int64, device=gpu)
    for window in (None, 128):
        ck, cv = cache_k.to(gpu), cache_v.to(gpu)
        x = d["x"].view(bs, 1, 2880).to(gpu)
        q = T.qkv_rope_cache_decode_forward(x, d["w"].to(gpu), d["b"].to(gpu), rope.sin, rope.cos, rope.max_context_length, ck, cv, offset,
                                            64, 8, 64, norm_scale=d["norm_scale"].to(gpu), norm_eps=1e-5)
        t = T.attention_decode(q.view(bs, 1, 8, 8, 64), ck, cv, sinks.to(gpu), 0.125, window, offset)
        y = T.out_residual_decode_forward(t, w_out.to(gpu), b_out.to(gpu), x.clone())
        # oracle chain, rounding to bf16 wherever a tensor crosses from one reference kernel to the next
        tn = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16()
        qr, kr, vr = O.qkv_rope_ref(tn, d["w"], d["b"], torch.full((bs,), slot, dtype=torch.int64))
        rk, rv = cache_k.clone(), cache_v.clone()
        rk[:, slot] = kr.bfloat16().view(bs, 8, 64)
        rv[:, slot] = vr.bfloat16().view(bs, 8, 64)
        tr = O.attention_decode_ref(qr.bfloat16().view(bs, 1, 8, 8, 64), rk, rv, sinks, 0.125, window, slot).bfloat16()
        yr = O.out_residual_ref(tr.view(bs, 4096), w_out, b_out, d["x"])
        close(t, tr.float())
        close(y.view(bs, 2880), yr)


def test_attention_block_prefill_chain(gpu):
    """The attention block of a prompt, in two chunks, as model.py:471-573 strings it together: RMSNorm, QKV + bias +
    RoPE with k / v written straight into the cache rows of the chunk, attention of the chunk's queries (read in place
    from the projection's output) over the cache so far, with sinks, full and windowed -- against the oracle chain."""
    n_ctx, chunk = 512, 200
    g = torch.Generator().manual_seed(91)
    sinks = torch.randn(64, generator=g).bfloat16()
    yarn = T.gpt_oss_yarn()
    for window in (None, 128):
        ck = torch.full((1, n_ctx, 8, 64), float("nan"), dtype=torch.bfloat16, device=gpu)     # slots never written stay NaN
        cv = torch.full((1, n_ctx, 8, 64), float("nan"), dtype=torch.bfloat16, device=gpu)
        rk = torch.zeros(1, 2 * chunk, 8, 64, dtype=torch.bfloat16)
        rv = torch.zeros(1, 2 * chunk, 8, 64, dtype=torch.bfloat16)
        for part in range(2):
            start = part * chunk
            d = O.make_inputs(chunk, seed=92 + part)
            pos = torch.arange(start, start + chunk, dtype=torch.int64)
            tn = T.rmsnorm_forward(d["x"].to(gpu), d["norm_scale"].to(gpu), 1e-5)
            q = torch.empty(chunk, 4096, dtype=torch.bfloat16, device=gpu)
            T.qkv_rope_forward(tn, d["w"].to(gpu), d["b"].to(gpu), 64, 8, 64, yarn=yarn, positions=pos.to(gpu), mode="prefill",
                               out=(q, ck[0, start:start + chunk].view(chunk, 512), cv[0, start:start + chunk].view(chunk, 512)))
            t = T.attention(q.view(1, chunk, 8, 8, 64), ck, cv, sinks.to(gpu), 0.125, window, torch.tensor([start], dtype=torch.int64, device=gpu))
            # oracle chain, rounding to bf16 wherever a tensor crosses from one reference kernel to the next
            tr = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16()
            qr, kr, vr = O.qkv_rope_ref(tr, d["w"], d["b"], pos)
            rk[0, start:start + chunk] = kr.bfloat16().view(chunk, 8, 64)
            rv[0, start:start + chunk] = vr.bfloat16().view(chunk, 8, 64)
            want = O.attention_ref(qr.bfloat16().view(1, chunk, 8, 8, 64), rk[:, :start + chunk], rv[:, :start + chunk], sinks, 0.125, window, start)
            close(ck[0, start:start + chunk].view(chunk, 512), kr)
            close(t, want)


@pytest.mark.parametrize("n_tokens", [1, 8, 300, 512, 513, 2048])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
def test_embedding_rmsnorm_one_launch(gpu, n_tokens, scale_dtype):
    """Gather + RMSNorm of the gathered rows in one launch (both row-count regimes of the norm kernel): the hidden state
    is bit-exact, the normalised rows equal the separate rmsnorm_forward bit for bit and the oracle within tolerance."""
    g = torch.Generator().manual_seed(n_tokens)
    table = (0.02 * torch.randn(5000, 2880, generator=g)).bfloat16()
    scale = (1 + 0.1 * torch.randn(2880, generator=g)).to(scale_dtype)
    for dt in (torch.int32, torch.int64):
        ids = torch.randint(0, 5000, (1, n_tokens), generator=g).to(dt)
        ids[0, 0], ids[0, -1] = 4999, 0
        x, t = T.embedding_rmsnorm_forward(ids.to(gpu), table.to(gpu), scale.to(gpu), 1e-5)
        assert x.shape == (1, n_tokens, 2880) and t.shape == x.shape
        x_ref = O.embedding_ref(table, ids)
        assert torch.equal(x.cpu(), x_ref)
        assert torch.equal(t, T.rmsnorm_forward(x, scale.to(gpu), 1e-5, out=torch.empty_like(x)))
        close(t, O.rmsnorm_ref(x_ref, scale.float(), 1e-5))


def test_embedding_rmsnorm_bad_ids_and_other_widths(gpu):
    g = torch.Generator().manual_seed(5)
    table = (0.02 * torch.randn(100, 256, generator=g)).bfloat16()
    scale = (1 + 0.1 * torch.randn(256, generator=g)).bfloat16()
    ids = torch.tensor([3, -1, 99, 100, 7], dtype=torch.int64)
    flag = torch.zeros(1, dtype=torch.int32, device=gpu)
    x, t = T.embedding_rmsnorm_forward(ids.to(gpu), table.to(gpu), scale.to(gpu), 1e-5, oob_flag=flag)
    assert flag.item() == 1
    good = torch.tensor([0, 2, 4])
    assert torch.equal(x.cpu()[good], table[ids[good]])
    assert x.cpu()[1].abs().max() == 0 and x.cpu()[3].abs().max() == 0 and t.cpu()[1].abs().max() == 0 and t.cpu()[3].abs().max() == 0
    close(t.cpu()[good], O.rmsnorm_ref(table[ids[good]], scale.float(), 1e-5))
    # a width the fused kernel does not take: composed from the two calls, same results
    table2 = (0.02 * torch.randn(50, 100, generator=g)).bfloat16()
    scale2 = torch.ones(100)
    ids2 = torch.randint(0, 50, (9,), generator=g, dtype=torch.int32)
    x2, t2 = T.embedding_rmsnorm_forward(ids2.to(gpu), table2.to(gpu), scale2.to(gpu), 1e-5)
    assert torch.equal(x2.cpu(), table2[ids2.long()])
    close(t2, O.rmsnorm_ref(table2[ids2.long()], scale2, 1e-5))


# ----------------------------------------------------------------------------------- MXFP4 checkpoint expansion
def _bits_equal_nan_aware(out, ref):
    out = out.cpu()
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(out), nan)
    assert torch.equal(out.view(torch.int16)[~nan], ref.view(torch.int16)[~nan])


def test_mxfp4_every_byte_and_scale(gpu):
    """All 256 byte values under all 256 scale bytes, bit for bit (denormal products at the low scales, inf at the
    top, 0 * inf = nan at scale 255 as torch.ldexp gives in the reference)."""
    blocks = torch.arange(256, dtype=torch.uint8).reshape(1, 16, 16).repeat(256, 1, 1)
    scales = torch.arange(256, dtype=torch.uint8).reshape(256, 1).repeat(1, 16)
    out = T.mxfp4_dequant(blocks.to(gpu), scales.to(gpu))
    assert out.shape == (256, 512) and out.dtype == torch.bfloat16
    _bits_equal_nan_aware(out, O.mxfp4_dequant_ref(blocks, scales))


@pytest.mark.parametrize("shape", [(1, 1), (1, 255), (257, 3), (4, 64, 90), (2, 5, 7, 11)])
def test_mxfp4_shapes(gpu, shape):
    g = torch.Generator().manual_seed(sum(shape))
    blocks = torch.randint(0, 256, (*shape, 16), dtype=torch.uint8, generator=g)
    scales = torch.randint(100, 140, shape, dtype=torch.uint8, generator=g)
    out = T.mxfp4_dequant(blocks.to(gpu), scales.to(gpu))
    assert out.shape == (*shape[:-1], shape[-1] * 32)
    _bits_equal_nan_aware(out, O.mxfp4_dequant_ref(blocks, scales))
    # expansion into a caller's buffer, and non-contiguous inputs
    dst = torch.empty(out.numel(), dtype=torch.bfloat16, device=gpu)
    res = T.mxfp4_dequant(blocks.to(gpu), scales.to(gpu), out=dst)
    assert res.data_ptr() == dst.data_ptr() and torch.equal(res, out)
    if len(shape) >= 2:
        bt = blocks.to(gpu).transpose(0, 1)
        st = scales.to(gpu).transpose(0, 1)
        _bits_equal_nan_aware(T.mxfp4_dequant(bt, st), O.mxfp4_dequant_ref(blocks.transpose(0, 1).contiguous(), scales.transpose(0, 1).contiguous()))


def test_mxfp4_empty(gpu):
    out = T.mxfp4_dequant(torch.empty(0, 3, 16, dtype=torch.uint8, device=gpu), torch.empty(0, 3, dtype=torch.uint8, device=gpu))
    assert out.shape == (0, 96)


def test_mxfp4_moe_weight_shape(gpu):
    """The gpt-oss-20b mlp1 weight, [32 experts, 5760, 2880] stored as [32, 5760, 90, 16] blocks: one expert against
    the oracle, the whole tensor through exact scaling (scale + 1 doubles every value) and block independence."""
    g = torch.Generator(device=gpu).manual_seed(11)
    blocks = torch.randint(0, 256, (32, 5760, 90, 16), dtype=torch.uint8, device=gpu, generator=g)
    scales = torch.randint(110, 130, (32, 5760, 90), dtype=torch.uint8, device=gpu, generator=g)
    out = T.mxfp4_dequant(blocks, scales)
    assert out.shape == (32, 5760, 2880)
    for e in (0, 31):
        _bits_equal_nan_aware(out[e], O.mxfp4_dequant_ref(blocks[e].cpu(), scales[e].cpu()))
    out2 = T.mxfp4_dequant(blocks, scales + 1)
    assert torch.equal(out2, out * 2)
    del out2
    # a reversed copy of the blocks expands to the reversed rows
    flip = T.mxfp4_dequant(blocks.flip(1), scales.flip(1))
    assert torch.equal(flip, out.flip(1))


def test_checkpoint_mxfp4_on_gpu(gpu, tmp_path):
    from safetensors.torch import save_file

    g = torch.Generator().manual_seed(21)
    blocks = torch.randint(0, 256, (4, 96, 6, 16), dtype=torch.uint8, generator=g)
    scales = torch.randint(115, 128, (4, 96, 6), dtype=torch.uint8, generator=g)
    bias = torch.randn(4, 96, generator=g).bfloat16()
    save_file({"block.2.mlp.mlp2_weight.blocks": blocks, "block.2.mlp.mlp2_weight.scales": scales}, str(tmp_path / "a.safetensors"))
    save_file({"block.2.mlp.mlp2_bias": bias}, str(tmp_path / "b.safetensors"))
    ck = T.Checkpoint(str(tmp_path), gpu)
    w = ck.get("block.2.mlp.mlp2_weight")
    assert w.is_cuda and w.shape == (4, 96, 192)
    _bits_equal_nan_aware(w, O.mxfp4_dequant_ref(blocks, scales))
    b = ck.get("block.2.mlp.mlp2_bias")
    assert b.is_cuda and torch.equal(b.cpu(), bias)
    dst = torch.empty(4, 96, 192, dtype=torch.bfloat16, device=gpu)
    assert ck.get("block.2.mlp.mlp2_weight", out=dst) is dst and torch.equal(dst, w)


# ----------------------------------------------------------------------------------- pooled outputs vs inputs
def test_pooled_outputs_never_alias_the_activations(gpu):
    """hidden == n_q_heads * head_dim: the normalised activations (a borrowed pool buffer of shape [rows, hidden]) and q
    have the same size. The projection must not be handed the buffer it is still reading as its output, neither when
    it normalises by a preceding launch itself nor when the caller passes a pooled rmsnorm result as x."""
    rows, hidden, nq, nkv, hd = 12, 4096, 64, 8, 64
    d = O.make_inputs(rows, seed=61, hidden=hidden, n_q_heads=nq, n_kv_heads=nkv, head_dim=hd)
    yarn = T.gpt_oss_yarn()
    t_ref = O.rmsnorm_ref(d["x"], d["norm_scale"].float(), 1e-5).bfloat16()
    qr, kr, vr = O.qkv_rope_ref(t_ref, d["w"], d["b"], d["positions"], n_q_heads=nq, n_kv_heads=nkv, head_dim=hd)
    xg, wg, bg, sg, pg = d["x"].to(gpu), d["w"].to(gpu), d["b"].to(gpu), d["norm_scale"].to(gpu), d["positions"].to(gpu)
    scratch_pool.clear()
    # (a) the call normalises by a preceding launch (this shape has no fused norm)
    q, k, v = T.qkv_rope_forward(xg, wg, bg, nq, nkv, hd, yarn=yarn, positions=pg, mode="decode", norm_scale=sg, norm_eps=1e-5)
    close(q, qr)
    close(k, kr)
    close(v, vr)
    # (b) the caller passes the pooled 2-D output of rmsnorm_forward as x
    t = T.rmsnorm_forward(xg, sg, 1e-5)
    assert t.data_ptr() == scratch_pool.get((rows, hidden), torch.bfloat16, gpu).data_ptr()
    q, k, v = T.qkv_rope_forward(t, wg, bg, nq, nkv, hd, yarn=yarn, positions=pg, mode="decode")
    assert q.data_ptr() != t.data_ptr()
    close(q, qr)
    close(k, kr)
    close(v, vr)
    # (c) the reference-signature decode call with a pooled [B, hidden] buffer viewed as [B, 1, hidden]
    t = T.rmsnorm_forward(xg, sg, 1e-5)
    q3, k3, v3 = T.qkv_decode_forward(t.view(rows, 1, hidden), wg, bg, nq * hd, nkv * hd)
    assert q3.data_ptr() != t.data_ptr()
    lin = O.linear_ref(t_ref, d["w"], d["b"])
    close(q3.view(rows, -1), lin[:, :nq * hd])
    close(k3.view(rows, -1), lin[:, nq * hd:(nq + nkv) * hd])
    close(v3.view(rows, -1), lin[:, (nq + nkv) * hd:])
    scratch_pool.clear()


# ----------------------------------------------------------------------------------- 24-layer per-token stack
N_STACK_LAYERS = 24


@pytest.fixture(scope="module")
def stack_weights(gpu):
    """24 distinct layer weight sets (bf16 N(0, 0.02), norm scales 1 + 0.1 N), seeded on the CPU; the GPU copies are made once."""
    g = torch.Generator().manual_seed(2024)
    cpu = {
        "w": [(0.02 * torch.randn(5120, 2880, generator=g)).bfloat16() for _ in range(N_STACK_LAYERS)],
        "b": [(0.02 * torch.randn(5120, generator=g)).bfloat16() for _ in range(N_STACK_LAYERS)],
        "attn": [(1 + 0.1 * torch.randn(2880, generator=g)).bfloat16() for _ in range(N_STACK_LAYERS)],
        "mlp": [(1 + 0.1 * torch.randn(2880, generator=g)).bfloat16() for _ in range(N_STACK_LAYERS)],
        "final": (1 + 0.1 * torch.randn(2880, generator=g)).bfloat16(),
    }
    dev = {key: ([t.to(gpu) for t in val] if isinstance(val, list) else val.to(gpu)) for key, val in cpu.items()}
    return cpu, dev


def _stack_inputs(batch, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(batch, 2880, generator=g).bfloat16()
    pos = torch.randint(0, 8192, (batch,), generator=g, dtype=torch.int64)
    sx = (2.0 * torch.randn(4 * batch, 5760, generator=g)).bfloat16()
    return x, pos, sx


def _check_stack(stack, final, cpu, x, pos, sx, what):
    """Every layer's q / k / v, MLP-norm output and SwiGLU output, and the final norm, against the oracle."""
    sw_ref = O.swiglu_ref(sx)
    for l in range(N_STACK_LAYERS):
        t_ref = O.rmsnorm_ref(x, cpu["attn"][l].float(), 1e-5).bfloat16()
        qr, kr, vr = O.qkv_rope_ref(t_ref, cpu["w"][l], cpu["b"][l], pos)
        for name, got, want in (("q", stack.q[l], qr), ("k", stack.k[l], kr), ("v", stack.v[l], vr),
                                ("mlp norm", stack.mlp_normed[l], O.rmsnorm_ref(x, cpu["mlp"][l].float(), 1e-5)),
                                ("swiglu", stack.swiglu_out[l], sw_ref)):
            try:
                close(got, want)
            except AssertionError as e:
                raise AssertionError(f"{what}: layer {l} {name}: {e}") from None
    close(final, O.rmsnorm_ref(x, cpu["final"].float(), 1e-5))


@pytest.mark.parametrize("batch", [1, 8, 32])
def test_layer_stack24_token_step(gpu, stack_weights, batch):
    """The whole per-token layer-kernel stack of a 24-layer gpt-oss-20b-shaped model -- per layer attention RMSNorm + QKV
    + bias + YaRN rotary (inside one kernel up to 16 rows, two launches at 32), MLP RMSNorm, SwiGLU on [4B, 5760]; then
    the final RMSNorm (model.py:471-526, 751-757, 918-923) -- with 24 distinct weight sets, run eagerly and as a
    captured HIP graph replayed with new inputs, every layer's outputs against the oracle."""
    from tritonllm_amd.stack import LayerKernelStack

    cpu, dev = stack_weights
    stack = LayerKernelStack(dev["w"], dev["b"], dev["attn"], dev["mlp"], dev["final"], T.gpt_oss_yarn(), batch, keep_layers=True)
    assert stack.launches_per_step() == N_STACK_LAYERS * (3 if batch <= 16 else 4) + 1
    x, pos, sx = _stack_inputs(batch, seed=700 + batch)
    xg, pg, sg = x.to(gpu), pos.to(gpu), sx.to(gpu)
    final = stack.token_step(xg, pg, sg)
    torch.cuda.synchronize()
    _check_stack(stack, final, cpu, x, pos, sx, f"eager B={batch}")

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        final_g = stack.token_step(xg, pg, sg)
    for rep in range(3):
        x, pos, sx = _stack_inputs(batch, seed=800 + 10 * batch + rep)
        for buf in (stack.q, stack.k, stack.v, stack.mlp_normed, stack.swiglu_out, stack.final):
            buf.fill_(float("nan"))                                    # nothing of the previous run may pass for a result
        xg.copy_(x.to(gpu))
        pg.copy_(pos.to(gpu))
        sg.copy_(sx.to(gpu))
        graph.replay()
        torch.cuda.synchronize()
        _check_stack(stack, final_g, cpu, x, pos, sx, f"graph replay {rep} B={batch}")


def test_layer_stack24_shared_buffers_and_unfused_norm(gpu, stack_weights):
    """The form the benchmark times (one output set reused by all layers) leaves the LAST layer's results behind, and the
    stack with the attention norm as its own launch agrees with the fused one."""
    from tritonllm_amd.stack import LayerKernelStack

    cpu, dev = stack_weights
    batch = 8
    x, pos, sx = _stack_inputs(batch, seed=900)
    outs = []
    for fuse in (True, False):
        stack = LayerKernelStack(dev["w"], dev["b"], dev["attn"], dev["mlp"], dev["final"], T.gpt_oss_yarn(), batch, fuse_norm=fuse)
        assert stack.launches_per_step() == N_STACK_LAYERS * (3 if fuse else 4) + 1
        final = stack.token_step(x.to(gpu), pos.to(gpu), sx.to(gpu))
        l = N_STACK_LAYERS - 1
        t_ref = O.rmsnorm_ref(x, cpu["attn"][l].float(), 1e-5).bfloat16()
        qr, kr, vr = O.qkv_rope_ref(t_ref, cpu["w"][l], cpu["b"][l], pos)
        close(stack.q[0], qr)
        close(stack.k[0], kr)
        close(stack.v[0], vr)
        close(stack.mlp_normed[0], O.rmsnorm_ref(x, cpu["mlp"][l].float(), 1e-5))
        close(final, O.rmsnorm_ref(x, cpu["final"].float(), 1e-5))
        outs.append((stack.q[0].clone(), stack.k[0].clone(), stack.v[0].clone()))
    for a, b in zip(*outs):
        close(a, b.float().cpu())
