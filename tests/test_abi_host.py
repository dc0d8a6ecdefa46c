"""CPU-side checks of the C-ABI boundary: the library loads, exports every symbol the
header declares, and rejects bad arguments on the host before anything is launched."""
import copy
import ctypes as C
import os
import pickle
import re
import subprocess
import sys
import threading
from itertools import chain, starmap

import numpy as np
import pytest
import torch

from tritonllm_amd import _lib, scratch_pool
from tritonllm_amd.yarn import YarnParams, gpt_oss_yarn

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_symbols():
    text = open(os.path.join(ROOT, "include", "tllm_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(tllm_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.lib()
    declared = _header_symbols()
    assert declared, "no declarations parsed"
    assert sorted(_lib.SIGNATURES) == declared
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.tllm_abi_version() == _lib.ABI_VERSION


def test_struct_layout_matches_header():
    assert C.sizeof(_lib.TllmYarn) == 128 * 4 + 4 + 4
    assert C.sizeof(_lib.TllmRope) == 8 * 8


def test_yarn_address_is_the_objects_own():
    """Copies of a YarnParams whose C struct has been used hand out their own struct's address."""
    y = gpt_oss_yarn()
    assert y._c_address == C.addressof(y.c_struct())
    for z in (copy.deepcopy(y), pickle.loads(pickle.dumps(y))):
        assert z._c_address == C.addressof(z.c_struct())
        assert bytes(_lib.TllmYarn.from_address(z._c_address)) == bytes(y.c_struct())


def test_scratch_pool_takes_any_integers():
    a = scratch_pool.get((np.int64(3), 5), torch.float32, "cpu")
    assert a.shape == (3, 5) and scratch_pool.get(torch.Size((3, 5)), torch.float32, torch.device("cpu")).data_ptr() == a.data_ptr()


def test_allocation_gives_up_the_interpreter_lock():
    """Another thread runs while the host side allocates (here: while the new buffer is filled). list() draws all three values
    without going back to the interpreter, so nothing else can let the thread in between them."""
    n, stop = [0], threading.Event()

    def count():
        while not stop.is_set():
            n[0] += 1

    thread = threading.Thread(target=count)
    torch.use_deterministic_algorithms(True)
    thread.start()
    try:
        args = ((1 << 27,), torch.float32, torch.device("cpu"))
        before, _, after = list(chain(map(n.__getitem__, [0]), starmap(_lib.host().pool_get, [args]), map(n.__getitem__, [0])))
    finally:
        stop.set()
        thread.join()
        torch.use_deterministic_algorithms(False)
        scratch_pool.clear()
    assert after > before


def test_cpu_buffers_need_no_library():
    """The scratch pool of other devices is torch alone: no library is loaded for it, and any shape that torch has is one. So is
    the out-projection of a prompt, F.linear, under torch's tracers as well."""
    code = '''if True:
        import torch
        from tritonllm_amd import OUT, _lib, scratch_pool
        _lib.LIB_PATH = _lib.HOST_PATH = "/nowhere.so"
        a = scratch_pool.get((2, 3), torch.float32, "cpu")
        assert scratch_pool.get((2, 3), torch.float32, torch.device("cpu")) is a
        assert scratch_pool.get((1,) * 17, torch.float32, "cpu").dim() == 17
        assert scratch_pool.stats() == {"num_buffers": 2, "total_bytes": 28}
        scratch_pool.clear()
        assert scratch_pool.stats() == {"num_buffers": 0, "total_bytes": 0}
        out = OUT(64, 32, device="cpu").requires_grad_(False)
        out.weight.normal_()
        out.bias.normal_()
        x = torch.randn(3, 64).bfloat16()
        want = torch.nn.functional.linear(x, out.weight, out.bias)
        for form in (out, torch.fx.symbolic_trace(out), torch.jit.trace(out, (x,))):
            assert torch.equal(form(x), want)
        '''
    subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True)


def _err():
    return _lib.lib().tllm_last_error().decode()


def test_argument_errors_are_reported_not_launched():
    lib = _lib.lib()
    assert lib.tllm_rmsnorm_bf16(None, None, 0, None, 4, 2880, 1e-5, None) == -1
    assert "null" in _err()
    assert lib.tllm_rmsnorm_bf16(None, None, 0, None, -1, 2880, 1e-5, None) == -1
    assert lib.tllm_rmsnorm_bf16(None, None, 0, None, 0, 2880, 1e-5, None) == 0     # empty input is a no-op
    assert lib.tllm_embedding_bf16(None, None, 0, None, 0, 2880, 10, None, None) == 0
    assert lib.tllm_embedding_bf16(None, None, 0, None, 3, 2880, 10, None, None) == -1
    assert lib.tllm_swiglu_bf16(None, None, 0, 2880, 5760, 1.702, 7.0, 1, 1, None) == 0
    assert lib.tllm_swiglu_bf16(None, None, 2, 2880, 100, 1.702, 7.0, 1, 1, None) == -1
    assert "x_row_stride" in _err()
    rope = _lib.TllmRope()
    assert lib.tllm_rope_bf16(None, None, 0, 64, 8, 64, C.byref(rope), None) == -1   # no yarn, no tables, max_ctx 0
    y = gpt_oss_yarn()
    rope.yarn = y.c_pointer()
    rope.max_ctx = 131072
    rope.tokens_per_batch = 1
    assert lib.tllm_rope_bf16(None, None, 0, 64, 8, 64, C.byref(rope), None) == 0
    assert lib.tllm_rope_bf16(None, None, 0, 64, 8, 128, C.byref(rope), None) == -2  # head_dim vs yarn.n_freq
    assert "n_freq" in _err()
    assert lib.tllm_rope_bf16(None, None, 0, 64, 8, 63, C.byref(rope), None) == -2
    qkv = lib.tllm_qkv_rope_decode_bf16
    assert qkv(None, None, None, None, None, None, 4096, 512, 512, 0, 8, 2880, 64, 8, 64, None, None) == -1
    assert qkv(None, None, None, None, None, None, 4096, 512, 512, 0, 8, 2880, 64, 8, 63, None, None) == -2
    assert lib.tllm_yarn_table_f32(None, None, 0, 0, None, None) == -1


def test_yarn_params_match_closed_form():
    y = gpt_oss_yarn()
    assert y.concentration == pytest.approx(1.3465735902799727, abs=1e-15)
    assert len(y.inv_freq) == 32 and y.inv_freq[0] == 1.0
    for i in (1, 5, 8):
        assert y.inv_freq[i] == pytest.approx(150000.0 ** (-i / 32), rel=2e-6)
    for i in (18, 25, 31):
        assert y.inv_freq[i] == pytest.approx(150000.0 ** (-i / 32) / 32, rel=2e-6)
    s = y.c_struct()
    assert s.n_freq == 32 and s.inv_freq[3] == torch.tensor(y.inv_freq[3], dtype=torch.float32).item()
    plain = YarnParams(head_dim=128, base=10000.0)
    assert plain.concentration == 1.0 and plain.inv_freq[1] == pytest.approx(10000.0 ** (-2 / 128), rel=2e-6)
    with pytest.raises(ValueError):
        YarnParams(head_dim=63, base=10000.0)


def test_yarn_params_agree_with_oracle_bitwise():
    from oracle import layers as O

    conc, inv = O.yarn_concentration_and_inv_freq()
    y = gpt_oss_yarn()
    assert conc == y.concentration
    assert inv.tolist() == list(y.inv_freq)


def test_ops_refuse_cpu_tensors():
    import tritonllm_amd as T

    x = torch.zeros(2, 2880, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="GPU only"):
        T.rmsnorm_forward(x, torch.ones(2880), 1e-5)
    with pytest.raises(RuntimeError, match="GPU only"):
        T.swiglu(torch.zeros(2, 8, dtype=torch.bfloat16))


def test_scratch_pool_returns_same_buffer():
    from tritonllm_amd import scratch_pool

    scratch_pool.clear()
    a = scratch_pool.get((2, 3), torch.float32, torch.device("cpu"))
    b = scratch_pool.get((2, 3), torch.float32, torch.device("cpu"))
    c = scratch_pool.get((2, 4), torch.float32, torch.device("cpu"))
    assert a.data_ptr() == b.data_ptr() and a.data_ptr() != c.data_ptr()
    assert scratch_pool.stats()["num_buffers"] == 2
    scratch_pool.clear()


def test_checkpoint_names_and_plain_tensors(tmp_path):
    """Host logic of the checkpoint reader (reference weights.py:17-66): key discovery over several files, the MoE
    name mapping, plain tensors on the CPU, and no CPU expansion of MXFP4 data."""
    from safetensors.torch import save_file

    from tritonllm_amd.weights import Checkpoint, _param_names

    assert _param_names("block.0.mlp.mlp1_weight") == ("block.0.mlp.mlp1_weight.blocks", "block.0.mlp.mlp1_weight.scales")
    assert _param_names("block.35.mlp.mlp2_weight") == ("block.35.mlp.mlp2_weight.blocks", "block.35.mlp.mlp2_weight.scales")
    assert _param_names("block.36.mlp.mlp2_weight") == "block.36.mlp.mlp2_weight"       # the reference maps 36 blocks
    assert _param_names("block.3.mlp.mlp1_bias") == "block.3.mlp.mlp1_bias"
    assert _param_names("block.3.attn.qkv.weight") == "block.3.attn.qkv.weight"
    assert _param_names("embedding.weight") == "embedding.weight"

    g = torch.Generator().manual_seed(0)
    a = torch.randn(4, 8, generator=g).bfloat16()
    b = torch.randn(3, generator=g)
    save_file({"embedding.weight": a}, str(tmp_path / "one.safetensors"))
    save_file({"block.0.mlp.mlp1_bias": b,
               "block.0.mlp.mlp1_weight.blocks": torch.zeros(2, 4, 3, 16, dtype=torch.uint8),
               "block.0.mlp.mlp1_weight.scales": torch.full((2, 4, 3), 127, dtype=torch.uint8)}, str(tmp_path / "two.safetensors"))
    (tmp_path / "ignored.txt").write_text("not a tensor file")
    ck = Checkpoint(str(tmp_path), torch.device("cpu"))
    assert sorted(ck.tensor_name_to_file) == ["block.0.mlp.mlp1_bias", "block.0.mlp.mlp1_weight.blocks", "block.0.mlp.mlp1_weight.scales",
                                              "embedding.weight"]
    assert torch.equal(ck.get("embedding.weight"), a)
    assert torch.equal(ck.get("block.0.mlp.mlp1_bias"), b)
    dst = torch.empty(3)
    assert ck.get("block.0.mlp.mlp1_bias", out=dst) is dst and torch.equal(dst, b)
    with pytest.raises(AssertionError, match="not found"):
        ck.get("block.1.mlp.mlp1_bias")
    with pytest.raises(AssertionError, match="not found"):
        ck.get("block.1.mlp.mlp1_weight")
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ck.get("block.0.mlp.mlp1_weight")


def test_mxfp4_argument_errors():
    lib = _lib.lib()
    assert lib.tllm_mxfp4_dequant_bf16(None, None, None, 0, None) == 0
    assert lib.tllm_mxfp4_dequant_bf16(None, None, None, 5, None) == -1
    assert lib.tllm_mxfp4_dequant_bf16(None, None, None, -1, None) == -1
    assert lib.tllm_mxfp4_dequant_bf16(C.c_void_p(8), C.c_void_p(1), C.c_void_p(16), 5, None) != 0   # blocks not 16-byte aligned
    assert "aligned" in _err()


def test_mxfp4_launches_hold_fewer_threads_than_a_grid_may():
    threads = _lib.lib().tllm_mxfp4_launch_threads
    assert [threads(n) for n in (0, 1, 128, 129)] == [0, 256, 256, 512]
    assert all(threads(n) < 1 << 32 for n in ((1 << 31) - 128, 1 << 31, 1 << 33, 1 << 40))


def test_attention_prefill_argument_errors():
    """Argument checks of the prefill attention entry point happen before anything touches the GPU."""
    f = _lib.lib().tllm_attention_prefill_bf16
    p = C.c_void_p(4096)

    def call(q=p, k=p, v=p, out=p, q_ts=4096, kv_ts=512, batch=1, n_q=16, n_kv=16, kvh=8, group=8, hd=64, scale=0.125, window=0, start=p):
        return f(q, k, v, None, out, n_q * q_ts, q_ts, n_q * 4096, 4096, n_kv * kv_ts, kv_ts, batch, n_q, n_kv, kvh, group, hd, scale, window,
                 start, 0, None)

    assert call(batch=0) == 0 and call(n_q=0) == 0                      # nothing to do
    assert call(hd=128) != 0 and "head_dim" in _err()
    assert call(scale=0.0) != 0 and "sm_scale" in _err()
    assert call(window=-1) != 0
    assert call(n_kv=0) != 0
    assert call(q=None) != 0 and "NULL" in _err()
    assert call(start=None) != 0
    assert call(k=C.c_void_p(4104)) != 0 and "aligned" in _err()
    assert call(q_ts=4000) != 0                                         # heads do not fit into a token's stride
    assert call(kv_ts=256) != 0


def test_attention_decode_shape_planning():
    """The host-side choice of workgroup shape and splits (no launch): small batches keep one KV head per workgroup."""
    hpw = _lib.lib().tllm_attention_decode_heads_per_workgroup
    splits = _lib.lib().tllm_attention_decode_splits
    assert [hpw(b, 8, 4096, 0) for b in (1, 4)] == [0, 0]
    assert hpw(8, 8, 4096, 0) == 4 and splits(8, 8, 4096, 0) == 16               # splits of 256 keys, few enough of them
    assert hpw(16, 8, 4096, 0) == 4 and splits(16, 8, 4096, 0) == 8
    assert hpw(32, 8, 4096, 0) == 4 and splits(32, 8, 4096, 0) == 4
    assert hpw(8, 8, 32768, 0) == 4 and splits(8, 8, 32768, 0) == 16             # the longer splits win over the wider workgroup
    assert hpw(8, 8, 131072, 0) == 8 and splits(8, 8, 131072, 0) == 32           # ... and the wider one a tie
    assert hpw(12, 8, 20000, 0) == 4 and splits(12, 8, 20000, 0) == 10           # 24 x 10 workgroups rather than 24 x 11 = 264
    assert hpw(3, 8, 4096, 0) == 0 and splits(3, 8, 4096, 0) == 10               # 24 x 10 here as well
    assert hpw(4, 8, 32768, 0) == 4 and splits(4, 8, 32768, 0) == 32
    assert hpw(2, 8, 32768, 0) == 4 and splits(2, 8, 32768, 0) == 64
    assert hpw(2, 8, 16384, 0) == 0
    assert hpw(1, 8, 131072, 0) == 0
    assert hpw(64, 8, 131072, 128) == 0 and splits(64, 8, 131072, 128) == 1      # a sliding window bounds the context
    # more than eight KV heads: where one split fewer is as good but leaves CUs without a workgroup, the splits stay
    assert [(hpw(b, n, c, 0), splits(b, n, c, 0)) for b, n, c in ((33, 16, 2048), (49, 16, 4096), (24, 32, 2048), (33, 24, 3000))] == [(4, 2)] * 4
    assert (hpw(38, 16, 3000, 0), splits(38, 16, 3000, 0)) == (8, 3)
    # one launch of eight wavefronts per KV head, as long as its few workgroups are not what takes longest
    assert [splits(b, 8, c, 0) for b, c in ((1, 512), (7, 512), (8, 640), (11, 640), (12, 800), (16, 800))] == [1] * 6
    assert all(splits(b, 8, c, 0) > 1 for b, c in ((8, 700), (8, 800), (9, 700), (10, 700), (11, 641)))
    for b in (1, 3, 8, 100):
        for ctx in (1, 127, 128, 129, 5000, 131072):
            s = splits(b, 8, ctx, 0)
            assert 1 <= s <= 64 and (s == 1 or ctx >= 128 * (s - 1))


def test_attention_prefill_shape_planning():
    """Key blocks are shared out between wavefronts where the launch is small and the walk long enough to pay for the meeting."""
    groups = _lib.lib().tllm_attention_prefill_key_groups
    assert [groups(1, n, n, 8, 8, 0) for n in (1, 16, 64)] == [1, 1, 1]              # one block: nothing to share
    assert [groups(b, 64, 64, 8, 8, w) for b in (4, 8) for w in (0, 128)] == [1] * 4
    assert groups(1, 97, 97, 8, 8, 0) == 2 and groups(4, 128, 128, 8, 8, 0) == 1     # two blocks: at one workgroup per CU
    assert [groups(1, n, n, 8, 8, 128) for n in (400, 512)] == [1, 1]                # a window's three blocks at two per CU
    assert [groups(1, n, n, 8, 8, 0) for n in (300, 400, 512)] == [2, 2, 2]
    assert [groups(1, 97, 1597, 8, 8, w) for w in (0, 128)] == [4, 4]
    assert groups(1, 777, 777, 8, 8, 0) == 1


def test_attention_prefill_shapes():
    """In chunks behind more than six blocks of keys, with a window from 322 on; workgroups of few heads while those of four are few."""
    shape = _lib.lib().tllm_attention_prefill_shape

    def of(b, n, n_kv, group=8, window=0):
        s = shape(b, n, n_kv, 8, group, window)
        return s >> 24, s >> 16 & 255, s >> 8 & 255, s & 255

    assert [of(3, 333, n)[0] for n in (384, 385)] == [0, 1] and [of(1, 2048, 2048, window=w)[0] for w in (128, 321, 322)] == [0, 0, 1]
    assert of(2, 700, 700) == of(2, 600, 600) == (1, 64, 2, 1)              # 352 and 320 workgroups of four heads
    assert of(3, 450, 450) == (1, 64, 4, 1) and of(3, 333, 333) == (0, 64, 2, 1)
    assert [of(1, n, n) for n in (1536, 2048)] == [(1, 64, 2, 1), (1, 64, 4, 1)]
    assert of(9, 650, 700, 2) == (1, 128, 2, 1) and of(8, 650, 700, 2, 128) == (0, 128, 2, 1) and of(2, 1000, 1100, 5) == (1, 128, 1, 1)
    assert of(1, 97, 1597) == (0, 64, 1, 4) and shape(0, 1, 1, 8, 8, 0) == 0


def test_qkv_decode_tiles_or_the_general_kernel():
    """Decode batches of more than 32 rows at widths other than 2880: GEMM tiles only where the general kernel's passes over the
    weight cost more than a tile's fixed time."""
    tile = _lib.lib().tllm_qkv_gemm_tile
    assert [tile(0, rows, hidden, nq, nkv, 64) for rows, hidden, nq, nkv in ((33, 256, 4, 2), (64, 512, 8, 2), (48, 1024, 12, 4), (64, 4096, 4, 2),
                                                                          (256, 1024, 4, 2), (128, 512, 12, 4))] == [0] * 6
    assert all(tile(0, rows, hidden, nq, nkv, 64) for rows, hidden, nq, nkv in ((40, 4096, 64, 8), (64, 1024, 64, 8), (448, 512, 12, 4), (128, 8192, 64, 8)))
    assert [tile(0, rows, 4096, 64, 8, hd) for rows, hd in ((32, 64), (40, 128))] == [0, 0]


def test_decode_general_streaming_wavefronts_follow_the_grid():
    """Four wavefronts stream a workgroup's weight rows while all workgroups are on the machine together, fewer, with less LDS,
    beyond that (fp8, 1536 wide, 400 rows 78 us with four, 37 with one); never more than K has phases for."""
    streams = _lib.lib().tllm_decode_general_streams
    assert [streams(rows, 1536, 5120, 1) for rows in (1, 8, 12, 32, 64, 400)] == [4, 4, 2, 2, 1, 1]
    assert [streams(rows, 1536, 5120, 0) for rows in (1, 8, 12, 32, 64)] == [4, 4, 4, 1, 1]
    assert [streams(rows, 4096, 2048, 1) for rows in (16, 32, 64, 150)] == [4, 4, 2, 1]
    assert [streams(8, k, 5120, fp8) for fp8 in (0, 1) for k in (128, 256, 512, 1024)] == [1, 2, 4, 4, 1, 1, 2, 4]


def test_walks_spread_only_behind_a_filled_row_tile():
    """The walks of a launch's row tiles are spread over K where the last row tile is filled far enough for the number of them, and for
    widths and weights where that was measured to be ahead."""
    spread = _lib.lib().tllm_gemm_tile_spread

    def rows_of(k, n, rows):
        return [r for r in rows if spread(r, k, n)]

    assert rows_of(2880, 5120, (111, 112, 128, 150, 151, 192, 193, 200, 219, 220, 256)) == [112, 128, 192, 220, 256]
    assert rows_of(5120, 2880, (113, 128, 130, 144, 159, 160, 192, 193, 219, 220, 256, 257, 271, 272, 320, 321, 327, 328, 385)) == [
        113, 128, 160, 192, 220, 256, 272, 320, 328, 385]
    assert rows_of(5120, 2560, (160, 167, 168, 192)) == [168, 192]             # 32 columns
    assert rows_of(8192, 1536, (192, 256, 300, 600)) == []
    assert rows_of(1024, 8192, (128, 200, 256, 300)) == [128]
    assert rows_of(2880, 5120, (513, 640)) == [513, 640] and rows_of(2048, 8192, (256, 640)) == []


def test_qkv_prefill_tiles_at_other_widths():
    """A prompt's route at K other than 2880: the fixed part of a launch counts once, whatever K is."""
    tile = _lib.lib().tllm_qkv_gemm_tile
    assert [tile(1, rows, 8192, 64, 8, 64) for rows in (2048, 4096, 8192)] == [0, 0, 0]
    assert tile(1, 2900, 4096, 64, 8, 64) == 0
    assert all(tile(1, rows, hidden, 64, 8, 64) for rows in (1, 97, 999) for hidden in (64, 512, 2880, 8192))
    # 2880 wide: smaller tiles up to 1536 rows and where a launch of the larger ones would need a round for little
    assert [bool(tile(1, rows, 2880, 64, 8, 64)) for rows in (97, 1536, 1537, 2048, 2049, 2816, 2817, 4096, 4097, 8192)] == \
        [True, True, False, False, True, True, False, False, True, False]


def test_logits_tiles_have_a_kernel_of_about_their_width():
    """fp8 tiles of 17 - 20 units beside more than 64 rows: one tile more where that leaves tiles of up to 15, one tile stays one."""
    units = _lib.lib().tllm_unembedding_tile_units
    assert [units(rows, 1, 2880, 151936) for rows in (64, 65, 96, 97, 128, 200)] == [19, 19, 19, 13, 13, 13]
    assert [units(rows, 1, 2048, 234000) for rows in (64, 96, 97)] == [20, 15, 15]
    assert [units(rows, 1, 2880, 70000) for rows in (96, 97, 128)] == [18, 18, 18] and units(96, 1, 2880, 163000) == 20
    assert [units(rows, 1, 2880, 201088) for rows in (64, 128)] == [25, 25] and [units(rows, 0, 2880, 201088) for rows in (49, 128)] == [17, 17]
    assert units(8, 0, 2880, 201088) == 0


def test_logits_of_a_small_vocabulary_stay_in_passes():
    tiled = _lib.lib().tllm_unembedding_decode_tiled
    assert [tiled(rows, 0, hidden, vocab) for rows, hidden, vocab in ((9, 4096, 1000), (16, 4096, 4000), (33, 2880, 1000), (64, 2880, 4096))] == [0] * 4
    assert [tiled(rows, 0, hidden, vocab) for rows, hidden, vocab in ((17, 4096, 1000), (65, 2880, 1000), (9, 4096, 8000), (33, 2880, 8000),
                                                                      (33, 2880, 201088))] == [1] * 5
    assert [tiled(16, 1, 4096, 1000), tiled(16, 1, 4096, 1001), tiled(33, 1, 2880, 1000), tiled(40, 0, 1024, 1000)] == [1, 0, 0, 1]
    assert [tiled(rows, 0, 2880, 201088) for rows in (8, 32)] == [0, 0]
