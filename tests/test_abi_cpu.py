"""No-GPU checks of the C-ABI library: it loads, exports every symbol the header declares, and
rejects bad arguments before touching the device."""
import ctypes
import os
import re

import pytest

from conftest import ROOT

HEADERS = [os.path.join(ROOT, "include", n) for n in ("llmops_hip.h", "llmops_hip_test.h")]
LIB = os.path.join(ROOT, "llama.cl_amd", "llmops", "libllmops_hip.so")


def declared_symbols():
    src = "".join(open(h).read() for h in HEADERS)
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(llmops_[A-Za-z0-9_]+)\s*\(", src)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} not built: run `python llama.cl_amd/build.py`")
    return ctypes.CDLL(LIB)


def test_header_declares_the_path():
    names = declared_symbols()
    for must in ("llmops_offline_FC_quant_Q4A", "llmops_offline_FC_dequant_Q4A", "llmops_FC_dynamic_quantize_x",
                 "llmops_fc_Q4A", "llmops_fc_Q4A_partials", "llmops_attention_rope", "llmops_rope_embed", "llmops_softmax"):
        assert must in names


def test_library_exports_every_declared_symbol(lib):
    missing = [n for n in declared_symbols() if not hasattr(lib, n)]
    assert not missing, missing


def test_python_binding_covers_every_declared_symbol():
    from llmops import _lib
    assert sorted(_lib.SIGNATURES) == declared_symbols()
    _lib.load()


def test_block_bytes(lib):
    lib.llmops_q4a_block_bytes.restype = ctypes.c_int64
    assert lib.llmops_q4a_block_bytes(32) == 640      # ops/op_fc.hpp:22-24 with G=32
    assert lib.llmops_q4a_block_bytes(128) == 2176
    assert lib.llmops_q4a_block_bytes(64) == 0


def test_argument_validation_without_device(lib):
    """Validation mirrors the reference's ASSERTs and runs before any HIP call, so it works with no GPU."""
    lib.llmops_last_error.restype = ctypes.c_char_p
    i64, vp = ctypes.c_int64, ctypes.c_void_p
    rc = lib.llmops_offline_FC_quant_Q4A(vp(16), i64(32), i64(64), i64(64), 64, vp(16), vp(0))
    assert rc == 1 and b"valid_group" in lib.llmops_last_error()
    rc = lib.llmops_fc_Q4A(vp(256), i64(1), i64(300), vp(256), i64(1), i64(1), 128, i64(32), vp(256), vp(256),
                           ctypes.c_size_t(1 << 20), vp(0))      # 300 activations cannot belong to one k-group of 128
    assert rc == 1 and b"K <= Kg * group_k" in lib.llmops_last_error()
    lib.llmops_fc_Q4A_workspace_bytes.restype = ctypes.c_size_t
    need = lib.llmops_fc_Q4A_workspace_bytes(i64(1), i64(4096), i64(128), i64(32), 128)
    assert need > 65536
    rc = lib.llmops_fc_Q4A(vp(256), i64(1), i64(4096), vp(256), i64(128), i64(32), 128, i64(4096), vp(256), vp(256),
                           ctypes.c_size_t(1024), vp(0))
    assert rc == 2 and b"workspace" in lib.llmops_last_error()
    rc = lib.llmops_attention_rope(vp(256), vp(256), vp(256), i64(1), i64(1), i64(32), i64(64), vp(256), i64(32), vp(256), 0,
                                   i64(2), i64(16), vp(256), 0, 0, vp(256), ctypes.c_size_t(1 << 30), vp(0))
    assert rc == 1 and b"S == 128" in lib.llmops_last_error()
    # the one-token kernels run on a (chunk, head) grid.  With the position by value more than 65535 heads in all take
    # the general kernels (GPU test); with the position in device memory they are refused before any launch
    rc = lib.llmops_attention_rope_decode(vp(256), vp(256), vp(256), i64(2200), i64(32), i64(128), vp(256), i64(64), vp(256), 0,
                                          i64(2), i64(16), vp(256), vp(256), 0, vp(256), ctypes.c_size_t(1 << 40), vp(0))
    assert rc == 1 and b"65535 heads" in lib.llmops_last_error()
    # int32 sums by tiles of 64 and 128 rows: a tile's rows are addressed with 32 bits
    for use_mfma, groups in ((1, 1 << 19), (2, 1 << 18)):
        rc = lib.llmops_fc_Q4A_partials(vp(256), i64(64), vp(256), i64(1), i64(groups), 128, vp(256), use_mfma, vp(0))
        assert rc == 1 and b"K must be below" in lib.llmops_last_error()
    # .. by the weight-streaming kernel: up to the 1024 rows that it takes
    rc = lib.llmops_fc_Q4A_partials(vp(256), i64(1025), vp(256), i64(1), i64(4), 128, vp(256), 3, vp(0))
    assert rc == 1 and b"rows <= 1024" in lib.llmops_last_error()
    rc = lib.llmops_fc_workspace_reset(vp(0), ctypes.c_size_t(1 << 20), vp(0))
    assert rc == 1 and b"workspace != nullptr" in lib.llmops_last_error()
    # the entry point that allocates nothing validates its arguments before it enqueues anything (no device here:
    # a launch would fail with a HIP error, not with this message)
    rc = lib.llmops_fc_Q4A_noalloc(vp(0), i64(1), i64(4096), vp(256), i64(128), i64(32), 128, i64(4096), vp(256), vp(0))
    assert rc == 1 and b"x != nullptr" in lib.llmops_last_error()


def test_test_hooks_are_refused_unless_the_process_asks_for_them():
    """The planner knobs, dump builds and calibration kernels of include/llmops_hip_test.h live in the product
    library; a process that was not started with LLMOPS_TEST_HOOKS=1 cannot use them."""
    import subprocess
    import sys
    code = (
        "import ctypes, sys\n"
        f"lib = ctypes.CDLL({LIB!r})\n"
        "lib.llmops_last_error.restype = ctypes.c_char_p\n"
        "vp, i64 = ctypes.c_void_p, ctypes.c_int64\n"
        "rc = lib.llmops_test_calib_read(vp(256), i64(1024), 4, vp(256), vp(0))\n"
        "msg = lib.llmops_last_error()\n"
        "lib.llmops_test_fc_set_tuning(64, 8)\n"
        "print(rc, msg.decode())\n"
    )
    env = {k: v for k, v in os.environ.items() if k != "LLMOPS_TEST_HOOKS"}
    out = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr
    assert out.stdout.startswith("1 ") and "LLMOPS_TEST_HOOKS=1" in out.stdout
    assert "test hooks are switched off" in out.stderr


def test_gemm_planner_choices(lib):
    """The prefill GEMM's planner is host arithmetic: what it chooses for the shapes its rules were measured
    on (row-tile factor 1, 2, 4 = 32, 64, 128 rows per workgroup; split-K factor), and that every plan covers K
    exactly once."""
    i64, ci = ctypes.c_int64, ctypes.c_int

    def plan(rows, N, K, G=128):
        rt, S = ci(0), ci(0)
        assert lib.llmops_test_gemm_plan(i64(rows), i64((N + 31) // 32), i64((K + G - 1) // G), G, ctypes.byref(rt),
                                         ctypes.byref(S)) == 0
        return rt.value, S.value

    # many rows: 128-row tiles, no split where they fill the machine (16 x 32 tiles are two to a compute unit)
    assert plan(2048, 11008, 4096) == (4, 1)
    assert plan(2048, 4096, 11008) == (4, 1)
    assert plan(2048, 4096, 512) == (4, 1)
    # few rows: 32-row tiles and as many splits as still leave runs of 4 k-groups (not 11 runs of 3)
    assert plan(32, 11008, 4096) == (1, 8)
    assert plan(64, 11008, 4096) == (1, 5)
    assert plan(128, 11008, 4096) == (2, 4)
    assert plan(128, 4096, 11008) == (1, 8)
    for rows in (17, 24, 40, 100, 255, 256, 300, 512, 1000, 4096):
        for N, K in ((4096, 4096), (11008, 4096), (4096, 11008), (352, 640), (22016, 4096), (64, 128)):
            rt, S = plan(rows, N, K)
            Kg = (K + 127) // 128
            assert rt in (1, 2, 4) and 1 <= S <= Kg
            per = (Kg + S - 1) // S
            assert (Kg + per - 1) // per == S     # S splits of `per` k-groups, the last possibly short, none empty
    assert lib.llmops_test_gemm_plan(i64(0), i64(1), i64(1), 128, None, None) != 0
    # a forced tile is the tile reported, and what is no tile is not forced
    try:
        for forced, want in ((1, 1), (2, 2), (4, 4), (8, 4), (3, 4), (0, 4)):
            lib.llmops_test_gemm_set_tuning(forced)
            assert plan(2048, 11008, 4096)[0] == want
    finally:
        lib.llmops_test_gemm_set_tuning(0)
    # group 32: 32-row tiles, stages of four k-groups
    assert plan(512, 11008, 4096, 32)[0] == 1 and plan(64, 4096, 4096, 32)[0] == 1


@pytest.mark.parametrize("form,sizes", [
    # (strips, k-groups): the last row count that measured faster in one launch, the first that did in separate ones
    ("residual", {(64, 4): (4, 6), (64, 16): (4, 5), (128, 32): (3, 4), (128, 86): (3, 4), (256, 32): (3, 4), (384, 32): (2, 3), (688, 32): (2, 3)}),
    ("residual sums", {(64, 4): (8, 9), (64, 16): (6, 8), (128, 32): (5, 6), (128, 86): (4, 5), (256, 32): (4, 5), (384, 32): (2, 3), (688, 32): (2, 3)}),
    ("norm", {(64, 4): (1, 3), (64, 16): (1, 3), (128, 32): (1, 3), (128, 86): (2, 3), (256, 32): (1, 3), (384, 32): (1, 2), (688, 32): (1, 2)}),
    ("norm sums", {(64, 4): (2, 3), (64, 16): (2, 3), (128, 32): (2, 3), (128, 86): (2, 3), (256, 32): (2, 3), (384, 32): (1, 2), (688, 32): (1, 2)}),
    ("norm sums_in", {(64, 4): (4, 5), (64, 16): (3, 5), (128, 32): (2, 3), (256, 32): (2, 3), (384, 32): (2, 3), (688, 32): (1, 2)}),
    ("glu", {(64, 4): (4, 5), (64, 16): (3, 5), (128, 32): (2, 3), (128, 86): (2, 3), (256, 32): (2, 3), (384, 32): (1, 2), (688, 32): (1, 2)}),
    ("glu sums", {(64, 4): (6, 8), (64, 16): (4, 6), (128, 32): (2, 4), (128, 86): (2, 4), (256, 32): (3, 4), (384, 32): (2, 3), (688, 32): (2, 3)})])
def test_rows_from_which_a_decode_projection_is_quantized_first(lib, form, sizes):
    opts, first = form.split(), ctypes.c_int(-1)
    i64 = ctypes.c_int64

    def separate(rows, strips, groups, group_k=128, glu=2 if "glu" in opts else 0):
        assert lib.llmops_test_fc_decode_route(i64(rows), i64(groups * group_k), i64(strips), i64(groups), group_k, int("norm" in opts),
                                               int("sums_in" in opts), glu, int("sums" in opts), ctypes.byref(first)) == 0
        return first.value

    for (strips, groups), (one, many) in sizes.items():
        assert [separate(r, strips, groups) for r in (1, one, many, 9)] == [0, 0, 1, 1], (form, strips, groups)
        # what the quantization and the product behind it do not take: one launch up to 8 rows
        assert not separate(8, 63, groups) and not separate(8, strips, groups, group_k=32)
        assert not separate(8, strips, groups, glu=1)
        if opts == ["norm"]:  # the FC in front hands on its sums of squares where this one is a single launch
            for rows in range(1, 10):
                assert lib.llmops_fc_Q4A_decode_wants_sumsq(i64(rows), i64(128 * groups), i64(strips), i64(groups), 128, 0) == 1 - separate(rows, strips, groups)


def test_python_ops_refuse_host_tensors():
    """The product path has no CPU fallback: host tensors raise instead of being computed elsewhere."""
    import torch
    import llmops
    with pytest.raises(RuntimeError, match="HIP device"):
        llmops.offline_FC_quant_Q4A(torch.zeros(32, 128))
    with pytest.raises(RuntimeError, match="HIP device"):
        llmops.fc_Q4A(torch.zeros(1, 1, 128), torch.zeros(1, 1, 2176, dtype=torch.int8), 32)


@pytest.mark.parametrize("native,why", [("None", "_host"), ("types.SimpleNamespace(built_for='torch 0.1, Python 3.10')", "torch 0.1")])
def test_calls_without_the_native_module(native, why):
    """Where _host.so is missing, or built for another torch, the Python functions take the calls, with their own errors, and
    say so once."""
    import subprocess
    import sys
    code = f"""
import sys, types, warnings
sys.path.insert(0, {os.path.dirname(os.path.dirname(LIB))!r})
sys.modules["llmops._host"] = {native}
import torch, llmops
llmops.__dict__.pop("_host", None)
if sys.modules["llmops._host"] is not None:
    llmops._host = sys.modules["llmops._host"]
with warnings.catch_warnings(record=True) as said:
    warnings.simplefilter("always")
    for call in (lambda: llmops.fc_Q4A(torch.zeros(1, 1, 128), torch.zeros(1, 1, 2176, dtype=torch.int8), 32),
                 lambda: llmops.attention_rope2(*[torch.zeros(1, 1, 128)] * 3, torch.zeros(64), torch.zeros(2, 1, 1, 4, 128), torch.zeros(1, dtype=torch.int32), 0, 0)):
        for _ in range(2):
            try:
                call()
            except RuntimeError as e:
                print(e)
print([str(w.message) for w in said])
"""
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr
    lines = out.stdout.splitlines()
    assert len(lines) == 5 and all("on the HIP device" in l for l in lines[:4])
    assert lines[4].count("_host.so does not load") == 1 and why in lines[4]


def test_kvcache_slot_manager():
    """KVCache.prepare mirrors chatllama/main.py:60-125: ring buffer, protected system slots, early stop."""
    import torch
    from llmops.opset import KVCache
    cfg = {"layer_num": 1, "head_num": 1, "head_size": 128}
    kv = KVCache(cfg, 1, 8, False, device="cpu")
    assert kv.prepare(3, -1, -1) and kv.slots.tolist() == [0, 1, 2] and kv.position_id == 0      # system prompt
    assert kv.prepare(2, 1, 0) and kv.slots.tolist() == [3, 4] and kv.position_id == 3
    assert kv.prepare(3, 2, 0) and kv.slots.tolist() == [5, 6, 7] and kv.cur_kv_len == 8
    # wraps around, skipping the protected system slots 0..2; sentence 1 may be overwritten
    assert kv.prepare(2, 3, 0) and kv.slots.tolist() == [3, 4] and kv.position_id == 8
    # sentence 2 holds the instruction: asked to fail rather than overwrite it
    assert not kv.prepare(1, 4, 2)
    assert kv.cur_kv_len == 8 and kv.slots.dtype == torch.int32


def test_tensor_attributes_the_reference_callers_use():
    """``weight.numel() * weight.item_size`` (chatllama/main.py:171-173) must work on what the ops return."""
    import torch
    import llmops  # noqa: F401  (adds the reference's spelling of the element size)
    t = torch.zeros(3, 5, dtype=torch.int8)
    assert t.item_size == 1 and torch.zeros(2, dtype=torch.float32).item_size == 4
    assert t.numel() * t.item_size == 15 and tuple(t.shape) == (3, 5) and t.clone().numpy().shape == (3, 5)


@pytest.mark.parametrize("rows,N,K,good", [
    (9, 12288, 4096, (6, 8)), (32, 22016, 4096, (4, 5, 6)), (96, 12288, 4096, (3, 5)), (16, 4096, 4096, (7, 8, 11)), (192, 3000, 5632, (7, 8)),
    (300, 2048, 2048, (3,)), (1024, 2048, 2048, (1,)), (300, 8192, 2048, (1,)), (128, 600, 11008, (15,)), (600, 1024, 512, (1,)), (9, 1024, 512, (4,))])
def test_group32_planner_measured_sizes(lib, rows, N, K, good):
    """Split-K factors of the group-32 product at sizes where these measured 3 % and more faster than most others."""
    i64, rt, S = ctypes.c_int64, ctypes.c_int(), ctypes.c_int()
    assert lib.llmops_test_gemm_plan(i64(rows), i64((N + 31) // 32), i64(K // 32), 32, ctypes.byref(rt), ctypes.byref(S)) == 0
    assert S.value in good


@pytest.mark.parametrize("half", [0, 1])
def test_attention_planner_measured_sizes(half):
    """Calls below 32 query tokens, and one token where the decode kernel is not taken: sizes at which one of the two
    kernels measured at least 15 % faster than the other (heads in all, tokens, cache rows; 1: a workgroup per query and
    chunk, 2: all tokens of a head together)."""
    from llmops import _lib
    lib = _lib.load()
    want = {1: [(4096, 1, 48), (4096, 1, 16), (512, 1, 16), (1024, 2, 16), (32, 8, 128), (32, 16, 32), (8, 2, 100), (4, 31, 48), (70000, 1, 16),
                (70000, 1, 64)],
            2: [(4, 1, 8192), (32, 16, 1516), (32, 31, 512), (256, 8, 500), (512, 8, 64), (1024, 6, 64), (4096, 8, 16), (4, 3, 8192)]}
    k, r, n = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    for kernel, sizes in want.items():
        for heads, tokens, kv in sizes:
            assert lib.llmops_test_attn_plan(1, tokens, heads, kv, kv - tokens, half, ctypes.byref(k), ctypes.byref(r), ctypes.byref(n)) == 0
            assert k.value == kernel and n.value == -(-kv // r.value), (heads, tokens, kv)


@pytest.mark.parametrize("heads,tokens,past,pieces32,pieces16", [
    (32, 32, 500, True, True), (32, 64, 100, False, False), (32, 256, 0, None, False), (32, 256, 300, True, True),
    (32, 200, 300, True, True), (16, 384, 100, True, True), (16, 512, 100, True, True), (16, 1024, 400, True, True), (32, 512, 300, True, True),
    (32, 512, 1500, True, True), (32, 2048, 0, False, False), (128, 512, 3500, False, False)])
def test_attention_planner_pieces_of_the_tiled_kernel(heads, tokens, past, pieces32, pieces16):
    """From 32 query tokens: the cache rows of a tile in several workgroups or in one, at sizes where one of the two measured
    faster (or where the tiles fill the chip); None: the same within 3 %."""
    from llmops import _lib
    lib = _lib.load()
    k, r, n = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    for half, several in ((0, pieces32), (1, pieces16)):
        kv = past + tokens
        assert lib.llmops_test_attn_plan(1, tokens, heads, kv, past, half, ctypes.byref(k), ctypes.byref(r), ctypes.byref(n)) == 0
        assert k.value == 3 and several in (None, n.value > 1) and r.value % 64 == 0 and (n.value - 1) * r.value < kv <= n.value * r.value
