"""Host model of the addresses of a prompt pass (LlamaDecoder.forward, fused plan, more than 8 rows, group 128): for every
launch the first and last byte of each pointer, from the launch's arguments and the kernels' index expressions, against the
size of the allocation behind it.  Plans and workspace sizes come from the library itself (no GPU needed)."""
import ctypes

import numpy as np
import pytest

COUNTERS = 3 << 20          # LLMOPS_FC_COUNTER_BYTES
BLK = 2176                  # a packed block of group 128


def up(v, a=256):
    return -(-v // a) * a


class Model:
    def __init__(self, lib):
        self.lib, self.seen, self.bad = lib, [], []

    def touch(self, launch, what, size, lo, hi):
        """bytes [lo, hi) of an allocation of `size` bytes"""
        self.seen.append((launch, what))
        if not (0 <= lo < hi <= size):
            self.bad.append((launch, what, lo, hi, size))


def product(m, name, rows, Ng, Kg, N, ws_bytes, y_bytes, y_off=0, w_bytes=None, w_off=0, residual=False):
    """launch_gemm on a workspace laid out as fc_layout lays it out"""
    rt, S = ctypes.c_int(), ctypes.c_int()
    assert m.lib.llmops_test_gemm_plan(rows, Ng, Kg, 128, ctypes.byref(rt), ctypes.byref(S)) == 0
    rt, S = rt.value, S.value
    off_xq = COUNTERS
    off_xd = up(off_xq + rows * Kg * 128)
    off_gs = up(off_xd + rows * Kg * 4)
    off_xst = up(off_gs + rows * Kg * 4)
    off_part = up(off_xst + rows * Kg * 8 + 256)
    w_bytes = Ng * Kg * BLK if w_bytes is None else w_bytes
    bm = rt * 32
    nbx, nby = -(-Ng // 4), -(-rows // bm)
    kper = -(-Kg // S)
    bx, by = np.arange(nbx)[:, None], np.arange(nby)[None, :]
    strips = np.minimum(Ng - 1, bx * 4 + np.array([0, 3])[:, None, None])
    row = np.minimum(rows - 1, by * bm + np.array([0, bm - 1])[:, None, None])
    launch = "%s: product of %d x %d strips, %d-row tiles, %d splits" % (name, rows, Ng, bm, S)
    assert kper * (S - 1) < Kg                                                  # every split has k-groups
    m.touch(launch, "codes", ws_bytes, off_xq + int(row.min()) * Kg * 128, off_xq + int(row.max()) * Kg * 128 + (Kg - 1) * 128 + 128)
    m.touch(launch, "pairs", ws_bytes, off_xst, off_xst + ((Kg - 1) * rows + int(row.max())) * 8 + 8)
    m.touch(launch, "weights", w_bytes, w_off + int(strips.min()) * Kg * BLK, w_off + (int(strips.max()) * Kg + Kg - 1) * BLK + BLK)
    if rt == 8:  # the min term reads eight k-groups of a row's sums and of a strip's mins at a time
        assert Kg >= 8 and rows * Kg * 128 < 1 << 31 and Ng * Kg * BLK < 1 << 31   # 32-bit offsets
        starts = np.minimum(np.concatenate([np.arange(z * kper, min(Kg, (z + 1) * kper), 32) for z in range(S)])[:, None] + 8 * np.arange(4), Kg - 8)
        m.touch(launch, "sums", ws_bytes, off_gs + int(starts.min()) * 4, off_gs + (int(row.max()) * Kg + int(starts.max())) * 4 + 32)
    in_kernel = S > 1 and rt != 8 and S <= 12 and nbx * nby <= 65536 // 4
    if S > 1:
        m.touch(launch, "partial sums", ws_bytes, off_part, off_part + ((S - 1) * rows * Ng * 32 + (rows - 1) * Ng * 32 + Ng * 32) * 4)
        if in_kernel:
            m.touch(launch, "counters", 65536, 0, (int(by.max()) * nbx + int(bx.max())) * 4 + 4)
        else:
            launch += ", then the sum"
    m.touch(launch, "result", y_bytes, y_off, y_off + ((rows - 1) * N + N) * 4)
    if residual:
        m.touch(launch, "residual", y_bytes, y_off, y_off + ((rows - 1) * N + N) * 4)
    return off_part


def quantization(m, name, rows, Kg, ws_bytes, x_bytes, glu=False):
    """rmsnorm_quant_kernel, quant_x_tile128_kernel: codes, scales or pairs, sums"""
    off_xq = COUNTERS
    off_xd = up(off_xq + rows * Kg * 128)
    off_gs = up(off_xd + rows * Kg * 4)
    off_xst = up(off_gs + rows * Kg * 4)
    K = Kg * 128
    m.touch(name, "input", x_bytes, 0, ((rows - 1) * (2 if glu else 1) * K + (2 * K if glu else K)) * 4)
    m.touch(name, "codes", ws_bytes, off_xq, off_xq + (rows - 1) * K + K)
    m.touch(name, "scales", ws_bytes, off_xd, off_xd + ((rows - 1) * Kg + Kg - 1) * 4 + 4)
    m.touch(name, "sums", ws_bytes, off_gs, off_gs + ((rows - 1) * Kg + Kg - 1) * 4 + 4)
    m.touch(name, "pairs", ws_bytes, off_xst, off_xst + ((Kg - 1) * rows + rows - 1) * 8 + 8)


def attention(m, rows, H, past, maxlen, half):
    S, e = 128, 2 if half else 4
    q_bytes, plane = rows * H * S * 4, H * maxlen * S * e
    ws_bytes = m.lib.llmops_attention_workspace_bytes(1, rows, H, S, maxlen)
    head = 65536
    k, r, n = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert m.lib.llmops_test_attn_plan(1, rows, H, maxlen, past, int(half), ctypes.byref(k), ctypes.byref(r), ctypes.byref(n)) == 0
    kv = min(past + rows, maxlen)
    name = "attention, kernel %d, %d pieces of %d rows" % (k.value, n.value, r.value)
    slot = np.arange(past, past + rows)
    for what, lo in (("k rows of the cache", 0), ("v rows of the cache", plane)):
        m.touch("rotation", what, 2 * plane, lo + int(slot.min()) * S * e, lo + ((H - 1) * maxlen + int(slot.max())) * S * e + S * e)
        m.touch(name, what, 2 * plane, lo, lo + ((H - 1) * maxlen + kv - 1) * S * e + S * e)
    for what in ("q", "k", "v"):
        m.touch("rotation", what, q_bytes, 0, (((rows - 1) * H + H - 1) * S + S - 1) * 4 + 4)
    part = head + up(maxlen * 4)
    if k.value == 3:
        m.touch("fill", "token of a cache row", ws_bytes, head, head + maxlen * 4)
        m.touch("rotation", "token of a cache row", part, head + int(slot.min()) * 4, head + int(slot.max()) * 4 + 4)
        m.touch(name, "token of a cache row", part, head, head + (kv - 1) * 4 + 4)
    if n.value > 1 or k.value < 3:
        m.touch(name, "records", ws_bytes, part, part + ((H * rows - 1) * n.value + n.value - 1) * 520 + 520)
    m.touch(name, "output", q_bytes, 0, ((rows - 1) * H + H - 1) * S * 4 + S * 4)


@pytest.mark.parametrize("rows", [33, 200, 300, 384, 512, 513, 1000, 2048])
@pytest.mark.parametrize("past,half", [(0, False), (700, True)])
def test_every_address_of_a_prompt_pass(rows, past, half):
    from llmops import _lib
    lib = _lib.load()
    m, H, F, V, heads, table = Model(lib), 4096, 11008, 55296, 32, 1024
    maxlen = max(256, up(past + rows))
    need = lambda Ng, Kg: lib.llmops_fc_Q4A_workspace_bytes(rows, Kg * 128, Ng, Kg, 128)
    m.touch("embedding", "output", rows * H * 4, 0, (rows - 1) * H * 4 + ((H // 4 - 1) * 4 + 4) * 4)
    m.touch("embedding", "rows", table * H, 0, (table - 1) * H + (H // 4 - 1) * 4 + 4)
    # q, k, v: three products of 128 strips on one quantization; the workspace is the larger of what whole and part need
    ws = max(need(384, 32), need(128, 32))
    quantization(m, "rmsnorm and quantization", rows, 32, ws, rows * H * 4)
    layouts = {product(m, "q, k, v part %d" % p, rows, 128, 32, H, ws, 3 * rows * H * 4, p * rows * H * 4, 384 * 32 * BLK, p * 128 * 32 * BLK)
               for p in range(3)}
    assert len(layouts) == 1
    attention(m, rows, heads, past, maxlen, half)
    quantization(m, "quantization of o's input", rows, 32, need(128, 32), rows * H * 4)
    product(m, "o", rows, 128, 32, H, need(128, 32), rows * H * 4, residual=True)
    quantization(m, "rmsnorm and quantization", rows, 32, need(688, 32), rows * H * 4)
    product(m, "gate and up", rows, 688, 32, 2 * F, need(688, 32), rows * 2 * F * 4)
    quantization(m, "silu * up and quantization", rows, 86, need(128, 86), rows * 2 * F * 4, glu=True)
    product(m, "down", rows, 128, 86, H, need(128, 86), rows * H * 4, residual=True)
    quantization(m, "rmsnorm and quantization", rows, 32, need(1728, 32), rows * H * 4)
    product(m, "logits", rows, 1728, 32, V, need(1728, 32), rows * V * 4)
    assert not m.bad, m.bad
    assert len(m.seen) > 60


def test_the_model_finds_a_workspace_that_is_too_small():
    """What the q|k|v product once did: a part's partial sums in a workspace sized for the whole."""
    from llmops import _lib
    lib = _lib.load()
    m = Model(lib)
    whole, part = (lib.llmops_fc_Q4A_workspace_bytes(512, 4096, n, 32, 128) for n in (384, 128))
    product(m, "q", 512, 128, 32, 4096, whole, 512 * 4096 * 4)
    assert [b[1] for b in m.bad] == ["partial sums"] and m.bad[0][3] <= part
    # (not even the module's smallest workspace, 16 MiB, held them)
    assert m.bad[0][3] > 16 << 20
