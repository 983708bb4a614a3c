"""Host model of the addresses of a prompt pass (LlamaDecoder.forward, fused plan, 33 tokens and more, group 128): for every
launch the first and last byte of each pointer, from the launch's arguments and the kernels' index expressions, against the
part of the allocation that is meant.  Plans and workspace sizes come from the library itself (no GPU needed)."""
import ctypes

import numpy as np
import pytest

COUNTERS = 3 << 20          # LLMOPS_FC_COUNTER_BYTES
TICKETS = 65536             # kTicketBytes: arrival counters, one per tile
BLK = 2176                  # a packed block of group 128
LANES = np.arange(64)


def up(v, a=256):
    return -(-v // a) * a


class Model:
    def __init__(self, lib):
        self.lib, self.seen, self.bad = lib, [], []

    def touch(self, launch, what, region, lo, hi):
        """bytes [lo, hi) that must lie in `region`: a size, or (first byte, end)"""
        first, end = region if isinstance(region, tuple) else (0, region)
        self.seen.append((launch, what))
        if not (first <= lo < hi <= end):
            self.bad.append((launch, what, lo, hi, first, end))

    def need(self, rows, Ng, Kg, G=128):
        return self.lib.llmops_fc_Q4A_workspace_bytes(rows, Kg * G, Ng, Kg, G)

    def plan(self, rows, Ng, Kg, G=128):
        rt, S = ctypes.c_int(), ctypes.c_int()
        assert self.lib.llmops_test_gemm_plan(rows, Ng, Kg, G, ctypes.byref(rt), ctypes.byref(S)) == 0
        return rt.value, S.value


def layout(rows, Kg, G, ws):
    """fc_layout: codes, scales, sums, pairs (and what the few-row product reads past them), partial sums"""
    at = {"codes": (COUNTERS, COUNTERS + rows * Kg * G)}
    off_gs = up(up(COUNTERS + rows * Kg * G) + rows * Kg * 4)
    off_xst = up(off_gs + rows * Kg * 4)
    at["pairs"] = (off_xst, off_xst + rows * Kg * 8)
    at["partial sums"] = (up(off_xst + rows * Kg * 8 + 256), ws)
    return at


def tiles_of_the_grid(nbx, nby):
    """(bx, by) of every workgroup that has a tile: runs of tiles per XCD, bands of 8 row blocks"""
    total, out = nbx * nby, []
    per = -(-total // 8)
    for block in range(8 * per):
        i = (block & 7) * per + (block >> 3)
        if i < total:
            band, in_band = divmod(i, 8 * nbx)
            rows_in_band = min(8, nby - band * 8)
            out.append((in_band // rows_in_band, band * 8 + in_band % rows_in_band))
    return out


def product(m, name, rows, Ng, Kg, N, ws_bytes, y_bytes, parts=1, residual=False):
    """launch_gemm, group 128: fc_gemm_tile_kernel (and gemm_reduce_kernel) on a workspace laid out as fc_layout does;
    results [parts][rows][N]"""
    rt, S = m.plan(rows, Ng, Kg)
    assert rt in (1, 2, 4)
    at = layout(rows, Kg, 128, ws_bytes)
    BM, per, Kp = 32 * rt, -(-Kg // S), Kg * 128
    nbx, nby = -(-Ng // 4), -(-rows // BM)
    launch = "%s: product of %d rows x %d strips, %d-row tiles, %d splits" % (name, rows, Ng, BM, S)
    assert (S - 1) * per < Kg <= S * per                                        # every split has k-groups, together all of them
    grid = tiles_of_the_grid(nbx, nby)
    assert len(grid) == nbx * nby and len(set(grid)) == len(grid) and max(grid) <= (nbx - 1, nby - 1)
    codes, pairs, weights = [], [], []
    for by in range(nby):
        row0 = by * BM
        # codes: wave w's copy i has rows (w * RT + i) * 8 + lane / 8, a 16-byte chunk of 128 per lane
        r = ((np.arange(4)[:, None, None] * rt + np.arange(rt)[:, None]) * 8 + (LANES >> 3)).ravel()
        chunk = np.tile(LANES & 7, 4 * rt) ^ ((r >> 1) & 7)
        assert len(set(zip(r, chunk))) == BM * 8 and r.max() == BM - 1
        off = (np.minimum(rows - 1, row0 + r) - row0) * Kp + chunk * 16
        assert 0 <= off.min() and off.max() < 1 << 32                           # 32-bit lane offsets
        codes += [row0 * Kp + off.min(), row0 * Kp + off.max() + (Kg - 1) * 128 + 16]
        # scales and sums: 64 rows to a copy, 4 bytes per lane, from the pairs [Kg][rows]
        row = np.minimum(rows - 1, row0 + np.arange(max(1, BM // 64))[:, None] * 64 + np.minimum(LANES, BM - 1))
        assert row.max() * 8 < 1 << 32
        pairs += [row.min() * 8, (Kg - 1) * rows * 8 + row.max() * 8 + 4 + 4]
    for bx in range(nbx):
        base, strip = bx * 4 * Kg * BLK, (np.minimum(Ng - 1, bx * 4 + np.arange(4)) - bx * 4) * Kg * BLK
        nib = strip[:, None, None] + (np.arange(2) * 1024)[:, None] + (2 * ((LANES >> 3) & 3) + (LANES >> 5)) * 128 + (LANES & 7) * 16
        assert len(set(nib[0].ravel())) == 128 and nib[0].max() + 16 == 2048    # a strip's nibbles, each once
        tail = strip[LANES >> 4] + (LANES & 15) * 4 + 2048                      # scales, and 64 bytes on the mins
        assert nib.max() < 1 << 32 and tail.max() + 64 < 1 << 32
        weights += [base + nib.min(), base + (Kg - 1) * BLK + max(nib.max() + 16, tail.max() + 64 + 4)]
    for what, seen, region in (("codes", codes, at["codes"]), ("pairs", pairs, at["pairs"]), ("weights", weights, (0, Ng * Kg * BLK))):
        m.touch(launch, what, region, region[0] + int(min(seen)), region[0] + int(max(seen)))
    # LDS: the last copies of a slot end where the slot's codes, nibbles, scales and row scales end
    stage = BM * 128 + 4 * 2048 + 256 + BM * 4
    smem = 3 * stage + 6 * BM * 4 + 6 * 256
    m.touch(launch, "LDS", smem, 0, 2 * stage + BM * 128 + 4 * 2 * 1024 + 256 + (max(1, BM // 64) - 1) * 256 + 4 * min(64, BM))
    m.touch(launch, "LDS", smem, 3 * stage, 3 * stage + 6 * BM * 4 + 5 * 256 + 64 * 4)
    assert smem <= 160 << 10 and {1: 4, 2: 3, 4: 2}[rt] * smem <= 160 << 10     # (as many workgroups to a compute unit as planned)
    Np, part_strips = Ng * 32, Ng // parts
    assert Ng % parts == 0 and (parts == 1 or N == part_strips * 32)
    last_strip = [((s // part_strips) * rows + rows - 1) * N + min(N, (s - s // part_strips * part_strips) * 32 + 32) for s in range(Ng)]
    if S > 1:
        first = at["partial sums"][0]
        if S <= 12 and nbx * nby <= TICKETS // 4:
            # a row block's sums strip by strip, pairs of rows in 16 bytes per lane, the last of an odd number by itself in 8
            ends = []
            for by in range(nby):
                tile_rows = min(BM, rows - by * BM)
                rr = np.arange(0, tile_rows, 2)
                end = np.where(rr + 1 < tile_rows, rr * 128 + 15 * 16 + 16, rr * 128 + 15 * 8 + 8).max()
                assert end == tile_rows * 128                                   # (a strip's place, filled)
                ends.append(((by * BM) * Np + (Ng - 1) * 32 * tile_rows) * 4 + int(end))
            m.touch(launch, "partial sums", at["partial sums"], first, first + (S - 1) * rows * Np * 4 + max(ends))
            m.touch(launch, "counters", TICKETS, 0, max(by * nbx + bx for bx, by in grid) * 4 + 4)
        else:
            m.touch(launch, "partial sums", at["partial sums"], first, first + ((S - 1) * rows * Np + (rows - 1) * Np + Np) * 4)
            launch += ", then the sum"
            m.touch(launch, "partial sums", at["partial sums"], first,
                    first + ((parts - 1) * N + (S - 1) * rows * Np + (rows - 1) * Np + (N + 3) // 4 * 4) * 4)
    m.touch(launch, "result", y_bytes, 0, max(last_strip) * 4)
    if residual:
        m.touch(launch, "residual", y_bytes, 0, max(last_strip) * 4)


def product_g32_part(m, name, rows, Ng, Kg, ws_bytes):
    """launch_gemm, group 32: partial sums [split][rows][Ng * 32], added by a second launch"""
    _, S = m.plan(rows, Ng, Kg, 32)
    at = layout(rows, Kg, 32, ws_bytes)["partial sums"]
    if S > 1:
        m.touch(name, "partial sums", at, at[0], at[0] + S * rows * Ng * 32 * 4)


def quantization(m, name, rows, Kg, ws_bytes, x_bytes, glu=False, norm=False):
    """rmsnorm_quant_kernel (norm), quant_x_tile128_kernel: codes and the pairs [Kg][rows], nothing else"""
    at, K = layout(rows, Kg, 128, ws_bytes), Kg * 128
    if norm:
        vpt = 1 if K <= 4096 else 2 if K <= 8192 else 4
        e = np.arange(vpt * 1024) * 4
        last = int(e[e < K].max()) + 4
        assert last == K
        m.touch(name, "norm weights", K * 4, 0, last * 4)
    else:
        # 8 rows x 1 or 4 k-groups to a workgroup; rows and k-groups past the end re-read the last and store nothing
        U = 4 if -(-rows // 8) * -(-Kg // 4) >= 1024 else 1
        kb = np.minimum(np.arange(-(-Kg // U) * U), Kg - 1)
        assert kb.max() == Kg - 1
    m.touch(name, "input", x_bytes, 0, ((rows - 1) * (2 if glu else 1) * K + (2 * K if glu else K)) * 4)
    m.touch(name, "codes", at["codes"], at["codes"][0], at["codes"][0] + (rows - 1) * K + K)
    m.touch(name, "pairs", at["pairs"], at["pairs"][0], at["pairs"][0] + ((Kg - 1) * rows + rows - 1) * 8 + 8)


def attention(m, rows, H, past, maxlen, half):
    S, e = 128, 2 if half else 4
    q_bytes, plane = rows * H * S * 4, H * maxlen * S * e
    ws_bytes = m.lib.llmops_attention_workspace_bytes(1, rows, H, S, maxlen)
    head = 65536
    part = head + up(maxlen * 4)
    k, r, n = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert m.lib.llmops_test_attn_plan(1, rows, H, maxlen, past, int(half), ctypes.byref(k), ctypes.byref(r), ctypes.byref(n)) == 0
    assert k.value == 3 and (n.value - 1) * r.value < min(past + rows, maxlen) <= n.value * r.value
    kv = min(past + rows, maxlen)
    slot = np.arange(past, past + rows)
    # rotation, cache update and, by workgroups of their own in front, the table of which token wrote a cache row
    tables = -(-kv // 64)
    table = np.arange(tables * 64)
    m.touch("rotation", "token of a cache row", (head, part), head, head + int(table[table < kv].max()) * 4 + 4)
    m.touch("rotation", "slots", rows * 4, 0, (rows - 1) * 4 + 4)
    for what, lo in (("k rows of the cache", 0), ("v rows of the cache", plane)):
        m.touch("rotation", what, (lo, lo + plane), lo + int(slot.min()) * S * e, lo + ((H - 1) * maxlen + int(slot.max())) * S * e + S * e)
    # behind that table the tiles' token ranges, the angles' cosines and sines, the records (what the launch asks the workspace for)
    turns = part + up(tables * 16)
    records = turns + rows * S * 4
    assert records + (H * rows * n.value * 520 if n.value > 1 else 0) <= ws_bytes
    m.touch("rotation", "token ranges of the tiles", (part, turns), part, part + tables * 16)
    m.touch("rotation", "cosines and sines", (turns, records), turns, turns + ((rows - 1) * S + 64 + 63) * 4 + 4)
    group_heads = np.arange(-(-H // 32) * 32)
    for what in ("k", "v"):
        m.touch("rotation", what, q_bytes, 0, (((rows - 1) * H + np.minimum(group_heads, H - 1).max()) * S + 64 + 60) * 4 + 16)
    name = "attention, %d pieces of %d rows" % (n.value, r.value)
    for what, lo in (("k rows of the cache", 0), ("v rows of the cache", plane)):
        m.touch(name, what, (lo, lo + plane), lo, lo + ((H - 1) * maxlen + kv - 1) * S * e + S * e)
    m.touch(name, "token of a cache row", (head, head + kv * 4), head, head + (kv - 1) * 4 + 4)  # (what the table's workgroups wrote)
    m.touch(name, "q", q_bytes, 0, ((rows - 1) * H + H - 1) * S * 4 + (64 + 60) * 4 + 16)
    m.touch(name, "cosines and sines", (turns, records), turns, turns + ((rows - 1) * S + 64 + 60) * 4 + 16)
    if n.value > 1:
        m.touch(name, "records", (records, ws_bytes), records, records + ((H * rows - 1) * n.value + n.value - 1) * 520 + 520)
    m.touch(name, "output", q_bytes, 0, ((rows - 1) * H + H - 1) * S * 4 + S * 4)


@pytest.mark.parametrize("rows", [33, 65, 200, 300, 383, 384, 512, 513, 1000, 2048])
@pytest.mark.parametrize("past,half", [(0, False), (700, True)])
def test_every_address_of_a_prompt_pass(rows, past, half):
    from llmops import _lib
    lib = _lib.load()
    m, H, F, V, heads, table = Model(lib), 4096, 11008, 55296, 32, 1024
    maxlen = max(256, up(past + rows))
    m.touch("embedding", "output", rows * H * 4, 0, (rows - 1) * H * 4 + ((H // 4 - 1) * 4 + 4) * 4)
    m.touch("embedding", "rows", table * H, 0, (table - 1) * H + (H // 4 - 1) * 4 + 4)
    # q, k, v: one product of 384 strips whose stores know the three parts (the call asks for a part's workspace too)
    ws = max(m.need(rows, 384, 32), m.need(rows, 128, 32))
    quantization(m, "rmsnorm and quantization", rows, 32, ws, rows * H * 4, norm=True)
    product(m, "q, k and v", rows, 384, 32, H, m.need(rows, 384, 32), 3 * rows * H * 4, parts=3)
    attention(m, rows, heads, past, maxlen, half)
    quantization(m, "quantization of o's input", rows, 32, m.need(rows, 128, 32), rows * H * 4)
    product(m, "o", rows, 128, 32, H, m.need(rows, 128, 32), rows * H * 4, residual=True)
    quantization(m, "rmsnorm and quantization", rows, 32, m.need(rows, 688, 32), rows * H * 4, norm=True)
    product(m, "gate and up", rows, 688, 32, 2 * F, m.need(rows, 688, 32), rows * 2 * F * 4)
    quantization(m, "silu * up and quantization", rows, 86, m.need(rows, 128, 86), rows * 2 * F * 4, glu=True)
    product(m, "down", rows, 128, 86, H, m.need(rows, 128, 86), rows * H * 4, residual=True)
    quantization(m, "rmsnorm and quantization", rows, 32, m.need(rows, 1728, 32), rows * H * 4, norm=True)
    product(m, "logits", rows, 1728, 32, V, m.need(rows, 1728, 32), rows * V * 4)
    assert not m.bad, m.bad
    assert len(m.seen) > 60


@pytest.mark.parametrize("rows,Ng,Kg,N,parts", [(45, 3, 1, 96, 1), (131, 7, 5, 210, 1), (300, 128, 86, 4090, 1), (97, 33, 8, 352, 3), (4096, 128, 32, 4096, 1)])
def test_ragged_products_stay_inside(rows, Ng, Kg, N, parts):
    """Rows, strips and columns that end inside a tile, a strip and a pair of rows; every split that the kernel finishes itself
    and one more than that, and a plan forced on every tile."""
    from llmops import _lib
    lib = _lib.load()
    m = Model(lib)
    try:
        for tile in (0, 1, 2, 4):
            for split in (0, 1, 2, 5, 12, 13):
                lib.llmops_test_gemm_set_tuning(tile)
                lib.llmops_test_gemm_set_split(split)
                product(m, "tile %d" % tile, rows, Ng, Kg, N, m.need(rows, Ng, Kg), parts * rows * N * 4, parts=parts, residual=parts == 1)
    finally:
        lib.llmops_test_gemm_set_tuning(0)
        lib.llmops_test_gemm_set_split(0)
    assert not m.bad, m.bad


def test_the_model_finds_a_workspace_that_is_too_small():
    """A part of q|k|v with groups of 32, which are products of their own, in a workspace sized for the whole; and partial sums
    of the tiled product with 256 bytes too few."""
    from llmops import _lib
    m = Model(_lib.load())
    whole, part = m.need(512, 384, 128, 32), m.need(512, 128, 128, 32)
    assert whole < part
    product_g32_part(m, "q", 512, 128, 128, part)
    assert not m.bad
    product_g32_part(m, "q", 512, 128, 128, whole)
    assert [b[1] for b in m.bad] == ["partial sums"] and m.bad[0][3] == part
    m.bad.clear()
    assert m.plan(300, 128, 86)[1] > 1
    product(m, "down", 300, 128, 86, 4096, m.need(300, 128, 86) - 256, 300 * 4096 * 4)
    assert [b[1] for b in m.bad] == ["partial sums"]


def streamed(m, name, rows, Ng, Kg, N, ws_bytes, y_bytes, build, parts=1):
    """launch_fc_rows: fc_stream_kernel on codes in the order of tile_code_offset; results [parts][rows][N]"""
    rt, sw, nw, halves = build
    at, Kp = layout(rows, Kg, 128, ws_bytes), Kg * 128
    blocks, units = -(-rows // (16 * rt)), -(-Ng // sw)
    launch = "%s: streamed product of %d rows x %d strips, %d row tiles, %d strips, %d waves%s" % (name, rows, Ng, rt, sw, nw, ", halves" if halves else "")
    per = 2 if halves else 1
    block = np.arange(-(-units // 8) * 8 * blocks * per)
    inn = block % (8 * blocks * per)
    nb0, rb, split = (block // (8 * blocks * per) * 8 + (inn & 7)) * sw, (inn >> 3) % blocks, (inn >> 3) // blocks
    live = nb0 < Ng
    seen = set(zip(nb0[live], rb[live], split[live]))
    assert len(seen) == live.sum() == units * blocks * per                       # every (strips, row block, half) once
    runs = []
    for sp in range(per):
        lo, hi = sp * Kg // per, (sp + 1) * Kg // per
        runs += [(lo + w * (hi - lo) // nw, lo + (w + 1) * (hi - lo) // nw) for w in range(nw)]
    assert [r[0] for r in runs] == [0] + [r[1] for r in runs][:-1] and runs[-1][1] == Kg   # the waves' runs cover K once
    # codes: what the quantization writes fills rows * Kp bytes, each chunk of 16 once, and the loads find a row's chunks
    row, g, jj = np.arange(rows), LANES >> 4, LANES & 15
    first, n = row & ~15, np.minimum(16, rows - (row & ~15))
    kbs = sorted({0, Kg // 2, Kg - 1})
    wrote = {}
    for kb in kbs:
        for chunk in range(8):
            for r, o in zip(row, first * Kp + ((kb * 8 + chunk) * n + (row - first)) * 16):
                assert o not in wrote
                wrote[o] = (r, kb, chunk)
    assert max(wrote) + 16 == at["codes"][1] - at["codes"][0] == rows * Kp
    for b in range(blocks):
        for t in range(rt):
            top = min(b * 16 * rt + 16 * t, (rows - 1) & ~15)
            cnt = min(16, rows - top)
            lane = top * Kp + (g * cnt + np.minimum(jj, cnt - 1)) * 16
            for kb in kbs:
                for h in range(2):
                    off = lane + (kb * 2 + h) * cnt * 64
                    assert off.max() < 1 << 32
                    assert [wrote[o] for o in off] == [(top + min(j, cnt - 1), kb, 4 * h + gg) for j, gg in zip(jj, g)]
    m.touch(launch, "codes", at["codes"], at["codes"][0], at["codes"][0] + max(wrote) + 16)
    lane_x = np.minimum(rows - 1, np.arange(blocks)[:, None] * 16 * rt + np.minimum(LANES, 16 * rt - 1)) * 8
    m.touch(launch, "pairs", at["pairs"], at["pairs"][0], at["pairs"][0] + (Kg - 1) * rows * 8 + int(lane_x.max()) + 8)
    lane_w = 2 * g * 128 + jj * 8 + 9 * 128
    assert lane_w.max() + 8 == 2048
    m.touch(launch, "weights", Ng * Kg * BLK, 0, (Ng - 1) * Kg * BLK + (Kg - 1) * BLK + 2048 + 64 + 15 * 4 + 4)
    assert nw * (32 // sw * (32 * sw + 8) * 4 + 512) <= 64 << 10                # LDS, static
    if halves:
        m.touch(launch, "exchange slots", COUNTERS - TICKETS, 0, ((rows - 1) * Ng + Ng - 1) * 32 * 8 + 32 * 8)
    part_strips = Ng // parts
    m.touch(launch, "result", y_bytes, 0, max(((s // part_strips) * rows + rows - 1) * N + min(N, (s % part_strips) * 32 + 32) for s in range(Ng)) * 4)


@pytest.mark.parametrize("Ng,Kg,N,parts", [(128, 32, 4096, 1), (384, 32, 4096, 3), (688, 32, 22016, 1), (128, 86, 4096, 1), (16, 4, 500, 1), (3, 1, 70, 1)])
def test_streamed_products_stay_inside(Ng, Kg, N, parts):
    """The route and the build that are chosen at 1 to 1024 rows, and every build forced at ragged ones; above 1024 rows never."""
    from llmops import _lib
    lib = _lib.load()
    m, out = Model(lib), [ctypes.c_int() for _ in range(4)]

    def chosen(rows):
        assert lib.llmops_test_fc_stream_plan(rows, Ng, Kg, *[ctypes.byref(o) for o in out]) == 0
        return tuple(o.value for o in out) if out[0].value else None

    took = []
    for rows in (1, 9, 16, 17, 32, 33, 48, 64, 65, 100, 128, 200, 512, 1000, 1025, 2048):
        build = chosen(rows)
        if build:
            took.append(rows)
            streamed(m, "chosen", rows, Ng, Kg, N, m.need(rows, Ng, Kg), parts * rows * N * 4, build, parts)
    assert 1025 not in took and 2048 not in took and 48 in took and 9 in took
    try:
        for rt in (1, 2, 3, 4):
            for sw in (1, 2):
                for nw in (4, 8):
                    for halves in (0, 1):
                        lib.llmops_test_fc_stream_set(rt, sw, nw, halves)
                        for rows in (9, 45, 131):
                            build = chosen(rows)
                            assert build[:3] == (rt, sw, nw)
                            streamed(m, "forced", rows, Ng, Kg, N, m.need(rows, Ng, Kg), parts * rows * N * 4, build, parts)
    finally:
        lib.llmops_test_fc_stream_set(0, 0, 0, 0)
    assert not m.bad, m.bad


@pytest.mark.parametrize("half", [False, True])
def test_an_attention_workspace_of_the_size_asked_holds_the_angles_beside_the_records(half):
    """The tiled prompt kernel rotates q from a table of angles that lies ahead of the records: whatever the heads, tokens and cache,
    a workspace of exactly the size asked has the room."""
    from llmops import _lib
    lib = _lib.load()
    for H in (1, 2, 3, 32):
        for rows in (32, 33, 127, 129, 500, 2048):
            for maxlen in (1, 33, 64, 128, 129, 192, 193, 256, 300, 1000, 4096):
                for past in (0, 1, 100, maxlen // 2, 2 * maxlen):
                    k, r, n = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
                    assert lib.llmops_test_attn_plan(1, rows, H, maxlen, past, int(half), ctypes.byref(k), ctypes.byref(r), ctypes.byref(n)) == 0
                    tables = -(-min(past + rows, maxlen) // 64)
                    need = 65536 + up(maxlen * 4) + up(tables * 16) + rows * 512 + (H * rows * n.value * 520 if n.value > 1 else 0)
                    assert k.value == 3 and need <= lib.llmops_attention_workspace_bytes(1, rows, H, 128, maxlen), (H, rows, maxlen, past)
