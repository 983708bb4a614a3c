"""Edges of the tiled product, of the weight-streaming one and of the launches that were folded together, against the oracle.
Outputs are fp32 sums of exact int32 group sums: 1e-5 of the largest, as elsewhere."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from conftest import max_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import llmops
    return llmops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _inputs(rows, N, K, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((1, rows, K)).astype(np.float32), (rng.standard_normal((N, K)) * 0.02).astype(np.float32),
            rng.standard_normal((1, rows, N)).astype(np.float32))


@pytest.mark.parametrize("tile", [1, 2, 4])
@pytest.mark.parametrize("rows,N,Kg,split", [
    (17, 33, 1, 1), (31, 64, 2, 1), (33, 130, 3, 3), (65, 257, 5, 2), (127, 96, 6, 3), (129, 160, 7, 7), (40, 1000, 13, 12), (131, 32, 25, 12)])
def test_tiled_product_edges(ops, orc, tile, rows, N, Kg, split):
    """Row counts around a tile and a row tile, odd ones (whose last row has a place of its own among the partial sums),
    columns that end inside a strip and strips inside a tile, runs of one k-group up, runs shorter and longer than the LDS slots and than the
    four k-groups whose min term is formed together; with the residual, and parts against the slices of the whole."""
    from llmops import _lib
    lib = _lib.load()
    x, w, res = _inputs(rows, N, 128 * Kg, rows + Kg)
    pw = orc.quant_w(w, 128)
    want = orc.fc(x, pw, N)
    lib.llmops_test_gemm_set_tuning(tile)
    lib.llmops_test_gemm_set_split(split)
    try:
        got = ops.fc_Q4A(dev(x), dev(pw), N).cpu().numpy()
        got_res = ops.fc_Q4A(dev(x), dev(pw), N, residual=dev(res)).cpu().numpy()
        strips = pw.shape[0] - pw.shape[0] % 3
        if strips:
            p3 = dev(pw[:strips])
            whole = ops.fc_Q4A_decode(dev(x), p3, strips * 32)
            parts = ops.fc_Q4A_decode(dev(x), p3, strips * 32, out_parts=3)
            assert torch.equal(torch.cat(list(parts), dim=-1), whole)
    finally:
        lib.llmops_test_gemm_set_tuning(0)
        lib.llmops_test_gemm_set_split(0)
    assert max_rel_err(got, want) <= 1e-5
    assert max_rel_err(got_res, want + res) <= 1e-5


@pytest.fixture(params=["tiled", "tiled, split", "streaming 1 1 8 0", "streaming 2 2 4 1", "streaming 3 1 4 0", "streaming 4 2 8 1"])
def product(request):
    """A product of more than 8 rows (group 128) pinned: the tiled kernel as planned or K in three, builds of the streaming kernel (row tiles,
    strips, waves, K in halves)."""
    from llmops import _lib
    lib, kind = _lib.load(), request.param.split()
    try:
        if kind[0] == "streaming":
            lib.llmops_test_fc_stream_set(*map(int, kind[1:]))
        else:
            lib.llmops_test_gemm_set_tuning(-1)
            lib.llmops_test_gemm_set_split(3 if len(kind) > 1 else 0)
        build = [ctypes.c_int(-1) for _ in range(4)]
        assert lib.llmops_test_fc_stream_plan(100, 16, 8, *[ctypes.byref(b) for b in build]) == 0
        assert [b.value for b in build] == (list(map(int, kind[1:])) if kind[0] == "streaming" else [0, -1, -1, -1])
        yield request.param
    finally:
        lib.llmops_test_fc_stream_set(0, 0, 0, 0)
        lib.llmops_test_gemm_set_tuning(0)
        lib.llmops_test_gemm_set_split(0)


@pytest.mark.parametrize("rows", [40, 300])
def test_product_sums_that_overflow(ops, orc, rows, product):
    """A row whose group sum is beyond fp32 although its values are not: infinite outputs where the min says so, in that
    row and nowhere else."""
    x, w, _ = _inputs(rows, 96, 640, 3)
    x[0, 7, 128:256] = 3e36
    pw = orc.quant_w(w, 128)
    want = orc.fc(x, pw, 96)
    got = ops.fc_Q4A(dev(x), dev(pw), 96).cpu().numpy()
    assert np.isinf(want[0, 7]).all() and np.array_equal(got[0, 7], want[0, 7])
    other = np.arange(rows) != 7
    assert max_rel_err(got[0, other], want[0, other]) <= 1e-5


@pytest.mark.parametrize("rows,Kg", [(37, 8), (131, 17)])
def test_product_rows_stay_their_own(ops, orc, rows, Kg, product):
    """Rows of ordinary, tiny, huge and zero activations side by side: each to 1e-5 of its own largest output (sums of Kg products carry
    Kg * 2^-24).  An infinity or a NaN in one row leaves the bits of all others as they are and no value of its own finite."""
    x, w, _ = _inputs(rows, 290, 128 * Kg, rows + Kg)
    x[0, 2:6] *= 1e-4
    x[0, 6:10] *= 30000.0
    x[0, 10] = 0.0
    x[0, 1, 128:256] = 0.0
    x[0, 17:20] *= 3000.0
    x[0, rows - 1] *= 1e-6
    pw = orc.quant_w(w, 128)
    want = orc.fc(x, pw, 290)[0]
    got = ops.fc_Q4A(dev(x), dev(pw), 290)[0]
    err, scale = np.abs(got.cpu().numpy() - want).max(axis=1), np.abs(want).max(axis=1)
    assert (err <= 1e-5 * scale).all() and (got[10] == 0.0).all()
    x[0, 3, 77], x[0, 35, 1000] = np.inf, np.nan
    hurt = ops.fc_Q4A(dev(x), dev(pw), 290)[0]
    rest = [r for r in range(rows) if r not in (3, 35)]
    assert torch.equal(hurt[rest], got[rest]) and not torch.isfinite(hurt[[3, 35]]).any()


@pytest.mark.parametrize("rows,N", [(9, 70), (33, 300)])
@pytest.mark.parametrize("Kg", [1, 2, 3, 4, 5, 6, 7, 10])
def test_group32_product_last_stage(ops, orc, rows, N, Kg):
    """The group-32 product's stages of four k-groups where the last has one, two, three or all of them, in the only stage and
    behind others: int32 sums exactly; outputs, a row of huge and one of zero activations among them, to 1e-5 of each row's
    own largest (sums of Kg products: Kg * 2^-24)."""
    x, w, res = _inputs(rows, N, 32 * Kg, rows + Kg)
    x[0, 2] *= 30000.0
    x[0, 3] = 0.0
    pw = orc.quant_w(w, 32)
    rng = np.random.default_rng(Kg)
    xq = rng.integers(-127, 128, (rows, 32 * Kg)).astype(np.int8)
    assert np.array_equal(ops.fc_Q4A_partials(dev(xq), dev(pw), use_mfma=1).cpu().numpy(), orc.fc_partials(xq, pw))
    want = orc.fc(x, pw, N)
    got = ops.fc_Q4A(dev(x), dev(pw), N).cpu().numpy()
    scale = np.abs(want[0]).max(axis=1, keepdims=True)
    assert (np.abs(got[0] - want[0]) <= 1e-5 * scale).all() and (got[0, 3] == 0.0).all()
    got = ops.fc_Q4A(dev(x), dev(pw), N, residual=dev(res)).cpu().numpy()
    assert (np.abs(got[0] - (want + res)[0]) <= 1e-5 * np.maximum(scale, np.abs(res[0]).max())).all()


@pytest.mark.parametrize("halves", [0, 1])
@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("strips", [1, 2])
@pytest.mark.parametrize("row_tiles", [1, 2, 3, 4])
def test_streaming_product_every_build(ops, orc, row_tiles, strips, waves, halves):
    """Every build of the weight-streaming product, forced: rows that end inside a row tile, one past it and past a row block, columns
    inside a strip, strips inside a pair (and fewer than the eight of a round of the XCDs), waves with no k-group, one and several; K in
    halves; residual; results in parts; the same bits again (the exchange slots are left empty); the int32 sums."""
    from llmops import _lib
    lib = _lib.load()
    lib.llmops_test_fc_stream_set(row_tiles, strips, waves, halves)
    try:
        for rows, N, Kg in ((9, 33, 1), (17, 290, 5), (16 * row_tiles + 1, 96, 9), (33, 130, 17), (129, 1000, 3)):
            x, w, res = _inputs(rows, N, 128 * Kg, rows + Kg)
            pw = orc.quant_w(w, 128)
            want = orc.fc(x, pw, N)
            tx, tw, tr = dev(x), dev(pw), dev(res)
            got = ops.fc_Q4A(tx, tw, N)
            assert max_rel_err(got.cpu().numpy(), want) <= 1e-5
            assert torch.equal(ops.fc_Q4A(tx, tw, N), got)
            assert max_rel_err(ops.fc_Q4A(tx, tw, N, residual=tr).cpu().numpy(), want + res) <= 1e-5
            if pw.shape[0] >= 3:
                p3 = dev(pw[:pw.shape[0] - pw.shape[0] % 3])
                whole = ops.fc_Q4A_decode(tx, p3, p3.shape[0] * 32)
                assert torch.equal(torch.cat(list(ops.fc_Q4A_decode(tx, p3, p3.shape[0] * 32, out_parts=3)), dim=-1), whole)
            # codes row by row: an input that does not start on 16 bytes takes the general quantization
            flat = torch.empty(tx.numel() + 2, device="cuda")
            flat[2:] = tx.flatten()
            assert max_rel_err(ops.fc_Q4A(flat[2:].view(tx.shape), tw, N).cpu().numpy(), want) <= 1e-5
            # the int32 sums: of codes row by row by themselves, of codes in the order of the loads through outputs that are exact
            xq = np.random.default_rng(rows).integers(-127, 128, (rows, 128 * Kg)).astype(np.int8)
            assert np.array_equal(ops.fc_Q4A_partials(dev(xq), tw, use_mfma=3).cpu().numpy(), orc.fc_partials(xq, pw))
            xe, we = oracle.closed_form_fc_inputs(rows, N, 128 * Kg, seed=rows)
            got = ops.fc_Q4A(dev(xe.reshape(1, rows, 128 * Kg)), ops.offline_FC_quant_Q4A(dev(we), 128), N).cpu().numpy()
            assert np.array_equal(got[0], (xe.astype(np.float64) @ we.astype(np.float64).T).astype(np.float32))
    finally:
        lib.llmops_test_fc_stream_set(0, 0, 0, 0)


@pytest.mark.parametrize("rows", [9, 16, 31, 33, 100, 500])
@pytest.mark.parametrize("N,K", [(512, 512), (4096, 4096), (2090, 1024)])
def test_streaming_product_exact_and_with_a_producer(ops, orc, rows, N, K):
    """Whatever build is chosen: whole-numbered inputs whose result is exact, and rmsnorm and silu(gate) * up in the quantization launch, whose
    codes are those of the separate operators: the same bits."""
    xe, we = oracle.closed_form_fc_inputs(rows, N, K, seed=rows)
    got = ops.fc_Q4A(dev(xe.reshape(1, rows, K)), ops.offline_FC_quant_Q4A(dev(we), 128), N).cpu().numpy()
    assert np.array_equal(got, (xe.astype(np.float64) @ we.astype(np.float64).T).astype(np.float32).reshape(1, rows, N))
    rng = np.random.default_rng(rows)
    pw = ops.offline_FC_quant_Q4A(dev((rng.standard_normal((N, K)) * 0.02).astype(np.float32)), 128)
    x, gu, nw = (dev(rng.standard_normal(s).astype(np.float32)) for s in ((1, rows, K), (1, rows, 2 * K), (K,)))
    assert torch.equal(ops.fc_Q4A_decode(x, pw, N, norm=(nw, 1e-5)), ops.fc_Q4A(ops.rmsnorm_out(x, nw, 1e-5), pw, N))
    assert torch.equal(ops.fc_Q4A_decode(gu, pw, N, glu_in=True), ops.fc_Q4A(ops.silu_mul(gu), pw, N))


@pytest.mark.parametrize("rows", [4, 32, 33, 128])
def test_input_that_does_not_start_on_16_bytes(ops, orc, rows):
    """The general quantization (codes row by row), on either side of the 32 rows from which the tiled kernel takes such an input."""
    x, w, res = _inputs(rows, 300, 1024, rows)
    pw = orc.quant_w(w, 128)
    flat = torch.empty(x.size + 2, device="cuda")
    flat[2:] = dev(x).flatten()
    view = flat[2:].view(x.shape)
    assert max_rel_err(ops.fc_Q4A(view, dev(pw), 300).cpu().numpy(), orc.fc(x, pw, 300)) <= 1e-5
    assert max_rel_err(ops.fc_Q4A(view, dev(pw), 300, residual=dev(res)).cpu().numpy(), orc.fc(x, pw, 300) + res) <= 1e-5


@pytest.mark.parametrize("N,Kg", [(70, 11), (96, 12), (4096, 32), (4128, 32), (8224, 31), (8224, 32)])
def test_rows_either_side_of_the_streaming_kernel(ops, orc, N, Kg):
    """fc_Q4A on either side of the lines between the kernel that quantizes on the fly (2 to 4 rows) and the weight-streaming one, and
    between that and the tiles (around 512 and 1024 rows)."""
    for rows in (2, 3, 4, 5, 8) + ((512, 513, 1024, 1025) if N < 100 else ()):
        x, w, res = _inputs(rows, N, 128 * Kg, rows + Kg)
        pw = orc.quant_w(w, 128)
        want = orc.fc(x, pw, N)
        assert max_rel_err(ops.fc_Q4A(dev(x), dev(pw), N).cpu().numpy(), want) <= 1e-5
        assert max_rel_err(ops.fc_Q4A(dev(x), dev(pw), N, residual=dev(res)).cpu().numpy(), want + res) <= 1e-5


@pytest.mark.parametrize("N,Kg,first", [(20, 24, 6), (33, 32, 6), (480, 63, 6), (256, 64, 5), (480, 64, 5), (512, 64, 4), (250, 23, 9), (96, 11, 9)])
def test_rows_from_which_few_strips_are_streamed(ops, orc, N, Kg, first):
    """Tensors of fewer than 64 strips: fc_Q4A quantizes first from `first` rows on (9: never, up to 8): the bits of that kernel from
    there, of the one-launch kernel below; both against the oracle."""
    from llmops import _lib
    lib = _lib.load()
    for rows in {max(2, first - 1), min(first, 8)}:
        x, w, _ = _inputs(rows, N, 128 * Kg, rows + Kg)
        pw = orc.quant_w(w, 128)
        got = {}
        for routing in (0, 9, 2):
            lib.llmops_test_fc_set_row_routing(routing, routing)
            try:
                got[routing] = ops.fc_Q4A(dev(x), dev(pw), N)
            finally:
                lib.llmops_test_fc_set_row_routing(0, 0)
            assert max_rel_err(got[routing].cpu().numpy(), orc.fc(x, pw, N)) <= 1e-5
        assert torch.equal(got[0], got[2 if rows >= first else 9]) and not torch.equal(got[2], got[9])


@pytest.mark.parametrize("rows", [3, 16, 17, 32])
@pytest.mark.parametrize("N,Kg", [(2048, 1), (2050, 15), (2048, 16), (2080, 35), (2048, 49), (8224, 33), (8224, 66)])
def test_few_row_product_runs(ops, orc, rows, N, Kg):
    """The weight-streaming product where a wave has one k-group, 2, 3, 4 or more of them, halves of K and all of it."""
    x, w, _ = _inputs(rows, N, 128 * Kg, rows + Kg)
    pw = orc.quant_w(w, 128)
    assert max_rel_err(ops.fc_Q4A(dev(x), dev(pw), N).cpu().numpy(), orc.fc(x, pw, N)) <= 1e-5


@pytest.mark.parametrize("rows", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("N,K,off", [(2048, 512, 0), (2048, 512, 2), (8224, 256, 0), (96, 512, 0)])
def test_two_to_eight_rows_with_a_producer(ops, orc, rows, N, K, off):
    """rmsnorm, silu(gate) * up and residual around the product of few rows against the separate operators, on either
    side of the rule that sends them to the quantization launch: rows, strips (64, more than 256, too few), an input that
    does not start on 16 bytes."""
    rng = np.random.default_rng(rows + N + off)
    pw = ops.offline_FC_quant_Q4A(dev((rng.standard_normal((N, K)) * 0.02).astype(np.float32)), 128)

    def shifted(shape):  # (a dense tensor that starts 4 * off bytes behind an allocation)
        flat = dev(rng.standard_normal(int(np.prod(shape)) + off).astype(np.float32))
        return flat[off:].view(shape)

    x, gu, nw = shifted((1, rows, K)), shifted((1, rows, 2 * K)), dev(rng.standard_normal(K).astype(np.float32))
    res = dev(rng.standard_normal((1, rows, N)).astype(np.float32))

    def close(got, want):
        assert max_rel_err(got.cpu().numpy(), want.cpu().numpy()) <= 1e-5

    close(ops.fc_Q4A_decode(x, pw, N, residual=res), ops.fc_Q4A(x, pw, N) + res)
    if off == 0:
        close(ops.fc_Q4A_decode(x, pw, N, norm=(nw, 1e-5)), ops.fc_Q4A(ops.rmsnorm_out(x, nw, 1e-5), pw, N))
    close(ops.fc_Q4A_decode(gu, pw, N, glu_in=True), ops.fc_Q4A(ops.silu_mul(gu), pw, N))
    y, ss = ops.fc_Q4A_decode(x, pw, N, residual=res, want_sumsq=True)
    pad = torch.nn.functional.pad(y.reshape(rows, N).double(), (0, -N % 32))
    assert ((ss.double() - (pad ** 2).reshape(rows, -1, 32).sum(-1)).abs() <= 1e-5 * ss.double().abs().clamp(min=1e-3)).all()


@pytest.mark.parametrize("cache_dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("qL,past,H", [(16, 300, 32), (31, 96, 32), (9, 1000, 32), (22, 200, 16), (23, 200, 16)])
def test_attention_does_not_read_the_rows_it_replaces(ops, qL, past, H, cache_dtype):
    """What the cache held where the call's own rows go, and behind them, must not matter, be it infinities or NaN; rotary
    pairs 64 dims apart (one launch for rotation and scores) and 32 (two)."""
    S, rows = 128, past + qL + 40
    gen = torch.Generator(device="cuda").manual_seed(qL)
    q, k, v = (torch.randn(1, qL, H * S, generator=gen, device="cuda") for _ in range(3))
    clean = torch.randn(2, 1, H, rows, S, generator=gen, device="cuda").to(cache_dtype)
    slots = torch.arange(past, past + qL, dtype=torch.int32, device="cuda")
    slots[2], slots[qL - 1] = 5, rows + 7  # one inside the old rows, one outside the cache
    for half in (64, 32):
        inv = 1.0 / (10000.0 ** (torch.arange(half, device="cuda").float() / half))
        outs = []
        for stale in (0.0, float("nan"), float("inf")):
            cache = clean.clone()
            cache[:, :, :, past:past + qL - 1] = stale
            cache[:, :, :, past + 2] = 1.0  # (row of no token: an old row like the others)
            cache[:, :, :, past + qL - 1:] = stale  # (behind all tokens but one that has no row)
            cache[:, :, :, past + qL - 1] = 1.0
            cache[:, :, :, 5] = stale
            a = [q.clone(), k.clone()]
            ops.attention_rope2(a[0], a[1], v, inv, cache, slots, past, 0)
            outs.append(a + [cache[:, :, :, :past + qL]])  # (what lies behind stays as it was)
        for o in outs[1:]:
            assert all(torch.equal(s, t) for s, t in zip(o, outs[0]))
        assert torch.isfinite(outs[0][0]).all()
