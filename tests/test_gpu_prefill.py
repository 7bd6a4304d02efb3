"""GPU tests of the prefill pieces (marked gpu): MFMA layouts, bucketing, the grouped GEMMs, the whole step."""
import numpy as np
import pytest

from dsgx10_amd import lib
from tests import gpu, orc

pytestmark = pytest.mark.gpu


def test_mfma_fp8_layout():
    """one 32x32x64 e4m3 MFMA, operands loaded as the prefill kernels load them, against an exact integer product"""
    rng = np.random.default_rng(5)
    vals = np.array([0.0, 1.0, -1.0, 2.0, -2.0, 3.0, 0.5, -4.0], dtype=np.float32)
    A = vals[rng.integers(0, len(vals), (32, 64))]
    B = vals[rng.integers(0, len(vals), (32, 64))]
    qa, qb = orc.f32_to_e4m3(A), orc.f32_to_e4m3(B)
    assert np.array_equal(orc.e4m3_table()[qa], A)
    raw = gpu.empty(64 * 16 * 4, 0xFF)
    lib.probe_mfma_fp8(gpu.dev(qa), gpu.dev(qb), raw)
    raw = gpu.host(raw, np.float32, (64, 16))
    D = A.astype(np.float64) @ B.astype(np.float64).T
    got = np.empty((32, 32), dtype=np.float64)
    for l in range(64):
        for r in range(16):
            got[8 * (r // 4) + 4 * (l // 32) + r % 4, l % 32] = raw[l, r]
    assert np.array_equal(got, D)


def test_mfma_fp8_k128_layout():
    """one 16x16x128 e4m3 MFMA with the prefill kernels' k order, against an exact integer product"""
    rng = np.random.default_rng(6)
    vals = np.array([0.0, 1.0, -1.0, 2.0, -2.0, 3.0, 0.5, -4.0], dtype=np.float32)
    A = vals[rng.integers(0, len(vals), (16, 128))]
    B = vals[rng.integers(0, len(vals), (16, 128))]
    raw = gpu.empty(64 * 16 * 4, 0xFF)
    lib.probe_mfma_fp8(gpu.dev(orc.f32_to_e4m3(A)), gpu.dev(orc.f32_to_e4m3(B)), raw, form=1)
    raw = gpu.host(raw, np.float32, (64, 16))
    got = np.empty((16, 16), dtype=np.float64)
    for l in range(64):
        for r in range(4):
            got[4 * (l // 16) + r, l % 16] = raw[l, r]
    assert np.array_equal(got, A.astype(np.float64) @ B.astype(np.float64).T)


def test_mfma_fp8_accuracy():
    """What the e4m3 MFMA's own sums are worth: against exact sums of 64 products, the error stays under 1e-4 of
    sum|terms| on data shaped like quantised activations and weights (the GEMV tolerance of the reference,
    test_experts.cu:352-361), but it is far from f32 rounding (a sequential f32 sum: ~1e-8)."""
    rng = np.random.default_rng(7)
    tab = orc.e4m3_table().astype(np.float64)
    worst = 0.0
    for it in range(4):
        qa = orc.f32_to_e4m3((rng.standard_normal((32, 64)) * 100).astype(np.float32))
        qb = orc.f32_to_e4m3((rng.standard_normal((32, 64)) * 100).astype(np.float32))
        raw = gpu.empty(64 * 16 * 4, 0xFF)
        lib.probe_mfma_fp8(gpu.dev(qa), gpu.dev(qb), raw)
        raw = gpu.host(raw, np.float32, (64, 16))
        A, B = tab[qa], tab[qb]
        got = np.empty((32, 32))
        for l in range(64):
            for r in range(16):
                got[8 * (r // 4) + 4 * (l // 32) + r % 4, l % 32] = raw[l, r]
        worst = max(worst, float((np.abs(got - A @ B.T) / (np.abs(A) @ np.abs(B).T)).max()))
    assert worst <= 1e-4, worst


# ---- the whole step against the oracle (FP8 weights, FP8 activations) ------------------------------------------------
from dsgx10_amd import abi  # noqa: E402
from tests import helpers  # noqa: E402


def _prefill(hl, x, idx, w, T, **kw):
    dl = hl.upload()
    ws = gpu.empty(lib.prefill_ws_bytes(dl.w, T), 0)
    yr, ys = gpu.empty(T * hl.H * 4, 0xFF), gpu.empty(T * hl.H * 4, 0xFF)
    lib.moe_prefill(dl.w, gpu.dev(x), gpu.dev(idx), gpu.dev(w), T, ws, yr, ys, **kw)
    return gpu.host(yr, np.float32, (T, hl.H)), gpu.host(ys, np.float32, (T, hl.H)), ws, dl


def test_mfma_fp8_block_rule_live():
    """the oracle's statement of the e4m3 MFMA's block sum (pinned on the CPU by tests/golden/mfma_fp8_k128.npz) against the
    instruction itself on fresh operands: every bit"""
    rng = np.random.default_rng(2718)
    for sa, sb, dens in ((104, 160, 1.0), (30, 300, 1.0), (104, 160, 0.1), (None, None, 1.0), (None, None, 0.05)):
        if sa is None:
            qa, qb = rng.integers(0, 256, (16, 128)).astype(np.uint8), rng.integers(0, 256, (16, 128)).astype(np.uint8)
            qa[(qa & 0x7F) == 0x7F] = 0x21
            qb[(qb & 0x7F) == 0x7F] = 0xA2
        else:
            qa = orc.f32_to_e4m3(np.clip(rng.standard_normal((16, 128)) * sa, -448, 448).astype(np.float32))
            qb = orc.f32_to_e4m3(np.clip(rng.standard_normal((16, 128)) * sb, -448, 448).astype(np.float32))
        qa[rng.random((16, 128)) > dens] = 0
        raw = gpu.empty(64 * 16 * 4, 0xFF)
        lib.probe_mfma_fp8(gpu.dev(qa), gpu.dev(qb), raw, 1)
        raw = gpu.host(raw, np.float32, (64, 16))
        got = np.empty((16, 16), np.float32)
        for l in range(64):
            for r in range(4):
                got[4 * (l // 16) + r, l % 16] = raw[l, r]
        want = orc.mfma_fp8_k128(qa, qb)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), int((got != want).sum())


@pytest.fixture
def unit_rule():
    """the oracle adds a 128-k block's products by the matrix unit's rule (orc_mfma_fp8_k128) instead of sequentially"""
    orc.set_fp8_block_rule(1)
    yield
    orc.set_fp8_block_rule(0)


@pytest.mark.parametrize("H,I,E,topk,T,shared", [(512, 256, 16, 4, 70, "fp8"), (256, 384, 4, 2, 300, None), (1024, 128, 8, 8, 129, "fp8")])
def test_prefill_fp8_against_oracle(H, I, E, topk, T, shared, unit_rule):
    hl = helpers.make_layer(abi.FMT_FP8, H, I, E, topk, min(E, 6), seed=3, shared=shared)
    x, _, idx, w = helpers.rows_and_routing(11, T, H, E, topk, 2.5)
    yr, ys, ws, dl = _prefill(hl, x, idx, w, T)
    v = lib.prefill_view(dl.w, ws, T)
    # the buckets: offsets are the expert counts' prefix sums, perm lists each expert's rows in row order
    P = T * topk
    off = gpu.host(gpu.view(ws, v.off, (E + 1) * 4), np.int32, (E + 1,))
    perm = gpu.host(gpu.view(ws, v.perm, P * 4), np.int32, (P,))
    cnt = np.bincount(idx.reshape(-1), minlength=E)
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(cnt)]))
    for e in range(E):
        assert np.array_equal(perm[off[e]:off[e + 1]], np.nonzero((idx == e).any(axis=1))[0])
    re = gpu.host(gpu.view(ws, v.re, P * 4), np.int32, (T, topk))
    rpos = gpu.host(gpu.view(ws, v.rpos, P * 4), np.int32, (T, topk))
    assert np.array_equal(re, np.sort(idx, axis=1))
    assert all(perm[rpos[t, r]] == t and off[re[t, r]] <= rpos[t, r] < off[re[t, r] + 1] for t in range(T) for r in range(topk))
    hg = gpu.host(gpu.view(ws, v.h, P * I * 2), np.uint16, (P, I))
    hsh = gpu.host(gpu.view(ws, v.hsh, T * I * 2), np.uint16, (T, I)) if shared else None
    nh = nbad = 0
    worst_sum = 0.0
    ref_r, ref_s = np.empty((T, H), np.float32), np.empty((T, H), np.float32)
    seq_r, seq_s = np.empty((T, H), np.float32), np.empty((T, H), np.float32)
    for t in range(T):
        # (1) gate/up + SwiGLU against the oracle that adds each 128-k block by the matrix unit's rule: the same sums, so h
        # differs only where the device's expf() and the host's round silu to different bf16 values (rare), by one step
        o = orc.moe_prefill_fp8_row(hl, x[t], idx[t], w[t])
        ref_r[t], ref_s[t] = o["yr"], o["ys"]
        mine = [hg[rpos[t, r]] for r in range(topk)] + [hsh[t] if shared else np.zeros(I, np.uint16)]
        for r in range(topk + (1 if shared else 0)):
            nbad += int((mine[r] != o["h"][r]).sum())
            nh += I
            a, b = orc.bf16_to_f32(mine[r]).astype(np.float64), orc.bf16_to_f32(o["h"][r]).astype(np.float64)
            step = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(b), 2.0 ** -100))) - 7)
            assert np.all(np.abs(a - b) <= step), np.abs(a - b).max()
        # (2) down + combine from the very h the GPU made: the GEMV tolerance of the reference (test_experts.cu:352-361)
        # against exact sums, and the f32 outputs bit for bit against the oracle's (same block sums, same order of adds)
        o = orc.moe_prefill_fp8_row(hl, x[t], idx[t], w[t], h_in=np.stack(mine))
        worst, bad = helpers.check_sums(yr[t], o["yr64"], o["yrmag"])
        assert bad == 0, (t, worst)
        worst_sum = max(worst_sum, worst)
        assert np.array_equal(yr[t].view(np.uint32), o["yr"].view(np.uint32)), (t, int((yr[t] != o["yr"]).sum()))
        if shared:
            worst, bad = helpers.check_sums(ys[t], o["ys64"], o["ysmag"])
            assert bad == 0, (t, worst)
            worst_sum = max(worst_sum, worst)
            assert np.array_equal(ys[t].view(np.uint32), o["ys"].view(np.uint32)), (t, int((ys[t] != o["ys"]).sum()))
        if t < 24:  # the contract with sequential f32 block sums (the reference's CPU stand-in), for the record below
            orc.set_fp8_block_rule(0)
            o0 = orc.moe_prefill_fp8_row(hl, x[t], idx[t], w[t])
            orc.set_fp8_block_rule(1)
            seq_r[t], seq_s[t] = o0["yr"], o0["ys"]
    assert nbad <= 0.002 * nh, (nbad, nh)
    print("fp8 prefill H=%d I=%d T=%d: h equal %.3f%%, staged |err|/sum|terms| %.2e, end-to-end rel-L2 routed %.2e%s, max-abs %.2e; "
          "against sequential f32 block sums (24 rows): rel-L2 routed %.2e"
          % (H, I, T, 100 - 100.0 * nbad / nh, worst_sum, helpers.rel_l2(yr, ref_r),
             " shared %.2e" % helpers.rel_l2(ys, ref_s) if shared else "", np.abs(yr - ref_r).max(), helpers.rel_l2(yr[:24], seq_r[:24])))
    # (3) end to end against the oracle's own h, the benchmark's bar: relative L2 1e-3, max-abs 2e-2, on the f32 outputs and
    # on their bf16 roundings
    helpers.check_outputs(yr, ref_r)
    if shared:
        helpers.check_outputs(ys, ref_s)
    # (4) the same chunk against the oracle with sequential f32 block sums: inside what evaluations whose sums differ by
    # 2e-6 of their sums of |terms| differ by (tests/test_oracle_moe.py records that spread at the benchmark's shape)
    assert helpers.rel_l2(yr[:24], seq_r[:24]) <= 6e-3
    if shared:
        assert helpers.rel_l2(ys[:24], seq_s[:24]) <= 6e-3


@pytest.mark.parametrize("topk", [5, 6])
def test_prefill_fp8_picks_a_row(topk, unit_rule):
    """the combine with a row's loads batched (4, 6 and 8 picks; the other tests have 4 and 8) and one after the other"""
    test_prefill_fp8_against_oracle(256, 256, 12, topk, 40, "fp8", unit_rule)


@pytest.mark.parametrize("H,I,T", [(512, 640, 20), (1280, 1152, 300)])
def test_prefill_fp8_scale_groups(H, I, T, unit_rule):
    """the rows' scales come for eight 128-k blocks at a time, in the widest tile for four: last groups that are not whole (5, 9 and 10
    blocks; 4 and 8 are one group, fewer are among the shapes above), tiles of a few rows and of 160"""
    test_prefill_fp8_against_oracle(H, I, 4, 2, T, "fp8", unit_rule)


@pytest.mark.parametrize("E,topk,T", [(3, 1, 1), (40, 8, 31), (40, 8, 33), (256, 8, 512), (256, 8, 513), (512, 2, 2048), (5, 1, 4096), (5, 1, 4097)])
def test_prefill_buckets_at_the_edges_of_one_workgroup(E, topk, T):
    """the bucketing as one launch (up to 4096 picks whose masks fit LDS) and as three: offsets, rows in token order, each row's picks in
    expert-id order, words of 32 rows that are full, one row more, and more words than lanes; the factors s2_down * w and the lists of
    tiles by what comes out: the rows that a chunk of some rows more (at 512 and 4096 rows beyond the one launch's picks) or fewer holds
    too have its bits, and some rows the oracle's, from the h that the GPU made"""
    H, I = 256, 128
    hl = helpers.make_layer(abi.FMT_FP8, H, I, E, topk, 3, seed=8, shared=None)
    hl.desc["s2"] = (0.5 + np.arange(3 * E, dtype=np.float32) % 7 / 5)  # (factors that tell the experts apart)
    x, _, idx, w = helpers.rows_and_routing(19, T + 1, H, E, topk, 1.0)
    more, _, _, _ = _prefill(hl, x, idx, w, T + 1)
    few = (T + 1) // 2
    fewer, _, _, _ = _prefill(hl, x[:few], idx[:few], w[:few], few)
    x, idx, w = x[:T], idx[:T], w[:T]
    yr, _, ws, dl = _prefill(hl, x, idx, w, T)
    assert np.array_equal(yr.view(np.uint32), more[:T].view(np.uint32)) and np.array_equal(yr[:few].view(np.uint32), fewer.view(np.uint32))
    v, P = lib.prefill_view(dl.w, ws, T), T * topk
    off = gpu.host(gpu.view(ws, v.off, (E + 1) * 4), np.int32, (E + 1,))
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(np.bincount(idx.reshape(-1), minlength=E))]))
    order = np.argsort(idx.reshape(-1), kind="stable")
    assert np.array_equal(gpu.host(gpu.view(ws, v.perm, P * 4), np.int32, (P,)), order // topk)
    pos = np.empty(P, np.int32)
    pos[order] = np.arange(P)
    by_e = np.argsort(idx, axis=1)
    assert np.array_equal(gpu.host(gpu.view(ws, v.re, P * 4), np.int32, (T, topk)), np.take_along_axis(idx, by_e, 1))
    rpos = np.take_along_axis(pos.reshape(T, topk), by_e, 1)
    assert np.array_equal(gpu.host(gpu.view(ws, v.rpos, P * 4), np.int32, (T, topk)), rpos)
    hg = gpu.host(gpu.view(ws, v.h, P * I * 2), np.uint16, (P, I))
    orc.set_fp8_block_rule(1)
    try:
        for t in sorted({0, T // 2, T - 1}):
            o = orc.moe_prefill_fp8_row(hl, x[t], idx[t], w[t], h_in=np.concatenate([hg[rpos[t]], np.zeros((1, I), np.uint16)]))
            assert np.array_equal(yr[t].view(np.uint32), o["yr"].view(np.uint32)), t
    finally:
        orc.set_fp8_block_rule(0)


def test_prefill_rows_do_not_depend_on_the_chunk():
    """a row's result is the same bits whatever else is in the chunk (bucket positions differ)"""
    H, I, E, topk = 256, 256, 8, 2
    hl = helpers.make_layer(abi.FMT_FP8, H, I, E, topk, 5, seed=4, shared="fp8")
    x, _, idx, w = helpers.rows_and_routing(12, 200, H, E, topk, 1.0)
    yr, ys, _, _ = _prefill(hl, x, idx, w, 200)
    yr2, ys2, _, _ = _prefill(hl, x[50:60], idx[50:60], w[50:60], 10)
    assert np.array_equal(yr[50:60], yr2) and np.array_equal(ys[50:60], ys2)


@pytest.mark.parametrize("H,I", [(256, 128), (1280, 1152)])
def test_prefill_fp8_tile_shapes_give_the_same_bits(H, I):
    """experts whose rows end at the edges of the tiles of 32 and 160 positions and of their 16-position tiles (and one row beyond): every
    row has the bits that it has alone in a chunk, in the smallest tile (with deep rings there)"""
    counts, topk = [1, 8, 9, 32, 33, 64, 65, 160, 161, 321], 1
    hl = helpers.make_layer(abi.FMT_FP8, H, I, len(counts), topk, 5, seed=14, shared="fp8")
    idx = np.repeat(np.arange(len(counts), dtype=np.int32), counts)[:, None].copy()
    T = len(idx)
    x, _, _, w = helpers.rows_and_routing(15, T, H, len(counts), topk, 1.0)
    yr, ys, _, dl = _prefill(hl, x, idx, w, T)
    ends = np.cumsum(counts)
    for t in sorted(set(int(v) for e, n in zip(ends, counts) for v in (e - n, e - 1 - n // 2, e - 1 - n % 16 * (n > 16), e - 1))):
        y1, s1, _, _ = _prefill(hl, x[t:t + 1], idx[t:t + 1], w[t:t + 1], 1)
        assert np.array_equal(yr[t].view(np.uint32), y1[0].view(np.uint32)), t
        assert np.array_equal(ys[t].view(np.uint32), s1[0].view(np.uint32)), t


@pytest.mark.parametrize("T,want", [
    (900, [0, 1, 17, 128, 129, 256, 257, 300, 421, 291]),       # (the rest of the picks over two more experts)
    (580, [159, 160, 161, 320, 321, 0, 1, 33, 5]),              # at the edges of the 160-position tiles
    (640, [160, 320, 0, 160, 480, 160]),                        # full tiles only: no remainders
    (274, [159, 1, 32, 33, 100, 0, 64, 159]),                   # remainders only
], ids=["any", "edges", "full", "remainders"])
def test_prefill_tile_order_does_not_change_a_bit(T, want):
    """dsgx_prefill_cfg::tile_order (the reference's prefill_tuning tord, ds41f engine/kernels/dsk.h:252) only changes which
    workgroup takes which tile: experts of no rows, of a few, of full tiles, of remainders and of both, every order, the same h, yr and
    ys as the order by expert id"""
    H, I, topk = 256, 256, 2
    # rows an expert as given (pairs (a, b), a < b, dealt so that the counts come out)
    if sum(want) < 2 * T:
        want = want + [(2 * T - sum(want)) // 2, (2 * T - sum(want) + 1) // 2]
    E = len(want)
    hl = helpers.make_layer(abi.FMT_FP8, H, I, E, topk, 5, seed=9, shared="fp8")
    x, _, _, w = helpers.rows_and_routing(21, T, H, E, topk, 1.0)
    left = list(want)
    idx = np.zeros((T, topk), np.int32)
    for t in range(T):
        a = int(np.argmax(left))
        left[a] -= 1
        b = int(np.argmax([v if j != a else -1 for j, v in enumerate(left)]))
        left[b] -= 1
        idx[t] = (a, b)
    assert min(left) == 0 and max(left) == 0 and (idx[:, 0] != idx[:, 1]).all()
    ref = None
    for order in (0, 1, 2, -1):
        yr, ys, ws, dl = _prefill(hl, x, idx, w, T, tile_order=order)
        h = gpu.host(gpu.view(ws, lib.prefill_view(dl.w, ws, T).h, T * topk * I * 2), np.uint16, (-1,))
        got = (yr.view(np.uint32), ys.view(np.uint32), h)
        if ref is None:
            ref = got
            assert np.isfinite(yr).all() and np.isfinite(ys).all() and (np.abs(yr).max(axis=1) > 0).all()
        assert all(np.array_equal(a, b) for a, b in zip(ref, got)), order
    with pytest.raises(lib.DsgxError):
        _prefill(hl, x, idx, w, T, tile_order=3)


@pytest.mark.parametrize("fmt,shared,T", [(abi.FMT_FP8, "fp8", 1), (abi.FMT_FP8, "fp8", 128), (abi.FMT_FP8, "fp8", 129), (abi.FMT_FP8, "fp8", 300)])
def test_prefill_shared_expert_in_the_routed_launches(fmt, shared, T):
    """a whole step runs the shared expert's tiles in the routed experts' launches: the bits of its own launches (phase 16)"""
    H, I, E, topk = 512, 256, 8, 2
    hl = helpers.make_layer(fmt, H, I, E, topk, 5, seed=33, shared=shared)
    x, _, idx, w = helpers.rows_and_routing(23, T, H, E, topk, 2.5)
    yr, ys, _, dl = _prefill(hl, x, idx, w, T)
    ws, r2, s2 = gpu.empty(lib.prefill_ws_bytes(dl.w, T), 0), gpu.empty(T * H * 4, 0xFF), gpu.empty(T * H * 4, 0xFF)
    dx, di, dw = gpu.dev(x), gpu.dev(idx), gpu.dev(w)
    for ph in (1, 2, 4, 8, 16):
        lib.moe_prefill(dl.w, dx, di, dw, T, ws, r2, s2, phases=ph)
    assert np.array_equal(gpu.host(r2, np.uint32, (T, H)), yr.view(np.uint32))
    assert np.array_equal(gpu.host(s2, np.uint32, (T, H)), ys.view(np.uint32))


@pytest.mark.parametrize("fmt,shared", [(abi.FMT_FP8, "fp8"), (abi.FMT_INT4, "bf16")], ids=["fp8", "int4-bf16"])
@pytest.mark.parametrize("H,I,T", [(256, 128, 1), (256, 384, 33), (1280, 4096, 250), (1280, 4096, 257), (1280, 4096, 520), (1280, 4096, 1400),
                                   (4096, 1152, 512), (4096, 1152, 700), (4096, 1152, 1030)])
def test_prefill_shared_expert_alone_in_every_shape(fmt, shared, H, I, T):
    """the shared expert as a phase of its own takes tiles of 32, 64 and 160 (FP8) or 128 (BF16) rows while they are one a CU, then two workgroups a
    CU in tiles whose height evens out their rounds: both GEMMs at each, ragged last tiles, K of 1 to 64 blocks, deeper stages than blocks
    of K: the bits that the rows have in the routed experts' launches"""
    E, topk = 3, 1
    hl = helpers.make_layer(fmt, H, I, E, topk, 1, seed=37, shared=shared)
    x, _, idx, w = helpers.rows_and_routing(39, T, H, E, topk, 2.5)
    yr, ys, _, dl = _prefill(hl, x, idx, w, T)
    ws, s2 = gpu.empty(lib.prefill_ws_bytes(dl.w, T), 0x5A), gpu.empty(T * H * 4, 0xFF)
    lib.moe_prefill(dl.w, gpu.dev(x), gpu.dev(idx), gpu.dev(w), T, ws, gpu.empty(T * H * 4), s2, phases=16)
    assert np.isfinite(ys).all() and (np.abs(ys).max(axis=1) > 0).all()
    assert np.array_equal(gpu.host(s2, np.uint32, (T, H)), ys.view(np.uint32))


def test_prefill_argument_errors():
    hl = helpers.make_layer(abi.FMT_BF16, 512, 256, 8, 2, 4, seed=1)
    dl = hl.upload()
    assert lib.prefill_ws_bytes(dl.w, 16) == 0
    with pytest.raises(lib.DsgxError):
        lib.moe_prefill(dl.w, gpu.empty(16), gpu.empty(16), gpu.empty(16), 16, gpu.empty(16), gpu.empty(16), gpu.empty(16))


# ---- bf16 activations (INT4 layers; FP8 layers with act_fp8 = 0): the decode contract row by row -----------------------
def _rows_are_decode_rows(fmt, H, I, E, topk, T, shared, seed, per_row=True, **kw):
    """a chunk row is a decode row (engine/experts/tests/test_prefill.inc:307-373): h and the outputs against the decode oracle.
    per_row: the benchmark's output bar (relative L2 1e-3, max-abs 2e-2) is applied to every row by itself; else to the
    chunk's output tensor as a whole (the FP8 test layers are random codes with a wide range of magnitudes: ONE h value
    that falls on the other side of a bf16 rounding, inside the range of valid f32 sums, moves a small row by 2e-3)."""
    hl = helpers.make_layer(fmt, H, I, E, topk, min(E, 5), seed=seed, shared=shared)
    x, _, idx, w = helpers.rows_and_routing(13, T, H, E, topk, 2.5)
    yr, ys, ws, dl = _prefill(hl, x, idx, w, T, **kw)
    v = lib.prefill_view(dl.w, ws, T)
    P = T * topk
    rpos = gpu.host(gpu.view(ws, v.rpos, P * 4), np.int32, (T, topk))
    re = gpu.host(gpu.view(ws, v.re, P * 4), np.int32, (T, topk))
    hg = gpu.host(gpu.view(ws, v.h, P * I * 2), np.uint16, (P, I))
    hsh = gpu.host(gpu.view(ws, v.hsh, T * I * 2), np.uint16, (T, I)) if shared else None
    assert np.array_equal(re, np.sort(idx, axis=1))
    exact = total = 0
    ref_yr, ref_ys = [], []
    for t in range(T):
        uni = orc.union(idx[t:t + 1], E)
        up = orc.moe_up(hl, x[t:t + 1], uni)
        mine = np.stack([hg[rpos[t, r]] for r in range(topk)] + ([hsh[t]] if shared else []))[:, None, :]
        hv = orc.bf16_to_f32(mine)
        assert np.all((hv >= up["lo"]) & (hv <= up["hi"])), "h outside the range of f32 sums"
        exact += int(((mine == up["h64"]) | ((hv == 0) & (orc.bf16_to_f32(up["h64"]) == 0))).sum())
        total += mine.size
        dn = orc.moe_down(hl, mine, idx[t:t + 1], w[t:t + 1], uni)
        worst, bad = helpers.check_sums(yr[t:t + 1], dn["yr64"], dn["yrmag"], 1e-4)
        assert bad == 0, worst
        full = orc.moe_down(hl, up["h32"], idx[t:t + 1], w[t:t + 1], uni)
        ref_yr.append(full["yr32"][0])
        if per_row:
            helpers.check_outputs(yr[t:t + 1], full["yr32"])
        if shared:
            worst, bad = helpers.check_sums(ys[t:t + 1], dn["ys64"], dn["ysmag"], 1e-4)
            assert bad == 0, worst
            ref_ys.append(full["ys32"][0])
            if per_row:
                helpers.check_outputs(ys[t:t + 1], full["ys32"])
    assert exact >= 0.995 * total, (exact, total)
    helpers.check_outputs(yr, np.stack(ref_yr))
    if shared:
        helpers.check_outputs(ys, np.stack(ref_ys))


@pytest.mark.parametrize("H,I,E,topk,T,shared", [(512, 256, 8, 2, 150, "bf16"), (256, 128, 16, 4, 37, None)])
def test_prefill_int4_against_oracle(H, I, E, topk, T, shared):
    _rows_are_decode_rows(abi.FMT_INT4, H, I, E, topk, T, shared, seed=6)


def test_prefill_int4_lds_staged_kernels_give_the_register_ring_kernels_bits():
    """the INT4 experts' grouped GEMMs (pf_gemm_i4.cuh: both operands staged in LDS by DMA, weights decoded a turn ahead) add
    in the k order of the kernel they replaced (k_pf_gemm16: register ring, kept behind DSGX_PF_I4_OLD=1): yr, ys and h equal
    bit for bit, on a chunk with full and ragged tiles"""
    import os
    H, I, E, topk, T = 512, 256, 4, 2, 300
    hl = helpers.make_layer(abi.FMT_INT4, H, I, E, topk, 4, seed=9, shared="bf16")
    x, _, idx, w = helpers.rows_and_routing(17, T, H, E, topk, 2.5)
    outs = []
    for old in ("0", "1"):
        os.environ["DSGX_PF_I4_OLD"] = old
        try:
            yr, ys, ws, dl = _prefill(hl, x, idx, w, T)
            v = lib.prefill_view(dl.w, ws, T)
            outs.append((yr.view(np.uint32), ys.view(np.uint32), gpu.host(gpu.view(ws, v.h, T * topk * I * 2), np.uint16, (-1,))))
        finally:
            os.environ.pop("DSGX_PF_I4_OLD", None)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("H,I,T", [(256, 128, 9), (256, 384, 20), (512, 640, 64), (768, 1152, 70), (1280, 256, 130)])
def test_prefill_int4_rings_at_the_edges_of_k_and_of_the_tiles(H, I, T):
    """pf_gemm_i4.cuh's rings (two blocks of scales and zero points a load, two of weights for up to 64 rows): one 128-k block, odd
    numbers of them, the shortest pairs; tiles of a few rows, of 64 and over - the register-ring kernel's bits"""
    import os
    E, topk = 4, 4
    hl = helpers.make_layer(abi.FMT_INT4, H, I, E, topk, 4, seed=23, shared=None)
    x, _, idx, w = helpers.rows_and_routing(29, T, H, E, topk, 2.5)
    outs = []
    for old in ("0", "1"):
        os.environ["DSGX_PF_I4_OLD"] = old
        try:
            yr, _, ws, dl = _prefill(hl, x, idx, w, T)
            v = lib.prefill_view(dl.w, ws, T)
            outs.append((yr.view(np.uint32), gpu.host(gpu.view(ws, v.h, T * topk * I * 2), np.uint16, (-1,))))
        finally:
            os.environ.pop("DSGX_PF_I4_OLD", None)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("I", [256, 384])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 48, 49, 65, 96, 97, 128, 129, 161])
def test_prefill_int4_tiles_of_every_height(I, T):
    """pf_gemm_i4.cuh's tiles: 16-row MFMAs for up to 64 positions (by sixteens, odd numbers of them too), 32-row ones for more (96, 128), K in
    pairs of 128-k blocks and an odd number of them, and each redone for large scales - the register-ring kernel's bits"""
    import os
    H, E, topk = 512, 3, 3
    for large in (False, True):
        if large:
            hl, x, idx, w = helpers.int4_layer_with_large_scales(H, I, E, topk, 61, T)
        else:
            hl = helpers.make_layer(abi.FMT_INT4, H, I, E, topk, 3, seed=67, shared=None)
            x, _, idx, w = helpers.rows_and_routing(71, T, H, E, topk, 2.5)
        outs = []
        for old in ("0", "1"):
            os.environ["DSGX_PF_I4_OLD"] = old
            try:
                yr, _, ws, dl = _prefill(hl, x, idx, w, T)
                v = lib.prefill_view(dl.w, ws, T)
                outs.append((yr.view(np.uint32), gpu.host(gpu.view(ws, v.h, T * topk * I * 2), np.uint16, (-1,))))
            finally:
                os.environ.pop("DSGX_PF_I4_OLD", None)
        for a, b in zip(*outs):
            assert np.array_equal(a, b), large


def test_prefill_int4_scales_above_the_fast_decodes_range():
    """scales of 2^116 and more make a workgroup do its tile once more by the routine for every scale: the bits of the
    register-ring kernel, which has that routine only, in tiles of 128 positions and in ragged ones"""
    import os
    H, I, E, topk, T = 512, 256, 4, 2, 300
    hl, x, idx, w = helpers.int4_layer_with_large_scales(H, I, E, topk, 61, T)
    outs = []
    for old in ("0", "1"):
        os.environ["DSGX_PF_I4_OLD"] = old
        try:
            yr, _, ws, dl = _prefill(hl, x, idx, w, T)
            v = lib.prefill_view(dl.w, ws, T)
            outs.append((yr, orc.bf16_to_f32(gpu.host(gpu.view(ws, v.h, T * topk * I * 2), np.uint16, (-1,)))))
        finally:
            os.environ.pop("DSGX_PF_I4_OLD", None)
    for a, b in zip(*outs):
        assert np.isfinite(a).all() and (a != 0).mean() > 0.9 and np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("H,I,E,topk,T,shared", [(512, 256, 8, 2, 150, "fp8"), (1024, 128, 16, 4, 37, None)])
def test_prefill_fp8_bf16_activations_against_oracle(H, I, E, topk, T, shared):
    """FP8 weights under the engine's own prefill contract (prefill.cu:337-352: bf16 activations, per 128-k block the sum
    from zero, then fma(S, sum, acc)): act_fp8 = 0"""
    _rows_are_decode_rows(abi.FMT_FP8, H, I, E, topk, T, shared, seed=8, per_row=False, act_fp8=False)


@pytest.mark.parametrize("fmt,H,I,E,topk,T,shared,kw", [
    (abi.FMT_INT4, 512, 256, 8, 2, 150, "bf16", {}),
    (abi.FMT_INT4, 256, 384, 4, 4, 300, None, {}),
    (abi.FMT_FP8, 512, 256, 8, 2, 150, "fp8", dict(act_fp8=False)),
    (abi.FMT_FP8, 1024, 128, 16, 4, 37, None, dict(act_fp8=False)),
])
def test_prefill_bf16_activations_every_bit_against_the_matrix_unit_oracle(fmt, H, I, E, topk, T, shared, kw):
    """with the bf16 MFMA's order of adds restated in the oracle (pinned on the CPU by tests/golden/mfma_bf16_k32.npz) the
    bf16-activation prefill is checked bit for bit: h of every pick and of the shared expert, yr, ys, on chunks with full
    and ragged tiles (INT4 experts: pf_gemm_i4.cuh; the BF16 and FP8 matrices: k_pf_gemm16)"""
    hl = helpers.make_layer(fmt, H, I, E, topk, min(E, 5), seed=21, shared=shared)
    x, _, idx, w = helpers.rows_and_routing(29, T, H, E, topk, 2.5)
    yr, ys, ws, dl = _prefill(hl, x, idx, w, T, **kw)
    v = lib.prefill_view(dl.w, ws, T)
    P = T * topk
    rpos = gpu.host(gpu.view(ws, v.rpos, P * 4), np.int32, (T, topk))
    hg = gpu.host(gpu.view(ws, v.h, P * I * 2), np.uint16, (P, I))
    hsh = gpu.host(gpu.view(ws, v.hsh, T * I * 2), np.uint16, (T, I)) if shared else None
    rows = list(range(T)) if T <= 40 else sorted(set(np.random.default_rng(1).integers(0, T, 24).tolist()) | {0, T - 1})
    for t in rows:
        o = orc.moe_prefill_b16_row_mfma(hl, x[t], idx[t], w[t])
        mine = np.stack([hg[rpos[t, r]] for r in range(topk)] + ([hsh[t]] if shared else []))
        assert np.array_equal(mine, o["h"]), (t, int((mine != o["h"]).sum()))
        assert np.array_equal(yr[t].view(np.uint32), o["yr"].view(np.uint32)), (t, int((yr[t] != o["yr"]).sum()))
        if shared:
            assert np.array_equal(ys[t].view(np.uint32), o["ys"].view(np.uint32)), (t, int((ys[t] != o["ys"]).sum()))


@pytest.mark.parametrize("H,I,T", [(256, 128, 1), (512, 384, 128), (1024, 256, 129), (256, 640, 300)])
def test_prefill_int4_bf16_shared_expert_tiles(H, I, T):
    """the BF16 shared expert's tiles (pf_gemm_b16.cuh: two 64-k turns of K and more; one row, one tile, one row over, a ragged third)
    bit for bit against the oracle that adds as the matrix unit does, and in launches of their own the bits that they have in
    the routed experts' launches"""
    E, topk = 8, 2
    test_prefill_bf16_activations_every_bit_against_the_matrix_unit_oracle(abi.FMT_INT4, H, I, E, topk, T, "bf16", {})
    hl = helpers.make_layer(abi.FMT_INT4, H, I, E, topk, 4, seed=27, shared="bf16")
    x, _, idx, w = helpers.rows_and_routing(31, T, H, E, topk, 2.5)
    yr, ys, _, dl = _prefill(hl, x, idx, w, T)
    ws, r2, s2 = gpu.empty(lib.prefill_ws_bytes(dl.w, T), 0x5A), gpu.empty(T * H * 4, 0xFF), gpu.empty(T * H * 4, 0xFF)
    for ph in (1, 2, 4, 8, 16):
        lib.moe_prefill(dl.w, gpu.dev(x), gpu.dev(idx), gpu.dev(w), T, ws, r2, s2, phases=ph)
    assert np.array_equal(gpu.host(r2, np.uint32, (T, H)), yr.view(np.uint32))
    assert np.array_equal(gpu.host(s2, np.uint32, (T, H)), ys.view(np.uint32))


def test_prefill_silu_at_the_ends_of_its_fast_division():
    """silu of the INT4 prefill's epilogue (common.cuh: silu_for_bf16) against the decode kernels', which divide by IEEE's division
    everywhere: h of a BF16 shared expert whose gates are given values, denormal results, zeros and overflowing divisors among them, from
    both (silu4, whose division has ends at +-60: test_dsk_prefill_silu_of_given_gates)"""
    H, I, E, topk = 256, 256, 8, 2
    hl = helpers.make_layer(abi.FMT_INT4, H, I, E, topk, 4, seed=27, shared="bf16")
    dl = hl.upload()
    v = np.concatenate([np.float32([0, -0.0, 1e-40, -1e-40, 59.75, -59.75, 60, -60, 60.25, -60.25, 87, -87, 88.5, -88.5, 103, -103, 1e30, -1e30, 1e38, -1e38]),
                        np.linspace(-70, 70, I - 20, dtype=np.float32)])
    bgu = np.zeros((2 * I, H), np.uint16)
    bgu[0::2, 0] = orc.f32_to_bf16(v)           # gate of channel c: v[c] x[0]
    bgu[1::2, 1] = orc.f32_to_bf16(np.float32([1.0]))[0]  # up: x[1]
    keep = gpu.dev(bgu)
    dl.w.sh.bgu = keep.data_ptr()
    x, _, idx, w = helpers.rows_and_routing(31, 1, H, E, topk, 2.5)
    x[:] = 0
    x[0, :2] = orc.f32_to_bf16(np.float32([1.0, 3.0]))
    ws, yr, ys = gpu.empty(lib.prefill_ws_bytes(dl.w, 1), 0), gpu.empty(H * 4), gpu.empty(H * 4)
    lib.moe_prefill(dl.w, gpu.dev(x), gpu.dev(idx), gpu.dev(w), 1, ws, yr, ys, act_fp8=False)
    pv = lib.prefill_view(dl.w, ws, 1)
    h = gpu.host(gpu.view(ws, pv.hsh, I * 2), np.uint16, (I,))
    _, _, wd = gpu.decode_layer(dl, x, idx, w, 1, up=1)
    assert np.array_equal(h, gpu.h_of(wd, dl, 1, topk)[-1][0])
    g = orc.bf16_to_f32(orc.f32_to_bf16(v)).astype(np.float64)
    with np.errstate(over="ignore"):
        ref = 3.0 * (g / (1.0 + np.exp(-g)))
    assert np.allclose(orc.bf16_to_f32(h), ref, rtol=2.0 ** -6, atol=1e-37)


def test_prefill_silu_of_every_finite_bf16_gate():
    """the prefill epilogues' silu (common.cuh: silu_for_bf16) rounds every bf16 gate to the bits of the decode kernels' (expf and IEEE's
    division): row t of a one-hot x picks column t of a BF16 shared expert's gate matrix, 256 rows x 256 channels; the up values are 1"""
    H, I, E, topk, T = 256, 256, 8, 2, 256
    hl = helpers.make_layer(abi.FMT_INT4, H, I, E, topk, 4, seed=27, shared="bf16")
    dl = hl.upload()
    v = np.arange(65536, dtype=np.uint16)
    v[(v & 0x7F80) == 0x7F80] = 0x3F80  # (one infinite or NaN weight would reach every row of its channel)
    bgu = np.zeros((2 * I, H), np.uint16)
    bgu[0::2] = v.reshape(I, H)
    bgu[1::2] = 0x3F80
    keep = gpu.dev(bgu)
    dl.w.sh.bgu = keep.data_ptr()
    _, _, idx, w = helpers.rows_and_routing(31, T, H, E, topk, 2.5)
    x = np.zeros((T, H), np.uint16)
    x[np.arange(T), np.arange(T)] = 0x3F80
    ws, yr, ys = gpu.empty(lib.prefill_ws_bytes(dl.w, T), 0), gpu.empty(T * H * 4), gpu.empty(T * H * 4)
    lib.moe_prefill(dl.w, gpu.dev(x), gpu.dev(idx), gpu.dev(w), T, ws, yr, ys, act_fp8=False)
    h = gpu.host(gpu.view(ws, lib.prefill_view(dl.w, ws, T).hsh, T * I * 2), np.uint16, (T, I))
    for t0 in range(0, T, 8):
        _, _, wd = gpu.decode_layer(dl, x[t0:t0 + 8], idx[t0:t0 + 8], w[t0:t0 + 8], 8, up=1)
        o = gpu.h_of(wd, dl, 8, topk)[-1]
        for m in range(8):
            assert np.array_equal(h[t0 + m], o[m]), t0 + m


def test_prefill_fp8_silu_of_given_gates_exact_and_by_the_plain_formula():
    """the FP8 prefill's silu rounds every bf16 gate met here - all significands of both signs, row by row of powers of two up to those that
    overflow - to the bits of the decode kernels'; with fast_act four gates are others, as dsgx.h lists them"""
    H, I, E, topk = 256, 512, 8, 2
    hl = helpers.make_layer(abi.FMT_FP8, H, I, E, topk, 4, seed=27, shared="fp8")
    dl = hl.upload()
    exps = np.arange(-22, 116)  # (beyond, the decode kernels' sums overflow before their scale of 2^-90)
    T = len(exps)
    code = lambda v: orc.f32_to_e4m3(np.asarray(v, np.float32))
    sig, sign = 128 + np.arange(I) % 128, np.where(np.arange(I) // 128 % 2 == 0, 1.0, -1.0)
    gate, up = np.zeros((I, H), np.uint8), np.zeros((I, H), np.uint8)
    gate[:, 0], gate[:, 1] = code(sign * (sig >> 4)), code(sign * (sig & 15))  # g = +-(256 hi + 16 lo) 2^e s
    up[:, 129] = code(1.0)
    gs, us = np.ones((I // 128, H // 128), np.float32), np.full((I // 128, H // 128), 2.0 ** -8, np.float32)
    gs[:2], gs[2:] = 2.0 ** 4, 2.0 ** -90
    keep = [gpu.dev(a) for a in (gate, gs, up, us)]
    dl.w.sh.g, dl.w.sh.gs, dl.w.sh.u, dl.w.sh.us = [k.data_ptr() for k in keep]
    x = np.zeros((T, H), np.float32)
    x[:, 0], x[:, 1], x[:, 2] = 256 * 2.0 ** exps, 16 * 2.0 ** exps, 448 * 2.0 ** exps  # (the largest makes the block's scale 2^e)
    x[:, 128], x[:, 129] = 448, 256
    x = orc.f32_to_bf16(x)
    _, _, idx, w = helpers.rows_and_routing(31, T, H, E, topk, 2.5)

    def prefill(fast):
        ws, yr, ys = gpu.empty(lib.prefill_ws_bytes(dl.w, T), 0), gpu.empty(T * H * 4), gpu.empty(T * H * 4)
        lib.moe_prefill(dl.w, gpu.dev(x), gpu.dev(idx), gpu.dev(w), T, ws, yr, ys, fast_act=fast)
        return gpu.host(gpu.view(ws, lib.prefill_view(dl.w, ws, T).hsh, T * I * 2), np.uint16, (T, I))
    h, hf = prefill(False), prefill(True)
    nan = lambda b: (b & 0x7FFF) > 0x7F80
    for t0 in range(0, T, 8):
        n = min(8, T - t0)
        _, _, wd = gpu.decode_layer(dl, x[t0:t0 + n], idx[t0:t0 + n], w[t0:t0 + n], n, up=1)
        hd = gpu.h_of(wd, dl, n, topk)[-1]
        assert np.array_equal(np.where(nan(hd), 0x7FC0, hd), np.where(nan(h[t0:t0 + n]), 0x7FC0, h[t0:t0 + n])), t0
    with np.errstate(over="ignore"):
        g = (sign * sig * 16.0 * np.repeat(gs[:, 0], 128)[None, :]) * 2.0 ** exps[:, None]
        g32 = g.astype(np.float32)
    assert nan(h[g32 == -np.inf]).all() and (h[g32 == np.inf] == 0x7F80).all() and np.isinf(g32).any()
    other = (h != hf) & ~(nan(h) & nan(hf))
    assert sorted(set(g[other].tolist())) == [-88.5, -88.0, -87.5, 5.9375]
    assert (hf[other & (g < 0)] == 0x8000).all()
