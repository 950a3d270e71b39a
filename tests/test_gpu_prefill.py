"""Prefill path (pre -> decode-fused grouped GEMM -> mid -> grouped GEMM -> post through the C ABI) against the float64
oracle and against the decode kernels run in 8-token slices (the reference's own cross-check, sm120/smoke_prefill.py)."""
import numpy as np
import pytest
import torch

from nestquant_amd import format as F, moe as M
from oracle import nq_oracle as O
from tests.test_gpu_moe import experts_on_gpu, oracle_layer, to_dev
from tests.util import oracle_plane, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"


def gumbel_topk(T, E, k, seed, skew=1.1):
    """Zipf(skew) expert popularity, k distinct experts per token (Gumbel top-k, as sm120/smoke_prefill.py:77-78)"""
    g = torch.Generator().manual_seed(seed)
    p = torch.arange(1, E + 1, dtype=torch.float64) ** -skew
    p = (p / p.sum())[torch.randperm(E, generator=g)]
    u = torch.rand(T, E, generator=g, dtype=torch.float64).clamp_min(1e-300)
    ids = torch.topk(p.log()[None] - torch.log(-torch.log(u)), k, dim=-1).indices
    w = torch.rand(T, k, generator=g) + 0.1
    return ids.to(DEV), (w / w.sum(1, keepdim=True)).half().to(DEV)


def sliced_decode(L, x, sel, rw):
    out = torch.empty(x.shape[0], x.shape[1], dtype=torch.float32, device=DEV)
    for i in range(0, x.shape[0], 8):
        L(x[i:i + 8], sel[i:i + 8].contiguous(), rw[i:i + 8].contiguous(), out=out[i:i + 8])
    return out


def test_small_prefill_vs_oracle_and_slices():
    H, I, NE, T, K = 512, 256, 10, 70, 4
    rk = [(0, 0), (3, 7), (6, 9), (8, 3), (0, 0), (1, 2), (4, 5), (0, 0), (7, 6), (0, 0)]
    ex = experts_on_gpu(H, I, NE, 40, nested_ids=(4, 7, 9), rk=rk, var_ids=(1, 4))
    planes = [(oracle_plane(e.gu), oracle_plane(e.dn), e.nested) for e in ex]
    signs = [e.signs.numpy() for e in ex]
    levels = [2, 4, 4, 4, 3, 4, 4, 4, 2, 0]
    to_dev(ex)
    L = M.MoELayer(NE, H, I, Bmax=8, topk=K)
    for e in range(NE):
        L.set(e, ex[e], levels[e])
    sel, rw = gumbel_topk(T, NE, K, seed=3)
    rw[5, 1] = 0
    g = torch.Generator().manual_seed(4)
    x = (torch.randn(T, H, generator=g) * 0.05).half().to(DEV)
    hits = torch.zeros(NE, dtype=torch.int32, device=DEV)
    L.hits_ptr = hits.data_ptr()
    for R in (None, 64):                                         # one pass, and row chunks that split experts
        hits.zero_()
        y = L.prefill(x, sel, rw, R=R)
        torch.cuda.synchronize()
        want = oracle_layer(planes, levels, signs, x, sel, rw)
        assert rel_err(y.cpu().numpy(), want) < 5e-5, R
        want_hits = torch.bincount(sel[rw != 0].flatten().cpu(), minlength=NE)
        assert hits.cpu().tolist() == want_hits.tolist()
    L.hits_ptr = 0
    ys = sliced_decode(L, x, sel, rw)
    torch.cuda.synchronize()
    assert rel_err(y.cpu().numpy(), ys.cpu().numpy()) < 2e-5


def test_full_shape_prefill_vs_decode_slices():
    """H 6144, I 2048, 16 experts (levels 2/3/4/0), 300 tokens with Zipf popularity: tiles of every height occur"""
    H, I, NE, T = 6144, 2048, 16, 300
    levels = [4, 2, 4, 3, 2, 4, 4, 2, 3, 4, 2, 4, 0, 4, 2, 3]
    nested = tuple(i for i in range(NE) if levels[i] == 3 or i % 2 == 0)
    ex = to_dev(experts_on_gpu(H, I, NE, 500, nested_ids=nested, rk=[(6, 7) if i == 5 else (0, 0) for i in range(NE)]))
    L = M.MoELayer(NE, H, I, Bmax=8)
    for e in range(NE):
        L.set(e, ex[e], levels[e])
    sel, rw = gumbel_topk(T, NE, 8, seed=9)
    g = torch.Generator().manual_seed(10)
    x = (torch.randn(T, H, generator=g) * 0.05).half().to(DEV)
    y = L.prefill(x, sel, rw)
    ys = sliced_decode(L, x, sel, rw)
    torch.cuda.synchronize()
    cnt = torch.bincount(sel.flatten().cpu(), minlength=NE).tolist()
    kinds = M.pf_tiles([(e, 0, c) for e, c in enumerate(cnt) if c])
    assert max(cnt) > 256 and len(kinds) >= 3                    # multi-tile experts and remainder tiles of several heights
    assert rel_err(y.cpu().numpy(), ys.cpu().numpy()) < 5e-5     # two summation orders, each ~1e-5 from exact
    # float64 oracle on a few tokens through HIP-decoded dense weights (the decoder is proved bit-exact elsewhere)
    from tests.test_gpu_moe import _dense_from_gpu
    dense = _dense_from_gpu(ex, levels); signs = [e.signs.cpu().numpy() for e in ex]
    idx = [0, 137, 299]
    want = O.moe_forward(dense, levels, lambda e: signs[e], x[idx].cpu().numpy(), sel[idx].cpu().numpy(), rw[idx].cpu().numpy(), dtype=np.float64)
    assert rel_err(y[idx].cpu().numpy(), want) < 5e-5


@pytest.fixture
def decoded_slots(monkeypatch):
    """how many slots of decoded weights each step since the last call has written, both projections of each: () -> [slots of a step, ...]. (Where slots are
    written, their experts' tiles are nq_pf_wide_k's: both hang on the planner's one decision, and the decode-fused kernel leaves them out.)"""
    steps, block = [], M._pf_block

    def kept(dev, need, extra, capturing=False):
        b, extra = block(dev, need, extra, capturing)
        b[need:].zero_()
        steps.append(b[need:])
        return b, extra
    monkeypatch.setattr(M, "_pf_block", kept)

    def written(H, I):
        torch.cuda.synchronize()
        out = []
        for b in steps:
            gu, dn = b.view(-1, 6 * H * I).split([4 * H * I, 2 * H * I], 1)
            assert torch.equal(gu.any(1), dn.any(1))
            out.append(int(gu.any(1).sum()))
        steps.clear()
        return out
    return written


def test_hot_expert_scratch_gives_the_same_bits(decoded_slots):
    """experts with more than one 256-row tile decoded once into the operand scratch (nq_pf_wdecode; the library itself gives a step this small none): the
    grouped GEMM multiplies the same operands in the same order, so the result is bitwise the one of the decode-fused tiles"""
    H, I, NE, T = 1024, 512, 6, 700
    levels = [4, 2, 3, 4, 2, 4]
    ex = to_dev(experts_on_gpu(H, I, NE, 900, nested_ids=(0, 2, 4)))
    L = M.MoELayer(NE, H, I, Bmax=8)
    for e in range(NE):
        L.set(e, ex[e], levels[e])
    sel, rw = gumbel_topk(T, NE, 2, seed=5)
    g = torch.Generator().manual_seed(6)
    x = (torch.randn(T, H, generator=g) * 0.05).half().to(DEV)
    assert M.PF_HOT_SLOTS == 0
    y0 = L.prefill(x, sel, rw)
    torch.cuda.synchronize()
    cnt = torch.bincount(sel.flatten().cpu(), minlength=NE)
    assert int((cnt >= M.PF_HOT_MIN).sum()) >= 2                  # several experts qualify
    try:
        M.PF_HOT_SLOTS = 1                                       # fewer slots than hot experts: the rest keep decoding per tile
        y1 = L.prefill(x, sel, rw)
        M.PF_HOT_SLOTS = 4
        y2 = L.prefill(x, sel, rw)
        torch.cuda.synchronize()
    finally:
        M.PF_HOT_SLOTS = 0
    assert decoded_slots(H, I) == [0, 1, min(4, int((cnt >= M.PF_HOT_MIN).sum()))]
    assert torch.equal(y0, y1) and torch.equal(y0, y2)
    ys = sliced_decode(L, x, sel, rw)
    torch.cuda.synchronize()
    assert rel_err(y0.cpu().numpy(), ys.cpu().numpy()) < 5e-5


@pytest.mark.parametrize("H,I", [(128, 128), (384, 256), (256, 640), (1024, 512)])        # one chunk; blocks of 128 weight rows; K = 128 .. 1024
def test_tiles_of_decoded_weights_give_the_bits_of_decode_fused_tiles(H, I, decoded_slots):
    """nq_pf_wdecode_k and nq_pf_wide_k at the edges of their tiles: one row more than a remainder that decodes in its GEMM, full tiles, a
    row beyond, several tiles; every level, window codes of several record lengths, sign planes; and the same in chunks of pair rows"""
    rows = [129, 255, 256, 257, 385, 512, 130, 700, 0, 1]
    rk = [(0, 0), (3, 7), (6, 9), (8, 3), (0, 0), (1, 2), (4, 5), (0, 0), (7, 6), (0, 0)]
    ex = to_dev(experts_on_gpu(H, I, len(rows), 77, nested_ids=(4, 7, 9), rk=rk, var_ids=(1, 4)))
    L = M.MoELayer(len(rows), H, I, Bmax=8, topk=1)
    for e, lv in enumerate([4, 4, 4, 4, 3, 2, 4, 4, 2, 4]):
        L.set(e, ex[e], lv)
    g = torch.Generator().manual_seed(78)
    sel = torch.repeat_interleave(torch.arange(len(rows)), torch.tensor(rows))[torch.randperm(sum(rows), generator=g)].view(-1, 1).to(DEV)
    rw = (torch.rand(sel.shape, generator=g) + 0.1).half().to(DEV)
    x = (torch.randn(sel.shape[0], H, generator=g) * 0.05).half().to(DEV)
    try:
        M.PF_HOT_SLOTS = -1
        want = L.prefill(x, sel, rw)
        assert decoded_slots(H, I) == [0]
        for M.PF_HOT_SLOTS, hot_min in ((10, 1), (3, 200)):
            hot, M.PF_HOT_MIN = M.PF_HOT_MIN, hot_min
            got = [L.prefill(x, sel, rw, R=R) for R in (None, 600)]
            M.PF_HOT_MIN = hot
            torch.cuda.synchronize()
            whole, cut = decoded_slots(H, I)                     # nine experts have rows, six of them 200 or more; of a chunk of 600 rows fewer
            assert whole == min(M.PF_HOT_SLOTS, 9 if hot_min == 1 else 6) and 0 < cut <= whole
            assert all(torch.equal(want, y) for y in got), (M.PF_HOT_SLOTS, hot_min)
    finally:
        M.PF_HOT_SLOTS, M.PF_HOT_MIN = 0, 257
    assert want.isfinite().all()


@pytest.mark.parametrize("H,I", [(256, 128), (384, 640)])
def test_decoded_weights_over_the_lists_of_the_plan(H, I):
    """nq_pf_plan, nq_pf_wdecode and nq_pf_gemm one by one, as a caller of the single entry points has them: list 4 with its gaps, decoded weights for some of its
    experts, the same bits as without, rows of other lists left alone"""
    from nestquant_amd import _lib
    Lb, rows, E = _lib.lib(), [300, 0, 129, 90, 1100, 40, 256, 770, 3], 9
    ex = to_dev(experts_on_gpu(H, I, 3, 90, nested_ids=(1,)))
    L = M.MoELayer(E, H, I, Bmax=2, topk=1)
    for e in range(E):
        L.set(e, ex[e % 3], 4 if e % 2 else 2)
    P, cnt = sum(rows), torch.tensor(rows, dtype=torch.int32, device=DEV)
    cap = E + P // 256 + 1
    tiles, hot = torch.empty(5, cap, 4, dtype=torch.int32, device=DEV), torch.empty(E, dtype=torch.int32, device=DEV)
    _lib.check(Lb.nq_pf_plan(cnt.data_ptr(), E, 0, P, tiles.data_ptr(), cap, hot.data_ptr(), 200, 3, _lib.stream_ptr()))
    torch.cuda.synchronize()
    assert hot.tolist() == [0, -1, -1, -1, 1, -1, 2, -1, -1]     # three slots for four experts of 200 rows
    g = torch.Generator().manual_seed(91)
    A0, A1 = [(torch.randn(P, max(H, I), generator=g) * 0.05).half().to(DEV) for _ in range(2)]
    wop = torch.zeros(3, 3 * H * I, dtype=torch.float16, device=DEV)
    for mode in (0, 1):
        _lib.check(Lb.nq_pf_wdecode(L.table.data_ptr(), hot.data_ptr(), E, mode, wop.data_ptr(), wop.numel() * 2, 3, H, I, _lib.stream_ptr()))
        C = [torch.full((P, 2 * I if mode == 0 else H), 7.0, device=DEV) for _ in range(2)]
        for c, w in zip(C, (None, wop.data_ptr())):
            _lib.check(Lb.nq_pf_gemm(L.table.data_ptr(), tiles[4].data_ptr(), cap, 256, mode | 4, A0.data_ptr(), A1.data_ptr(), c.data_ptr(), E, H, I, w, _lib.stream_ptr()))
        torch.cuda.synchronize()
        assert torch.equal(*C)
        tall = torch.zeros(P, dtype=torch.bool)
        for e, r0, n, _ in tiles[4].tolist():
            tall[r0:r0 + n] |= e >= 0
        assert torch.equal((C[1] != 7).any(1).cpu(), tall) and 0 < int(tall.sum()) < P


def test_slots_beyond_a_grid_are_decoded():
    """an expert with a slot of decoded weights beyond the 65535 of one launch (6.4 GB of the smallest shape's): the bytes of slot 0"""
    from nestquant_amd import _lib
    H = I = 128
    slots = 65540
    ex = to_dev(experts_on_gpu(H, I, 2, 89))
    L = M.MoELayer(2, H, I, Bmax=2, topk=1)
    for e in range(2):
        L.set(e, ex[e], 4)
    wop = torch.zeros(slots, 3 * H * I, dtype=torch.float16, device=DEV)
    for hot in ((0, 1), (slots - 1, 65534)):
        h = torch.tensor(hot, dtype=torch.int32, device=DEV)
        for mode in (0, 1):
            _lib.check(_lib.lib().nq_pf_wdecode(L.table.data_ptr(), h.data_ptr(), 2, mode, wop.data_ptr(), wop.numel() * 2, slots, H, I, _lib.stream_ptr()))
    torch.cuda.synchronize()
    assert wop[0].any() and wop[1].any() and not wop[2].any() and not wop[65535].any()
    assert torch.equal(wop[slots - 1], wop[0]) and torch.equal(wop[65534], wop[1])


@pytest.mark.parametrize("bm,rows", [(64, (33, 48, 49, 64)), (128, (1, 65, 80, 81, 96, 97, 112, 113, 128)), (256, (40, 129, 144, 145, 160, 161, 176, 177, 192, 193, 208, 209, 224, 225, 240, 241, 256))])
def test_bodies_of_tall_tiles_give_the_bits_of_16_row_tiles(bm, rows):
    """nq_pf_gemm picks a body by a tile's rows: at the edges of each body the rows come out as in tiles of 16 (which are held against the oracle
    above), and nothing is written beyond them; levels 2 to 4, mask mode and another base window code"""
    from nestquant_amd import _lib
    H, I = 256, 384
    ex = [F.Expert(H, I, seed=6100 + i, dev="cpu", nm_gu=(1 if i == 3 else None), nm_dn=(2 if i == 3 else None), rk_gu=(0, 3, 7, 6, 9)[i], rk_dn=(0, 9, 3, 8, 0)[i],
                   nested=i == 1, var=i in (1, 3), bk_gu=int(i == 4), bk_dn=int(i == 4)) for i in range(5)]
    to_dev(ex)
    L = M.MoELayer(5, H, I, Bmax=4, topk=1)
    for e, lv in enumerate([2, 3, 4, 4, 4]):
        L.set(e, ex[e], lv)
    g = torch.Generator().manual_seed(bm)
    A0, A1 = [(torch.randn(300, max(H, I), generator=g) * 0.05).half().to(DEV) for _ in range(2)]

    def run(mode, kind, tiles, height):
        C = torch.full((300, 2 * I if mode == 0 else H), 7.0, device=DEV)
        t = torch.tensor(tiles, dtype=torch.int32, device=DEV)
        _lib.check(_lib.lib().nq_pf_gemm(L.table.data_ptr(), t.data_ptr(), len(tiles), height, mode | kind, A0.data_ptr(), A1.data_ptr(), C.data_ptr(), 5, H, I, None, None))
        torch.cuda.synchronize()
        return C

    for n in rows:
        for e in range(5):
            for mode in (0, 1):
                kind = 2 * (e >= 3)
                want = run(mode, kind, [[e, 8 + r, min(16, n - r), 0] for r in range(0, n, 16)], 16)
                assert torch.equal(run(mode, kind, [[e, 8, n, 0]], bm), want), (n, e, mode)
                assert want[8:8 + n].isfinite().all() and bool((want[:8] == 7).all() and (want[8 + n:] == 7).all() and (want[8:8 + n] != 7).any(1).all())


def test_a_step_takes_decoded_weights_where_they_pay(decoded_slots):
    """the rule's first step (eight experts of 1100 rows: 32 tiles of a shape whose units are then 512): equal bits with all experts above
    level 2, and with one below, which leaves too few tiles"""
    H = I = 2048
    E, T = 8, 1100
    assert M._lib.lib().nq_pf_wide_slots(T, 8, 8 * T, E, H, I, 1, M.C.byref(M.C.c_int32())) == E
    ex = to_dev(experts_on_gpu(H, I, 4, 79, nested_ids=(1, 3)))
    L = M.MoELayer(E, H, I, Bmax=8, topk=8)
    g = torch.Generator().manual_seed(80)
    sel = torch.stack([torch.randperm(E, generator=g) for _ in range(T)]).to(DEV)
    rw = torch.softmax(torch.randn(T, 8, generator=g), -1).half().to(DEV)
    x = (torch.randn(T, H, generator=g) * 0.05).half().to(DEV)
    for levels in ([4, 4, 4, 3, 4, 4, 4, 3], [4, 4, 4, 3, 2, 4, 4, 3]):
        for e in range(E):
            L.set(e, ex[e % 4], levels[e])
        got = L.prefill(x, sel, rw)
        try:
            M.PF_HOT_SLOTS = -1
            want = L.prefill(x, sel, rw)
        finally:
            M.PF_HOT_SLOTS = 0
        torch.cuda.synchronize()
        assert decoded_slots(H, I) == [0 if 2 in levels else E, 0]
        assert torch.equal(got, want) and got.isfinite().all()


def test_prefill_argument_errors_and_empty():
    L = M.MoELayer(4, 256, 256, Bmax=2, topk=2)
    tb = L.table
    with pytest.raises(RuntimeError, match="tile height"):
        t = torch.tensor([[0, 0, 4, 0]], dtype=torch.int32, device=DEV)
        buf = torch.zeros(8, 512, dtype=torch.float16, device=DEV); c = torch.zeros(8, 512, device=DEV)
        from nestquant_amd import _lib
        _lib.check(_lib.lib().nq_pf_gemm(tb.data_ptr(), t.data_ptr(), 1, 48, 0, buf.data_ptr(), buf.data_ptr(), c.data_ptr(), 4, 256, 256, None, None))
    x = torch.zeros(12, 256, dtype=torch.float16, device=DEV)
    sel = torch.zeros(12, 2, dtype=torch.int64, device=DEV); sel[:, 1] = 1
    rw = torch.full((12, 2), 0.5, dtype=torch.float16, device=DEV)
    y = L.prefill(x, sel, rw)                                    # every expert at level 0: output is zero, nothing faults
    torch.cuda.synchronize()
    assert not y.any()


def test_device_tile_planner_matches_host_lists():
    """nq_pf_plan against pf_tiles (the host construction the reference's prefill uses) for random expert counts and chunk
    windows: the same set of tiles per height, everything else marked as skipped"""
    from nestquant_amd import _lib
    g = torch.Generator().manual_seed(21)
    for E, scale in ((7, 40), (256, 300), (300, 5), (64, 2000)):
        cnt = (torch.rand(E, generator=g) ** 3 * scale).int()
        cnt[torch.randint(0, E, (max(1, E // 5),), generator=g)] = 0
        if E == 64:
            cnt[3] = 256; cnt[4] = 512; cnt[5] = 257; cnt[6] = 16; cnt[7] = 17
        P = int(cnt.sum())
        start = torch.cumsum(cnt, 0) - cnt
        for lo, n in ((0, P), (P // 3, P // 2), (0, 0), (P - 1, 1)) if P else ((0, 0),):
            segs = []
            for e in range(E):
                u, v = max(int(start[e]), lo), min(int(start[e] + cnt[e]), lo + n)
                if v > u:
                    segs.append((e, u - lo, v - u))
            want = {bm: sorted(map(tuple, t.tolist())) for bm, t in M.pf_tiles(segs).items()}
            cap = E + n // 256 + 1
            tiles = torch.full((5, cap, 4), 77, dtype=torch.int32, device=DEV)
            _lib.check(_lib.lib().nq_pf_plan(cnt.to(DEV).data_ptr(), E, lo, n, tiles.data_ptr(), cap, None, 0, 0, None))
            torch.cuda.synchronize()
            t = tiles.cpu()
            for i in range(5):
                used = t[i, : (E if i < 4 else cap)]
                live = used[used[:, 0] >= 0]
                assert sorted(map(tuple, live.tolist())) == want.get(16 << i, []), (E, lo, n, i)
                assert bool((used[used[:, 0] < 0][:, 0] == -1).all())
                covered = sum(r for _, _, r, _ in live.tolist())
            total = sum(int(t[i, : (E if i < 4 else cap)][t[i, : (E if i < 4 else cap), 0] >= 0][:, 2].sum()) for i in range(5))
            assert total == n
    with pytest.raises(RuntimeError, match="cap"):
        _lib.check(_lib.lib().nq_pf_plan(cnt.to(DEV).data_ptr(), 64, 0, 1024, tiles.data_ptr(), 64, None, 0, 0, None))


def test_prefill_on_a_side_stream_matches_the_default_stream():
    """prefill() forks its grouped-GEMM launches onto side streams and joins them again: the result must not depend on which
    stream the caller is on, nor on work the caller queued right before and after it"""
    H, I, NE, T = 512, 256, 8, 200
    ex = to_dev(experts_on_gpu(H, I, NE, 640, rk=[(3, 9)] * NE))
    L = M.MoELayer(NE, H, I, Bmax=8, topk=4)
    for e in range(NE):
        L.set(e, ex[e], (4, 2, 4, 4, 2, 4, 0, 4)[e])
    sel, rw = gumbel_topk(T, NE, 4, seed=3)
    g = torch.Generator().manual_seed(4)
    x = (torch.randn(T, H, generator=g) * 0.05).half().to(DEV)
    want = L.prefill(x, sel, rw).clone()
    torch.cuda.synchronize()
    s2 = torch.cuda.Stream()
    with torch.cuda.stream(s2):
        x2 = x * 1.0                                                # produced on the side stream just before the call
        got = L.prefill(x2, sel, rw)
        got2 = got * 2.0                                            # consumed on it right after
    s2.synchronize()
    assert torch.equal(got, want) and torch.equal(got2, want * 2.0)
    for _ in range(3):                                              # back to back: the scratch is reused, nothing overtakes
        assert torch.equal(L.prefill(x, sel, rw), want)


def test_row_restricted_pre_and_mid_cover_the_rows_of_their_heights_exactly():
    """nq_pf_pre_rows / nq_pf_mid_rows over the five single-height masks write, together, bitwise what nq_pf_pre / nq_pf_mid
    write, each launch only the rows of tiles of its height (everything else keeps the fill value), with the height of a row
    taken from the host construction of the tile lists"""
    from nestquant_amd import _lib
    Lb = _lib.lib()
    H, I, E = 256, 512, 12
    ex = to_dev(experts_on_gpu(H, I, E, 900, rk=[(0, 3)] * E))
    L = M.MoELayer(E, H, I, Bmax=8, topk=2)
    for e in range(E):
        L.set(e, ex[e], 4 if e % 3 else 2)
    g = torch.Generator().manual_seed(77)
    cnt = torch.tensor([0, 5, 16, 17, 40, 64, 100, 129, 256, 300, 513, 31])
    pe = torch.repeat_interleave(torch.arange(E), cnt).int()
    pe[3] = -1; pe[40] = E + 2                                   # rows of no valid expert: height 256 by convention
    n = int(cnt.sum())
    T = 50
    pt = torch.randint(0, T, (n,), generator=g).int()
    x = (torch.randn(T, H, generator=g) * 0.3).half().to(DEV)
    acc = torch.randn(n, 2 * I, generator=g).to(DEV)
    pe_d, pt_d = pe.to(DEV), pt.to(DEV)
    cap = E + n // 256 + 1
    tiles = torch.empty(5, cap, 4, dtype=torch.int32, device=DEV)
    _lib.check(Lb.nq_pf_plan(cnt.int().to(DEV).data_ptr(), E, 0, n, tiles.data_ptr(), cap, None, 0, 0, None))
    # height class of every row from the host lists
    start = torch.cumsum(cnt, 0) - cnt
    cls = torch.full((n,), 4)
    for bm, t in M.pf_tiles([(e, int(start[e]), int(cnt[e])) for e in range(E) if cnt[e]]).items():
        for e, r0, rows, _ in t.tolist():
            cls[r0:r0 + rows] = bm.bit_length() - 5
    cls[3] = cls[40] = 4
    assert sorted(set(cls.tolist())) == [0, 1, 2, 3, 4]

    def pre(rows_mask):
        xg = torch.full((n, H), 7.0, dtype=torch.float16, device=DEV); xu = torch.full_like(xg, 7.0)
        a = (x.data_ptr(), pt_d.data_ptr(), pe_d.data_ptr(), n, L.table.data_ptr(), xg.data_ptr(), xu.data_ptr(), None, E, H, I)
        _lib.check(Lb.nq_pf_pre(*a, None) if rows_mask is None else Lb.nq_pf_pre_rows(*a, tiles.data_ptr(), cap, rows_mask, None))
        return xg.cpu(), xu.cpu()

    def mid(rows_mask):
        h = torch.full((n, I), 7.0, dtype=torch.float16, device=DEV)
        a = (acc.data_ptr(), pe_d.data_ptr(), n, L.table.data_ptr(), h.data_ptr(), None, None, E, H, I)
        _lib.check(Lb.nq_pf_mid(*a, None) if rows_mask is None else Lb.nq_pf_mid_rows(*a, tiles.data_ptr(), cap, rows_mask, None))
        return (h.cpu(),)

    for fn in (pre, mid):
        whole = fn(None)
        for k in range(5):
            part = fn(1 << k)
            for w, q in zip(whole, part):
                mine = cls == k
                assert torch.equal(q[mine], w[mine]) and bool((q[~mine] == 7.0).all()), (fn.__name__, k)
        assert all(torch.equal(a, b) for a, b in zip(fn(31), whole))


@pytest.mark.parametrize("T,E,K,Bmax,xd,wd,sd", [
    (13, 40, 4, 4, torch.bfloat16, torch.float32, torch.int32),        # first grouped size, one-launch plan, rows of every height it has
    (150, 7, 3, 2, torch.float32, torch.bfloat16, torch.int64),        # 64 rows per expert and more: several short tiles of one expert
    (229, 300, 8, 8, torch.float16, torch.float16, torch.int32),       # more experts than a workgroup of the sort has threads' worth of groups
    (5600, 4, 3, 4, torch.float16, torch.float32, torch.int64),        # more pairs than the sort keeps in LDS at a time
])
def test_grouped_step_equals_the_decode_slices(T, E, K, Bmax, xd, wd, sd):
    """moe.forward between the decode call and the long prompts: caller dtypes, ids outside the table, zero weights, an expert at
    level 0, hits -- against fp32 decode slices of the same layer"""
    grouped_step_against_slices(256, 256, T, E, K, Bmax, xd, wd, sd)


@pytest.mark.parametrize("H,I,T,E,K,Bmax,xd,wd,sd", [
    (2560, 2304, 383, 9, 8, 4, torch.float32, torch.bfloat16, torch.int64),     # just beyond the one-launch plan: tall tiles on side streams
    (2048, 1024, 5500, 4, 2, 8, torch.bfloat16, torch.float32, torch.int32),    # many 256-row tiles
])
def test_tall_grouped_step_equals_the_decode_slices(H, I, T, E, K, Bmax, xd, wd, sd):
    grouped_step_against_slices(H, I, T, E, K, Bmax, xd, wd, sd)


def grouped_step_against_slices(H, I, T, E, K, Bmax, xd, wd, sd):
    ex = to_dev(experts_on_gpu(H, I, min(E, 12), 70, nested_ids=(1, 3)))
    L = M.MoELayer(E, H, I, Bmax=Bmax, topk=K)
    for e in range(E):
        L.set(e, ex[e % len(ex)], 0 if e == 2 else 4 if ex[e % len(ex)].nested else 2)
    hits = torch.zeros(E, dtype=torch.int32, device=DEV)
    L.hits_ptr = hits.data_ptr()
    g = torch.Generator().manual_seed(T)
    sel = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(min(T, 256))]).repeat(-(-T // 256), 1)[:T]
    sel[3, 0], sel[T // 2, 1], sel[5] = -1, E + 3, 2
    w = torch.rand(T, K, generator=g) + 0.05
    w[::7, 0] = 0
    x = (torch.randn(T, H, generator=g) * 0.3).to(DEV).to(xd)
    sel, w = sel.to(DEV).to(sd), w.to(DEV).to(wd)
    y = M.forward(L, None, x, w, sel)
    want_hits = hits.clone()
    assert y.dtype == xd and bool(torch.isfinite(y.float()).all())
    want = torch.empty(T, H, dtype=torch.float32, device=DEV)
    hits.zero_()
    for i in range(0, T, Bmax):
        L(x[i:i + Bmax], sel[i:i + Bmax], w[i:i + Bmax], out=want[i:i + Bmax])
    torch.cuda.synchronize()
    assert torch.equal(hits, want_hits)
    tol = {torch.float32: 5e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[xd]
    assert rel_err(y.float().cpu().numpy(), want.cpu().numpy()) < tol
    assert not y[5].any()                                         # all its picks at level 0


@pytest.mark.parametrize("R", [None, 500])
def test_tiles_of_every_list_of_a_tall_step(R):
    """remainders at the edges of the three lists that the GEMMs are launched on, with and without full tiles before them, at levels 0, 2 and 4 (above
    2 first), in one pass and in chunks of pair rows that cut experts: equal to the decode kernels, the same bits without side streams"""
    H, I = 2560, 2304
    rows = [1, 0, 64, 65, 128, 129, 256, 257, 16, 255, 40, 192, 3]
    ex = to_dev(experts_on_gpu(H, I, 6, 83, nested_ids=(1, 3)))
    L = M.MoELayer(len(rows), H, I, Bmax=8, topk=1)
    for e in range(len(rows)):
        L.set(e, ex[e % 6], 0 if e == 8 else 4 if ex[e % 6].nested or e in (2, 4, 11) else 2)
    g = torch.Generator().manual_seed(84)
    sel = torch.repeat_interleave(torch.arange(len(rows)), torch.tensor(rows))[torch.randperm(sum(rows), generator=g)].view(-1, 1).to(DEV)
    rw = (torch.rand(sel.shape, generator=g) + 0.1).half().to(DEV)
    x = (torch.randn(sel.shape[0], H, generator=g) * 0.3).half().to(DEV)
    got = L.prefill(x, sel, rw, R=R)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = L.prefill(x, sel, rw, R=R)
    graph.replay()
    want = sliced_decode(L, x, sel, rw)
    torch.cuda.synchronize()
    assert torch.equal(got, held)
    assert rel_err(got.cpu().numpy(), want.cpu().numpy()) < 5e-5 and not got[sel.flatten() == 8].any()


@pytest.mark.parametrize("E,T,R", [(3, 1000, None), (3, 1000, 900), (2, 1600, None), (16, 520, None)])
def test_tile_lists_are_read_to_their_end_only(E, T, R):
    """steps whose rows could make more tiles than their lists hold (few experts, no remainders to speak of), in memory that is full of valid
    tiles of expert 0 and of nothing finite: every row is computed, none by an entry that is not the step's"""
    H, I, K = 2048, 1024, min(E, 8)
    ex = to_dev(experts_on_gpu(H, I, 2, 87, nested_ids=(1,)))
    L = M.MoELayer(E, H, I, Bmax=8, topk=K)
    for e in range(E):
        L.set(e, ex[e % 2], 4 if e % 2 else 2)
    g = torch.Generator().manual_seed(88)
    sel = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).to(DEV)
    rw = (torch.rand(T, K, generator=g) + 0.1).half().to(DEV)
    x = (torch.randn(T, H, generator=g) * 0.3).half().to(DEV)
    want = sliced_decode(L, x, sel, rw)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    n = 4 * T * K * (2 * H + 3 * I) + (1 << 22)                   # beyond the step's scratch
    for junk in ([0, 0, 256, 0], [-1, -1, -1, -1]):              # as floats, 0xffffffff is NaN
        torch.tensor(junk, dtype=torch.int32, device=DEV).repeat(n // 2)
        got = L.prefill(x, sel, rw, R=R)
        torch.cuda.synchronize()
        assert rel_err(got.cpu().numpy(), want.cpu().numpy()) < 5e-5, junk


@pytest.mark.parametrize("H,I,n", [(128, 128, 1), (640, 384, 37), (2176, 512, 2050), (256, 768, 4100)])
def test_row_kernels_against_a_float64_hadamard(H, I, n):
    """nq_pf_pre and nq_pf_mid where chunks do not fill a wavefront's four and where a workgroup takes one, two, more rows"""
    from nestquant_amd import _lib
    Lb = _lib.lib()
    E, T = 3, 11
    ex = to_dev(experts_on_gpu(H, I, E, 31))
    L = M.MoELayer(E, H, I, Bmax=4, topk=1)
    for e in range(E):
        L.set(e, ex[e], 2)
    g = torch.Generator().manual_seed(n)
    pe, pt = torch.randint(-1, E, (n,), generator=g).int().sort().values, torch.randint(0, T, (n,), generator=g).int()
    x, acc = (torch.randn(T, H, generator=g) * 0.3).half(), torch.randn(n, 2 * I, generator=g)
    xg = torch.full((n, H), 7.0, dtype=torch.float16, device=DEV); xu, h = torch.full_like(xg, 7.0), torch.full((n, I), 7.0, dtype=torch.float16, device=DEV)
    xd, ad, ped, ptd = x.to(DEV), acc.to(DEV), pe.to(DEV), pt.to(DEV)
    _lib.check(Lb.nq_pf_pre(xd.data_ptr(), ptd.data_ptr(), ped.data_ptr(), n, L.table.data_ptr(), xg.data_ptr(), xu.data_ptr(), None, E, H, I, None))
    _lib.check(Lb.nq_pf_mid(ad.data_ptr(), ped.data_ptr(), n, L.table.data_ptr(), h.data_ptr(), None, None, E, H, I, None))
    had = torch.ones(1, 1, dtype=torch.float64)
    for _ in range(7):
        had = torch.cat([torch.cat([had, had], 1), torch.cat([had, -had], 1)])
    wht = lambda v: (v.view(n, -1, 128) @ had / 128**0.5).view(n, -1)
    place = torch.tensor([((c >> 5) * 4 + (c >> 1 & 3)) * 8 + 2 * (2 * (c >> 3 & 1) + (c & 1)) + (c >> 4 & 1) for c in range(128)])
    bop = lambda v: torch.empty_like(v).view(n, -1, 128).index_copy_(2, place, v.view(n, -1, 128)).view(n, -1)
    sg = torch.stack([e.signs.cpu().double() for e in ex])[pe.clamp(min=0).long()]
    live = (pe >= 0).double()[:, None]
    xs = x.double()[pt.long()]
    for got, su in ((xg, sg[:, :H]), (xu, sg[:, 2 * H + 3 * I:])):
        assert rel_err(got.cpu().double().numpy(), (bop(wht(xs * su)) * live).numpy()) < 5e-4
    gate, up = wht(acc[:, :I].double().contiguous()) * sg[:, H:H + I], wht(acc[:, I:].double().contiguous()) * sg[:, H + I:H + 2 * I]
    want = bop(wht(torch.nn.functional.silu(gate) * up * sg[:, H + 2 * I:H + 3 * I])) * live
    assert rel_err(h.cpu().double().numpy(), want.numpy()) < 5e-4


class _StepSpy:
    """the library, remembering of each nq_pf_step call where its scratch is and which events it records"""

    def __init__(s):
        from nestquant_amd import _lib
        s.lib, s.calls = _lib.lib(), []

    def __getattr__(s, name):
        return getattr(s.lib, name)

    def nq_pf_step(s, ref, stream):
        a = ref._obj
        s.calls.append((a.xg, a.y + a.rows * a.H * 4, set(a.events)))
        return s.lib.nq_pf_step(ref, stream)


@pytest.mark.parametrize("H,I,T,E,K", [(256, 256, 40, 40, 4), (2560, 2304, 383, 8, 8)])      # the one-launch plan, and the tall tiles on side streams
def test_steps_on_two_streams_share_no_scratch_and_no_event(H, I, T, E, K):
    """two layers of one shape, each on a stream of its own, with both steps in flight at once (a sleep in front of each): no
    common scratch or event, and the results of the layers one after the other"""
    spy, layers, want = _StepSpy(), [], []
    ex = to_dev(experts_on_gpu(H, I, min(E, 4), 310, nested_ids=(1, 3)))
    for i in range(2):
        L = M.MoELayer(E, H, I, Bmax=4, topk=K, mod=spy)
        for e in range(E):
            L.set(e, ex[(e + 3 * i) % len(ex)], 2)
        g = torch.Generator().manual_seed(50 + i)
        sel, rw = gumbel_topk(T, E, K, seed=8 + i)
        layers.append((L, (torch.randn(T, H, generator=g) * 0.3).to(DEV), rw, sel))
        want.append(M.forward(L, None, *layers[i][1:]))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for L, *a in layers:
        for s in streams:
            with torch.cuda.stream(s):
                M.forward(L, None, *a)                            # the streams' first step
    torch.cuda.synchronize()
    for _ in range(3):
        del spy.calls[:]
        got = []
        for (L, *a), s in zip(layers, streams):
            with torch.cuda.stream(s):
                torch.cuda._sleep(20_000_000)
                got.append(M.forward(L, None, *a))
        assert not streams[0].query()                             # the first step has not run when the second one is enqueued
        (lo, hi, ev), (lo2, hi2, ev2) = spy.calls
        assert (hi <= lo2 or hi2 <= lo) and not ev & ev2
        torch.cuda.synchronize()
        assert all(torch.equal(g, w) for g, w in zip(got, want))


def test_scratch_is_as_large_as_pf_bytes_says():
    for H, I, R in ((256, 128, 1), (6144, 2048, 777)):
        S = None
        before = torch.cuda.memory_allocated()
        S = M.pf_scratch(torch.device(DEV), H, I, R)
        assert 0 <= torch.cuda.memory_allocated() - before - M.pf_bytes(H, I, R) < 2 << 20       # the allocator's rounding
        assert S["rows"] == R and {n: tuple(S[n].shape) for n in S if n not in ("rows", "wop")} == dict(
            xg=(R, H), xu=(R, H), acc=(R, 2 * I), h=(R, I), y=(R, H), zg=(R, 4), zd=(R, 4))
        assert S["wop"] is None and M.pf_scratch(torch.device(DEV), H, I, R)["xg"].data_ptr() != S["xg"].data_ptr()


def test_a_step_takes_no_more_than_pf_bytes_says():
    """the most that a step holds of the allocator's memory while it runs: pf_bytes and its lists, decoded weights among them"""
    H = I = 2048
    E, T = 8, 1100
    L = M.MoELayer(E, H, I, Bmax=8, topk=8)
    x, out = torch.zeros(T, H, dtype=torch.float16, device=DEV), torch.empty(T, H, device=DEV)
    sel, rw = torch.arange(E, device=DEV).repeat(T, 1), torch.ones(T, E, dtype=torch.float16, device=DEV)
    slots = M._lib.lib().nq_pf_wide_slots(T, 8, 8 * T, E, H, I, 1, M.C.byref(M.C.c_int32()))
    L.prefill(x, sel, rw, out)                                   # side streams and the like are there
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    L.prefill(x, sel, rw, out)
    took, lists = torch.cuda.max_memory_allocated() - before, M._lib.lib().nq_pf_meta_bytes(T, 8, 8 * T, E)
    assert slots == E and took >= M._pf_offsets(H, I, 8 * T)[1] + slots * 6 * H * I
    # the bound is for any number of experts: five slots more than this layer's eight; 2 MB of the allocator's rounding
    assert took <= M.pf_bytes(H, I, 8 * T) + lists + (2 << 20) and M.pf_bytes(H, I, 8 * T) - took < 6 * 6 * H * I


def test_a_step_that_cannot_have_decoded_weights_runs_without(monkeypatch):
    """the first allocation of a step refused: the same bits in the smaller block, and the next step asks for that one only"""
    H = I = 2048
    E, T = 8, 1100
    ex = to_dev(experts_on_gpu(H, I, 2, 79, nested_ids=(1,)))
    L = M.MoELayer(E, H, I, Bmax=8, topk=8)
    for e in range(E):
        L.set(e, ex[e % 2], 4)
    g = torch.Generator().manual_seed(81)
    x = (torch.randn(T, H, generator=g) * 0.05).half().to(DEV)
    sel, rw = torch.arange(E, device=DEV).repeat(T, 1), (torch.rand(T, E, generator=g) + 0.1).half().to(DEV)
    want, asked, empty = L.prefill(x, sel, rw), [], torch.empty
    limit = M._pf_offsets(H, I, 8 * T)[1] + 6 * H * I            # one expert's decoded weights

    def short(*a, **kw):
        if kw.get("dtype") == torch.uint8 and len(a) == 1:
            asked.append(a[0])
            if a[0] > limit:
                raise torch.OutOfMemoryError("refused")
        return empty(*a, **kw)
    monkeypatch.setattr(M, "_PF_SHORT", {})
    monkeypatch.setattr(M.torch, "empty", short)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: (1 << 20, 1 << 38))
    got = [L.prefill(x, sel, rw) for _ in range(2)]
    torch.cuda.synchronize()
    assert len(asked) == 3 and asked[0] - asked[1] == E * 6 * H * I and asked[2] == asked[1] <= limit
    assert all(torch.equal(y, want) for y in got) and want.isfinite().all()


@pytest.mark.parametrize("H,I,T,E,K", [(256, 256, 13, 40, 3), (2560, 2304, 383, 8, 8)])      # the one-launch plan, and the tall tiles on side streams
def test_a_captured_grouped_step_equals_the_eager_one(H, I, T, E, K):
    """the same kernels under capture: equal bits on every replay, with new inputs in the graph's buffers, longer and shorter eager
    steps and foreign memory in between"""
    ex = to_dev(experts_on_gpu(H, I, min(E, 4), 610, nested_ids=(1, 3)))
    L = M.MoELayer(E, H, I, Bmax=4, topk=K)
    for e in range(E):
        L.set(e, ex[e % len(ex)], 4 if ex[e % len(ex)].nested else 2)
    MB = M.Mailbox(L)
    g = torch.Generator().manual_seed(T)
    x = (torch.randn(T, H, generator=g) * 0.3).to(DEV).bfloat16()
    sel, w = gumbel_topk(T, E, K, seed=2)
    M.forward(L, MB, x, w, sel)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()                                     # the step's first call on this stream is the captured one
    M._PF_SIDE.pop((0, st.cuda_stream), None)
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr, stream=st):
        y = M.forward(L, MB, x, w, sel)
    assert (0, st.cuda_stream) not in M._PF_SIDE                 # and it stays on the stream
    for i in range(4):
        x.copy_((torch.randn(T, H, generator=g) * 0.3).to(DEV))
        s2, w2 = gumbel_topk(T, E, K, seed=3 + i)
        sel.copy_(s2); w.copy_(w2)
        for n in (T, 3 * T, 700 + 900 * i):                      # a longer step each time: its scratch is new memory
            xe = (torch.randn(n, H, generator=g) * 0.3).to(DEV)
            se, we = gumbel_topk(n, E, K, seed=n)
            M.forward(L, MB, xe, we, se)
        want = M.forward(L, MB, x, w, sel)
        junk = [torch.full((1 << 18,), float("nan"), device=DEV) for _ in range(8)]
        y.fill_(float("nan"))
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
        del junk


def test_a_captured_prompt_equals_the_eager_one():
    """prefill() captured: the tall tiles one after the other on the graph's stream"""
    H, I, T, E = 2560, 2304, 1500, 8
    ex = to_dev(experts_on_gpu(H, I, 4, 620, nested_ids=(1, 3)))
    L = M.MoELayer(E, H, I, Bmax=4)
    for e in range(E):
        L.set(e, ex[e % 4], 4 if ex[e % 4].nested else 2)
    x = (torch.randn(T, H, generator=torch.Generator().manual_seed(3)) * 0.3).to(DEV).half()
    sel, w = gumbel_topk(T, E, 8, seed=2)
    want = L.prefill(x, sel, w)
    torch.cuda.synchronize()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        y = L.prefill(x, sel, w)
    for _ in range(3):
        y.fill_(float("nan"))
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(L.prefill(x, sel, w), want)


@pytest.mark.parametrize("H,I", [(640, 384), (256, 1024)])
def test_row_kernels_keep_infinities_and_nan_in_their_chunk(H, I):
    """nq_pf_pre and nq_pf_mid over rows with infinities, NaN, sums beyond fp16 and gates whose exponential overflows: what float64
    gives in the 128 columns they share a Hadamard with, nothing anywhere else"""
    from nestquant_amd import _lib
    Lb = _lib.lib()
    E, n = 2, 12
    ex = to_dev(experts_on_gpu(H, I, E, 33))
    L = M.MoELayer(E, H, I, Bmax=4, topk=1)
    for e in range(E):
        L.set(e, ex[e], 2)
    g = torch.Generator().manual_seed(H)
    x, acc = (torch.randn(n, H, generator=g) * 0.3).half(), torch.randn(n, 2 * I, generator=g)
    clean = x.clone(), acc.clone()
    inf, nan = float("inf"), float("nan")
    for r, v in enumerate((inf, -inf, nan)):
        x[r, 5 + 128 * (r % 2)] = v; acc[r, 200 + r] = v; acc[r + 3, I + 7 + r] = v
    x[3, 130], x[3, 140] = inf, inf                              # inf - inf in half of the outputs
    x[4, :128] = 65504.0                                         # their sum does not fit fp16
    acc[6, :128] = -200.0; acc[7, 128:256] = 200.0               # exp(200) does not fit fp32; the gate is 0, or the value itself
    pe, pt = torch.arange(n).mul(E).div(n, rounding_mode="floor").int().to(DEV), torch.arange(n).int().to(DEV)

    def run(x, acc):
        xg = torch.full((n, H), 7.0, dtype=torch.float16, device=DEV); xu, h = torch.full_like(xg, 7.0), torch.full((n, I), 7.0, dtype=torch.float16, device=DEV)
        xd, ad = x.to(DEV), acc.to(DEV)
        _lib.check(Lb.nq_pf_pre(xd.data_ptr(), pt.data_ptr(), pe.data_ptr(), n, L.table.data_ptr(), xg.data_ptr(), xu.data_ptr(), None, E, H, I, None))
        _lib.check(Lb.nq_pf_mid(ad.data_ptr(), pe.data_ptr(), n, L.table.data_ptr(), h.data_ptr(), None, None, E, H, I, None))
        return [t.cpu().double() for t in (xg, xu, h)]
    had = torch.ones(1, 1, dtype=torch.float64)
    for _ in range(7):
        had = torch.cat([torch.cat([had, had], 1), torch.cat([had, -had], 1)])
    wht = lambda v: ((v.reshape(n, -1, 1, 128) * had).sum(-1) / 128**0.5).reshape(n, -1)      # sums, no products with zero
    place = torch.tensor([((c >> 5) * 4 + (c >> 1 & 3)) * 8 + 2 * (2 * (c >> 3 & 1) + (c & 1)) + (c >> 4 & 1) for c in range(128)])
    bop = lambda v: torch.empty_like(v).view(n, -1, 128).index_copy_(2, place, v.view(n, -1, 128)).view(n, -1)
    sg = torch.stack([e.signs.cpu().double() for e in ex])[pe.cpu().long()]

    def want(x, acc):
        xs = x.double()
        gate, up = wht(acc[:, :I].double()) * sg[:, H:H + I], wht(acc[:, I:].double()) * sg[:, H + I:H + 2 * I]
        act = torch.nn.functional.silu(gate) * up
        return [bop(wht(xs * sg[:, :H])).half().double(), bop(wht(xs * sg[:, 2 * H + 3 * I:])).half().double(),
                bop(wht(act * sg[:, H + 2 * I:H + 3 * I])).half().double()]
    for got, base, ref in zip(run(x, acc), run(*clean), want(x, acc)):
        for kind in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(kind(got), kind(ref)), kind.__name__
        ok = torch.isfinite(ref)
        assert 0 < int((~ok).sum()) < ok.numel() // 2 and rel_err(got[ok].numpy(), ref[ok].numpy()) < 5e-4
        same = (got == base).view(n, -1, 128).all(-1)            # whole chunks
        assert bool(same[8:].all()) and int((~same).sum()) <= 12


@pytest.mark.parametrize("H,I,T,E,K", [(256, 256, 40, 40, 4), (2560, 2304, 383, 8, 8)])      # the one-launch plan, and the tall tiles on side streams
def test_a_token_that_is_not_finite_is_its_own_affair(H, I, T, E, K):
    """NaN or an infinity in a token's activations or weights reaches that token's result, as in the decode call, and no other's"""
    ex = to_dev(experts_on_gpu(H, I, 4, 710, nested_ids=(1, 3)))
    L = M.MoELayer(E, H, I, Bmax=4, topk=K)
    for e in range(E):
        L.set(e, ex[e % 4], 4 if ex[e % 4].nested else 2)
    g = torch.Generator().manual_seed(T)
    x = (torch.randn(T, H, generator=g) * 0.3).to(DEV)
    sel, w = gumbel_topk(T, E, K, seed=4)
    w = w.float()
    clean = M.forward(L, None, x, w, sel)
    x[1, 3], x[T // 2, H - 1], w[T - 1, 0], w[6, 1] = float("nan"), float("inf"), float("inf"), float("nan")
    hit = torch.zeros(T, dtype=torch.bool, device=DEV)
    hit[[1, T // 2, T - 1, 6]] = True
    y = M.forward(L, None, x, w, sel)
    slices = torch.cat([L(x[i:i + 4], sel[i:i + 4], w[i:i + 4]).clone() for i in range(0, T, 4)])
    torch.cuda.synchronize()
    assert torch.equal(y[~hit], clean[~hit])
    assert torch.equal(torch.isfinite(y), torch.isfinite(slices)) and not torch.isfinite(y[hit]).any()


@pytest.mark.parametrize("T,E,K,sd", [(1, 1, 1, torch.int32), (16, 4096, 32, torch.int64), (171, 5, 3, torch.int32), (73, 256, 7, torch.int64), (128, 300, 8, torch.int32),
                                      (4096, 256, 8, torch.int32), (2049, 63, 64, torch.int64), (33001, 1000, 8, torch.int32)])
def test_pairs_are_sorted_by_expert_in_pair_order(monkeypatch, T, E, K, sd):
    """the sort of a grouped step against torch's stable one: a share of 512 pairs per workgroup, one more or fewer, several such
    blocks per workgroup, ids of one bit and of thirteen, ids outside the table (a group behind all others), one popular expert"""
    L = M.MoELayer(E, 128, 128, Bmax=1, topk=K)                      # every row of the table at level 0: nothing is decoded
    g = torch.Generator().manual_seed(T)
    sel = torch.randint(-1, E + 1, (T, K), generator=g)
    sel[torch.rand(T, K, generator=g) < 0.3] = E // 2
    rw = (torch.rand(T, K, generator=g) > 0.2).float()
    hits = torch.zeros(E, dtype=torch.int32, device=DEV)
    L.hits_ptr = hits.data_ptr()
    made, empty = [], torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: made.append(empty(*a, **k)) or made[-1])
    M._pf_step(L, torch.ones(T, 128, dtype=torch.float16, device=DEV), sel.to(DEV, sd), rw.to(DEV), torch.zeros(T, 128, device=DEV), R=T * K)
    monkeypatch.undo()
    P, key = T * K, torch.where((sel < 0) | (sel >= E), E, sel).reshape(-1)
    block = next(t for t in made if t.dtype == torch.uint8).cpu()
    at, parts = M._pf_offsets(128, 128, P)[1], []
    for n in (E, P, P, P):
        parts.append(block[at:at + 4 * n].view(torch.int32).long())
        at += (4 * n + 15) // 16 * 16
    cnt, pe, pt, pos = parts
    order = torch.argsort(key, stable=True)
    assert torch.equal(cnt, torch.bincount(key, minlength=E + 1)[:E])
    assert torch.equal(pos[order], torch.arange(P)) and torch.equal(pt, order // K)
    assert torch.equal(pe, torch.where(key[order] < E, key[order], -1))
    assert torch.equal(hits.cpu().long(), torch.bincount(key[rw.reshape(-1) != 0], minlength=E + 1)[:E])
