"""The encoder's GPU searches against their torch form on the CPU: the same states, ties included."""
import pytest
import torch

from nestquant_amd import _lib, encode as EN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 2])
@pytest.mark.parametrize("T,L", [(1, 256), (3, 256), (2, 1), (2, 2), (3, 17), (5, 33), (300, 6)])
def test_viterbi_search_equals_the_torch_form(T, L, K):
    """one ring and more rings than are searched at a time; rings shorter, equal and longer than a block of the walk back; targets
    far outside the codebook and on a coarse grid, where equal costs have to go to the smallest predecessor"""
    g = torch.Generator().manual_seed(100 * T + L + K)
    w = torch.randn(T, L, generator=g) * 1.3
    w[::2] = (w[::2] * 2).round() / 2
    w[-1, : max(1, L // 3)] = 9.0
    lut = EN.codebook()
    want = EN.viterbi_ring(w, lut, K)
    assert torch.equal(EN.viterbi_ring(w.cuda(), lut.cuda(), K).cpu(), want)
    if L == 256:
        assert torch.equal(EN.viterbi_rings(w.cuda(), K).cpu(), EN.viterbi_rings(w, K))


@pytest.mark.parametrize("K", [1, 2])
@pytest.mark.parametrize("T,slots,L,position", [(3, 2, 40, False), (4, 3, 9, True), (5, 2, 1, False), (6, 5, 2, True), (7, 3, 33, True), (9, 4, 17, False), (22, 4, 5, True)])
def test_viterbi_search_pass_by_pass(T, slots, L, position, K):
    """more rings than the scratch holds at a time, with a last round that is at most half full: its rings and those before by passes, the same
    states as with a scratch for all of them (whole rings)"""
    g = torch.Generator().manual_seed(T + L)
    w, lut = (torch.randn(T, L, generator=g) * 1.3).cuda(), EN.codebook().cuda()
    def run(n):
        st, scratch = torch.full((T, L), -1, dtype=torch.int64, device="cuda"), torch.empty(n * L * 1024, dtype=torch.int32, device="cuda")
        _lib.check(_lib.lib().nq_viterbi(w.data_ptr(), T, L, K, lut.data_ptr(), st.data_ptr(), scratch.data_ptr(), scratch.numel() * 4, int(position), _lib.stream_ptr()))
        return st.cpu()
    assert torch.equal(run(slots), run(T))


def test_viterbi_ties_on_a_coarse_codebook():
    """a codebook of nine values: many states tie at every step"""
    g = torch.Generator().manual_seed(7)
    lut = EN.codebook().round().clamp(-4, 4)
    w = torch.randint(-3, 4, (4, 64), generator=g).float()
    for K in (1, 2):
        assert torch.equal(EN.viterbi_ring(w.cuda(), lut.cuda(), K).cpu(), EN.viterbi_ring(w, lut, K))


@pytest.mark.parametrize("T,L", [(1, 256), (5, 256), (3, 1), (2, 2), (9, 16), (4, 77)])
def test_second_plane_search_equals_the_torch_form(T, L):
    """plane P4 with P3 frozen: a partly filled last workgroup, rings of one step up, equal costs"""
    g = torch.Generator().manual_seed(T * 1000 + L)
    w = torch.randn(T, L, generator=g)
    w[::2] = w[::2].round()
    a = torch.randint(0, 256, (T, L), generator=g)
    for lut in (EN.codebook(), EN.codebook().round().clamp(-2, 2)):
        assert torch.equal(EN.viterbi_ring_given_p3(w.cuda(), a.cuda(), lut.cuda()).cpu(), EN.viterbi_ring_given_p3(w, a, lut))
    if L == 256:
        st3 = torch.randint(0, 1 << 16, (T, L), generator=g)
        got, want = EN.viterbi_rings_given_p3(w.cuda(), st3.cuda()), EN.viterbi_rings_given_p3(w, st3)
        assert all(torch.equal(p.cpu(), q) for p, q in zip(got, want))


@pytest.mark.parametrize("U,K,signed,metric", [(1, 2, False, None), (5, 1, True, None), (7, 2, True, "columns"), (3, 1, False, "both"), (2, 2, True, "one")])
def test_block_word_fit_equals_the_torch_form(U, K, signed, metric):
    """a refinement stage with plain, column and two-sided cost on the GPU against the same stage in torch on the CPU: the trellis
    targets may differ in the last bit (sums in another order), so states are given; words and values are then the same"""
    g = torch.Generator().manual_seed(10 * U + K)
    target = torch.randn(U, 8, 256, generator=g)
    target[0] *= 1e-3
    base = torch.randint(0, 1 << 16, (U, 8, 256), generator=g)
    res = torch.randint(0, 1 << 16, (U, 8, 256), generator=g)
    near = EN.codebook()[base] + 0.1 * torch.rand(U, 1, 1, generator=g) * EN.codebook()[res]      # a stage that has something to fit
    target[-1] = near[-1]
    sign = (torch.randint(0, 2, (U, 8, 1), generator=g) * 2 - 1).float() if signed else None
    spd = lambda n, *b: (lambda X: X @ X.transpose(-1, -2) / n + torch.eye(n, dtype=torch.float64))(torch.randn(*b, n, n, generator=g, dtype=torch.float64))
    Da = None if metric is None else spd(128) if metric == "one" else spd(128, U)
    Do = spd(16, U) if metric == "both" else None

    def cost(E):
        idx = EN.ring_index().reshape(-1)
        X = torch.empty(U, 2048, dtype=torch.float64); X[:, idx] = E.reshape(U, 2048)
        X = X.reshape(U, 128, 16).transpose(1, 2)
        Y = X @ Da
        return ((Y if Do is None else Do @ Y) * X).sum((1, 2))
    want = EN.encode_residual(target, base, K, sign=sign, states=res, cost=None if Da is None else cost)
    dev = lambda t: None if t is None else t.cuda()
    got = EN.encode_residual(target.cuda(), base.cuda(), K, sign=dev(sign), states=res.cuda(), metric=None if Da is None else (Da.cuda(), dev(Do)))
    for k in ("Mb", "N", "Q"):
        assert torch.equal(got[k].cpu(), want[k]), k
    assert torch.allclose(got["delta"].cpu(), want["delta"], rtol=1e-12)
    # the targets of the stage's own search
    lut = EN.codebook()
    r = (target if sign is None else target * sign).double() - lut[base].double()
    s0 = r.square().mean((1, 2)).sqrt().clamp_min(1e-12) / 1.1
    out = torch.empty_like(target, device="cuda")
    from nestquant_amd import _lib
    args = [t if t is None else t.cuda().contiguous() for t in (target, sign, base, lut)]
    _lib.check(_lib.lib().nq_fit_residual(*[None if t is None else t.data_ptr() for t in args], 1.1, U, out.data_ptr(), None))
    torch.cuda.synchronize()
    assert torch.allclose(out.cpu(), (r / s0[:, None, None]).float(), rtol=2e-7, atol=0)


def test_viterbi_search_looks_at_its_codebook():
    """a short codebook raises as the torch form does; one that fp32 cannot hold, or of another layout, takes the torch form"""
    g = torch.Generator().manual_seed(3)
    w = torch.randn(2, 9, generator=g)
    lut = EN.codebook()
    for bad in (lut[:65535], lut[:16], lut[:0]):
        for dev in ("cpu", "cuda"):
            with pytest.raises(IndexError):
                EN.viterbi_ring(w.to(dev), bad.to(dev))
    with pytest.raises(RuntimeError):
        EN.viterbi_ring(w.cuda(), lut)                            # on another device
    near = lut.double() + 1e-9 * torch.randn(1 << 16, generator=g, dtype=torch.float64)
    for other in (near, lut.half(), lut.repeat(2), lut.repeat_interleave(2)[::2], (lut * 16).round().int()):
        assert torch.equal(EN.viterbi_ring(w.cuda(), other.cuda()).cpu(), EN.viterbi_ring(w, other)), other.dtype


def test_second_plane_search_looks_at_its_inputs():
    """windows of another shape, type or device and short codebooks do on the GPU what they do in torch on the CPU"""
    g = torch.Generator().manual_seed(4)
    w, lut = torch.randn(3, 6, generator=g), EN.codebook()
    win = lambda *s: torch.randint(0, 256, s, generator=g)
    for a in (win(1, 6), win(3, 9), win(3, 6).int(), win(3, 6).short()):
        assert torch.equal(EN.viterbi_ring_given_p3(w.cuda(), a.cuda(), lut.cuda()).cpu(), EN.viterbi_ring_given_p3(w, a, lut)), (a.shape, a.dtype)
    near = lut.double() + 1e-9 * torch.randn(1 << 16, generator=g, dtype=torch.float64)
    assert torch.equal(EN.viterbi_ring_given_p3(w.cuda(), win(3, 6).cuda().fill_(5), near.cuda()).cpu(), EN.viterbi_ring_given_p3(w, win(3, 6).fill_(5), near))
    for bad in (win(3, 5), win(2, 6), win(6), torch.rand(3, 6)):
        with pytest.raises((IndexError, RuntimeError)):
            EN.viterbi_ring_given_p3(w.cuda(), bad.cuda(), lut.cuda())
    with pytest.raises(RuntimeError):
        EN.viterbi_ring_given_p3(w.cuda(), win(3, 6), lut.cuda())
    with pytest.raises(IndexError):
        EN.viterbi_ring_given_p3(w.cuda(), win(3, 6).cuda(), lut.cuda()[:4096])


def test_block_word_fit_looks_at_its_inputs():
    """states, signs and scales of another type or shape do on the GPU what they do in torch on the CPU: int32 states count as the
    same states, broadcast ones are broadcast, others raise"""
    g = torch.Generator().manual_seed(5)
    U = 3
    st, res = (torch.randint(0, 1 << 16, (U, 8, 256), generator=g) for _ in range(2))
    target = EN.codebook()[st] + 0.2 * EN.codebook()[res]
    sign = (torch.randint(0, 2, (U, 8, 1), generator=g) * 2 - 1).float()
    dev = lambda t: t.cuda() if isinstance(t, torch.Tensor) else t
    want = EN.encode_residual(target, st, 1, states=res)
    for a, b in ((st.int(), res), (st, res.int())):
        got = EN.encode_residual(target.cuda(), a.cuda(), 1, states=b.cuda())
        assert all(torch.equal(got[k].cpu(), want[k]) for k in ("Mb", "N", "Q", "states"))
    for base, kw in ((st[:1], dict(states=res)), (st, dict(states=res[:1])), (st, dict(states=res, sign=sign[:1])),
                     (st, dict(states=res, sign=sign.expand(U, 8, 256))), (st, dict(states=res, sign=sign.double())),
                     (st, dict(states=res, scale=torch.tensor([1.0, 1.1, 1.2]))), (st.transpose(1, 2).contiguous().transpose(1, 2), dict(states=res))):
        want = EN.encode_residual(target, base, 1, **kw)
        got = EN.encode_residual(target.cuda(), base.cuda(), 1, **{k: dev(v) for k, v in kw.items()})
        assert got["Q"].dtype == want["Q"].dtype and all(torch.equal(got[k].cpu(), want[k]) for k in ("Mb", "N", "Q")), (base.shape, list(kw))
    for base, b in ((st[:2], res), (st[:, :4], res), (st.reshape(U, 2048), res), (st, res[:, :, :128]), (st.float(), res), (st, res.float())):
        with pytest.raises((RuntimeError, NotImplementedError)):
            EN.encode_residual(target.cuda(), base.cuda(), 1, states=b.cuda())
    with pytest.raises(RuntimeError):
        EN.encode_residual(target.cuda(), st.cuda(), 1, states=res)                   # on another device


def test_side_stream_of_a_fit_outlives_another_threads_clean_up(monkeypatch):
    """a thread that drops the kept side streams between two steps of another one"""
    class Emptied(dict):
        def __setitem__(s, k, v):
            super().__setitem__(k, v)
            s.clear()
    monkeypatch.setattr(EN, "_SIDE", Emptied())
    W = torch.randn(128, 128, generator=torch.Generator().manual_seed(2)).cuda()
    a = EN.encode_nested(W)
    monkeypatch.undo()
    b = EN.encode_nested(W)
    assert all(torch.equal(a[k], b[k]) for k in ("base", "p3", "d3", "p4", "d4"))


@pytest.mark.parametrize("K", [1, 2])
def test_searches_over_targets_that_are_not_finite(K):
    """an infinite or NaN target makes every path equally dear from its step on: ties to the smallest predecessor, as in torch"""
    g = torch.Generator().manual_seed(K)
    w = torch.randn(4, 24, generator=g)
    w[0, 3], w[1, 20], w[2, 11], w[3, 0] = float("inf"), -float("inf"), float("nan"), 3e20      # whose square is infinite
    lut = EN.codebook()
    assert torch.equal(EN.viterbi_ring(w.cuda(), lut.cuda(), K).cpu(), EN.viterbi_ring(w, lut, K))
    a = torch.randint(0, 256, (4, 24), generator=g)
    assert torch.equal(EN.viterbi_ring_given_p3(w.cuda(), a.cuda(), lut.cuda()).cpu(), EN.viterbi_ring_given_p3(w, a, lut))


@pytest.mark.parametrize("K", [1, 2])
@pytest.mark.parametrize("scale", [1e-21, 3e-20, 1e18])
def test_searches_at_the_ends_of_the_range_of_costs(K, scale):
    """costs that are zero, subnormal or close to overflow order as they do in torch, ties included (L 17 and 40: one block of the walk
    back and a remainder, two blocks and a remainder)"""
    g = torch.Generator().manual_seed(K)
    lut = EN.codebook().round().clamp(-5, 5) * scale
    for L in (17, 40):
        w = torch.randint(-6, 7, (3, L), generator=g).float() * scale
        assert torch.equal(EN.viterbi_ring(w.cuda(), lut.cuda(), K).cpu(), EN.viterbi_ring(w, lut, K))


@pytest.mark.parametrize("N,K,signed,nested", [(16, 128, False, False), (48, 384, True, True), (128, 256, True, False), (32, 128, False, True)])
def test_planes_are_packed_as_in_torch(N, K, signed, nested):
    """records, block words, sign bytes and matrices of a fit, from whole rings of random bits, at one unit and at several strips and chunks;
    a ring that does not close, in any plane, raises as it does in torch"""
    g = torch.Generator().manual_seed(N + K)
    U = (N // 16) * (K // 128)

    def states(k):
        sym = torch.randint(0, 1 << k, (U * 8, 256), generator=g)
        return sum(sym[:, (torch.arange(256) + i) % 256] << (k * i) for i in range(16 // k)).reshape(U, 8, 256)
    word = lambda n: torch.randint(0, n, (U,), generator=g)
    e = lambda k: dict(states=states(k), Q=torch.randn(U, 8, 256, generator=g), Mb=word(256), N=word(256))
    fits = {3: e(1), 4: e(2)}
    if nested:
        fits["4n"] = dict(e(2), p4_bits=torch.randint(0, 2, (U, 8, 256), generator=g))
    sign = (torch.randint(0, 2, (U, 8, 1), generator=g) * 2 - 1).float() if signed else None
    st2 = states(2)
    dev = lambda f: {k: {n: t.cuda() for n, t in v.items()} for k, v in f.items()}
    put = lambda t: None if t is None else t.cuda()
    want, got = EN.pack_planes({}, N, K, st2, fits, sign), EN.pack_planes({}, N, K, st2.cuda(), dev(fits), put(sign))
    assert want.keys() == got.keys()
    for k in want:
        assert (want[k] is None and got[k] is None) or (want[k].dtype == got[k].dtype and torch.equal(want[k], got[k].cpu())), k
    if signed:                                                   # a type that the kernel does not read
        got = EN.pack_planes({}, N, K, st2.cuda(), dev(fits), sign.cuda().double())
        assert torch.equal(got["Q"].cpu(), want["Q"].double()) and torch.equal(got["base"].cpu(), want["base"])
    for lvl in (2, 3, 4):
        f, s = {k: dict(v) for k, v in fits.items()}, st2.clone()
        broken = s if lvl == 2 else f[lvl]["states"].clone()
        broken[U - 1, 7, 255] ^= 1 << 15                          # the last state's first bit, whose ring it closes
        if lvl != 2:
            f[lvl]["states"] = broken
        for args in ((s, f, sign), (s.cuda(), dev(f), put(sign))):
            with pytest.raises(AssertionError, match="tail-biting"):
                EN.pack_planes({}, N, K, *args)


@pytest.mark.parametrize("N,K", [(128, 128), (256, 384), (384, 128)])
def test_prepared_weights_equal_the_torch_form(N, K):
    """scales, signs, rotated targets and their ring order; 16-bit and strided weights, a channel of zeros, values that are not finite. The torch form is what a
    float64 weight takes; sums in another order leave 1e-16, which a rounding to fp16 or fp32 shows once in 1e8"""
    g = torch.Generator().manual_seed(N + K)
    W = torch.randn(N, K, generator=g).cuda()
    dead, wild = W.clone(), W.clone()
    dead[:, 5] = 0; dead[7] = 0
    wild[3, 9] = float("inf"); wild[100, 100] = float("nan")
    for w in (W, W.half(), W.bfloat16(), torch.randn(K, N, generator=g).cuda().t(), dead, wild):
        got, want = EN.prepare(w, 11), EN.prepare(w.double(), 11)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num()), w.dtype
        for n in (1, 2):
            rings = EN._prepare_gpu(w, 11, n)[3].nan_to_num()
            assert torch.equal(rings[: N * K // 256], EN.to_rings(got[2]).nan_to_num()) and (n == 1 or torch.equal(rings[N * K // 256:], EN.to_rings(-got[2]).nan_to_num()))


def test_weights_of_more_rows_than_a_launch_takes_have_the_torch_form():
    """8.4 million rows; a view, nothing of it is read"""
    W = torch.zeros(1, 128, device="cuda")
    assert EN._plain_weight(W.expand(65535 * 128, 128)) and not EN._plain_weight(W.expand(65536 * 128, 128))


def test_transformed_weights_take_the_torch_form():
    """a weight with a tangent keeps it, vmap and jvp go through prepare as on the CPU, a gradient comes back: against the same on a float64 weight, which
    no kernel takes; 4 ulp of fp32 for the sums' other order"""
    fw = torch.autograd.forward_ad
    g = torch.Generator().manual_seed(31)
    W, V = torch.randn(2, 128, 256, generator=g).cuda(), torch.randn(2, 128, 256, generator=g).cuda()
    close = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm()) < 2.0**-21
    with fw.dual_level():
        got, want = (EN.prepare(fw.make_dual(W[0].to(t), V[0].to(t)), 3) for t in (torch.float32, torch.float64))
        for a, b in zip(got, want):
            assert torch.equal(fw.unpack_dual(a).primal, fw.unpack_dual(b).primal)
        assert close(fw.unpack_dual(got[2]).tangent, fw.unpack_dual(want[2]).tangent)
        assert fw.unpack_dual(EN.encode_level2(fw.make_dual(W[0], V[0]), 3)["target"]).tangent is not None
    target = lambda w: EN.prepare(w, 3)[2]
    assert close(torch.func.jvp(target, (W[0],), (V[0],))[1], torch.func.jvp(target, (W[0].double(),), (V[0].double(),))[1])
    for a, *b in zip(torch.func.vmap(lambda w: EN.prepare(w, 3), randomness="same")(W), *(EN.prepare(w, 3) for w in W)):
        assert torch.equal(a, torch.stack(b))
    a, b = (torch.func.grad(lambda w: (target(w) * V[1]).sum())(w) for w in (W[0], W[0].double()))
    assert close(a, b)


def test_orientation_of_rings_equals_the_torch_form():
    """each ring fitted as it is and negated: the better of the two, the first where they are equal (a ring of zeros, whose two searches give one path)"""
    g = torch.Generator().manual_seed(12)
    rings = torch.randn(24, 256, generator=g).cuda()
    rings[3] = 0
    got, sign = EN.base_rings(rings, var=True)
    lut = EN.codebook("cuda")
    st = EN.viterbi_rings(torch.cat([rings, -rings]))
    e = (lut[st] - torch.cat([rings, -rings])).double().square().sum(1)
    neg = e[24:] < e[:24]
    assert 0 < int(neg.sum()) < 24 and torch.equal(sign[:, 0], 1.0 - 2.0 * neg.float()) and sign.shape == (24, 1)
    assert torch.equal(got, torch.where(neg[:, None], st[24:], st[:24]))


@pytest.mark.parametrize("m", [1, 2, 5])
def test_block_factors_on_the_gpu(m):
    """L D L^T is the matrix, as far as 64 bits hold it; a matrix that is not positive definite is reported with the order of its first minor that is not"""
    g = torch.Generator().manual_seed(m)
    n = 128 * m
    X = torch.randn(2 * n, n, generator=g, dtype=torch.float64) * (1 + torch.arange(n)) ** -0.5
    H = (X.T @ X / n).cuda()

    def factors(H):
        D, Lc = torch.empty(m, 128, 128, dtype=torch.float64, device="cuda"), [torch.empty(n - 128 * (i + 1), 128, dtype=torch.float64, device="cuda") for i in range(m - 1)]
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        EN._block_ldl_gpu(H, D, Lc, bad)
        L = torch.eye(n, dtype=torch.float64, device="cuda")
        for i, c in enumerate(Lc):
            L[128 * (i + 1):, 128 * i: 128 * (i + 1)] = c
        return L, D, int(bad)
    before = H.clone()
    L, D, bad = factors(H)
    L0, D0 = EN.block_ldl(H)
    assert bad == 0 and torch.equal(H, before)
    assert float((L @ torch.block_diag(*D) @ L.T - H).norm() / H.norm()) < 4e-15
    assert float((D - D0).norm() / D0.norm()) < 1e-13 and float((L - L0).norm() / L0.norm()) < 1e-12
    for at in (0, n // 2 + 3, n - 1):
        B = H.clone()
        B[at, at] = -1.0
        assert factors(B)[2] == int(torch.linalg.cholesky_ex(B.cpu()).info) == at + 1
    assert factors(H * float("nan"))[2] == 1


@pytest.mark.parametrize("var", [False, True])
def test_nested_fit_equals_the_torch_form(var):
    """encode_nested of a weight whose rings, with `var` the negated ones too, come from nq_enc_prepare, and of the same in float64, which takes the
    torch form: the same bytes"""
    W = torch.randn(128, 256, generator=torch.Generator().manual_seed(51)).cuda()
    got, want = (EN.encode_nested(w, seed=6, var=var) for w in (W, W.double()))
    assert got.keys() == want.keys() and (got["var"] is not None) == var
    for k, w in want.items():
        assert (w is None and got[k] is None) or (got[k].dtype == w.dtype and torch.equal(got[k], w)), k
    assert not var or 0 < int((got["var"] != 0).sum())


@pytest.mark.parametrize("N,K,var", [(128, 128, True), (128, 384, False), (256, 256, True)])
def test_hessian_aware_fit_equals_the_torch_form(N, K, var):
    """encode_ldlq with its glue in kernels and level 3 at its own pace against the torch form (which a float64 weight takes): the same bytes, errors to
    the rounding of other sums; a metric that is not positive definite raises as there"""
    g = torch.Generator().manual_seed(N + K)
    W = torch.randn(N, K, generator=g).cuda()
    X = torch.randn(4 * K, K, generator=g) * (1 + torch.arange(K)) ** -0.25
    H = (X.T @ X / (4 * K)).cuda()
    got, want = EN.encode_ldlq(W, H, seed=5, var=var), EN.encode_ldlq(W.double(), H, seed=5, var=var)
    assert got.keys() == want.keys()
    for k, w in want.items():
        if k == "proxy":
            assert all(abs(got[k][l] - w[l]) < 1e-12 * w[l] for l in (2, 3, 4))
        elif k == "eta":
            assert all(float((got[k][l] - w[l]).abs().max()) < 1e-12 for l in (2, 3, 4))
        elif k in ("Hr", "D"):
            assert got[k].shape == w.shape and float((got[k] - w).norm() / w.norm()) < 1e-13
        else:
            assert (w is None and got[k] is None) or (got[k].dtype == w.dtype and torch.equal(got[k], w)), k
    for bad in (-H, H * float("nan")):
        for w in (W, W.double()):
            with pytest.raises(torch.linalg.LinAlgError):
                EN.encode_ldlq(w, bad)


def test_a_metric_that_is_not_positive_definite_is_reported_after_the_first_search(monkeypatch):
    """not after a whole fit: one search here, and the one under which the torch form factorises"""
    g = torch.Generator().manual_seed(41)
    W, searches, search = torch.randn(128, 512, generator=g).cuda(), [], EN._viterbi_gpu
    monkeypatch.setattr(EN, "_viterbi_gpu", lambda *a: (searches.append(a[0].shape[0]), search(*a))[1])
    bad = torch.eye(512, device="cuda")
    bad[200, 200] = -1e4                                         # below zero after the damping too
    with pytest.raises(torch.linalg.LinAlgError):
        EN.encode_ldlq(W, bad)
    assert len(searches) <= 2
    EN.encode_ldlq(W, torch.eye(512, device="cuda"))
    assert len(searches) > 8
