"""Decode salience export (sal[e] += (rsf w)^2 |x|^2 per pick): the oracle against exact known answers and an independent
float64 closed form on the CPU; the HIP kernel against the oracle on the GPU -- exactly where every partial sum is exact (rows
of small powers of two), to fp32 rounding of the squared norm (1e-5 relative) otherwise."""
import numpy as np
import pytest
import torch

from oracle import nq_oracle as O


def closed_form(x, w, ids, rsf, E):
    out = np.zeros(E)
    xn = (x.astype(np.float64) ** 2).sum(1)
    for t in range(ids.shape[0]):
        for k in range(ids.shape[1]):
            e = int(ids[t, k])
            if float(w[t, k]) != 0.0 and 0 <= e < E:
                out[e] += (rsf * float(w[t, k])) ** 2 * xn[t]
    return out


def test_oracle_known_answers():
    E, H = 16, 6144
    x = np.ones((2, H), np.float16); x[1] *= 2                       # |x|^2 = 6144 and 4 * 6144, every partial sum exact
    w = np.array([[0.5, 0.25, 0.0, 1.0], [0.5, 0.5, 0.5, 0.5]], np.float16)
    ids = np.array([[3, 5, 7, 3], [5, 5, 99, -1]])                   # duplicates in a token and across tokens, ids outside the table
    acc = np.zeros(E); acc[3] = 1.5
    touched = O.salience(x, w, ids, 2.0, acc)
    want = np.zeros(E)
    want[3] = 1.5 + (1.0 + 4.0) * 6144                                 # (2 * 0.5)^2 + (2 * 1)^2
    want[5] = 0.25 * 6144 + 2 * 1.0 * 4 * 6144
    assert np.array_equal(acc, want) and touched == [3, 5]            # expert 7 had weight 0; 99 and -1 are outside the table
    assert np.array_equal(closed_form(x, w, ids, 2.0, E), want - np.eye(E)[3] * 1.5)
    # a second call keeps adding
    O.salience(x[:1], w[:1], ids[:1], 1.0, acc)
    assert acc[3] == want[3] + (0.25 + 1.0) * 6144 and acc[5] == want[5] + 0.0625 * 6144


@pytest.mark.parametrize("H", [6144, 100, 8, 2056])
def test_oracle_matches_float64_closed_form(H):
    rng = np.random.default_rng(H)
    E, T, K = 32, 5, 8
    x = (rng.standard_normal((T, H)) * 0.7).astype(np.float16)
    w = rng.random((T, K)).astype(np.float16); w[2, 3] = 0
    ids = rng.integers(0, E, (T, K))
    acc = np.zeros(E)
    O.salience(x, w, ids, 2.5, acc)
    assert np.allclose(acc, closed_form(x, w, ids, 2.5, E), rtol=3e-7, atol=0)        # rsf * w is an fp32 product in the oracle, as in the kernels


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_hip_salience(dtype):
    from nestquant_amd import salience as SA
    g = torch.Generator().manual_seed(11)
    E, K = 256, 8
    # exact cases: rows of +-1 and +-2 (every partial sum is a small integer), weights that are powers of two
    S = SA.Salience(E, rsf=2.0)
    want = np.zeros(E)
    for T, H, cut in ((2, 6144, 0), (8, 6144, 0), (3, 100, 0), (4, 2048, 1), (1, 8, 0)):
        sign = torch.randint(0, 2, (T, H + 16), generator=g) * 2 - 1
        big = (sign * (1 + torch.arange(T)[:, None] % 2)).to(dtype)
        x = big[:, cut:cut + H]                                       # cut = 1: rows off 16-byte alignment
        w = (0.5 ** torch.randint(0, 4, (T, K), generator=g)).half(); w[0, 1] = 0
        ids = torch.randint(0, E, (T, K), generator=g); ids[-1, 0] = E + 3; ids[0, 2] = ids[0, 5]
        touched = O.salience(x.float().numpy(), w.numpy(), ids.numpy(), 2.0, want)
        S(x.cuda(), w.cuda(), ids.cuda()) if cut == 0 else SA.sal(big.cuda()[:, cut:cut + H], w.cuda(), ids.cuda(), 2.0, S.acc, S.host)
        torch.cuda.synchronize()
        got = S.acc.cpu().numpy()
        assert np.array_equal(got, want), (T, H, cut, np.abs(got - want).max())
        assert np.array_equal(S.host.numpy()[touched], want[touched])
    # general values: fp32 rounding of the squared norm
    S = SA.Salience(E, rsf=2.5)
    want = np.zeros(E)
    for T, H, cut in ((1, 6144, 0), (8, 6144, 0), (3, 100, 0), (4, 2048, 1), (5, 4096, 8), (7, 2056, 0)):
        big = (torch.randn(T, H + 16, generator=g) * 0.7).to(dtype)
        x = big[:, cut:cut + H]
        w = torch.rand(T, K, generator=g).half(); w[0, 1] = 0
        ids = torch.randint(0, E, (T, K), generator=g); ids[-1, 0] = E + 3; ids[0, 2] = ids[0, 5]
        xo = x.float().half().float().numpy() if dtype != torch.bfloat16 else x.float().numpy()
        touched = O.salience(xo, w.numpy(), ids.numpy(), 2.5, want)
        S(x.cuda(), w.cuda(), ids.cuda()) if cut == 0 else SA.sal(big.cuda()[:, cut:cut + H], w.cuda(), ids.cuda(), 2.5, S.acc, S.host)
        torch.cuda.synchronize()
        got = S.acc.cpu().numpy()
        assert np.allclose(got, want, rtol=1e-5, atol=0), (T, H, cut, np.abs(got / np.maximum(want, 1e-30) - 1).max())
        assert np.array_equal(S.host.numpy()[touched], got[touched])
        assert np.array_equal(got == 0, want == 0)                     # skipped picks touch nothing
        want = got.copy()                                              # the running sums continue from the device's values
    # int32 ids and bf16 / fp32 weights read as the casts would leave them
    x = (torch.randn(2, 512, generator=g)).to(dtype).cuda()
    w32 = torch.rand(2, K, generator=g); ids = torch.randint(0, E, (2, K), generator=g)
    a = SA.Salience(E, 1.0); b = SA.Salience(E, 1.0)
    a(x, w32.half().cuda(), ids.cuda()); b(x, w32.cuda(), ids.int().cuda())
    torch.cuda.synchronize()
    assert torch.equal(a.acc, b.acc) and a.acc.sum() > 0


@pytest.mark.gpu
def test_salience_errors_and_forward_hook():
    from nestquant_amd import format as F, moe as M, salience as SA
    S = SA.Salience(8)
    x = torch.zeros(9, 128, dtype=torch.float16, device="cuda")
    w = torch.ones(9, 2, dtype=torch.float16, device="cuda"); ids = torch.zeros(9, 2, dtype=torch.int64, device="cuda")
    with pytest.raises(RuntimeError, match="at most 8"):
        S(x, w, ids)
    with pytest.raises(RuntimeError, match="nqsal"):
        S(x[:2].double(), w[:2], ids[:2])
    with pytest.raises(RuntimeError, match="nqsal"):
        SA.sal(x[:2], w[:2], ids[:2], 1.0, S.acc.float(), S.host)
    S(x[:0], w[:0], ids[:0])                                          # no tokens: nothing to do
    # the serving step feeds it: steps of up to Bmax tokens and the slices of steps of up to 16
    H, I, E = 256, 128, 4
    L = M.MoELayer(E, H, I, Bmax=4, topk=2)
    for e in range(E):
        ex = F.Expert(H, I, seed=e, dev="cpu"); ex.gu.to("cuda"); ex.dn.to("cuda"); ex.signs = ex.signs.cuda()
        L.keep = getattr(L, "keep", []) + [ex]
        L.set(e, ex, 2)
    g = torch.Generator().manual_seed(3)
    S = SA.Salience(E, rsf=1.5)
    want = np.zeros(E)
    for T in (3, 4, 11, 16, 17):
        xt = torch.randn(T, H, generator=g).bfloat16().cuda()
        wt = torch.rand(T, 2, generator=g).cuda(); it = torch.stack([torch.randperm(E, generator=g)[:2] for _ in range(T)]).int().cuda()
        M.forward(L, None, xt, wt, it, sal=S)
        if T <= 16:
            for i in range(0, T, 4):
                O.salience(xt[i:i + 4].float().cpu().numpy(), wt[i:i + 4].half().cpu().numpy(), it[i:i + 4].cpu().numpy(), 1.5, want)
    torch.cuda.synchronize()
    assert np.allclose(S.acc.cpu().numpy(), want, rtol=1e-5, atol=0) and np.array_equal(S.host.numpy(), S.acc.cpu().numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,H,xd", [(1, 1, 128, torch.float16), (2, 3, 1152, torch.bfloat16), (8, 8, 384, torch.float32), (3, 8, 6144, torch.bfloat16)])
def test_salience_inside_the_layer_call_is_the_launch_in_front_of_it(T, K, H, xd):
    """NqMoeArgs.with_salience: the routing launch exports what nq_sal exports, call after call, and the layer's result is the same"""
    from nestquant_amd import format as F, moe as M, salience as SA
    I, E = 128, 9
    L = M.MoELayer(E, H, I, Bmax=8, topk=K)
    keep = []
    for e in range(E):
        ex = F.Expert(H, I, seed=e, dev="cuda", gen_dev="cuda"); keep.append(ex)
        L.set(e, ex, 2)
    g = torch.Generator().manual_seed(T)
    A, B = SA.Salience(E, rsf=2.5), SA.Salience(E, rsf=2.5)
    for _ in range(3):
        x = torch.randn(T, H, generator=g).to(xd).cuda()
        w = torch.rand(T, K, generator=g).cuda(); w[0, 0] = 0
        ids = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).int().cuda()
        ids[-1, -1] = E + 1 if K > 1 else 0
        A(x, w, ids)
        y = L(x, ids, w).clone()
        assert torch.equal(L(x, ids, w, sal=B), y)
    torch.cuda.synchronize()
    assert A.acc.sum() > 0 or K == 1
    # the two launches have 512 and 256 threads, so their fp32 norms add up in different orders
    assert torch.allclose(A.acc, B.acc, rtol=1e-6, atol=0) and torch.equal(B.host, B.acc.cpu())


def _host_salience(cls, E):
    s = object.__new__(cls)                                       # without the pinned mirror, which needs a GPU
    s.acc, s.host, s.rsf = torch.zeros(E, dtype=torch.float64), torch.zeros(E, dtype=torch.float64), 1.0
    return s


class _LayerStub:
    """what moe.forward asks of a layer for a decode call; remembers which salience the call was to export"""
    H, E, Bmax, G = 128, 6, 4, 4

    def __call__(s, x, sel, rw, out=None, mailbox=None, sal=None):
        s.sal = sal
        return out


def test_a_salience_with_a_call_of_its_own_is_called():
    from nestquant_amd import moe as M, salience as SAL
    x, w, ids = torch.zeros(2, 128), torch.ones(2, 3), torch.zeros(2, 3, dtype=torch.int64)

    class Doubled(SAL.Salience):
        def __call__(s, x, w, ids):
            calls.append(s)

    class Other:
        acc = torch.zeros(6, dtype=torch.float64)

        def __call__(s, x, w, ids):
            calls.append(s)
    for own in (_host_salience(Doubled, 6), Other()):
        calls, L = [], _LayerStub()
        M.forward(L, None, x, w, ids, sal=own)
        assert calls == [own] and L.sal is None
    L, plain = _LayerStub(), _host_salience(SAL.Salience, 6)
    M.forward(L, None, x, w, ids, sal=plain)
    assert L.sal is plain


def test_salience_operands_are_looked_at_either_way():
    """what the salience call refuses is not left to the routing launch, which would not notice"""
    from nestquant_amd import moe as M, salience as SAL
    x, w, ids = torch.zeros(2, 128, dtype=torch.float16), torch.ones(2, 3, dtype=torch.float16), torch.zeros(2, 3, dtype=torch.int64)
    for acc, ww in ((torch.zeros(6), w), (torch.zeros(6, dtype=torch.int64), w), (torch.zeros(12, dtype=torch.float64)[::2], w),
                    (torch.zeros(6, dtype=torch.float64), w[:, :2])):
        s = _host_salience(SAL.Salience, 6)
        s.acc = acc
        with pytest.raises(RuntimeError):
            M.forward(_LayerStub(), None, x, ww, ids, sal=s)


def test_layer_call_looks_at_its_salience(monkeypatch):
    """the routing launch indexes accumulator and mirror by expert: a shorter or otherwise typed one is refused by the host"""
    from nestquant_amd import _lib, moe as M, salience as SAL

    class Lib:
        calls = 0

        def nq_moe_forward(s, raw, stream):
            s.calls += 1
            return 0
    monkeypatch.setattr(_lib, "stream_ptr", lambda: 0)
    L = M.MoELayer(6, 128, 128, Bmax=2, topk=2, dev="cpu", mod=Lib())
    x, sel, rw = torch.zeros(1, 128, dtype=torch.float16), torch.zeros(1, 2, dtype=torch.int64), torch.ones(1, 2, dtype=torch.float16)
    f64 = lambda n: torch.zeros(n, dtype=torch.float64)
    for acc, host, w in ((f64(5), f64(6), rw), (f64(6), f64(5), rw), (torch.zeros(6), f64(6), rw), (f64(6), torch.zeros(6), rw),
                         (f64(12)[::2], f64(6), rw), (f64(6), f64(6), rw[:, :1].contiguous())):
        s = _host_salience(SAL.Salience, 6)
        s.acc, s.host = acc, host
        with pytest.raises(RuntimeError):
            L(x, sel, w, sal=s)
    assert L.M.calls == 0
    L(x, sel, rw, sal=_host_salience(SAL.Salience, 6))
    assert L.M.calls == 1
