"""NestQuant grouped MoE layer on MI355X: device table, workspaces, launch wrappers.

Host-side mirror of the reference's Python op surface (sm120/moe.py): `entry` :216-229, `MoELayer` :231-260,
`prefill` :282-326, `Mailbox` :329-342, `dense_W` :156-166, `H128` :168-172, `Expert.ref` :196-210, `moe_ref` :344-351. The kernels behind it are the HIP kernels of
libnq_moe_hip.so, reached through ctypes with raw device pointers; there is no CPU path in this module.
"""
import ctypes as C
import os

import numpy as np
import torch

from . import _lib
from .format import (CODE_L3, CODE_L4B, CODE_L4N, RK_OF, RKP, TBL_W, Expert, Proj, all_MbN, make_flags, pack_words, popc, proj_sizes,  # noqa: F401
                     rbits, split_bits, step_off, unpack_words)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def had_dn(ex):
    """down-projection input Hadamard width (absent = 128)"""
    return int(getattr(ex, "had_dn", 128) or 128)


def base_code(p):
    return int(getattr(p, "bk", 0) or 0)


def H128(dev="cuda", n=128):
    """normalised Sylvester Hadamard matrix of order n"""
    H = torch.ones(1, 1)
    while H.shape[0] < n:
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)], 0)
    return (H / n**0.5).to(dev)


def _entry_words(ex, level):
    """table row (TBL_W integers) of expert `ex` at `level` (0, 2, 3, 4). Level 3 points at the one-bit plane p3 (code 10); level 4
    points, for experts built with nested=True, at the planes P3 and P4 read as one record (code 11: concatenated, or code 12
    for experts built with interleave=True: interleaved bit by bit), otherwise at the wide residual plane p4 (code rk)."""
    e = [0] * TBL_W                                  # a list first: setting elements of a tensor one by one takes 30 us
    e[0] = level
    nested = bool(getattr(ex, "nested", False))
    l3 = level == 3
    if l3 and not nested and any(getattr(p, "p3", None) is None for p in (ex.gu, ex.dn)):
        raise ValueError("level 3 needs an expert with the one-bit planes p3 / d3")
    for off, p in ((1, ex.gu), (5, ex.dn)):
        e[off] = p.base.data_ptr()
        if nested:
            slot = p.slot
            e[off + 1] = slot.data_ptr()
            e[off + 2] = (p.d3 if l3 else p.d4n).data_ptr()
        elif l3:
            e[off + 1] = p.p3.data_ptr()
            e[off + 2] = p.d3.data_ptr()
        else:
            e[off + 1] = 0 if p.p4 is None else p.p4.data_ptr()      # None: resident-only expert, a record slot supplies them
            e[off + 2] = 0 if p.d4 is None else p.d4.data_ptr()
        if getattr(p, "flags", None) is not None:
            e[off + 3] = p.flags.data_ptr()
    e[9] = ex.signs.data_ptr()
    if nested or l3:
        e[10] = e[11] = CODE_L3 if l3 else int(getattr(ex, "l4code", CODE_L4N))
    else:
        e[10], e[11] = ex.gu.rk, ex.dn.rk
    for i, p in ((12, ex.gu), (13, ex.dn)):
        v = getattr(p, "var", None)
        e[i] = 0 if v is None else v.data_ptr()
    lr = getattr(ex, "lr", None)
    if lr is not None:
        e[14] = lr.data_ptr(); e[15] = ex.lr4.data_ptr(); e[16] = ex.rg; e[17] = ex.rd
    w = had_dn(ex)
    e[18] = 0 if w == 128 else w
    e[19] = base_code(ex.gu) | base_code(ex.dn) << 8
    return e


def entry(ex, level):
    """_entry_words as an int64 tensor (host)"""
    return torch.from_numpy(np.array(_entry_words(ex, level), dtype=np.int64))


def validate_row(row, H, I):
    """raise RuntimeError if the row uses a field or code the kernels do not implement"""
    r = row.to("cpu", torch.int64).contiguous()
    _lib.check(_lib.lib().nq_validate_row(C.cast(r.data_ptr(), C.POINTER(C.c_int64)), H, I))


def rk_codes():
    """[gate|up mask, down mask] of compiled residual window codes"""
    out = (C.c_uint32 * 4)()
    _lib.check(_lib.lib().nq_codes(out))
    return [int(out[0]), int(out[1])]


def occ(mode, sb, shm, any_rows=False):
    """(resident workgroups per CU, registers per lane, spill bytes per lane) of the decode kernel `mode` (0 gate|up, 1 down) of a
    call with a routing launch, launched with sb wavefronts per workgroup and shm bytes of dynamic LDS; the reference's M.occ (sm120/nqmoe.cu:930-937)"""
    out = (C.c_int * 3)()
    _lib.check(_lib.lib().nq_occ(mode, int(any_rows), sb, shm, out))
    return tuple(out)


def bk_codes():
    out = (C.c_uint32 * 4)()
    _lib.check(_lib.lib().nq_codes(out))
    return [int(out[2]), int(out[3])]


def dequant(row_dev, proj, H, I, level=0, out=None):
    """HIP dense decode of one projection from a table row on the device -> fp16 [N, K]"""
    N, K = (2 * I, H) if proj == 0 else (H, I)
    if out is None:
        out = torch.empty(N, K, dtype=torch.float16, device=row_dev.device)
    _lib.check(_lib.lib().nq_dequant(_ptr(row_dev), proj, level, H, I, _ptr(out), _lib.stream_ptr()))
    return out


def dense_W(ex, proj, level, dtype=torch.float16):
    """dense rotated-domain weights [N, K] of projection `proj` (0 gate|up, 1 down) of expert `ex`, decoded on the GPU"""
    row = (C.c_int64 * TBL_W)(*_entry_words(ex, level))
    L = _lib.lib()
    N, K = (2 * ex.I, ex.H) if proj == 0 else (ex.H, ex.I)
    rc = L.nq_validate_row(row, ex.H, ex.I)
    out = None
    if not rc:                                                   # the row goes along as a kernel argument: no copy to the device
        out = torch.empty(N, K, dtype=torch.float16, device=ex.signs.device)
        rc = L.nq_dequant_row(row, proj, 0, ex.H, ex.I, out.data_ptr(), _lib.stream_ptr())
    _lib.check(rc)
    return out if dtype == torch.float16 else out.to(dtype)


# caller element types the decode kernels read / write directly (codes of include/nq_moe_hip.h)
_DT_IN = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}
_DT_SEL = {torch.int64: 0, torch.int32: 1}
_DT_OUT = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


_LONE = {}


def _lone_picks(dev, E):
    """(ids int32 [>= E, 8] with row e = e, ones fp16 [8]) of a device: the routing of a lone projection of expert e for up to eight
    tokens. Constants, made with the first layer of a device and whole before another stream or a capture may see them."""
    k = str(dev)
    t = _LONE.get(k)
    if t is None or t[0].shape[0] < E:
        n = max(E, 256)
        t = (torch.arange(n, dtype=torch.int32, device=dev)[:, None].repeat(1, 8), torch.ones(8, dtype=torch.float16, device=dev))
        if t[0].is_cuda:
            torch.cuda.current_stream(t[0].device).synchronize()
        _LONE[k] = t
    return t


class MoELayer:
    """Device table [E, TBL_W] + workspaces for up to Bmax tokens; table rows are flipped in place (graph-safe).

    Same constructor, attributes and call signature as the reference's MoELayer (sm120/moe.py:231-260). Differences that
    a caller can observe: acc_gu / acc_d hold per-k-slice partial sums ([NY, S, 2I] and [NY, S, H]) instead of
    atomically accumulated [S, 2I] / [S, H], so they are not zero between calls and outputs are bitwise repeatable;
    cnt_gu / cnt_d / cnt_h are arrival counters (zero on entry, zero on exit; cnt_h counts the 128-column groups of a
    512-column block when in_had_down = 512); zd carries the low-rank plane's z_d partial sums from the gate|up launch to
    the down launch and needs no zeroing; wq exists for attribute compatibility only (no work queue here) and stays zero."""

    def __init__(s, E, H, I, nm_gu=0, nm_dn=0, Bmax=4, topk=8, G=4, dev="cuda", mod=None):
        if G not in (4, 2):
            raise NotImplementedError("rings of G = 4 lanes (every artifact) or G = 2 (the reference's test variant) only")
        s.M = mod or _lib.lib()
        s.E, s.H, s.I, s.nm_gu, s.nm_dn, s.G, s.Bmax, s.topk = E, H, I, nm_gu, nm_dn, G, Bmax, topk
        s.table = torch.zeros(E, TBL_W, dtype=torch.int64, device=dev)
        S = Bmax * topk
        f32, i32 = torch.float32, torch.int32
        s.cfg_gu, s.cfg_dn = s.default_cfg(H, I)
        s._tuned, s._cfgs = True, {}                  # cfg_for picks the k-slice lengths by the call's size; set_cfg switches that off
        s.h = torch.zeros(S, I, dtype=torch.float16, device=dev)
        s.cnt_gu = torch.zeros(max(S * (I // 128), _lib.CNT_STEP * 2 * I // 128), dtype=i32, device=dev); s.cnt_d = torch.zeros(_lib.CNT_STEP * H // 128, dtype=i32, device=dev)
        s.wq = torch.zeros(4, dtype=i32, device=dev)
        s.zd = torch.zeros(S * (I // 128) * 4, dtype=f32, device=dev); s.cnt_h = torch.zeros(S * (I // 128), dtype=i32, device=dev)
        s.out = torch.zeros(Bmax, H, dtype=f32, device=dev)
        s.route = torch.zeros(_lib.ROUTE_WS_BYTES, dtype=torch.uint8, device=dev)    # the routing launch's result for the projection launches
        s.xrot = torch.zeros(S, 2, H, dtype=torch.float16, device=dev)               # and the rotated activations of every pick
        s._lone, s._lone_views = _lone_picks(s.table.device, E), {}                  # proj_gemv
        s.hits_ptr = 0
        s.rare_rows = False                           # set once a row in mask mode or with a base window code other than 0 is
                                                      # installed (set / Mailbox.post): the decode call then runs the kernel that
                                                      # carries their loops and prefill also launches its variant kernel. A caller
                                                      # that writes such rows into the table itself must set it, else the tokens
                                                      # that pick them come out NaN
        s._alloc_partials()

    # k-slice lengths. A projection launch has (row blocks) x (k-slices) x (runs of distinct experts) workgroups, and about 1024 of
    # them fill the chip (four per CU for gate|up, five for down): fewer leave CUs idle, and every further one costs a head (run
    # header, activations, first records) of 2 to 4 us. So a slice is as long as keeps the launch at that number, with a run for
    # every pick (an upper bound), at most 24 chunks for gate|up and 4 for down (whose finisher and SwiGLU staging favour short
    # slices at every count). Measured best at H = 6144, I = 2048, top-8: 12 chunks at one token, 24 above, down 4; the rule gives
    # these. The reference keeps tables of measured lengths per GPU (sm120/serve/nq_vllm.py:32-33).
    @staticmethod
    def _slice(C, blocks, runs, slots, most):
        want = min(most, max(1, blocks * C * runs // slots))
        return max(d for d in range(1, want + 1) if C % d == 0)

    @staticmethod
    def default_cfg(H, I, runs=8):
        """[cpw, sb, nst]: k-slice of cpw * nst chunks, sb wavefronts per block; for a call of `runs` picks"""
        sb = lambda N: max(d for d in (4, 2, 1) if (N // 32) % d == 0 and (I // 32) % d == 0)
        gu, dn = sb(2 * I), sb(H)
        return ([1, gu, MoELayer._slice(H // 128, 2 * I // 32 // gu, runs, 1024, 24)],
                [1, dn, MoELayer._slice(I // 128, H // 32 // dn, runs, 1280, 4)])

    def cfg_for(s, T):
        """(cfg_gu, cfg_dn) for a decode call of T tokens: default_cfg for its picks, unless set_cfg has replaced the defaults"""
        if not s._tuned:
            return s.cfg_gu, s.cfg_dn
        c = s._cfgs.get(T)
        if c is None:
            c = s._cfgs[T] = s.default_cfg(s.H, s.I, T * s.topk)
        return c

    def _ny(s, cfg, C):
        return C // (cfg[0] * cfg[2])

    def _alloc_partials(s, cfg_gu=None, cfg_dn=None):
        """Partial-sum workspaces for the given (default: the layer's) tilings. At construction they are sized for the finest
        k-split among the layer's own tilings (cfg_for, 1 .. Bmax tokens), so the calls a serving loop makes never re-size them. A call
        that brings a finer split of its own replaces them -- graphs captured before hold the old addresses and must be
        captured again -- and that is refused while the stream is capturing (an allocation cannot be captured)."""
        S, dev = s.Bmax * s.topk, s.table.device
        ny_gu, ny_dn = s._ny(cfg_gu or s.cfg_gu, s.H // 128), s._ny(cfg_dn or s.cfg_dn, s.I // 128)
        first = getattr(s, "acc_gu", None) is None
        if first:
            own = [s.cfg_for(T) for T in range(1, s.Bmax + 1)]
            ny_gu = max([ny_gu] + [s._ny(c[0], s.H // 128) for c in own])
            ny_dn = max([ny_dn] + [s._ny(c[1], s.I // 128) for c in own])
        grow_gu, grow_dn = first or s.acc_gu.shape[0] < ny_gu, first or s.acc_d.shape[0] < ny_dn
        if (grow_gu or grow_dn) and not first and torch.cuda.is_current_stream_capturing():
            raise RuntimeError("this call's k-split needs larger partial-sum workspaces than the layer holds; make one call with "
                               "these tilings (or set_cfg) before capturing")
        if grow_gu:
            s.acc_gu = torch.zeros(ny_gu, S, 2 * s.I, dtype=torch.float32, device=dev)
        if grow_dn:
            s.acc_d = torch.zeros(ny_dn, S, s.H, dtype=torch.float32, device=dev)

    def set_cfg(s, cfg_gu=None, cfg_dn=None):
        """change the default tilings (may replace the partial-sum workspaces: graphs captured before must be captured again)"""
        s.cfg_gu, s.cfg_dn = list(cfg_gu or s.cfg_gu), list(cfg_dn or s.cfg_dn)
        s._tuned = False
        s._alloc_partials()

    def set(s, e, ex, level):
        row = entry(ex, level)
        if s.G != 4 and (row[12] or row[13]):
            raise ValueError("sign-variant planes are defined for rings of G = 4 lanes only (reference sm120/moe.py:143)")
        validate_row(row, s.H, s.I)
        s.rare_rows |= bool(row[4] or row[8] or row[19])
        s.table[e].copy_(row.to(s.table.device), non_blocking=False)

    def __call__(s, x, sel, rw, out=None, force_level=0, which=3, cfg_gu=None, cfg_dn=None, table=None, static_ws=False, mailbox=None, hoist=False, sal=None):
        """x [B, H], sel [B, topk], rw [B, topk] -> fp32 [B, H] (s.out[:B] unless `out` is given). As in the reference x
        and rw are fp16 and sel int64; the kernels also take x / rw in bf16 or fp32, sel in int32 and `out` in fp16 or
        bf16, with the roundings of x.half(), rw.half() and out.to(dtype) (the casts the reference's caller launches as
        separate kernels, sm120/serve/nq_vllm.py:522,560).
        table: optional [E, TBL_W] override. Everything is enqueued on torch's current stream; nothing syncs.
        mailbox: a Mailbox of this layer, served by the call without a launch of its own: the call's last projection launch
        applies it (table rows and the device copy of `applied`) after the call's routing has read the table, and the routing
        launch of the next call publishes `applied_host`. Rows that land while this call runs are used, and reported done, from
        the next call on -- when `mailbox.apply()` at the head of the next call would have done both. After the last call of
        a sequence one `mailbox.apply()` publishes what that call applied.
        hoist: experts without a sign plane (rows of the common kind) multiply the integers 1024 + S / 1024 + F and apply the value
        map to the sums, so no weight is rounded to fp16: ~4 % faster, ~5e-4 from the default's result (NqMoeArgs.hoist_value_map;
        off by default).
        sal: a salience.Salience, fed with this call's x, sel and rw by the call's routing launch (what `sal(x, rw, sel)` in front of
        the call does with a launch of its own; at most 8 picks per token).
        static_ws: go through nq_moe_forward_static, which ignores this layer's workspaces and uses the library's built-in
        device scratch instead (for callers that must not allocate; calls on one GPU then share that scratch)."""
        assert x.dtype in _DT_IN and rw.dtype in _DT_IN and sel.dtype in _DT_SEL, (x.dtype, rw.dtype, sel.dtype)
        assert x.is_contiguous() and sel.is_contiguous() and rw.is_contiguous()
        B, topk = sel.shape
        out = s.out[:B] if out is None else out
        assert out.dtype in _DT_OUT and out.is_contiguous(), out.dtype
        tb = s.table if table is None else table
        tg, td = s.cfg_for(B)
        cg, cd = cfg_gu or tg, cfg_dn or td
        if not static_ws and (cfg_gu or cfg_dn):
            s._alloc_partials(cg, cd)                # grows only when a call brings a finer k-split than any before
        # one struct.pack instead of sixty attribute stores on a ctypes structure: 4 us less host time per call
        mb = (0, 0, 0, 0, 0) if mailbox is None else (tb.data_ptr(), mailbox.stage.data_ptr(), mailbox.seq.data_ptr(), mailbox.applied.data_ptr(),
                                                      mailbox.applied_host.data_ptr())
        if sal is not None and not (sal.acc.dtype == sal.host.dtype == torch.float64 and sal.acc.is_contiguous() and sal.host.is_contiguous()
                                    and sal.acc.numel() >= tb.shape[0] <= sal.host.numel() and rw.numel() == sel.numel()):
            raise RuntimeError("salience: acc and its host mirror must be contiguous float64 with an entry per expert, rw one weight per pick")
        sl = (0, 0, 0, 0.0) if sal is None else (1, sal.acc.data_ptr(), sal.host.data_ptr(), sal.rsf)
        if which & 2 and s.cnt_d.numel() >= _lib.CNT_STEP * x.shape[1] // 128:       # room for the down launch's counters to stand apart
            which |= 16
        raw = _lib.PACK_MOE_ARGS(
            x.data_ptr(), sel.data_ptr(), rw.data_ptr(), tb.data_ptr(), out.data_ptr(), s.acc_gu.data_ptr(), s.h.data_ptr(), s.acc_d.data_ptr(),
            s.cnt_gu.data_ptr(), s.cnt_d.data_ptr(), s.hits_ptr or 0,
            s.acc_gu.numel(), s.acc_d.numel(), s.h.numel(), out.numel(), s.cnt_gu.numel(), s.cnt_d.numel(),
            B, topk, tb.shape[0], x.shape[1], s.I, cg[0], cg[1], cg[2], cg[3] if len(cg) > 3 else 0, cd[0], cd[1], cd[2], cd[3] if len(cd) > 3 else 0,
            force_level, which, _DT_IN[x.dtype], _DT_SEL[sel.dtype], _DT_IN[rw.dtype], _DT_OUT[out.dtype],
            s.cnt_h.data_ptr(), s.cnt_h.numel(), s.zd.data_ptr(), s.zd.numel(),
            int(table is None and not s.rare_rows), s.G,             # common_rows; a caller's own table: unknown
            s.route.data_ptr(), s.route.numel(), s.xrot.data_ptr(), s.xrot.numel(), *mb, int(bool(hoist)), *sl, 0)
        rc = (s.M.nq_moe_forward_static if static_ws else s.M.nq_moe_forward)(raw, _lib.stream_ptr())
        if rc:
            _lib.check(rc)
        return out


PF_TILES = (16, 32, 64, 128, 256)            # token-tile heights the grouped GEMM is compiled for
# Experts with many pair rows can be decoded once per call into a scratch of decoded weights (6 H I bytes each), whose tiles a GEMM of
# their own multiplies, instead of once per tile; see nq_pf_wdecode. Same bits either way. With PF_HOT_SLOTS = 0 the library says for which
# steps and experts (nq_pf_wide_slots); > 0: every expert of at least PF_HOT_MIN rows, at most this many; < 0: none.
PF_HOT_MIN, PF_HOT_SLOTS = 257, 0


_PF_REGIONS = ("xg", "xu", "acc", "h", "y", "zg", "zd")


def _pf_offsets(H, I, R):
    """byte offsets of _PF_REGIONS in a block for R pair rows, each on 256 bytes, and the block's size"""
    at, off = 0, []
    for row in (2 * H, 2 * H, 8 * I, 2 * I, 4 * H, 16, 16):
        off.append(at)
        at += -(-R * row // 256) * 256
    return off, at


def _pf_slots(R):
    """slots of the decoded-weight scratch for R pair rows"""
    return max(0, min(PF_HOT_SLOTS, R // PF_HOT_MIN))


def pf_bytes(H, I, R, G=0):
    """bytes of scratch that a step of up to R pair rows at a time takes beside its lists (nq_pf_meta_bytes): the regions of pf_scratch and the decoded
    weights. With PF_HOT_SLOTS = 0 the most that the library gives any step of such chunks, whatever its tokens, picks and experts. (G is accepted for
    signature compatibility: the decoded-weight scratch is sized by the rows, not by a group of experts)"""
    slots = _pf_slots(R)
    if PF_HOT_SLOTS == 0 and R > 0:                  # a step of one pair more than a chunk holds, over more experts than could take a slot
        slots = _lib.lib().nq_pf_wide_slots(min(R + 1, 2**31 - 1), 1, R, R, H, I, 1, C.byref(C.c_int32()))
    return _pf_offsets(H, I, R)[1] + slots * 6 * H * I


def pf_scratch(dev, H, I, R, G=0):
    """Prefill scratch for R pair rows on `dev`, not initialised: xg | xu fp16 [R, H], acc fp32 [R, 2I], h fp16 [R, I], y fp32
    [R, H], the low-rank plane's zg | zd fp32 [R, 4], and wop: decoded weights of up to PF_HOT_SLOTS hot experts (None without; what a step takes by the
    library's own choice is not in it, see pf_bytes).
    A set belongs to whoever asks for it, and every step takes one of its own from torch's allocator: what another layer, stream
    or thread has in flight, or a captured graph holds, is never shared. Unlike the reference (sm120/moe.py:262-274), which
    keeps one set per device and decodes every expert of a group into it, only experts with several tiles go through
    decoded weights; the others are decoded in registers inside the grouped GEMM."""
    f16, f32 = torch.float16, torch.float32
    off, size = _pf_offsets(H, I, R)
    block, slots = torch.empty(size, dtype=torch.uint8, device=dev), _pf_slots(R)
    S = {n: block[o:o + R * w * dt.itemsize].view(dt).view(R, w)
         for n, o, w, dt in zip(_PF_REGIONS, off, (H, H, 2 * I, I, H, 4, 4), (f16, f16, f32, f16, f32, f32, f32))}
    return dict(S, rows=R, wop=torch.empty(slots, 3 * H * I, dtype=f16, device=dev) if slots else None)


def pf_tiles(segs):
    """segs [(expert, first row, rows)] -> {tile height: int32 [n, 4] rows (expert, row0, rows, 0)}. Rows of an expert are
    cut into 256-row tiles; the remainder takes the smallest compiled height that holds it."""
    out = {bm: [] for bm in PF_TILES}
    for e, r0, n in segs:
        while n > 0:
            take = min(n, PF_TILES[-1])
            bm = next(b for b in PF_TILES if b >= take)
            out[bm].append((e, r0, take, 0))
            r0 += take; n -= take
    return {bm: torch.tensor(v, dtype=torch.int32) for bm, v in out.items() if v}


_PF_SIDE = {}


def _pf_side(dev, stream):
    """(streams, events, their handles): three side streams (default priority) and four events for steps that the caller puts on
    `stream` of `dev`. An event is only ever recorded on one stream, so of two threads on one stream each waits for its own
    work, at most for more; steps on different streams share no event (streams of torch's pool may coincide, which only orders
    more). At most 64 sets are kept."""
    k = (dev.index, stream)
    S = _PF_SIDE.get(k)
    if S is None:
        with torch.cuda.device(dev):
            side, ev = [torch.cuda.Stream(device=dev) for _ in range(3)], [torch.cuda.Event() for _ in range(4)]
            for e in ev:
                e.record(side[0])                    # a torch event exists from its first record on
        S = (side, ev, (C.c_void_p * 3)(*[st.cuda_stream for st in side]), (C.c_void_p * 4)(*[e.cuda_event for e in ev]))
        if len(_PF_SIDE) >= 64:
            _PF_SIDE.clear()
        _PF_SIDE[k] = S
    return S


# Device index -> free bytes of the driver from which on a step there asks for decoded weights again, after it could not have them
_PF_SHORT = {}


def _pf_block(dev, need, extra, capturing=False):
    """(a block of need + extra bytes, extra), or a block of `need` bytes and 0 where the device has no more. The refusal costs the allocator its cached
    blocks and the host a wait for the device, so it is paid once and not by every step: the next steps do not ask before the driver has as much
    more to give as was refused (3 us a step to find out; a step that is being captured neither asks then nor leaves word)."""
    short = _PF_SHORT.get(dev.index) if extra else None
    if extra and (short is None or (not capturing and torch.cuda.mem_get_info(dev)[0] >= short)):
        try:
            block = torch.empty(need + extra, dtype=torch.uint8, device=dev)
            _PF_SHORT.pop(dev.index, None)
            return block, extra
        except torch.OutOfMemoryError:
            refused = not capturing
    else:
        refused = False
    block = torch.empty(need, dtype=torch.uint8, device=dev)
    if refused:
        _PF_SHORT[dev.index] = torch.cuda.mem_get_info(dev)[0] + need + extra
    return block, 0


def _pf_step(s, x, sel, rw, out, R=None, table=None):
    """one nq_pf_step call: x [T, H], sel and rw [T, k], out [T, H] in any of the types the decode kernels take and write"""
    T, k = sel.shape
    H, I, E, dev, Lb = s.H, s.I, s.E, x.device, s.M
    tb = s.table if table is None else table
    P = T * k
    if P == 0:
        return out.zero_()
    R = min(P, R or int(os.environ.get("NQ_PF_ROWS", "32768")))
    nb = Lb.nq_pf_meta_bytes(T, k, R, E)
    if nb < 0:
        raise RuntimeError(Lb.nq_last_error().decode())
    # decoded-weight scratch: rows of the common kind only (the variant kernel of the others decodes in the GEMM)
    off, size = _pf_offsets(H, I, R)
    meta_at, wop_at = size, size + -(-nb // 256) * 256
    stream = _lib.stream_ptr()
    # a step that is being captured stays on its stream: streams of torch's pool may coincide with one that somebody is using
    held = None if torch.cuda.is_current_stream_capturing() else _pf_side(dev, stream)
    slots, hot_min, advised = 0, C.c_int32(PF_HOT_MIN), PF_HOT_SLOTS == 0
    if not s.rare_rows and table is None:            # rows of the common kind only: the variant kernel of the others decodes in the GEMM
        if advised:
            slots = Lb.nq_pf_wide_slots(T, k, R, E, H, I, held is not None, C.byref(hot_min))
        elif P >= PF_HOT_MIN:
            slots = _pf_slots(R)
    # one block per call, the step's own: it goes back to the allocator in the order of the caller's stream, which the side streams join
    block, wop_bytes = _pf_block(dev, wop_at, slots * 6 * H * I, held is None)
    whole = out if out.dtype == torch.float32 or R == P else torch.empty(T, H, dtype=torch.float32, device=dev)   # chunks add up in fp32
    a, at = _lib.NqPfArgs(), block.data_ptr()
    a.x, a.sel, a.rw, a.table, a.out, a.hits = x.data_ptr(), sel.data_ptr(), rw.data_ptr(), tb.data_ptr(), whole.data_ptr(), s.hits_ptr or None
    a.meta, a.meta_bytes = at + meta_at, nb
    a.xg, a.xu, a.acc, a.h, a.y, a.zg, a.zd = (at + o for o in off)
    if wop_bytes:
        a.wop, a.wop_bytes, a.wop_slots, a.hot_min = at + wop_at, wop_bytes, slots, hot_min.value
    if held is not None:
        a.side, a.events = held[2], held[3]
    a.T, a.topk, a.E, a.H, a.I, a.rows = T, k, E, H, I, R
    a.x_dtype, a.sel_dtype, a.rw_dtype, a.out_dtype = _DT_IN[x.dtype], _DT_SEL[sel.dtype], _DT_IN[rw.dtype], _DT_OUT[whole.dtype]
    # mask mode / other base codes run in their own kernel variant; a caller's own table may hold such rows, so it gets both, and
    # a lone variant is told so: should it meet a row of the other kind after all, the result is NaN, not stale scratch
    a.variants = (3 if (s.rare_rows or table is not None) else 1) | (4 if advised else 0)
    _lib.check(Lb.nq_pf_step(C.byref(a), stream))
    return out if whole is out else out.copy_(whole)


def prefill(s, x, sel, rw, out=None, R=None, G=None, table=None):
    """T > Bmax tokens (reference sm120/moe.py:282-326): pairs sorted by expert, each routed expert decoded inside the
    grouped GEMMs at the level of its live table row, same math as the decode path (fp32 accumulation order differs).
    No host synchronisation (the reference's prefill reads the expert counts back; here the sort and the tile lists are
    built on the device), but for what torch's allocator does when the device runs out of memory. Exports routing hits like the decode kernel. A call's scratch is its own (pf_scratch; the reference's calls
    share one set per device, sm120/moe.py:262-274) and its side streams belong to the caller's stream."""
    if s.G != 4:
        raise NotImplementedError("prefill decodes rings of G = 4 lanes only (as the reference's pf_decode)")
    assert x.dtype == torch.float16 and rw.dtype == torch.float16 and sel.dtype == torch.int64, (x.dtype, rw.dtype, sel.dtype)
    assert x.is_contiguous()
    out = torch.empty(x.shape[0], s.H, dtype=torch.float32, device=x.device) if out is None else out
    return _pf_step(s, x, sel.contiguous(), rw.contiguous(), out, R, table)


class Mailbox:
    """Graph-safe table updates (reference sm120/moe.py:329-342): call apply() on the compute stream before the layer;
    stage rows from a side stream with post(). One outstanding op per expert."""

    def __init__(s, layer):
        E, dev = layer.E, layer.table.device
        s.L = layer
        s.stage = torch.zeros(E, TBL_W, dtype=torch.int64, device=dev)
        s.seq = torch.zeros(E, dtype=torch.int32, device=dev)
        s.applied = torch.zeros(E, dtype=torch.int32, device=dev)
        s.applied_host = torch.zeros(E, dtype=torch.int32).pin_memory()
        s.hseq = [0] * E
        s.pins = []

    def apply(s):
        _lib.check(s.L.M.nq_mailbox(s.L.table.data_ptr(), s.stage.data_ptr(), s.seq.data_ptr(), s.applied.data_ptr(),
                                    s.applied_host.data_ptr(), s.L.E, _lib.stream_ptr()))

    def post(s, e, row, stream):
        """enqueue on `stream`, after any plane copy already enqueued there: stage[e] = row; seq[e] += 1"""
        assert s.done(e), "one outstanding op per expert"
        validate_row(row, s.L.H, s.L.I)
        s.L.rare_rows |= bool(row[4] or row[8] or row[19])
        s.hseq[e] += 1
        r = row.pin_memory(); q = torch.tensor([s.hseq[e]], dtype=torch.int32).pin_memory()
        s.pins += [r, q]
        if len(s.pins) > 4096:                       # rows whose copies completed long ago
            del s.pins[:2048]
        with torch.cuda.stream(stream):
            s.stage[e].copy_(r, non_blocking=True)
            s.seq[e:e + 1].copy_(q, non_blocking=True)

    def done(s, e):
        return int(s.applied_host[e]) == s.hseq[e]


MoELayer.prefill = prefill


PF_MIN = 384         # tokens from which a step goes through prefill() (reference NQ_PF_MIN, sm120/serve/nq_vllm.py:187)
# Steps of more than GROUP_MIN tokens that would take more than three slices go through the grouped kernels of prefill() too, eagerly
# and under graph capture alike (a step's scratch comes from torch's allocator, which hands out the graph's own memory then).
# The reference slices up to 383 tokens into decode calls, and each slice decodes its experts anew: 48 tokens
# name 200 distinct experts, their twelve slices of four 360. Measured at E = 256, top-8, Bmax 4 (slices / grouped): 9 tokens
# 522 / 478 us, 16: 934 / 707, 48: 2650 / 1200, 201: 10900 / 1530, 383: 20800 / 1600. At the other end, 512 x 256 with 4 experts, top-4,
# Bmax 8: 33 tokens 139 / 35; between them ten shapes from 256 x 128 to 6144 x 2048, 4 to 256 experts, top-2 to top-8, Bmax 1 to 8, 13
# to 65 tokens: grouped is ahead at every one, eagerly and in a graph.
GROUP_MIN = 12


def forward(layer, mailbox, x, topk_weights, topk_ids, pf_min=PF_MIN, sal=None):
    """One MoE layer step as the reference's serving caller runs it (sm120/serve/nq_vllm.py:520-574): apply the mailbox,
    then up to Bmax tokens in one decode call, more than three slices' worth through the grouped kernels of prefill(), pf_min
    tokens or more through prefill() (under graph capture in slices, as the reference's caller does), anything between in slices of
    Bmax tokens. x [T, H] in fp16 / bf16 / fp32, weights [T, topk] likewise, ids int64 / int32;
    returns [T, H] in x's dtype. The decode calls read the caller's dtypes and write the result dtype themselves. `sal`: an
    optional salience.Salience, fed by the decode steps as the reference does (every step of up to Bmax tokens, the slices of
    a step of up to 16 tokens; longer steps count as prefill and are left out)."""
    T = x.shape[0]
    x, w, ids = x.contiguous(), topk_weights.contiguous(), topk_ids.contiguous()
    odt = x.dtype if x.dtype in _DT_OUT else torch.float32
    if 0 < T <= layer.Bmax:
        # a Salience whose call is its own, with operands that call would take: exported by the layer call itself
        inside = getattr(type(sal).__call__, "layer_can", False) and ids.shape[1] <= 8 and sal.acc.numel() == layer.E \
            and sal.acc.dtype == torch.float64 and sal.acc.is_contiguous() and w.numel() == ids.numel() == T * ids.shape[1]
        if sal is not None and not inside:
            sal(x, w, ids)
        return layer(x, ids, w, out=torch.empty(T, layer.H, dtype=odt, device=x.device), mailbox=mailbox,   # applied by the call's last launch, for the next step
                     sal=sal if inside else None)
    if mailbox is not None:
        mailbox.apply()
    if T == 0:
        return torch.empty(0, layer.H, dtype=odt, device=x.device)
    out = torch.empty(T, layer.H, dtype=odt, device=x.device)
    plain = layer.G == 4 and x.dtype in _DT_IN and w.dtype in _DT_IN and ids.dtype in _DT_SEL
    if T >= pf_min:
        grouped = not torch.cuda.is_current_stream_capturing()
    else:                                            # what the slices refuse stays refused
        grouped = T > max(GROUP_MIN, 3 * layer.Bmax) and plain and layer.E <= 4096
    if grouped:
        if not plain:
            return layer.prefill(x.half(), ids.long(), w.half()).to(x.dtype)
        _pf_step(layer, x, ids, w, out)
        for i in range(0, T if sal is not None and T <= 16 and T < pf_min else 0, layer.Bmax):
            sal(x[i:i + layer.Bmax], w[i:i + layer.Bmax], ids[i:i + layer.Bmax])
        return out
    for i in range(0, T, layer.Bmax):
        j = min(T, i + layer.Bmax)
        layer(x[i:j], ids[i:j], w[i:j], out=out[i:j])
        if sal is not None and T <= 16:
            sal(x[i:j], w[i:j], ids[i:j])
    return out


def _lr_parts(ex, level):
    """the low-rank factors of `ex` as fp32 matrices, read back from the two table buffers (lr = V_g | U2_g | U2_u | V_d | U2_d,
    lr4 = U4_g | U4_u | U4_d): (V_g [rg, H], U_g [rg, I], U_u [rg, I], V_d [rd, I], U_d [rd, H]) with U = U2 (+ U4 at level 4)"""
    H, I, rg, rd = ex.H, ex.I, ex.rg, ex.rd
    cut = lambda t, sizes: [c.float() for c in torch.split(t[: sum(sizes)], sizes)]
    Vg, U2g, U2u, Vd, U2d = cut(ex.lr, [rg * H, rg * I, rg * I, rd * I, rd * H])
    Ug, Uu, Ud = U2g, U2u, U2d
    if level == 4:
        U4g, U4u, U4d = cut(ex.lr4, [rg * I, rg * I, rd * H])
        Ug, Uu, Ud = Ug + U4g, Uu + U4u, Ud + U4d
    return Vg.view(rg, H), Ug.view(rg, I), Uu.view(rg, I), Vd.view(rd, I), Ud.view(rd, H)


def expert_ref(ex, x, level, G=4):
    """One expert's MLP through dense weights (reference Expert.ref, sm120/moe.py:196-210): x [T, H] fp32 -> [T, H] fp32 on the
    expert's device. The weights are decoded by the HIP decoder (bit-exact values); rotations, products and sums are plain
    torch fp32 with the two fp16 roundings of the activations, so this is the slow, transparent twin of the fused kernels that
    check scripts compare them with. Rings of G = 4 lanes."""
    if G != 4:
        raise NotImplementedError("the dense decoder reads rings of G = 4 lanes")
    H, I, dev = ex.H, ex.I, ex.signs.device
    x = x.to(dev, torch.float32)
    had = lambda v, n=128: (v.reshape(*v.shape[:-1], -1, n) @ H128(dev, n)).reshape(v.shape)
    su_g, sv_g, sv_u, su_d, sv_o, su_u = torch.split(ex.signs.float(), [H, I, I, I, H, H])
    Wgu, Wdn = dense_W(ex, 0, level, torch.float32), dense_W(ex, 1, level, torch.float32)
    g = had(had(x * su_g).half().float() @ Wgu[:I].T) * sv_g
    u = had(had(x * su_u).half().float() @ Wgu[I:].T) * sv_u
    lowrank = getattr(ex, "lr", None) is not None
    if lowrank:
        Vg, Ug, Uu, Vd, Ud = _lr_parts(ex, level)
        z = x @ Vg.T
        g, u = g + z @ Ug, u + z @ Uu
    sw = torch.nn.functional.silu(g) * u
    y = had(had(sw * su_d, had_dn(ex)).half().float() @ Wdn.T) * sv_o
    if lowrank:
        y = y + (sw @ Vd.T) @ Ud
    return y


def moe_ref(experts, levels, x, sel, rw, G=4):
    """The layer through expert_ref (reference moe_ref, sm120/moe.py:344-351): out[t] = sum over the picks of rw * expert(x[t]),
    picks of level <= 0 or weight 0 skipped. Every distinct routed expert is decoded once and applied to all its tokens."""
    T, H = x.shape
    y = torch.zeros(T, H, dtype=torch.float32, device=x.device)
    xf, w = x.float(), rw.float()
    for e in sorted(set(sel.flatten().tolist())):
        if not 0 <= e < len(experts) or levels[e] <= 0:
            continue
        hit = (sel == e) & (w != 0)
        rows = hit.any(1).nonzero().flatten()
        if rows.numel():
            y[rows] += (w * hit)[rows].sum(1, keepdim=True) * expert_ref(experts[e], xf[rows], levels[e], G).to(x.device)
    return y


Expert.ref = expert_ref


def proj_gemv(layer, x, e=0, cfg=None):
    """Raw fused decode+GEMV of the gate|up projection of expert e for every token of x [B, H] (B <= 8), without the
    SwiGLU finisher: returns fp32 [B, 2I] = W_gu . fp16(Hadamard(x * su)) (rows < I rotated with su_g, the rest with su_u)."""
    B = x.shape[0]
    C_ = layer.H // 128
    # One launch (nq_proj) for rows of the common kind where nobody counts the picks; what that leaves, and what it would refuse, goes through
    # a layer call of one run and the sum of its slices. At 6144 x 4096, eight tokens: 10.7 / 13.7 / 13.8 us a call at levels 2 / 3 / 4, three
    # launches 20.4 / 19.0 / 19.0.
    lone = not layer.rare_rows and not layer.hits_ptr and 0 <= e < layer.E and 0 < B <= min(8, layer.Bmax) and x.dtype in _DT_IN \
        and x.is_contiguous() and x.shape == (B, layer.H) and layer.cnt_gu.numel() >= 2 * layer.I // 128
    if cfg is None:
        # one run: about 512 workgroups and slices of two or three chunks at the full shape are where heads, decode and the number
        # of partial sums balance, as far as the layer's workspace holds that many slices
        sb = layer.cfg_gu[1]
        n = MoELayer._slice(C_, 2 * layer.I // 32 // sb, 1, 512, 24)
        n = next(d for d in range(n, C_ + 1) if C_ % d == 0 and C_ // d <= layer.acc_gu.shape[0])
        cfg = [1, sb, n]
    n = 2 * layer.I
    if lone and len(cfg) == 3 and cfg[0] >= 1 and cfg[2] >= 1 and C_ % (cfg[0] * cfg[2]) == 0:
        if C_ // (cfg[0] * cfg[2]) * B * n > layer.acc_gu.numel():
            layer._alloc_partials(cfg)
        out = torch.empty(B, n, dtype=torch.float32, device=x.device)
        rc = layer.M.nq_proj(x.data_ptr(), _DT_IN[x.dtype], B, layer.table.data_ptr() + 8 * TBL_W * e, layer.H, layer.I, layer.G, cfg[0] * cfg[2], cfg[1],
                             layer.acc_gu.data_ptr(), layer.acc_gu.numel(), layer.cnt_gu.data_ptr(), layer.cnt_gu.numel(), out.data_ptr(), _lib.stream_ptr())
        if rc:
            _lib.check(rc)
        return out
    picks = layer._lone_views.get((B, e))
    if picks is None:
        if 0 <= e < layer.E and B <= 8:
            picks = layer._lone_views[B, e] = (layer._lone[0][e, :B].view(B, 1), layer._lone[1][:B].view(B, 1))
        else:                                                     # the layer call has its answer to both
            picks = torch.full((B, 1), e, dtype=torch.int64, device=x.device), torch.ones(B, 1, dtype=torch.float16, device=x.device)
    sel, rw = picks
    layer(x, sel, rw, which=1 | 8, cfg_gu=list(cfg))              # 8: the launch ends with its partial sums
    ny = C_ // (cfg[0] * cfg[2])                                  # partial sums are laid out [k-slice][B * topk of the call][2I]
    out = torch.empty(B, n, dtype=torch.float32, device=x.device)
    _lib.check(layer.M.nq_sum_slices(layer.acc_gu.data_ptr(), ny, B * n, out.data_ptr(), _lib.stream_ptr()))
    return out
