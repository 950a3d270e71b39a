"""The C-ABI library loads without a GPU and exports every symbol include/nq_moe_hip.h declares; host-only entry
points (validation, code masks, error text) behave as documented. No compute call is made here."""
import ctypes as C
import os
import re

import pytest
import torch

from nestquant_amd import _lib
from nestquant_amd.format import TBL_W

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "nq_moe_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(nq_[a-z0-9_]+)\s*\(", text)))


def test_library_is_built():
    assert os.path.exists(_lib.LIB_PATH), "run `python -m nestquant_amd.build`"


def test_every_declared_symbol_is_exported_and_bound():
    L = _lib.lib()
    names = declared_symbols()
    assert len(names) >= 6
    for n in names:
        assert hasattr(L, n), n
        assert n in _lib.SIGNATURES, f"{n} has no ctypes signature"
    assert sorted(_lib.SIGNATURES) == names
    assert L.nq_abi_version() == 3


def _row(**kw):
    r = torch.zeros(TBL_W, dtype=torch.int64)
    r[0] = 2; r[1] = r[5] = r[9] = 0x1000
    for k, v in kw.items():
        r[int(k[1:])] = v
    return r


def _validate(r, H=256, I=256):
    return _lib.lib().nq_validate_row(C.cast(r.data_ptr(), C.POINTER(C.c_int64)), H, I)


def test_validate_row_accepts_supported_rows():
    assert _validate(_row()) == 0
    assert _validate(_row(f0=0, f1=0, f5=0, f9=0)) == 0                                   # level 0: nothing else looked at
    assert _validate(_row(f0=4, f2=8, f3=8, f6=8, f7=8, f10=7, f11=3)) == 0
    assert _validate(_row(f0=3, f2=8, f3=8, f6=8, f7=8, f10=10, f11=10)) == 0
    assert _validate(_row(f0=4, f2=8, f3=8, f6=8, f7=8, f10=11, f11=11, f12=8, f18=128)) == 0
    assert _validate(_row(f0=4, f2=8, f3=8, f6=8, f7=8, f10=12, f11=12)) == 0            # P3 and P4 interleaved
    assert _validate(_row(f19=1)) == 0 and _validate(_row(f19=0x101)) == 0 and _validate(_row(f19=0x100)) == 0   # K = 1.75 base


@pytest.mark.parametrize("bad,word", [
    (dict(f0=1), "level"), (dict(f0=5), "level"), (dict(f0=3, f2=8, f3=8, f6=8, f7=8, f10=10, f11=10, f4=8), "mask mode"), (dict(f0=4, f2=8, f3=8, f6=8, f7=8, f10=11, f11=11, f8=8), "mask mode"),
    (dict(f14=8), "low-rank"), (dict(f16=2), "low-rank"), (dict(f18=512), "in_had_down"), (dict(f19=2), "base code"), (dict(f19=0x10001), "base code"),
    (dict(f0=4), "residual planes"), (dict(f0=4, f2=8, f3=8, f6=8, f7=8, f10=13), "out of range"),
    (dict(f0=3, f2=8, f3=8, f6=8, f7=8, f10=0, f11=10), "level 3"), (dict(f0=4, f2=8, f3=8, f6=8, f7=8, f10=10), "level 4"),
    (dict(f1=0), "null base"),
])
def test_validate_row_rejects_unimplemented_fields(bad, word):
    """a field the kernels do not implement is an error, never silently ignored"""
    assert _validate(_row(**bad)) != 0
    assert word in _lib.lib().nq_last_error().decode()


def test_shape_errors_and_code_masks():
    assert _validate(_row(), H=200) != 0 and "multiples of 128" in _lib.lib().nq_last_error().decode()
    out = (C.c_uint32 * 4)()
    assert _lib.lib().nq_codes(out) == 0
    assert out[0] == out[1] == 0x1FFF and out[2] == out[3] == 3
    with pytest.raises(RuntimeError, match="multiples of 128"):
        _lib.check(_validate(_row(), I=100))


def test_argument_checks_run_before_any_device_work():
    """bad arguments are refused on the host, with a message, before anything is launched (so this runs without a GPU)"""
    L = _lib.lib()
    err = lambda: L.nq_last_error().decode()
    buf = (C.c_char * 4096)()
    base = C.addressof(buf)
    base += (-base) % 64                                           # a 64-byte aligned address inside the buffer
    a = _lib.NqMoeArgs()
    for f in ("x", "sel", "rw", "table", "out", "acc_gu", "h", "acc_d", "cnt_gu", "cnt_d", "cnt_h", "zd"):
        setattr(a, f, base)
    a.B, a.topk, a.E, a.H, a.I = 1, 8, 256, 6144, 2048
    a.cfg_gu = (C.c_int32 * 4)(1, 4, 12, 0); a.cfg_dn = (C.c_int32 * 4)(1, 4, 4, 0)
    a.which = 3
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "workspace too small" in err()
    a.x = base + 2
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "16-byte aligned" in err()
    a.x = base; a.B = 9
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "B=9" in err()
    a.B = 1; a.cfg_gu = (C.c_int32 * 4)(1, 3, 12, 0)
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "bad cfg" in err()
    a.cfg_gu = (C.c_int32 * 4)(1, 4, 12, 0); a.G = 3
    a.route_ws = base
    a.acc_gu_elems = a.acc_d_elems = a.h_elems = a.out_elems = a.cnt_gu_elems = a.cnt_d_elems = a.cnt_h_elems = a.zd_elems = 1 << 40
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "route_ws" in err()
    a.route_ws_bytes = _lib.ROUTE_WS_BYTES
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "xrot" in err()
    a.xrot, a.xrot_elems = base, 1 << 40
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "G=3" in err()
    a.G = 4; a.mb_table = base
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "mailbox needs" in err()
    a.mb_table = None; a.G = 3
    a.G = 0; a.common_rows = 2
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "common_rows" in err()
    a.common_rows = 0; a.hoist_value_map = 2
    assert L.nq_moe_forward(C.byref(a), None) != 0 and "hoist_value_map" in err()
    a.hoist_value_map = 0
    assert L.nq_pf_plan(base, 256, 0, 1024, base, 256, None, 0, 0, None) != 0 and "cap" in err()
    assert L.nq_pf_plan(base, 256, 0, 1024, base + 4, 512, None, 0, 0, None) != 0 and "aligned" in err()
    assert L.nq_pf_gemm(base, base, 1, 48, 0, base, base, base, 4, 256, 256, None, None) != 0 and "tile height" in err()
    assert L.nq_pf_gemm(base, base, 1, 16, 0, base + 8, base, base, 4, 256, 256, None, None) != 0 and "aligned" in err()
    assert L.nq_pf_plan(base, 256, 0, 1024, base, 512, base, 0, 4, None) != 0 and "hot_min" in err()
    assert L.nq_pf_wdecode(base, base, 4, 0, base, 100, 2, 256, 256, None) != 0 and "scratch" in err()
    assert L.nq_pf_wdecode(base, base, 4, 0, base, 100, 1 << 20, 256, 256, None) != 0 and "scratch" in err()     # any number of slots
    assert L.nq_pf_pre(base + 2, base, base, 1, base, base, base, None, 4, 256, 256, None) != 0 and "aligned" in err()
    assert L.nq_pf_pre_rows(base, base, base, 1, base, base, base, None, 4, 256, 256, base, 3, 1, None) != 0 and "cap" in err()
    assert L.nq_pf_pre_rows(base, base, base, 1, base, base, base, None, 4, 256, 256, base, 4, 32, None) != 0 and "heights" in err()
    assert L.nq_pf_pre_rows(base, base, base, 1, base, base, base, None, 4, 256, 256, base, 4, 0, None) == 0          # no height: nothing to do
    assert L.nq_pf_mid_rows(base, base, 1, base, base, None, None, 4, 256, 256, None, 4, 1, None) != 0 and "null" in err()
    assert L.nq_pf_mid_rows(base, base, 1, base, base, None, None, 4, 256, 256, base + 8, 4, 1, None) != 0 and "aligned" in err()
    assert L.nq_sal(base, 0, 64, base, 0, base, 0, 9, 64, 8, 16, 1.0, base, base, None) != 0 and "at most 8" in err()
    assert L.nq_dequant(base, 2, 0, 256, 256, base, None) != 0 and "proj" in err()
    assert L.nq_mailbox(None, base, base, base, None, 4, None) != 0 and "null" in err()


def test_encoder_entry_points_refuse_bad_arguments():
    """shapes, chunks and pointers that the kernels index without looking"""
    L = _lib.lib()
    err = lambda: L.nq_last_error().decode()
    b = 64
    assert L.nq_enc_prepare(b, 100, 128, b, b, b, b, b, None, 0, None) != 0 and "multiples of 128" in err()
    assert L.nq_enc_prepare(b, 65536 * 128, 128, b, b, b, b, b, None, 0, None) != 0 and "65535" in err()        # more blocks of rows than a grid holds
    assert L.nq_enc_prepare(b, 128, 128, None, b, b, b, b, None, 0, None) != 0 and "null" in err()
    assert L.nq_enc_hessian(b, 64, b, b, None) != 0 and "multiple of 128" in err()
    assert L.nq_enc_inverse(b, 127, b, b, 0, None) != 0 and "lda" in err()
    assert L.nq_enc_targets(b, 128, 256, 2, None, 2, 0.3, b, b, 0, None) != 0 and "chunk" in err()
    assert L.nq_enc_targets(b, 128, 256, 0, None, 1, 0.3, b, b, 1, None) != 0 and "negated" in err()
    assert L.nq_enc_base(b, 4, 1, b, b, b, None, 128, 0, b, b, b, b, b, b, None) != 0 and "null" in err()
    assert L.nq_enc_base(b, 0, 1, None, None, None, None, 128, 0, None, None, None, None, None, None, None) == 0
    assert L.nq_enc_feed(b, b, b, b, b, b, 128, 256, -1, b, b, b, b, b, b, None) != 0 and "chunk" in err()


def test_which_steps_are_given_decoded_weights():
    """nq_pf_wide_slots: none for steps of short tiles, of few tokens, of too few tiles to fill the GPU, of shapes that would be padded; no
    more than 2 GB; nothing for sizes that a step refuses"""
    L = _lib.lib()
    m = C.c_int32(0)

    def slots(T, topk, E, H, I, rows=32768, side=1):
        return L.nq_pf_wide_slots(T, topk, rows, E, H, I, side, C.byref(m))
    assert slots(4096, 8, 256, 6144, 2048) == 2**31 // (6 * 6144 * 2048) and m.value == 640
    assert slots(1100, 8, 8, 2048, 2048) == 8
    assert slots(1024, 8, 8, 2048, 2048) == 8 and slots(1023, 8, 8, 2048, 2048) == 0          # 32 tiles of 256 rows
    assert slots(639, 64, 8, 6144, 2048) == 0
    assert slots(1000, 8, 256, 6144, 2048) == 0                  # at most 32 rows per expert on average
    assert slots(4096, 8, 16, 256, 512) == 0                     # little work
    assert slots(1100, 8, 280, 6144, 2048, side=0) == 0 and slots(1100, 8, 280, 6144, 2048) > 0    # without side streams short tiles go further
    assert slots(4096, 8, 64, 4096, 1152) == 0 and slots(4096, 8, 64, 4096, 1024) > 0
    assert slots(4096, 8, 256, 6144, 2048, rows=4096) == 0       # chunks of few rows
    for bad in ((-1, 8, 16, 2048, 1024), (4096, 0, 16, 2048, 1024), (4096, 8, 0, 2048, 1024), (4096, 8, 16, 2000, 1024), (4096, 8, 16, 2048, 0)):
        assert slots(*bad) == 0
    assert L.nq_pf_wide_slots(4096, 8, 32768, 256, 6144, 2048, 1, None) == 0


def test_pf_bytes_covers_the_decoded_weights_of_every_step():
    """pf_bytes knows the rows of a chunk only: it holds what nq_pf_wide_slots gives any step of such chunks, and is no larger than the largest of them"""
    from nestquant_amd import moe as M
    assert M.PF_HOT_SLOTS == 0
    L, m = _lib.lib(), C.c_int32()
    for H, I in ((6144, 2048), (2048, 2048), (4096, 1024), (4096, 1152), (512, 256)):
        for R in (1, 640, 4096, 8191, 8192, 8800, 16384, 32768):
            plain = M._pf_offsets(H, I, R)[1]
            given = [L.nq_pf_wide_slots(T, k, R, E, H, I, side, C.byref(m)) for k in (1, 2, 8) for T in (R // k, R // k + 1, 4096, 40000)
                     for E in (2, 16, 64, 256, 4096) for side in (0, 1) if min(T * k, R) == R]
            assert M.pf_bytes(H, I, R) == plain + max(given) * 6 * H * I, (H, I, R)
    assert M.pf_bytes(6144, 2048, 32768) - M._pf_offsets(6144, 2048, 32768)[1] == 28 * 6 * 6144 * 2048


def test_counters_apart_are_asked_for_and_checked():
    """which bit 4 needs NQ_CNT_STEP * H / 128 counters and the down launch; without it H / 128 are enough, and no capacity changes what they mean"""
    L = _lib.lib()
    err = lambda: L.nq_last_error().decode()
    buf = (C.c_char * 4096)()
    base = C.addressof(buf)
    base += (-base) % 64
    a = _lib.NqMoeArgs()
    for f in ("x", "sel", "rw", "table", "out", "acc_gu", "h", "acc_d", "cnt_gu", "cnt_d", "cnt_h", "zd"):
        setattr(a, f, base)
    a.B, a.topk, a.E, a.H, a.I = 1, 8, 256, 6144, 2048
    a.cfg_gu = (C.c_int32 * 4)(1, 4, 12, 0); a.cfg_dn = (C.c_int32 * 4)(1, 4, 4, 0)
    a.acc_gu_elems = a.acc_d_elems = a.h_elems = a.out_elems = a.cnt_gu_elems = a.cnt_h_elems = a.zd_elems = 1 << 40
    for which, elems, want in ((3, 47, "cnt_d"), (3, 48, "route_ws"), (3 | 16, 48 * _lib.CNT_STEP - 1, "cnt_d"), (3 | 16, 48 * _lib.CNT_STEP, "route_ws"),
                               (2 | 16, 48 * _lib.CNT_STEP, "route_ws"), (16, 1 << 40, "which=16"), (1 | 16, 1 << 40, "which=17"), (32, 1 << 40, "which=32")):
        a.which, a.cnt_d_elems = which, elems
        assert L.nq_moe_forward(C.byref(a), None) != 0 and want in err(), (which, elems, err())


def test_stream_engine_refuses_bad_arguments_before_touching_the_gpu(tmp_path):
    """the checks of the reference's Engine constructor (streaming/nqstream.cu:76,77,81): record size a multiple of 4 KiB,
    at least as many host entries as reads in flight, the record file must exist"""
    from nestquant_amd.stream_engine import Engine
    f = tmp_path / "r.bin"
    f.write_bytes(b"\0" * 8192)
    with pytest.raises(RuntimeError, match="4096"):
        Engine(str(f), 4095, 8, 2, 0)
    with pytest.raises(RuntimeError, match="n_host"):
        Engine(str(f), 4096, 3, 4, 0)
    with pytest.raises(RuntimeError, match="n_host"):
        Engine(str(f), 4096, 4, 3, 0, alt_path=str(f), qd_alt=2)
    with pytest.raises(RuntimeError, match="open .*missing.bin"):
        Engine(str(tmp_path / "missing.bin"), 4096, 4, 2, 0)
