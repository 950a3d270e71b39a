"""moe.forward's choice between the decode call, slices of it and the grouped kernels, on the CPU with a stub layer."""
import pytest
import torch

from nestquant_amd import moe as M


class Stub:
    def __init__(s, G=4, E=64, Bmax=4):
        s.G, s.E, s.Bmax, s.H, s.calls = G, E, Bmax, 128, []

    def __call__(s, x, sel, rw, out=None, **kw):
        assert x.dtype in M._DT_IN and rw.dtype in M._DT_IN and sel.dtype in M._DT_SEL
        s.calls.append(x.shape[0])
        return out

    def prefill(s, x, sel, rw):
        s.calls.append("prefill")
        return x.float()


def route(monkeypatch, layer, T, capturing=False, xd=torch.float16, wd=torch.float16, sd=torch.int64, **kw):
    monkeypatch.setattr(M, "_pf_step", lambda s, x, sel, rw, out, *a: s.calls.append("grouped"))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    M.forward(layer, None, torch.zeros(T, 128, dtype=xd), torch.ones(T, 2, dtype=wd), torch.zeros(T, 2, dtype=sd), **kw)
    return layer.calls


@pytest.mark.parametrize("xd,wd,sd", [(torch.float64, torch.float16, torch.int64), (torch.float16, torch.float64, torch.int64),
                                      (torch.float16, torch.float16, torch.int16)])
def test_types_that_the_slices_refuse_are_refused_below_the_prompts(monkeypatch, xd, wd, sd):
    for T in (5, 13, 383):
        with pytest.raises(AssertionError):
            route(monkeypatch, Stub(), T, xd=xd, wd=wd, sd=sd)
    assert route(monkeypatch, Stub(), 384, xd=xd, wd=wd, sd=sd) == ["prefill"]         # cast, as they always were


def test_which_steps_are_grouped(monkeypatch):
    one = lambda T, **kw: route(monkeypatch, Stub(**kw), T)
    assert one(4) == [4] and one(12) == [4, 4, 4] and one(13) == one(383) == one(384) == ["grouped"]
    assert one(24, Bmax=8) == [8, 8, 8] and one(25, Bmax=8) == ["grouped"]
    assert one(14, G=2) == [4, 4, 4, 2] and one(384, G=2) == ["prefill"]
    assert one(13, E=4097) == [4, 4, 4, 1]
    # under capture: the same route below pf_min, slices from there on
    assert route(monkeypatch, Stub(), 13, capturing=True) == ["grouped"]
    assert route(monkeypatch, Stub(), 384, capturing=True) == [4] * 96


def test_memory_that_was_refused_is_not_asked_for_by_every_step(monkeypatch):
    """the block of a step with decoded weights: a refusal is met once, the steps after it take the smaller block at once until the driver has
    as much more to give; a captured step neither asks the driver nor leaves word; other devices are not concerned"""
    dev, other = torch.device("cuda", 3), torch.device("cuda", 4)
    asked, driver, have = [], [], {3: 150, 4: 1000}

    def empty(n, dtype, device):
        assert dtype == torch.uint8
        asked.append((device.index, n))
        if n > have[device.index]:
            raise torch.OutOfMemoryError("no")
        return ("block", n)

    def info(d):
        driver.append(d.index)
        return have[d.index], 10**6
    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(torch.cuda, "mem_get_info", info)
    monkeypatch.setattr(M, "_PF_SHORT", {})
    block = lambda *a: (M._pf_block(*a), asked.copy(), driver.copy(), asked.clear(), driver.clear())[:3]
    assert block(dev, 100, 0) == ((("block", 100), 0), [(3, 100)], [])
    assert block(dev, 100, 80, True) == ((("block", 100), 0), [(3, 180), (3, 100)], [])            # captured: refused, no word left
    assert block(dev, 100, 80) == ((("block", 100), 0), [(3, 180), (3, 100)], [3])
    assert block(dev, 100, 80) == ((("block", 100), 0), [(3, 100)], [3])                           # not asked again
    assert block(dev, 100, 80, True) == ((("block", 100), 0), [(3, 100)], [])
    assert block(other, 100, 80) == ((("block", 180), 80), [(4, 180)], [])
    have[3] = 329                                                # 150 + 180 - 1
    assert block(dev, 100, 80)[1] == [(3, 100)]
    have[3] = 330
    assert block(dev, 100, 80) == ((("block", 180), 80), [(3, 180)], [3])
    assert block(dev, 100, 80) == ((("block", 180), 80), [(3, 180)], [])
    have[3] = 50
    with pytest.raises(torch.OutOfMemoryError):                  # not even the smaller one
        M._pf_block(dev, 100, 80)
    assert not M._PF_SHORT
