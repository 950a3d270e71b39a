"""The encoder's GPU searches against their torch form on the CPU: the same states, ties included."""
import pytest
import torch

from nestquant_amd import encode as EN

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


def test_viterbi_ties_on_a_coarse_codebook():
    """a codebook of nine values: many states tie at every step"""
    g = torch.Generator().manual_seed(7)
    lut = EN.codebook().round().clamp(-4, 4)
    w = torch.randint(-3, 4, (4, 64), generator=g).float()
    for K in (1, 2):
        assert torch.equal(EN.viterbi_ring(w.cuda(), lut.cuda(), K).cpu(), EN.viterbi_ring(w, lut, K))
