"""GPU parity of dag_multihead_links (through the C ABI) against the CPU oracle."""
import pytest
import torch

import da_transformer_amd as dagx
from oracle import torch_native as tn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NEG_INF = float("-inf")
# the kernels compute in fp32 and round once to the storage dtype
FWD_TOL = {torch.float32: (1e-5, 1e-5), torch.float16: (2e-3, 2e-3), torch.bfloat16: (1.6e-2, 1.6e-2)}
GRAD_RTOL = {torch.float32: 1e-4, torch.float16: 1e-2, torch.bfloat16: 2e-2}


def _case(B, L, H, dtype, seed=0, scale=2.0, ragged=True):
    gen = torch.Generator().manual_seed(seed)
    content = (torch.randn(B, L, L, H, generator=gen) * scale).to(dtype)
    gates = torch.log_softmax(torch.randn(B, L, H, generator=gen), -1)
    if ragged:
        lens = torch.randint(2, L + 1, (B,), generator=gen)
        lens[0] = L
    else:
        lens = torch.full((B,), L)
    return content, gates, lens


def _mask(lens, L):
    return (torch.arange(L)[None, None, :] < lens[:, None, None]) & torch.ones(L, L, dtype=torch.bool).triu(1)[None]


def _compare(got, want, rtol, atol):
    finite = want > NEG_INF
    assert torch.equal(got > NEG_INF, finite), "different set of allowed transitions"
    assert not torch.isnan(got).any()
    assert torch.allclose(got[finite], want[finite], rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,L,H,translen", [(3, 17, 8, 5), (2, 70, 4, 100), (2, 300, 16, 64), (1, 1024, 8, 1023),
                                            (1, 600, 16, 599), (1, 1024, 16, 1023), (1, 498, 4, 497), (1, 786, 4, 785),
                                            (1, 257, 8, 256), (3, 259, 16, 257), (1, 513, 8, 512), (1, 515, 4, 513), (5, 3, 8, 2)])
def test_forward_and_backward_match_oracle(dtype, B, L, H, translen):
    content, gates, lens = _case(B, L, H, dtype)
    mask = _mask(lens, L)
    vend = lens[:, None].expand(-1, L).contiguous()
    # oracle in float64 on the same (rounded) inputs
    c64 = content.double().requires_grad_(); g64 = gates.double().requires_grad_()
    want = tn.multihead_links(c64, g64, mask, translen)
    weight = torch.randn(want.shape, generator=torch.Generator().manual_seed(5)).to(dtype)
    (want.masked_fill(want == NEG_INF, 0.0) * weight.double()).sum().backward()

    c = content.to(DEV).clone().requires_grad_(); g = gates.to(DEV).clone().requires_grad_()
    work = c * 1          # a non-leaf the operator may consume
    got = dagx.dag_multihead_links(work, g, vend.to(DEV), translen)
    assert got.dtype == dtype and got.shape == want.shape
    rtol, atol = FWD_TOL[dtype]
    _compare(got.detach().cpu().double(), want.detach(), rtol, atol)
    (got.masked_fill(got == NEG_INF, 0.0) * weight.to(DEV)).sum().backward()
    tol = GRAD_RTOL[dtype]
    for mine, ref in ((c.grad, c64.grad), (g.grad, g64.grad)):
        mine = mine.cpu().double()
        assert not torch.isnan(mine).any()
        assert torch.allclose(mine, ref, rtol=tol, atol=tol * ref.abs().max().item())
    # nothing outside the allowed transitions carries a gradient
    assert (c.grad.cpu()[~mask] == 0).all()


def test_bound_end_and_helpers():
    B, L, H = 2, 40, 8
    content, gates, _ = _case(B, L, H, torch.float32, seed=7, ragged=False)
    gen = torch.Generator().manual_seed(8)
    bound_end = torch.minimum(torch.arange(L)[None, :] + torch.randint(0, 9, (B, L), generator=gen), torch.tensor(L - 1))
    mask = (torch.arange(L)[None, None, :] <= bound_end[:, :, None]) & torch.ones(L, L, dtype=torch.bool).triu(1)[None]
    want = tn.multihead_links(content.double(), gates.double(), mask, 16)
    got = dagx.dag_multihead_links(content.to(DEV), gates.to(DEV), dagx.valid_end_from_bound(bound_end.to(DEV)), 16)
    _compare(got.cpu().double(), want, 1e-5, 1e-5)
    # decoder tokens with trailing padding
    pad = 1
    tokens = torch.full((B, L), 5); tokens[1, 30:] = pad
    vend = dagx.valid_end_from_tokens(tokens.to(DEV), pad)
    assert vend.shape == (B, L) and int(vend[0, 0]) == L and int(vend[1, 3]) == 30
    tokens[0, 4] = pad
    with pytest.raises(RuntimeError):
        dagx.valid_end_from_tokens(tokens.to(DEV), pad)


def test_feeds_dag_loss_and_extreme_scores():
    """The links go straight into dag_loss; huge score ranges and an all -inf head stay NaN-free."""
    B, L, H, T = 2, 64, 8, 9
    content, gates, lens = _case(B, L, H, torch.float32, seed=11, scale=30.0)
    content[0, 3, :, 2] = NEG_INF                      # head 2 of node 3 has no finite score
    mask = _mask(lens, L)
    vend = lens[:, None].expand(-1, L).contiguous()
    # (the reference's log_softmax turns such a head into NaN; here it simply drops out of the mixture,
    #  which the oracle reproduces with a -inf gate and harmless finite scores)
    c_ref = content.double().clone(); c_ref[0, 3, :, 2] = 0.0
    g_ref = gates.double().clone(); g_ref[0, 3, 2] = NEG_INF
    want = tn.multihead_links(c_ref, g_ref, mask, L - 1)
    got = dagx.dag_multihead_links(content.to(DEV), gates.to(DEV), vend.to(DEV), L - 1)
    _compare(got.cpu().double(), want, 1e-4, 1e-4)
    match = torch.log_softmax(torch.randn(B, T, L, generator=torch.Generator().manual_seed(2)), -1).to(DEV)
    tl = torch.tensor([T, 4]).to(DEV)
    ol = lens.clamp(min=T).to(DEV)
    vend2 = ol[:, None].expand(-1, L).contiguous()
    c = content.to(DEV).clamp(min=-100).requires_grad_()
    links = dagx.dag_multihead_links(c * 1, gates.to(DEV), vend2, L - 1)
    loss = dagx.dag_loss(match, links, ol, tl)
    loss.sum().backward()
    assert torch.isfinite(loss).all() and torch.isfinite(c.grad).all() and c.grad.abs().sum() > 0


@pytest.mark.parametrize("B,L,H", [(2, 120, 4), (1, 300, 8), (1, 700, 16)])
def test_scores_that_leave_the_float32_range(B, L, H):
    """Score ranges of several hundred: most positions are less likely than 2^-100, where the kernels turn from plain
    sums of probabilities to sums against the largest term -- with and without a head that reaches no position.  The
    tolerances: scores of 300 are rounded to 2^-16 relative to 1, and every probability with them."""
    content, gates, lens = _case(B, L, H, torch.float32, seed=L, scale=60.0)
    gates[:, ::3] = gates[:, ::3] * 30
    gates[0, 5, 1] = NEG_INF
    mask = _mask(lens, L)
    vend = lens[:, None].expand(-1, L).contiguous()
    c64 = content.double().requires_grad_(); g64 = gates.double().requires_grad_()
    want = tn.multihead_links(c64, g64, mask, L - 1)
    weight = torch.randn(want.shape, generator=torch.Generator().manual_seed(5))
    (want.masked_fill(want == NEG_INF, 0.0) * weight.double()).sum().backward()
    c = content.to(DEV).requires_grad_(); g = gates.to(DEV).requires_grad_()
    got = dagx.dag_multihead_links(c * 1, g, vend.to(DEV), L - 1)
    _compare(got.detach().cpu().double(), want.detach(), 1e-5, 2e-4)
    (got.masked_fill(got == NEG_INF, 0.0) * weight.to(DEV)).sum().backward()
    for mine, ref in ((c.grad, c64.grad), (g.grad, g64.grad)):
        ref = ref.nan_to_num(0.0)                          # (the oracle's gate of -inf)
        assert torch.allclose(mine.cpu().double(), ref, rtol=2e-4, atol=2e-4 * ref.abs().max().item())


def test_full_size_properties():
    """B=64, L=512, H=8 (the headline graph size): size-independent properties instead of the oracle.
    Every node with a successor gets a distribution over its transitions; the gradient of any function
    of the links sums to zero over a head's window (softmax) and the gate gradients sum to the incoming
    gradient mass of the node."""
    B, L, H = 64, 512, 8
    gen = torch.Generator(device=DEV).manual_seed(1)
    content = torch.randn(B, L, L, H, device=DEV, generator=gen) * 3
    gates = torch.log_softmax(torch.randn(B, L, H, device=DEV, generator=gen), -1).requires_grad_()
    lens = torch.randint(2, L + 1, (B,), device=DEV, generator=gen); lens[0] = L
    vend = lens[:, None].expand(-1, L).contiguous()
    c = content.requires_grad_()
    links = dagx.dag_multihead_links(c * 1, gates, vend, L - 1)
    total = torch.logsumexp(links.detach().float(), -1)                     # [B, L]
    has_next = torch.arange(L, device=DEV)[None, :] < (lens - 1)[:, None]
    assert torch.allclose(total[has_next], torch.zeros_like(total[has_next]), atol=2e-5)
    assert (total[~has_next] == NEG_INF).all()
    weight = torch.randn(links.shape, device=DEV, generator=gen)
    (links.masked_fill(links == NEG_INF, 0.0) * weight).sum().backward()
    assert torch.isfinite(c.grad).all() and torch.isfinite(gates.grad).all()
    per_head = c.grad.sum(2)                                                # sum over targets: [B, L, H]
    scale = c.grad.abs().sum(2).clamp(min=1.0)
    assert (per_head.abs() <= 1e-4 * scale).all()
    mass = (weight * (links.detach() > NEG_INF)).sum(-1)                    # incoming gradient of each node
    assert torch.allclose(gates.grad.sum(-1), mass, rtol=1e-4, atol=1e-3)


def test_argument_errors():
    c = torch.zeros(1, 8, 8, 3, device=DEV); g = torch.zeros(1, 8, 3, device=DEV)
    v = torch.full((1, 8), 8, device=DEV)
    with pytest.raises(RuntimeError, match="heads"):
        dagx.dag_multihead_links(c, g, v, 4)
    with pytest.raises(RuntimeError, match="valid_end"):
        dagx.dag_multihead_links(torch.zeros(1, 8, 8, 4, device=DEV), torch.zeros(1, 8, 4, device=DEV), v.int(), 4)


def test_scores_reused_after_backward_fail_loudly():
    """The backward writes the gradient over the scores; a node that had saved them for its own backward must
    raise rather than differentiate through gradient values."""
    B, L, H = 1, 40, 8
    content, gates, lens = _case(B, L, H, torch.float32, seed=3)
    vend = lens[:, None].expand(-1, L).contiguous().to(DEV)
    c = content.to(DEV).clone().requires_grad_()
    work = c * 1
    other_use = (work * work).sum()                    # saves `work` for its backward
    links = dagx.dag_multihead_links(work, gates.to(DEV), vend, L - 1)
    total = links.masked_fill(links == NEG_INF, 0.0).sum() + other_use
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        total.backward()


def _run_backward(content, gates, vend, translen, weight):
    """links, and the gradients of (links * weight).sum() over the allowed transitions, all on the CPU."""
    c = content.to(DEV).requires_grad_(); g = gates.to(DEV).requires_grad_()
    got = dagx.dag_multihead_links(c * 1, g, vend.to(DEV), translen)
    got.backward(weight.to(DEV))
    return got.detach().cpu(), c.grad.cpu(), g.grad.cpu()


@pytest.mark.parametrize("gate", [3.0, 25.0, 80.0])
@pytest.mark.parametrize("B,L,H", [(2, 120, 4), (1, 300, 8), (1, 700, 16)])
def test_gates_above_zero(B, L, H, gate):
    """Gates need not be log-probabilities.  In every third row a probability that is below the smallest float32 number
    (gate 25, 80) carries its position once its gate has been added, while the other heads keep the position's sum above
    2^-100: head 0 stands at -63.5 there, the others at -68 each.  The other rows: random scores, one gate above 0.
    Scores of 150 times log2(e), added to a normaliser of that size, are rounded to 2^-17 each: a few 1e-5 in a link."""
    content, gates, lens = _case(B, L, H, torch.float32, seed=L, scale=25.0, ragged=False)
    gates[:, 1::3, H - 1] = gate
    content[:, ::3] = -68.0
    content[:, ::3, :, 0] = -63.5 - gate
    for i in range(0, L - 1, 3):
        content[:, i, i + 1] = 0.0
    gates[:, ::3] = 0.0
    gates[:, ::3, 0] = gate
    vend = lens[:, None].expand(-1, L).contiguous()
    c64 = content.double().requires_grad_(); g64 = gates.double().requires_grad_()
    want = tn.multihead_links(c64, g64, _mask(lens, L), L - 1)
    weight = torch.randn(want.shape, generator=torch.Generator().manual_seed(5))
    (want.masked_fill(want == NEG_INF, 0.0) * weight.double()).sum().backward()
    got, dc, dg = _run_backward(content, gates, vend, L - 1, weight)
    _compare(got.double(), want.detach(), 1e-5, 5e-5)
    for mine, ref in ((dc, c64.grad), (dg, g64.grad)):
        assert torch.allclose(mine.double(), ref, rtol=2e-4, atol=2e-4 * ref.abs().max().item())


@pytest.mark.parametrize("L,H", [(40, 4), (300, 8), (700, 16)])
def test_not_a_number_and_infinity_are_not_hidden(L, H):
    """A NaN or an infinity among the scores or gates of a node reaches all gradients of that node and no other's, so that
    a loss scaler sees it; in the forward a NaN score stays at its position, a NaN gate takes the row and a gate of +inf
    makes its links +inf."""
    content, gates, lens = _case(1, L, H, torch.float32, seed=L, ragged=False)
    vend = lens[:, None].expand(-1, L).contiguous()
    weight = torch.randn(1, L, L - 1, generator=torch.Generator().manual_seed(5))
    clean = _run_backward(content, gates, vend, L - 1, weight)
    content[0, 2, L - 5, 1] = float("nan"); gates[0, 5, 1] = float("nan")
    content[0, 7, 20, 2] = float("inf"); gates[0, 9, 3] = float("inf")
    got, dc, dg = _run_backward(content, gates, vend, L - 1, weight)
    assert torch.equal(torch.isnan(got[0, 2]), torch.arange(L - 1) == L - 5 - 3)
    assert torch.isnan(got[0, 5, :L - 6]).all() and (got[0, 9, :L - 10] == float("inf")).all()
    for i in (2, 5, 7, 9):
        assert torch.isnan(dc[0, i, i + 1:]).all() and (dc[0, i, :i + 1] == 0).all() and torch.isnan(dg[0, i]).all()
    rest = torch.tensor([i not in (2, 5, 7, 9) for i in range(L)])
    for mine, ref in zip((got, dc, dg), clean):
        assert torch.equal(mine[0, rest], ref[0, rest])


@pytest.mark.parametrize("L,H", [(40, 4), (300, 8), (700, 16)])
def test_large_gradients_of_unlikely_transitions(L, H):
    """An incoming gradient of 1e30 at transitions down to e^-69: the gradient over the probability leaves the float32
    range, its product with a head's probability does not.  (Scores of 100: probabilities to a few 1e-5, as above.)"""
    content, gates, lens = _case(1, L, H, torch.float32, seed=L, scale=18.0, ragged=False)
    c64 = content.double().requires_grad_(); g64 = gates.double().requires_grad_()
    want = tn.multihead_links(c64, g64, _mask(lens, L), L - 1)
    weight = torch.randn(want.shape, generator=torch.Generator().manual_seed(5)) * 1e30
    (want.masked_fill(want == NEG_INF, 0.0) * weight.double()).sum().backward()
    _, dc, dg = _run_backward(content, gates, lens[:, None].expand(-1, L).contiguous(), L - 1, weight)
    for mine, ref in ((dc, c64.grad), (dg, g64.grad)):
        assert torch.allclose(mine.double(), ref, rtol=2e-4, atol=2e-4 * ref.abs().max().item())
