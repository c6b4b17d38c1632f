"""The chunked sweeps of dag_loss, in float32 and float64, and of dag_best_alignment at the sizes where they can go wrong:
graphs one node short of, at and one past a block of 64 and a group's last block, targets one step around a chunk of four, transition windows around a block,
transitions that start at an odd element of their tensor or are its very first and last ones, one sample alone."""
import math

import pytest
import torch

import da_transformer_amd as dagx
from da_transformer_amd import _native as nat
from da_transformer_amd.custom_ops.dag_loss import DagLossFunc, _clean_workspaces, _sweep_offsets
from oracle import torch_native as tn
from helpers import random_problem
from test_gpu_dag import DEV, hip_loss_and_grads, oracle_loss_and_grads, assert_close, RTOL

pytestmark = pytest.mark.gpu
F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("B,L,T,translen,dtype", [
    (1, 2, 2, 1, F32), (3, 2, 2, 1, F16), (2, 5, 5, 1, F32), (1, 20, 6, None, F16),
    (1, 63, 5, None, F32), (2, 64, 2, None, F16), (1, 65, 6, 63, F16), (3, 65, 9, 64, BF16), (2, 66, 10, 1, F32),
    (1, 127, 13, 65, F32), (2, 129, 17, 2, BF16), (1, 320, 8, None, F16), (2, 321, 9, 128, F32), (1, 385, 33, 63, F16),
    (2, 449, 30, 32, F32), (1, 511, 14, None, BF16), (2, 513, 7, 257, F32), (1, 705, 12, 130, F16), (2, 1024, 11, None, F32),
    (1, 1023, 64, 200, F16),
    (65, 320, 8, None, F16), (65, 1022, 20, 64, F16)])   # no room for groups of at most four blocks: five, eight
def test_edges_of_blocks_chunks_and_windows(B, L, T, translen, dtype, wide):
    match, links_sq, ol, tl = random_problem(L + T, B + 1, L, T, dtype=F32, ragged=False, translen=translen)
    if translen is not None:      # a path of T_b nodes spans at most (T_b - 1) translen transitions
        ol = torch.minimum(ol, (tl - 1) * translen + 1).clamp_(min=1)
    if B > 1:
        tl[1] = max(1, T - 1)
        ol[1] = max(int(tl[1]), int(ol[1]) - 3) if translen is None else int(tl[1])
    match, links = match.to(dtype), tn.extract_valid_links(links_sq, translen).to(dtype)
    ol, tl = ol[:B], tl[:B]
    g = torch.linspace(-1.0, 2.0, B)
    rloss, rgm, rgl = oracle_loss_and_grads(match[1:], links[1:], ol, tl, g)
    # views from the second sample on: contiguous, the first element anywhere in a four-byte word
    before = nat.lib().dagx_loss_float64_first(int(wide))
    try:
        loss, gm, gl = hip_loss_and_grads(match.to(DEV)[1:], links.to(DEV)[1:], ol, tl, g)
    finally:
        nat.lib().dagx_loss_float64_first(before)
    if B * L * links.shape[2] >= 4:       # the sweeps' own result (but for a sample without a path)
        assert (DagLossFunc.last_sample_flags.cpu()[torch.isfinite(rloss)] == (2 if wide else 0)).all()
    # per step a chain of at most 64 products a tile, two exponentials and the partial sums: 6e-7 of the cell
    fin = torch.isfinite(rloss)
    assert torch.equal(torch.isfinite(loss), fin)
    assert ((loss.double() - rloss)[fin].abs() <= 6e-7 * T + 2e-7 * rloss[fin].abs()).all(), (loss, rloss)
    assert_close(gm.float(), rgm, RTOL[dtype], "grad_match")
    assert_close(gl.float(), rgl, RTOL[dtype], "grad_links")


# Batches in which samples of some lengths get more workgroups than those of others, with the table of groups that the float32 and the
# float64 sweeps of a call take, 0: as many for every sample (test_sweep_tables.py works it out from the same lengths).
TABLE_BATCHES = [
    # B, L, T, shortest, dtype, tables
    (3, 650, 24, 1, F32, (2, 2)), (16, 760, 24, 570, F32, (2, 2)), (16, 768, 21, 768, F16, (2, 2)), (20, 760, 24, 760, F32, (1, 1)),
    (20, 765, 24, 400, BF16, (2, 2)), (24, 768, 24, 768, F32, (0, 0)), (5, 1024, 98, 700, F32, (0, 0)), (64, 390, 12, 1, F16, (0, 1)),
    (16, 1024, 128, 768, F32, (1, 1)), (16, 1000, 131, 750, F16, (1, 2)), (14, 1010, 130, 760, BF16, (1, 2)), (16, 1024, 130, 1024, F32, (0, 0)),
    (1, 800, 60, 800, F32, (2, 2)), (2, 523, 104, 400, F32, (2, 2))]


def table_lengths(B, L, T, shortest):
    ol = torch.randint(shortest, L + 1, (B,), generator=torch.Generator().manual_seed(B))
    tl = torch.full((B,), T)
    ol[0] = L
    tl = torch.minimum(tl, ol)
    if B > 4:
        ol[2], tl[3] = 0, T + 1          # samples without a length, among the others
    return ol, tl


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("B,L,T,shortest,dtype", [batch[:5] for batch in TABLE_BATCHES])
def test_batches_whose_samples_get_different_numbers_of_workgroups(B, L, T, shortest, dtype, wide):
    match, links_sq, _, _ = random_problem(L + B, B, L, T, dtype=F32, ragged=False)
    ol, tl = table_lengths(B, L, T, shortest)
    cols = torch.arange(L).view(1, 1, L) < ol.view(B, 1, 1)
    links_sq = torch.log_softmax(links_sq.masked_fill(~cols, -1e30), -1).masked_fill(~cols | ~torch.isfinite(links_sq), float("-inf"))
    match, links = match.to(dtype), tn.extract_valid_links(links_sq).to(dtype)
    good = (ol >= 1) & (tl <= T) & (tl <= ol)
    g = torch.linspace(0.5, 2.0, B)
    rloss, rgm, rgl = oracle_loss_and_grads(match[good], links[good], ol[good], tl[good], g[good])
    before = nat.lib().dagx_loss_float64_first(int(wide))
    try:
        for _ in range(2):               # the pipeline words are left as they were found
            loss, gm, gl = hip_loss_and_grads(match.to(DEV), links.to(DEV), ol, tl, g)
    finally:
        nat.lib().dagx_loss_float64_first(before)
    fin = torch.isfinite(rloss)
    assert (DagLossFunc.last_sample_flags.cpu()[good][fin] == (2 if wide else 0)).all()
    assert torch.isneginf(loss[~good]).all() and torch.equal(torch.isfinite(loss[good]), fin)
    # as above: 6e-7 of a cell and step
    assert ((loss[good].double() - rloss)[fin].abs() <= 6e-7 * T + 2e-7 * rloss[fin].abs()).all()
    assert_close(gm.float()[good], rgm, RTOL[dtype], "grad_match")
    assert_close(gl.float()[good], rgl, RTOL[dtype], "grad_links")


def mixed_lengths():
    T, L = 130, 1024
    ol = torch.randint(768, L + 1, (16,), generator=torch.Generator().manual_seed(3))
    ol[0] = L
    return T, L, ol


@pytest.mark.parametrize("with_grad", [True, False])
def test_some_samples_of_a_batch_with_tables_go_on_to_the_float64_sweeps(with_grad):
    """The float32 and the float64 launch of a call have groups, and so a layout of the workspace, of their own; the float64 launch
    passes over the samples that the float32 launch settled."""
    T, L, ol = mixed_lengths()
    B = len(ol)
    peaked = torch.arange(B) % 3 == 1
    cols = torch.arange(L).view(1, 1, L) < ol.view(B, 1, 1)
    gen = torch.Generator().manual_seed(11)
    sq = torch.randn(B, L, L, generator=gen) * torch.where(peaked, 20.0, 1.0).view(B, 1, 1)
    sq = tn.restore_valid_links(tn.extract_valid_links(sq))
    dead = ~(torch.isfinite(sq) & cols)
    links = tn.extract_valid_links(torch.log_softmax(sq.masked_fill(dead, -1e30), -1).masked_fill(dead, float("-inf")))
    match = torch.randn(B, T, L, generator=gen) - 2.0
    tl = torch.full((B,), T)
    g = torch.linspace(0.5, 2.0, B)
    rloss, rgm, rgl = oracle_loss_and_grads(match, links, ol, tl, g)
    assert torch.isfinite(rloss).all()
    for _ in range(2):
        if with_grad:
            loss, gm, gl = hip_loss_and_grads(match, links, ol, tl, g)
            assert_close(gm, rgm, RTOL[F32], "grad_match")
            assert_close(gl, rgl, RTOL[F32], "grad_links")
        else:
            with torch.no_grad():
                loss = dagx.dag_loss(match.to(DEV), links.to(DEV), ol.to(DEV), tl.to(DEV)).cpu()
        flags = DagLossFunc.last_sample_flags.cpu()
        assert (flags[~peaked] == 0).all() and (flags[peaked] == 2).any(), flags
        # the float32 sweeps' bound as above; the float64 ones' read-outs agree to 1e-8 of the value and 5e-5
        assert ((loss.double() - rloss).abs() <= 6e-7 * T + 2e-7 * rloss.abs()).all(), (loss, rloss)
        assert all(int(ws.count_nonzero()) == 0 for ws in _clean_workspaces.values())


@pytest.mark.parametrize("B,L,T,translen,dtype", [
    (1, 2, 2, 1, F32), (3, 2, 2, 1, F16), (2, 5, 5, 1, F32), (1, 63, 5, None, F16), (2, 64, 2, None, F32), (1, 65, 6, 63, BF16),
    (3, 65, 9, 64, F32), (2, 129, 17, 2, F16), (1, 257, 8, None, F32), (2, 320, 9, 128, F16), (1, 321, 33, 63, F32),
    (2, 449, 30, 32, BF16), (1, 511, 14, None, F32), (2, 513, 7, 257, F16), (1, 705, 12, 130, F32), (2, 1024, 11, None, F16),
    (1, 1023, 64, 200, F32),
    # up to three blocks of 64 nodes in chunks where T is at least 6 ceil(L / 64) + 8, else step by step
    (1, 64, 13, None, F32), (2, 128, 20, None, F32), (2, 129, 25, None, F32), (1, 129, 26, None, F16),
    # in chunks, of more than three blocks
    (2, 448, 50, None, F16), (2, 449, 56, 100, F32), (1, 513, 62, 257, F16), (1, 705, 80, 130, F32), (2, 1024, 104, None, F16),
    # few workgroups a sample: groups of several blocks (of eight in the last), one and two stages a block
    (65, 250, 33, None, F32), (65, 512, 66, None, F16), (129, 1022, 130, 64, F16),
    # of more than three blocks in chunks from 2 ceil(L / 64) + 22 on, where transitions span at most three blocks from 4 ceil(L / 64) + 14 on,
    # of eight blocks with a workgroup each from 43 on
    (2, 256, 29, None, F32), (2, 256, 30, None, F16), (1, 300, 31, None, F32), (3, 300, 32, 200, F32), (65, 500, 37, None, F16), (65, 500, 38, None, F32),
    (3, 500, 42, None, F32), (3, 500, 43, None, F16),
    (2, 1024, 53, None, F16), (2, 1024, 54, None, F32), (1, 700, 57, 192, F32), (2, 700, 58, 192, F16), (2, 1000, 78, 100, F32), (1, 700, 44, 193, F16),
    # step by step, one workgroup a sample: twelve and eleven blocks in eight waves, and as many tiles as make the fetching wave take some; a
    # single block more than waves
    (129, 768, 40, 64, F32), (129, 700, 57, 64, F16), (129, 576, 30, 64, BF16)])
def test_alignment_at_edges_of_blocks_chunks_and_windows(B, L, T, translen, dtype):
    match, links_sq, ol, tl = random_problem(L + T, B + 1, L, T, dtype=F32, ragged=False, translen=translen)
    if translen is not None:      # a path of T_b nodes spans at most (T_b - 1) translen transitions
        ol = torch.minimum(ol, (tl - 1) * translen + 1).clamp_(min=1)
    if B > 1:
        tl[1] = max(1, T - 1)
        ol[1] = max(int(tl[1]), int(ol[1]) - 3) if translen is None else int(tl[1])
    match, links = match.to(dtype), tn.extract_valid_links(links_sq, translen).to(dtype)
    ol, tl = ol[:B], tl[:B]
    # coarse scores: many ties, which the lowest predecessor has to win
    match, links = (match * 4).round() / 4, (links * 4).round() / 4
    got = dagx.dag_best_alignment(match.to(DEV)[1:], links.to(DEV)[1:], ol.to(DEV), tl.to(DEV)).cpu()
    some = sorted({0, min(1, B - 1), B // 2, B - 1})
    want = tn.torch_dag_best_alignment(match[1:][some].float(), tn.restore_valid_links(links[1:][some].float()), ol[some], tl[some])
    assert torch.equal(got[some], want)


@pytest.mark.parametrize("B,L,T", [(2, 64, 13), (2, 129, 25), (65, 250, 33), (65, 512, 66), (1, 1000, 110)])   # steps, chunks of both spacings
def test_alignment_of_subnormal_scores(B, L, T):
    """The sums of scores are formed by matrix instructions, which keep every bit of subnormal ones: whole multiples of the smallest."""
    match, links_sq, ol, tl = random_problem(L, B, L, T, dtype=F32)
    links = tn.extract_valid_links(links_sq, None)
    match, links = (match * 8).round() * 2.0 ** -149, (links * 8).round() * 2.0 ** -149
    assert 0 < match.abs().max() < 2.0 ** -126
    got = dagx.dag_best_alignment(match.to(DEV), links.to(DEV), ol.to(DEV), tl.to(DEV)).cpu()
    some = sorted({0, B // 2, B - 1})
    want = tn.torch_dag_best_alignment(match[some], tn.restore_valid_links(links[some]), ol[some], tl[some])
    assert torch.equal(got[some], want)


def alignment_by_the_rule(match, square, out_len, tgt_len):
    """One sample in float32: the first largest candidate wins, a sum that is no number is no candidate, and an end without a finite or
    infinite score above -inf has no path."""
    neg = float("-inf")
    cells = torch.full((square.shape[0],), neg)
    cells[0] = match[0, 0]
    came_from = []
    for t in range(1, tgt_len):
        sums = cells.unsqueeze(1) + square
        best, first = sums.masked_fill(sums.isnan(), neg).max(0)
        came_from.append(first)
        cells = best + match[t]
    path = torch.full((square.shape[0],), -1)
    node = out_len - 1
    if not cells[node] > neg:
        return path
    path[node] = tgt_len - 1
    for t in range(tgt_len - 1, 0, -1):
        node = int(came_from[t - 1][node])
        path[node] = t - 1
    return path


def with_extremes(kind, x, gen):
    """Some of the scores replaced: 'lowest' what masks stand for -inf with, whose sums overflow to it; 'huge' sums that overflow on either
    side; 'special' infinities and NaN."""
    pick = torch.rand(x.shape, generator=gen)
    if kind == "lowest":
        return x.masked_fill((pick < 0.5) & torch.isfinite(x), torch.finfo(x.dtype).min)
    if kind == "huge":
        return torch.where(pick < 0.3, x * 3e37, x)
    x = x.masked_fill(pick < 2e-3, float("inf"))
    return x.masked_fill(pick > 0.98, float("nan"))


@pytest.mark.parametrize("kind,dtype", [("lowest", F32), ("lowest", BF16), ("huge", F32), ("special", F32), ("special", F16)])
@pytest.mark.parametrize("B,L,T", [(3, 64, 20), (3, 200, 18), (65, 250, 33), (260, 130, 12), (65, 512, 66), (2, 1000, 24)])
def test_alignment_of_lowest_overflowing_infinite_and_undefined_scores(B, L, T, kind, dtype):
    gen = torch.Generator().manual_seed(L + T)
    match, links_sq, ol, tl = random_problem(L, B, L, T, dtype=F32)
    links = with_extremes(kind, tn.extract_valid_links(links_sq, None).to(dtype), gen)
    match = with_extremes(kind, match.to(dtype), gen)
    match[:, 0, 0] = -1.0
    some = sorted({0, 1, B // 2, B - 1})
    want = torch.stack([alignment_by_the_rule(match[b].float(), tn.restore_valid_links(links[b:b + 1].float())[0], int(ol[b]), int(tl[b])) for b in some])
    assert (want >= 0).any(1).all()
    for mode in (0, 1, 2):      # the sweeps; one workgroup a sample; the sweeps, and every sample done again
        before = nat.lib().dagx_force_log_domain(mode)
        try:
            got = dagx.dag_best_alignment(match.to(DEV), links.to(DEV), ol.to(DEV), tl.to(DEV)).cpu()
        finally:
            nat.lib().dagx_force_log_domain(before)
        assert torch.equal(got[some], want), mode


@pytest.mark.parametrize("kind", ["lowest", "huge", "special"])
@pytest.mark.parametrize("B,L,steps", [(3, 64, 10), (3, 64, 20), (3, 250, 12), (65, 512, 64), (2, 1000, 24), (260, 100, 30)])
def test_viterbi_decoding_of_lowest_overflowing_infinite_and_undefined_scores(B, L, steps, kind):
    """The sweeps against the table by one workgroup a sample."""
    gen = torch.Generator().manual_seed(L + steps)
    _, links_sq, ol, _ = random_problem(L, B, L, 4, dtype=F32)
    links = with_extremes(kind, tn.extract_valid_links(links_sq, None), gen).to(DEV)
    scores = with_extremes(kind, torch.randn(B, L, generator=gen) - 2.0, gen).to(DEV)
    tokens = torch.randint(4, 50, (B, L), generator=gen).to(DEV)
    out = []
    for mode in (0, 1):
        before = nat.lib().dagx_force_log_domain(mode)
        try:
            out.append(dagx.dag_viterbi_decode(links, (scores, tokens), ol.to(DEV), 2 * L / steps, 1.0, True, 1))
        finally:
            nat.lib().dagx_force_log_domain(before)
    assert out[0].nodes.shape[1] == steps
    for name in ("output_tokens", "pred_length", "nodes"):
        assert torch.equal(getattr(out[0], name), getattr(out[1], name)), name


@pytest.mark.parametrize("B,L,T,translen,dtype,first", [
    (1, 4, 4, 1, F32, 0), (2, 4, 4, 3, F16, 1), (3, 5, 5, 1, F16, 3), (2, 6, 6, 2, F32, 2), (2, 63, 32, 2, F16, 1), (3, 64, 64, 1, F32, 1),
    (2, 65, 40, 3, BF16, 3), (1, 66, 66, 1, F16, 0), (3, 127, 64, 3, F32, 3), (2, 129, 129, 1, BF16, 1), (2, 130, 70, 2, F32, 2),
    (2, 195, 100, 2, F16, 3), (1, 321, 200, 3, F32, 1)])
def test_staged_walks_at_the_ends_of_a_sample_and_with_windows_of_one_to_three(B, L, T, translen, dtype, first):
    """The walk stages transitions four neighbouring elements a load.  Loads that would leave the sample are moved inside; what stands
    in front of the tensor, behind it and in the samples beside it, here better than any transition, is nobody's successor."""
    gen = torch.Generator().manual_seed(L + T)
    links = (torch.randn(B, L, translen, generator=gen) * 4).round() / 4 - 2.0
    node = torch.arange(L).view(1, L, 1)
    links = links.masked_fill(node + torch.arange(1, translen + 1) >= L, 40.0 if translen > 1 else float("-inf"))
    match = (torch.randn(B, T, L, generator=gen) * 4).round() / 4
    ol = torch.full((B,), min(L, (T - 1) * translen + 1))
    tl = torch.full((B,), T)
    links, match = links.to(dtype), match.to(dtype)
    room = torch.full((first + links.numel() + 8,), 40.0, dtype=dtype, device=DEV)
    room[first:first + links.numel()] = links.to(DEV).reshape(-1)
    got = dagx.dag_best_alignment(match.to(DEV), room[first:first + links.numel()].view(links.shape), ol.to(DEV), tl.to(DEV)).cpu()
    inside = links.float().masked_fill(node + torch.arange(1, translen + 1) >= ol.view(B, 1, 1), float("-inf"))
    want = tn.torch_dag_best_alignment(match.float(), tn.restore_valid_links(inside), ol, tl)
    assert torch.equal(got, want)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("B,L,T,translen,score", [
    (2, 640, 41, 639, 0.0),        # hundreds of predecessors with transitions of 1 feed every cell: sums of up to 2^9 cells
    (2, 1024, 102, 1023, -0.01), (3, 200, 22, 64, 0.0),
    (2, 130, 9, 129, None), (3, 512, 64, 511, None), (65, 321, 30, 320, None)])
def test_tables_are_relative_to_the_largest_cell_of_their_block(B, L, T, translen, score, wide):
    """What the gradients rely on, in every step and not only in those that scale their cells: a residual is never above 0, and
    the largest one of a block with a live cell lies within a binade below it."""
    match, links_sq, ol, tl = random_problem(L + T, B, L, T, dtype=F32, ragged=False, translen=translen)
    if score is not None:
        links_sq = torch.where(torch.isfinite(links_sq), torch.tensor(score), links_sq)
        match = torch.where(torch.isfinite(match), torch.tensor(score), match)
    ol = torch.minimum(ol, (tl - 1) * translen + 1)
    ol[B - 1] = max(T, L - 37)
    links = tn.extract_valid_links(links_sq, translen)
    before = nat.lib().dagx_loss_float64_first(int(wide))
    try:
        loss = DagLossFunc.apply(match.to(DEV).requires_grad_(), links.to(DEV), ol.to(DEV), tl.to(DEV))
    finally:
        nat.lib().dagx_loss_float64_first(before)
    assert (DagLossFunc.last_sample_flags.cpu() == (2 if wide else 0)).all()
    hats, offs = (x.cpu() for x in loss.grad_fn.saved_tensors[:2])
    NBK = (L + 63) // 64
    nhat, noff = _sweep_offsets(B, T, L)
    for direction in range(2):
        hat = hats[direction * nhat:(direction + 1) * nhat].view(B, T, L)
        off = offs[direction * noff:(direction + 1) * noff].view(B, T, NBK)
        for b in range(B):
            n, steps = int(ol[b]), int(tl[b])
            cells = hat[b, :steps, :n].flip(1) if direction else hat[b, :steps, :n]      # by position
            cells = torch.nn.functional.pad(cells, (0, -n % 64), value=float("-inf")).view(steps, -1, 64)
            top, alive = cells.amax(2), torch.isfinite(off[b, :steps, :cells.shape[1]])
            assert (top[alive] <= 0).all(), (direction, b, top[alive].max())
            # (a logarithm of a fraction in [1/2, 1), two float32 roundings)
            assert (top[alive] >= -math.log(2.0) - 1e-6).all(), (direction, b, top[alive].min())
