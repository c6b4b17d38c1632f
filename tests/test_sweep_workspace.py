"""The loss forward's workspace: what dagx_workspace_bytes asks for does not shrink as graphs grow, so a buffer for the largest graph
serves smaller ones; the words of further workgroups come out of what a caller has beyond that."""
import importlib

import pytest
import torch

from da_transformer_amd import _native as nat
from helpers import random_problem
from oracle import torch_native as tn

ops = importlib.import_module("da_transformer_amd.custom_ops.dag_loss")   # (the package exports a function of that name)
DEV = "cuda:0"
KBLK, TILES, GROUPS = 64, 24, 11


def _groups(L, translen, most):
    """Workgroups of a sweep: contiguous blocks of 64 nodes, at most 24 64x64 tiles (the diagonal among them) and `most` blocks each."""
    NB, W = -(-L // KBLK), -(-translen // KBLK)
    groups, tiles, blocks = 1, 0, 0
    for j in range(NB):
        c = j - max(0, j - W) + 1
        if tiles + c > TILES or blocks == most:
            groups, tiles, blocks = groups + 1, 0, 0
        tiles, blocks = tiles + c, blocks + 1
    return groups if groups <= GROUPS else 0


def _bytes(B, L, translen):
    four = _groups(L, translen, 4)
    C = four if 0 < 2 * (-(-B // 8) * 8) * four <= 256 else _groups(L, translen, 8)
    return 4 * ((16 + 2 * B * C + 2 * B + 1) // 2 * 2) + 16 * B


@pytest.mark.parametrize("translen", [None, 1, 64, 200, 450])
def test_what_is_asked_for_is_what_the_fewest_workgroups_need(translen):
    lib = nat.lib()
    for B in [*range(1, 66), 81, 128]:
        last = 0
        for L in range(2, 1025, 13):
            for T in (2, L // 5 + 2, L):
                need = lib.dagx_workspace_bytes(nat.OP_LOSS_FWD, B, T, L, translen or L - 1)
                assert need == _bytes(B, L, translen or L - 1), (B, T, L)
            if translen is None:
                assert need >= last, (B, L)
            last = need
            if B <= 64:   # every number of workgroups has room in what dag_loss allocates
                assert 4 * (16 + 2 * B * GROUPS + 2 * B) + 16 * B <= ops._SMALLEST_WORKSPACE


def _problem(B, L, T):
    match, links_sq, ol, tl = random_problem(L + B, B, L, T, dtype=torch.float32, ragged=True)
    return [x.to(DEV).contiguous() for x in (match, tn.extract_valid_links(links_sq), ol, tl)]


def _loss(p, ws, nbytes):
    m, lk, ol, tl = p
    B, T, L = m.shape
    hats = torch.empty(2, B, T, L, device=DEV)
    offs = torch.empty(2, B, T, -(-L // KBLK), dtype=torch.float64, device=DEV)
    logz, loss = torch.empty(2, B, dtype=torch.float64, device=DEV), torch.empty(B, device=DEV)
    flags = torch.empty(B, dtype=torch.int32, device=DEV)
    nat.check(nat.lib().dagx_loss_fwd(
        m.data_ptr(), nat.dtype_code(m), nat.strides3(m), lk.data_ptr(), nat.dtype_code(lk), ol.data_ptr(), tl.data_ptr(), B, T, L,
        lk.shape[2], hats[0].data_ptr(), hats[1].data_ptr(), offs[0].data_ptr(), offs[1].data_ptr(), logz.data_ptr(), loss.data_ptr(),
        flags.data_ptr(), 1, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert int(ws.count_nonzero()) == 0
    return loss


@pytest.mark.gpu
def test_a_buffer_for_the_largest_graph_serves_smaller_ones():
    ws = torch.zeros(8192, dtype=torch.uint8, device=DEV)
    largest = nat.workspace_bytes(nat.OP_LOSS_FWD, 16, 128, 1024, 1023)
    for B, L, T in [(16, 1024, 128), (16, 960, 96), (16, 700, 90), (16, 330, 40), (3, 700, 90)]:
        p = _problem(B, L, T)
        few, many = _loss(p, ws, largest), _loss(p, ws, ws.numel())
        # both are within 6e-7 of a cell and step of the exact value (tests/test_gpu_dag_chunks.py)
        assert ((few - many).abs() <= 2 * (6e-7 * T + 2e-7 * few.abs())).all(), (B, L, T)
    ws = torch.zeros(8192, dtype=torch.uint8, device=DEV)
    largest = nat.workspace_bytes(nat.OP_LOSS_FWD, 64, 64, 512, 511)
    _loss(_problem(64, 400, 80), ws, largest)
    need = nat.workspace_bytes(nat.OP_LOSS_FWD, 64, 80, 400, 399)
    with pytest.raises(RuntimeError, match="workspace"):
        _loss(_problem(64, 400, 80), ws, need - 1)


@pytest.mark.gpu
def test_a_batch_of_smaller_graphs_keeps_the_buffer():
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        kept = None
        for B, L, T in [(64, 512, 20), (64, 400, 20), (8, 700, 70), (16, 1024, 100)]:
            ops.dag_loss(*_problem(B, L, T))
            ws = ops._clean_workspaces[(0, nat.raw_stream(0))]
            assert kept is None or ws is kept, (B, L)
            kept = ws
    stream.synchronize()
