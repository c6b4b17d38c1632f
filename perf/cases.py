"""What a user of these operators has them do, as cases that can be timed: training steps of the DAG loss from a toy
graph to a thousand nodes, scoring, alignment, the fused log-softmax + gather, the whole criterion step, the link
predictor's tail and decoding of a batch and of a single sentence.

A case is a dict of plain values; `listed()` gives the fixed ones, `draw(rng)` one more from the same ranges,
`prepare(case, seed)` the inputs on the GPU, `run(state)` one pass through the public functions, `work(case)` the
bytes and operations a pass cannot do without and `tolerance(case)` how far two correct implementations may differ.

Shared fields: B samples, L graph nodes, T target tokens, window (longest transition, L - 1 = no limit), dtype,
ragged (lengths drawn between three quarters and all of L and T, as a length-bucketed batch has them; false: all
full), peak (standard deviation of the transition logits: 1 at the start of training, 10 for a trained model, whose
token log-probabilities spread five times as far and which has a few nodes pinned to targets by glancing).
"""
import math

import torch

import da_transformer_amd as dagx

NEG_INF = float("-inf")
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
PAD = 1

# the most a drawn case may hold: pair updates, logits and link scores of the largest listed case of its kind
MOST_CELLS = 16 * 1024 * 1024 * 256
MOST_LOGITS = 64 * 512 * 40000
MOST_CRITERION_LOGITS = 16 * 1024 * 30522
MOST_SCORES = 64 * 512 * 512 * 8


def listed():
    return [
        # a unit test, a debugging run or the last small bucket of an epoch: launches and host time count
        dict(name="loss_tiny", kind="loss", B=4, L=64, T=16, window=63, dtype="float32", ragged=False, peak=1, grad=True, storage="btl"),
        # the operator's headline shape: a full batch of mid-length sentences in mixed precision
        dict(name="loss_base", kind="loss", B=64, L=512, T=64, window=511, dtype="float16", ragged=False, peak=1, grad=True, storage="btl"),
        # limited transitions (--max-transition-length 32), odd batch, a graph size that is no multiple of 64
        dict(name="loss_window", kind="loss", B=81, L=400, T=50, window=32, dtype="float32", ragged=True, peak=1, grad=True, storage="btl"),
        # long documents: match is the transposed view of the gather's output, as the criterion passes it
        dict(name="loss_long", kind="loss", B=16, L=1024, T=256, window=1023, dtype="float32", ragged=True, peak=1, grad=True, storage="blt"),
        # the same graphs late in training, where probabilities are sharply peaked
        dict(name="loss_trained", kind="loss", B=16, L=1024, T=256, window=1023, dtype="float32", ragged=True, peak=10, grad=True, storage="btl"),
        # validation: scores of a ragged batch without gradients
        dict(name="loss_score", kind="loss", B=40, L=328, T=41, window=327, dtype="bfloat16", ragged=True, peak=1, grad=False, storage="blt"),
        # the glancing step's alignment
        dict(name="align_base", kind="align", B=64, L=512, T=64, window=511, dtype="float32", ragged=True, peak=1, storage="blt"),
        # log-probabilities of the targets out of a full batch of logits, forward and backward
        dict(name="gather_base", kind="gather", B=64, L=512, T=64, V=40000, dtype="float16"),
        # everything the criterion runs for one training step: glancing pass, then loss and backward to logits and links
        dict(name="criterion_long", kind="criterion", B=16, L=1024, T=256, V=30522, dtype="float16", ragged=True),
        # transition log-probabilities from the link predictor's per-head scores, forward and backward
        dict(name="links_base", kind="links", B=64, L=512, H=8, window=511, dtype="float32", ragged=True),
        # offline decoding of a test set in batches
        dict(name="decode_batch", kind="decode", B=64, L=512, V=40000, dtype="float16", strategy="jointviterbi", ragged=True),
        # serving: one sentence at a time, latency is what the user sees
        dict(name="decode_single", kind="decode", B=1, L=184, V=40000, dtype="float16", strategy="lookahead", ragged=False),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _graph(rng, most_cells):
    """B, L, T and the window of a drawn graph batch."""
    L = _log_int(rng, 24, 1024)
    T = max(4, min(256, round(L / rng.uniform(3.0, 10.0))))
    B = _log_int(rng, 1, max(1, min(128, most_cells // (L * L * T))))
    window = L - 1 if rng.random() < 0.7 else _log_int(rng, min(L - 1, max(8, math.ceil(4 * L / T))), L - 1)
    return dict(B=B, L=L, T=T, window=window, ragged=rng.random() < 0.7)


def draw(rng):
    kind = rng.choices(["loss", "align", "gather", "criterion", "links", "decode"], [8, 3, 3, 2, 3, 4])[0]
    dtype = rng.choice(["float32", "float16", "bfloat16"])
    if kind in ("loss", "align"):
        case = dict(kind=kind, dtype=dtype, peak=10 if rng.random() < 0.3 else 1, storage=rng.choice(["btl", "blt"]),
                    **_graph(rng, MOST_CELLS))
        return dict(case, grad=rng.random() < 0.8) if kind == "loss" else case
    if kind in ("gather", "criterion"):
        graph = _graph(rng, MOST_CELLS)
        V = _log_int(rng, 1000, 60000)
        most = MOST_LOGITS if kind == "gather" else MOST_CRITERION_LOGITS
        if dtype == "float32":
            most //= 2
        case = dict(kind=kind, L=graph["L"], T=graph["T"], V=V, dtype=dtype, B=max(1, min(graph["B"], most // (graph["L"] * V))))
        return dict(case, ragged=graph["ragged"]) if kind == "criterion" else case
    if kind == "links":
        H, L = rng.choice([4, 8, 16]), _log_int(rng, 24, 1024)
        B = _log_int(rng, 1, max(1, min(128, MOST_SCORES // (L * L * H))))
        window = L - 1 if rng.random() < 0.7 else _log_int(rng, 8, L - 1)
        return dict(kind=kind, B=B, L=L, H=H, window=window, dtype=dtype, ragged=rng.random() < 0.7)
    L, V = _log_int(rng, 32, 1024), _log_int(rng, 1000, 60000)
    B = 1 if rng.random() < 0.4 else _log_int(rng, 2, max(2, min(64, MOST_LOGITS // (2 * L * V))))
    strategy = rng.choice(["viterbi", "jointviterbi", "lookahead", "greedy"])
    return dict(kind=kind, B=B, L=L, V=V, dtype=dtype, strategy=strategy, ragged=B > 1 and rng.random() < 0.7)


# ---- inputs -----------------------------------------------------------------------------------------------------

def _lengths(case, gen, dev):
    B, L, T = case["B"], case["L"], case.get("T", 1)
    if not case.get("ragged", False):
        out_len, tgt_len = torch.full((B,), L), torch.full((B,), T)
    else:
        out_len = torch.randint(max(2, (3 * L) // 4), L + 1, (B,), generator=gen)
        tgt_len = torch.randint(max(2, (3 * T) // 4), max(2, T) + 1, (B,), generator=gen)
        out_len[0], tgt_len[0] = L, T
    return out_len.to(dev), torch.minimum(tgt_len, out_len).to(dev)


def _links(case, out_len, gen, dev, scale, dtype):
    """[B, L, window]: log-softmax over every node's successors inside its sample, -inf beyond (what a link predictor emits)."""
    B, L, W = case["B"], case["L"], case.get("window", case["L"] - 1)
    reach = torch.arange(L, device=dev).view(1, L, 1) + torch.arange(1, W + 1, device=dev).view(1, 1, W)
    links = torch.empty(B, L, W, dtype=dtype, device=dev)
    at_once = max(1, (1 << 25) // (L * W))
    for b in range(0, B, at_once):
        part = out_len[b:b + at_once].view(-1, 1, 1)
        logits = torch.randn(part.shape[0], L, W, generator=gen, device=dev).mul_(scale).masked_fill_(reach >= part, NEG_INF)
        links[b:b + at_once] = torch.log_softmax(logits, -1).nan_to_num_(NEG_INF, neginf=NEG_INF)
    return links


def _match(case, out_len, tgt_len, gen, dev, dtype):
    """[B, T, L]: log-probability of every target at every node, from logits of standard deviation 1 (5 late in training)
    over a vocabulary of 8000; late in training a few targets are pinned to a node."""
    B, L, T = case["B"], case["L"], case["T"]
    std = 5.0 if case["peak"] > 1 else 1.0
    rest = min(math.log(8000.0) + std * std / 2, std * math.sqrt(2 * math.log(8000.0)) + 1.0)
    logits = torch.randn(B, T, L, generator=gen, device=dev).mul_(std)
    match = logits - torch.logaddexp(torch.logsumexp(logits, 1, keepdim=True), torch.tensor(rest, device=dev))
    if case["peak"] > 1:
        for k in (1, 2, 3):
            t = ((k * tgt_len) // 4).clamp_(min=1)
            node = torch.minimum(torch.maximum((t * out_len) // tgt_len, t), out_len - 2)
            keep = (t < tgt_len - 1) & (node >= t)
            hit = (torch.arange(T, device=dev).view(1, T, 1) == t.view(B, 1, 1)) & keep.view(B, 1, 1)
            match = torch.where(hit, torch.where(torch.arange(L, device=dev).view(1, 1, L) == node.view(B, 1, 1), 0.0, NEG_INF), match)
    match = match.to(dtype)
    # "blt": the values lie as [B, L, T] and the operators get the transposed view, as from the gather
    return match.transpose(1, 2).contiguous().transpose(1, 2) if case["storage"] == "blt" else match


class _Produced(torch.autograd.Function):
    """Stands for the layer that wrote a tensor: the operators may take the tensor's storage for its gradient, which
    they may not do with a leaf.  No copy either way."""

    @staticmethod
    def forward(ctx, leaf):
        return leaf.detach()

    @staticmethod
    def backward(ctx, grad):
        return grad


def _logits(case, gen, dev, std):
    return torch.empty(case["B"], case["L"], case["V"], dtype=DTYPES[case["dtype"]], device=dev).normal_(0.0, std, generator=gen)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen, host = torch.Generator(dev).manual_seed(seed), torch.Generator().manual_seed(seed)
    dtype, kind = DTYPES[case["dtype"]], case["kind"]
    B, L = case["B"], case["L"]
    out_len, tgt_len = _lengths(case, host, dev)
    state = dict(kind=kind, out_len=out_len, tgt_len=tgt_len)
    if kind in ("loss", "align"):
        grad = kind == "loss" and case["grad"]
        state["match"] = _match(case, out_len, tgt_len, gen, dev, dtype).requires_grad_(grad)
        state["links"] = _links(case, out_len, gen, dev, case["peak"], dtype).requires_grad_(grad)
        # the gradient of -(loss / target length).mean() under a loss scale of 128
        state["grad"] = (-128.0 / (B * tgt_len)).float() if grad else None
    elif kind == "gather":
        # both directions run in the logits' own storage, so a further pass finds the last one's gradient there
        state["logits"] = _logits(case, gen, dev, 2.0).requires_grad_()
        state["targets"] = torch.randint(4, case["V"], (B, case["T"]), generator=gen, device=dev)
        state["grad"] = torch.randn(B, case["T"], L, generator=gen, device=dev).transpose(1, 2)
    elif kind == "criterion":
        state["first_logits"] = _logits(case, gen, dev, 1.0)
        state["logits"] = _logits(case, gen, dev, 1.0).requires_grad_()
        state["links"] = _links(case, out_len, gen, dev, 1.0, torch.float32).requires_grad_()
        targets = torch.randint(4, case["V"], (B, case["T"]), generator=gen, device=dev)
        state["targets"] = targets.masked_fill(torch.arange(case["T"], device=dev) >= tgt_len.view(B, 1), PAD)
        state["decoder_input"] = torch.full((B, L), 3, device=dev).masked_fill(torch.arange(L, device=dev) >= out_len.view(B, 1), PAD)
        state["rand"] = torch.rand(B, L, generator=gen, device=dev)
    elif kind == "links":
        state["scores"] = torch.empty(B, L, L, case["H"], dtype=dtype, device=dev).normal_(generator=gen).requires_grad_()
        state["gates"] = torch.log_softmax(torch.randn(B, L, case["H"], generator=gen, device=dev), -1).requires_grad_()
        state["valid_end"] = out_len.view(B, 1).expand(B, L).contiguous()
        state["window"] = case["window"]
        state["grad"] = torch.randn(B, L, case["window"], generator=gen, device=dev).to(dtype)
    else:
        state["logits"] = _logits(case, gen, dev, 2.0)
        state["links"] = _links(case, out_len, gen, dev, 1.0, torch.float32)
        state["strategy"] = case["strategy"]
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------

def _run_loss(s):
    loss = dagx.dag_loss(s["match"], s["links"], s["out_len"], s["tgt_len"])
    if s["grad"] is None:
        return loss
    return (loss.detach(),) + torch.autograd.grad(loss, (s["match"], s["links"]), s["grad"])


def _run_gather(s):
    ids = s["targets"].unsqueeze(1).expand(-1, s["logits"].shape[1], -1)
    _, selected = dagx.dag_logsoftmax_gather_inplace(_Produced.apply(s["logits"]), ids)
    return (selected.detach(),) + torch.autograd.grad(selected, s["logits"], s["grad"])


def _run_criterion(s):
    ids = s["targets"].unsqueeze(1).expand(-1, s["logits"].shape[1], -1)
    out_len, tgt_len = s["out_len"], s["tgt_len"]
    with torch.no_grad():
        _, match, best_tokens = dagx.dag_logsoftmax_gather_argmax(s["first_logits"], ids)
        path = dagx.dag_best_alignment(match.transpose(1, 2), s["links"], out_len, tgt_len)
        glance = dagx.dag_glat_glance(path, s["targets"], best_tokens, s["decoder_input"], tgt_len, 0.5, rand=s["rand"])
    _, match = dagx.dag_logsoftmax_gather_inplace(_Produced.apply(s["logits"]), ids)
    match = dagx.dag_force_alignment(match.transpose(1, 2), glance.next_force_emit)
    loss = dagx.dag_loss(match, s["links"], out_len, tgt_len)
    # a scale of B * 128 on the mean: what a loss scaler does to keep half-precision gradients away from zero
    total = -(loss / tgt_len).sum() * 128.0
    return (path, glance.glat_prev_output_tokens, total.detach()) + torch.autograd.grad(total, (s["logits"], s["links"]))


def _run_links(s):
    links = dagx.dag_multihead_links(_Produced.apply(s["scores"]), s["gates"], s["valid_end"], s["window"])
    return (links.detach(),) + torch.autograd.grad(links, (s["scores"], s["gates"]), s["grad"])


def _run_decode(s):
    best = dagx.dag_logsoftmax_max(s["logits"])
    if s["strategy"] in ("lookahead", "greedy"):
        got = dagx.dag_lookahead_decode(s["links"], best, s["out_len"], 1.0, s["strategy"] == "greedy", PAD)
    else:
        got = dagx.dag_viterbi_decode(s["links"], best, s["out_len"], 8.0, 1.0, s["strategy"] == "jointviterbi", PAD)
    # tokens come as wide as the longest output: padded here to one width; the scores are ones by definition
    tokens = torch.nn.functional.pad(got.output_tokens, (0, got.nodes.shape[1] - got.output_tokens.shape[1]), value=PAD)
    return (tokens, got.nodes) + ((got.pred_length,) if len(got) == 4 else ())


_RUN = {"loss": _run_loss, "align": lambda s: dagx.dag_best_alignment(s["match"], s["links"], s["out_len"], s["tgt_len"]),
        "gather": _run_gather, "criterion": _run_criterion, "links": _run_links, "decode": _run_decode}


def run(state):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without -------------------------------------------------------------------------------

def _mean_lengths(case):
    if case.get("ragged", False) and case["B"] > 1:
        return 0.875 * case["L"], max(2.0, 0.875 * case.get("T", 1))
    return float(case["L"]), float(case.get("T", 1))


def _pairs(L, W):
    """Transitions i < j <= i + W between L nodes."""
    W = min(W, L - 1)
    return W * (L - 1) - W * (W - 1) / 2


def work(case):
    B, L, size = case["B"], case["L"], 4 if case["dtype"] == "float32" else 2
    nodes, steps = _mean_lengths(case)
    kind = case["kind"]
    if kind in ("loss", "align"):
        pairs = B * _pairs(nodes, case["window"])
        inputs = B * nodes * steps * size + pairs * size
        if kind == "align":      # an addition and a maximum per pair and step
            return {"bytes": inputs + 8 * B * L, "flops": 2 * pairs * (steps - 1)}
        if not case["grad"]:     # one sweep
            return {"bytes": inputs + 4 * B, "flops": 2 * pairs * (steps - 1)}
        outputs = B * case["T"] * L * size + B * L * case["window"] * size
        return {"bytes": inputs + outputs + 4 * B, "flops": 3 * 2 * pairs * (steps - 1)}
    if kind == "gather":         # logits read once, their gradient written once
        logits, picked = B * L * case["V"], B * L * case["T"]
        return {"bytes": 2 * logits * size + 8 * B * case["T"] + 8 * picked, "flops": 6 * logits}
    if kind == "criterion":
        logits, pairs = B * L * case["V"], B * _pairs(nodes, L - 1)
        links = 4 * (pairs + B * L * (L - 1))
        return {"bytes": 3 * logits * size + links, "flops": 10 * logits + 4 * 2 * pairs * (steps - 1)}
    if kind == "links":
        H, pairs = case["H"], B * _pairs(nodes, case["window"])
        forward = pairs * H * size + B * L * case["window"] * size
        return {"bytes": forward + B * L * case["window"] * size + B * L * L * H * size + 8 * B * L * H, "flops": 16 * pairs * H}
    pairs = B * _pairs(nodes, L - 1)
    sweep = (2 * pairs * max(1, 2 * L // 8 - 1)) if case["strategy"].endswith("viterbi") else 2 * pairs
    return {"bytes": B * L * case["V"] * size + 4 * pairs + 8 * B * L, "flops": 3 * B * L * case["V"] + sweep}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------

def _square(links):
    """[B, L, L]: links[b, i, d] at (i, i + d + 1), -inf elsewhere."""
    B, L, W = links.shape
    d = torch.arange(L, device=links.device).view(1, L) - torch.arange(L, device=links.device).view(L, 1) - 1
    inside = (d >= 0) & (d < W)
    full = links.gather(2, d.clamp(0, W - 1).expand(B, L, L))
    return full.masked_fill_(~inside, NEG_INF)


def _exact_loss(case, s):
    match, edges = s["match"].detach().double(), _square(s["links"].detach().double())
    B, T, L = match.shape
    last, end = s["tgt_len"] - 1, s["out_len"] - 1
    rows = torch.arange(B, device=match.device)
    alpha = torch.full_like(match, NEG_INF)
    alpha[:, 0, 0] = match[:, 0, 0]
    for t in range(1, T):
        alpha[:, t] = torch.logsumexp(alpha[:, t - 1].unsqueeze(2) + edges, 1) + match[:, t]
    z = alpha[rows, last, end]
    if s["grad"] is None:
        return z
    scale = s["grad"].double().view(B, 1)
    grad_match, grad_edges = torch.zeros_like(match), torch.zeros_like(edges)
    stop = torch.where(torch.arange(L, device=match.device) == end.view(B, 1), 0.0, NEG_INF).double()
    beta = torch.full_like(stop, NEG_INF)       # log-probability of what follows node and step
    for t in reversed(range(T)):
        if t + 1 < T:
            ahead = edges + (match[:, t + 1] + beta).unsqueeze(1)
            share = (alpha[:, t] - z.view(B, 1)).unsqueeze(2) + ahead
            grad_edges += torch.exp(share) * scale.unsqueeze(2)
            beta = torch.logsumexp(ahead, 2)
        beta = torch.where((last == t).view(B, 1), stop, beta)
        grad_match[:, t] = torch.exp(alpha[:, t] + beta - z.view(B, 1)) * scale
    W = s["links"].shape[2]
    j = torch.arange(L, device=match.device).view(L, 1) + torch.arange(1, W + 1, device=match.device).view(1, W)
    grad_links = grad_edges.gather(2, j.clamp(max=L - 1).expand(B, L, W)).masked_fill_(j >= L, 0.0)
    return z, grad_match, grad_links


def _exact_gather(case, s):
    logits = s["logits"].detach().double()
    ids = s["targets"].unsqueeze(1).expand(-1, logits.shape[1], -1)
    lse = torch.logsumexp(logits, -1, keepdim=True)
    selected, grad = logits.gather(-1, ids) - lse, s["grad"].double()
    out = (logits - lse).exp_().mul_(-grad.sum(-1, keepdim=True))
    return selected, out.scatter_add_(-1, ids, grad)


def _exact_links(case, s):
    B, L, W = case["B"], case["L"], case["window"]
    i, j = torch.arange(L, device="cuda").view(L, 1), torch.arange(L, device="cuda").view(1, L)
    shifted = (i + torch.arange(1, W + 1, device="cuda").view(1, W))
    links, grad_scores, grad_gates = [], [], []
    for b in range(B):
        scores = s["scores"][b].detach().double().requires_grad_()
        gates = s["gates"][b].detach().double().requires_grad_()
        allowed = (j > i) & (j <= i + W) & (j < s["valid_end"][b].view(L, 1))
        some = allowed.any(1)
        logp = torch.log_softmax(scores.masked_fill(~allowed.unsqueeze(2), -1e30), 1) + gates.unsqueeze(1)
        mixed = torch.logsumexp(logp, 2)
        keep = (allowed & some.view(L, 1)).gather(1, shifted.clamp(max=L - 1)) & (shifted < L)
        mine = mixed.gather(1, shifted.clamp(max=L - 1))
        grads = torch.autograd.grad(mine, (scores, gates), s["grad"][b].double().masked_fill(~keep, 0.0))
        links.append(mine.detach().masked_fill(~keep, NEG_INF))
        grad_scores.append(grads[0])
        grad_gates.append(grads[1])
    return torch.stack(links), torch.stack(grad_scores), torch.stack(grad_gates)


def exact(case, seed):
    """What run() returns for these inputs in float64 by plain torch.  None where the outputs are whole numbers, and for
    the criterion, whose gradients hang on a path and on targets forced along it (its parts are cases of their own)."""
    made = {"loss": _exact_loss, "gather": _exact_gather, "links": _exact_links}.get(case["kind"])
    return None if made is None else made(case, prepare(case, seed))


def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("align", "decode"):
        return "exact"           # float32 scores in a stated order of operations: the same tokens and nodes
    if kind == "criterion":      # a path through float32 scores may turn at a near tie; gradients in the logits' type
        return {"rel": 1e-2 if dtype == "bfloat16" else 2e-3, "differ": 0.005}
    if dtype == "float32":
        # the loss and its posteriors are differences of sums of some hundred nats; the others plain 32-bit sums
        return {"rel": 1e-4 if kind == "loss" else 3e-5}
    if kind == "loss" and not case["grad"]:
        return {"rel": 1e-5}     # float32 whatever the inputs' type
    return {"rel": 1e-2 if dtype == "bfloat16" else 2e-3}
