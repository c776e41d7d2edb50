"""The work that users of this package have it do, as cases that can be timed and compared.

A case is one pass through the public entry points:

  step   a training step's share of the loss: ``TransducerLoss()`` forward, then the gradients of
         the summed costs with respect to both score arrays
  loss   the costs alone, as on a validation set
  align  the best alignment, ``criterion.viterbi``
  calls  the C++ interface's ``forward`` and ``backward`` on a log-normaliser that the caller has

Sizes: B utterances, T frames, U labels (so U + 1 rows of predictions), V symbols.  ``short`` is
the shortest utterance as a share of the longest, in frames and in labels (1.0: all at full
length).  Scores are normal with standard deviation ``sigma``, or uniform on [0, 1) for sigma 0.
"""
import math

import torch

from transducer_amd import TransducerLoss

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
DEVICE = "cuda"


def _case(name, op, B, T, U, V, dtype="f32", sigma=1.0, short=1.0):
    return dict(name=name, op=op, B=B, T=T, U=U, V=V, dtype=dtype, sigma=sigma, short=short)


def listed():
    return [
        # unit tests, toy tasks and the last, small batches of an epoch: launches and host work
        _case("step tiny", "step", 4, 50, 10, 32, short=0.5),
        # character models on long utterances: the lattice walks are the step
        _case("step characters", "step", 8, 2000, 100, 100),
        # word pieces, a spread-out batch, scores as peaked as a trained model's
        _case("step pieces", "step", 8, 2000, 100, 1000, sigma=2.0, short=0.5),
        # encoders that subsample in time, 16-bit projections, a vocabulary of no round size
        _case("step short odd f16", "step", 32, 400, 101, 4097, dtype="f16", sigma=2.0, short=0.5),
        # the benchmark's shape: large vocabulary, large batch
        _case("step words", "step", 32, 2000, 100, 10000, short=0.75),
        # the same as a model trained in bfloat16 calls it
        _case("step words bf16", "step", 32, 2000, 100, 10000, dtype="bf16", short=0.75),
        # whole recordings: long frame and label axes, small batch
        _case("step recordings", "step", 8, 10000, 400, 1000),
        # a validation pass over a batch of word pieces
        _case("loss pieces", "loss", 32, 2000, 100, 2000, sigma=0.0),
        # a C++ caller with its own log-normaliser, the reference's kernel benchmark
        _case("calls characters", "calls", 8, 10000, 400, 32),
        # one utterance aligned while somebody waits for it
        _case("align one", "align", 1, 500, 40, 1000, sigma=2.0),
        # alignment of a corpus, batch by batch
        _case("align words", "align", 32, 2000, 100, 10000, short=0.75),
        # the same for word pieces in 16 bits
        _case("align pieces bf16", "align", 16, 1500, 80, 2001, dtype="bf16", sigma=2.0, short=0.5),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["step", "step", "step", "loss", "align", "align", "calls"])
    while True:
        B = _log_uniform(rng, 1, 32)
        T = _log_uniform(rng, 50, 10000)
        U = _log_uniform(rng, 10, 400)
        # the C++ calls serve small vocabularies: their caller forms the normaliser densely
        V = _log_uniform(rng, 32, 1000 if op == "calls" else 10000)
        # labels do not outnumber frames, and no array or table is larger than the listed ones'
        if U <= T and B * T * V <= 640e6 and B * T * U <= 32e6 and B * T * U * V <= 5e10:
            break
    dtype = "f32" if op == "calls" else rng.choice(["f32", "f32", "bf16", "f16"])
    # uniform scores are a benchmark's: over thousands of frames of them fp32 alphas leave only the
    # first digit of the gradients (0.2 off those in fp64 at T=5000) and tie alignments, so only
    # the costs are compared on them
    sigma = rng.choice([0.0, 1.0, 2.0, 3.0] if op == "loss" else [1.0, 2.0, 3.0])
    case = _case("", op, B, T, U, V, dtype, sigma, rng.choice([0.5, 0.75, 1.0]))
    del case["name"]
    return case


def _lengths(n, longest, short, gen):
    low = max(1, int(math.ceil(longest * short)))
    out = torch.randint(low, longest + 1, (n,), generator=gen, device=DEVICE, dtype=torch.int32)
    return out


def _log_norms(emissions, predictions):
    """log sum_v exp(E[b,t,v] + P[b,u,v]), formed in fp64: what a caller of the C++ interface
    brings along."""
    out = []
    for e, p in zip(emissions.double(), predictions.double()):
        me, mp = e.max(1, keepdim=True)[0], p.max(1, keepdim=True)[0]
        sums = torch.matmul((e - me).exp(), (p - mp).exp().t().contiguous())
        out.append((sums.log() + me + mp.t()).float())
    return torch.stack(out)


def prepare(case, seed):
    B, T, U, V = case["B"], case["T"], case["U"], case["V"]
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def scores(rows):
        shape = (B, rows, V)
        if case["sigma"] == 0.0:
            x = torch.rand(shape, generator=gen, device=DEVICE)
        else:
            x = torch.randn(shape, generator=gen, device=DEVICE).mul_(case["sigma"])
        return x.to(DTYPES[case["dtype"]])

    state = dict(op=case["op"], emissions=scores(T), predictions=scores(U + 1))
    state["labels"] = torch.randint(1, V, (B, U), generator=gen, device=DEVICE, dtype=torch.int32)
    # the padded sizes are those of the longest utterance
    state["input_lengths"] = _lengths(B, T, case["short"], gen)
    state["label_lengths"] = _lengths(B, U, case["short"], gen)
    state["input_lengths"][0] = T
    state["label_lengths"][B - 1] = U
    state["criterion"] = TransducerLoss(allow_bf16=case["dtype"] == "bf16",
                                        allow_fp16=case["dtype"] == "f16")
    if case["op"] == "step":
        state["emissions"].requires_grad_()
        state["predictions"].requires_grad_()
    elif case["op"] == "align":
        # entries past an utterance's labels come back unwritten: what the caller blanks out
        state["padding"] = (torch.arange(U, device=DEVICE)[None, :] >=
                            state["label_lengths"][:, None])
    elif case["op"] == "calls":
        shape = (B, T, U + 1)
        state.update(costs=torch.zeros(B, device=DEVICE), alphas=torch.zeros(shape, device=DEVICE),
                     lngrads=torch.zeros(shape, device=DEVICE),
                     egrads=torch.zeros_like(state["emissions"]),
                     pgrads=torch.zeros_like(state["predictions"]),
                     log_norms=_log_norms(state["emissions"], state["predictions"]))
        state["sizes"] = (B, T, U + 1, V)
    return state


def run(state):
    scores = state["emissions"], state["predictions"]
    lengths = state["input_lengths"], state["label_lengths"]
    if state["op"] == "step":
        costs = state["criterion"](*scores, state["labels"], *lengths)
        egrads, pgrads = torch.autograd.grad(costs.sum(), scores)
        return {"costs": costs.detach(), "egrads": egrads, "pgrads": pgrads}
    if state["op"] == "loss":
        with torch.no_grad():
            return state["criterion"](*scores, state["labels"], *lengths)
    if state["op"] == "align":
        paths = state["criterion"].viterbi(*scores, *lengths)
        return paths.masked_fill_(state["padding"], -1)
    from transducer_amd import _transducer
    ptr = {k: v.data_ptr() for k, v in state.items() if isinstance(v, torch.Tensor)}
    _transducer.forward(ptr["emissions"], ptr["predictions"], ptr["costs"], ptr["alphas"],
                        ptr["log_norms"], ptr["labels"], ptr["input_lengths"],
                        ptr["label_lengths"], *state["sizes"], 0, True)
    _transducer.backward(ptr["emissions"], ptr["predictions"], ptr["egrads"], ptr["pgrads"],
                         ptr["lngrads"], ptr["alphas"], ptr["log_norms"], ptr["labels"],
                         ptr["input_lengths"], ptr["label_lengths"], *state["sizes"], 0, True)
    return {k: state[k] for k in ("costs", "alphas", "egrads", "pgrads", "lngrads")}


def work(case):
    """One pass on utterances of mean length: scores and labels in, results out, and two
    operations per cell and symbol for each contraction (normaliser, two gradients) or for the
    search of the best label.  Gradients are written at their padded size."""
    B, T, U, V = case["B"], case["T"], case["U"], case["V"]
    share = 1.0 if B == 1 else (1.0 + case["short"]) / 2
    frames, rows = share * T, share * U + 1
    cells = B * frames * rows
    size = 4 if case["dtype"] == "f32" else 2
    scores = size * B * (frames + rows) * V
    padded = size * B * (T + U + 1) * V
    ints = 4 * B * (U + 2)
    if case["op"] == "step":
        return {"bytes": scores + padded + ints + 4 * B, "flops": 6.0 * V * cells}
    if case["op"] == "loss":
        return {"bytes": scores + ints + 4 * B, "flops": 2.0 * V * cells}
    if case["op"] == "align":
        return {"bytes": scores + ints, "flops": 4.0 * V * cells}
    # of the scores only the blank and the label entry of each frame and row are needed; the
    # normaliser comes in twice, the alphas go out and come in, the gradients go out
    return {"bytes": 4.0 * (4 * cells + B * T * (U + 1)) + 4.0 * (2 * cells + 3 * B * (T + U)) +
            padded, "flops": 60.0 * cells}


def tolerance(case):
    """About four times the distance of the results from those of the same path in fp64, measured
    on the listed cases and eighty drawn ones.  What holds it: an fp32 alpha is a running sum over
    every frame before it, and the gradients are exponentials of differences of alphas.  That
    error grows with the number of steps, up to 2e-6 a step (T=500, U=200: 1.1e-3; T=10000,
    U=400: 1.9e-2), and the costs' own with it (5e-5 at T=5000).  16-bit gradients are rounded
    once more.  Labels of an alignment were the fp64 path's, every one, for normal scores; the
    three-call interface returns the same bits for the same normaliser."""
    steps = case["T"] + case["U"]
    if case["op"] == "step":
        unit = {"f32": 0.0, "f16": 2.5e-4, "bf16": 2e-3}[case["dtype"]]
        return {"rel": 4 * (1e-5 + unit + 1.5e-6 * steps)}
    if case["op"] == "loss":
        return {"rel": 4 * (1e-6 + 8e-9 * steps)}
    return "exact"
