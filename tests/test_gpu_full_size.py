"""The benchmark configurations at their full sizes (B=8/32, T=2000, U=100, V up to 10000).

The CPU oracle needs minutes for the largest one, so there the device result is held to
properties that do not depend on size -- rows of a gradient sum to zero, padding stays exactly
zero, the upstream factor is linear, an utterance's result does not depend on what else is in
the batch (bit for bit) -- and to the oracle on ONE utterance cut out of the batch.  The smaller
configurations go through the oracle whole."""
import numpy as np
import pytest

from util import (RTOL, ATOL, DeviceCase, assert_close, dev, gpu_backward, gpu_forward,
                  gpu_log_norms, gpu_loss, gpu_viterbi, ptr, violations)

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import oracle  # noqa: E402
from transducer_amd import capi  # noqa: E402
from transducer_amd.synthetic import CONFIGS, lengths, make_inputs  # noqa: E402


def unpack(d):
    return tuple(d[k] for k in ("emissions", "predictions", "labels", "input_lengths",
                                "label_lengths"))


class DeviceBatch(object):
    """Inputs of one configuration drawn on the device (torch's generator: these tests check
    properties and cut-outs, not fixtures, so the host generator's minutes are not needed)."""

    def __init__(self, cfg, seed, near_ties=False):
        g = torch.Generator(device="cuda:0")
        g.manual_seed(seed)
        self.B, self.T, self.U, self.V = cfg.B, cfg.T, cfg.U + 1, cfg.V
        self.E = torch.randn((cfg.B, cfg.T, cfg.V), generator=g, device="cuda:0") * cfg.sigma
        self.P = torch.randn((cfg.B, cfg.U + 1, cfg.V), generator=g, device="cuda:0") * cfg.sigma
        self.labels = torch.randint(1, cfg.V, (cfg.B, cfg.U), generator=g, device="cuda:0",
                                    dtype=torch.int32)
        il, ll = lengths(cfg, np.random.Generator(np.random.Philox(key=seed)))
        self.il_h, self.ll_h = il, ll
        self.il, self.ll = dev(il), dev(ll)
        if near_ties:  # a tenth of the entries of every frame repeat another column's value
            k = cfg.V // 10
            for b in range(cfg.B):
                dst = torch.randint(1, cfg.V, (cfg.T, k), generator=g, device="cuda:0")
                src = torch.randint(1, cfg.V, (cfg.T, k), generator=g, device="cuda:0")
                self.E[b].scatter_(1, dst, self.E[b].gather(1, src))

    @property
    def dims(self):
        return (self.B, self.T, self.U, self.V)

    def cut(self, b):
        """Utterance b as a batch of one with the same padded sizes."""
        c = DeviceBatch.__new__(DeviceBatch)
        c.B, c.T, c.U, c.V = 1, self.T, self.U, self.V
        c.E, c.P = self.E[b:b + 1].contiguous(), self.P[b:b + 1].contiguous()
        c.labels = self.labels[b:b + 1].contiguous()
        c.il_h, c.ll_h = self.il_h[b:b + 1].copy(), self.ll_h[b:b + 1].copy()
        c.il, c.ll = dev(c.il_h), dev(c.ll_h)
        return c

    def host(self):
        return (self.E.cpu().numpy(), self.P.cpu().numpy(), self.labels.cpu().numpy(),
                self.il_h, self.ll_h)


def loss_on_device(c, deltas=None, blank=0):
    """Whole loss through the C interface; results stay on the device."""
    B, T, U, V = c.dims
    nbytes = capi.load().rnnt_hip_loss_workspace_bytes(B, T, U, V)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda:0")
    costs = torch.full((B,), float("nan"), device="cuda:0")
    eg = torch.full_like(c.E, float("nan"))
    pg = torch.full_like(c.P, float("nan"))
    capi.call("rnnt_hip_loss_forward", ptr(c.E), ptr(c.P), ptr(c.labels), ptr(c.il), ptr(c.ll),
              ptr(costs), ptr(ws), nbytes, B, T, U, V, blank, None)
    capi.call("rnnt_hip_loss_backward", ptr(c.E), ptr(c.P), ptr(c.labels), ptr(c.il), ptr(c.ll),
              ptr(deltas), ptr(eg), ptr(pg), ptr(ws), nbytes, B, T, U, V, blank, None)
    torch.cuda.synchronize()
    return costs, eg, pg


def log_norms_on_device(c):
    B, T, U, V = c.dims
    LN = torch.full((B, T, U), float("nan"), device="cuda:0")
    capi.call("rnnt_hip_log_norms", ptr(c.E), ptr(c.P), ptr(LN), ptr(c.il), ptr(c.ll),
              B, T, U, V, None)
    return LN


def viterbi_on_device(c, LN, blank=0):
    B, T, U, V = c.dims
    out = torch.full((B, U - 1), -1, dtype=torch.int32, device="cuda:0")
    capi.call("rnnt_hip_viterbi", ptr(c.E), ptr(c.P), ptr(LN), ptr(out), ptr(c.il), ptr(c.ll),
              B, T, U, V, blank, None)
    torch.cuda.synchronize()
    return out


def decode_on_device(c, blank=0):
    """The fused best-path entry (log-normaliser + best path, what criterion.viterbi calls)."""
    B, T, U, V = c.dims
    out = torch.full((B, U - 1), -1, dtype=torch.int32, device="cuda:0")
    capi.call("rnnt_hip_viterbi_decode", ptr(c.E), ptr(c.P), ptr(c.il), ptr(c.ll), ptr(out),
              B, T, U, V, blank, None)
    torch.cuda.synchronize()
    return out


def ulp_error(got, truth, il, ll):
    """Largest |got - truth| over the cells inside the utterances, in units of the fp32 spacing
    at the true value (0.5 = correctly rounded)."""
    worst = 0.0
    for b in range(got.shape[0]):
        t = truth[b, :il[b], :ll[b] + 1]
        g = got[b, :il[b], :ll[b] + 1].astype(np.float64)
        if t.size:
            ulp = np.spacing(np.abs(t).astype(np.float32)).astype(np.float64)
            worst = max(worst, float((np.abs(g - t) / ulp).max()))
    return worst


def oracle_on_log_norms(E, P, labels, il, ll, LN):
    """The oracle's lattice recursions and dense gradient accumulation (transducer_cpu.cpp,
    test.h:82-113) on a log-normaliser supplied from outside."""
    costs, alphas = oracle.forward(E, P, LN, labels, il, ll)
    eg, pg, lng = oracle.backward(E, P, np.nan_to_num(alphas), LN, labels, il, ll)
    eg, pg = oracle.accumulate_grads(E, P, eg, pg, lng, LN, il, ll)
    return costs, eg, pg


# The device's log-normaliser against the fp64 value, in fp32 spacings of LN at the worst cell of
# a configuration.  Measured: 2.2 at V=100 (where LN lies in [4,8) and a spacing is 4.8e-7; the
# reference's own sequential fp32 sum, test.h:51-80, is 2.3 off there), 1.3-1.5 at V=10000.
# 0.5 would be correct rounding; the reference's gradients leave the tolerance from about 4 on.
LN_ULP_BAR = 2.5

# ------------------------------------------------------------------ headline configuration
# fraction of gradient entries of the cut-out utterance outside rel 1e-4 / abs 1e-5 end to end
# (each side with its own log-normaliser): (egrads, pgrads)
# measured: 0.0001 % / 0 at V=10000, 0 / 0 at V=10001
CUT_OUT_BAR = (2e-4, 2e-4)


@pytest.mark.parametrize("V", [10000, 10001])
def test_headline_configuration_properties_and_one_utterance_against_the_oracle(V):
    """V = 10001: the same at a vocabulary whose rows do not start on 16-byte boundaries (every
    row of the [B,T,V] arrays then comes in through the loads at the element's own alignment)."""
    c = DeviceBatch(CONFIGS["cfg4"]._replace(V=V), seed=3)
    B, T, U, V = c.dims
    costs, eg, pg = loss_on_device(c)
    assert torch.isfinite(costs).all() and (costs > 0).all()
    assert torch.isfinite(eg).all() and torch.isfinite(pg).all()

    # padding: frames past an utterance and label positions past it hold exact zeros
    tmask = torch.arange(T, device="cuda:0")[None, :] >= c.il[:, None]
    umask = torch.arange(U, device="cuda:0")[None, :] > c.ll[:, None]
    assert not eg[tmask].any() and not pg[umask].any()

    # every row of a gradient sums to zero: sum_v softmax = 1 and the occupancy of a node equals
    # the sum of its two outgoing moves
    # (relative to the row's size: with T >> U nearly all of an utterance's waiting happens at
    # one label position, whose blank entry reaches ~ -T_b as a sequential fp32 sum)
    se = eg.double().sum(-1).abs()
    sp = pg.double().sum(-1).abs()
    ae = eg.double().abs().sum(-1)
    ap = pg.double().abs().sum(-1)
    assert float(ae[~tmask].min()) > 1e-3  # the rows are not trivially zero
    print("largest |row sum| / sum |row|: egrads %.3g, pgrads %.3g"
          % (float((se / (ae + 1e-30)).max()), float((sp / (ap + 1e-30)).max())))
    assert bool((se <= 1e-5 + 2e-5 * ae).all())
    assert bool((sp <= 1e-5 + 2e-5 * ap).all())

    # the upstream factor: exact doubling
    two = torch.full((B,), 2.0, device="cuda:0")
    costs2, eg2, pg2 = loss_on_device(c, deltas=two)
    assert torch.equal(costs2, costs)
    assert torch.equal(eg2, 2.0 * eg) and torch.equal(pg2, 2.0 * pg)
    del eg2, pg2

    # an utterance alone gives the same bits as inside the batch
    shortest = int(np.argmin(c.il_h.astype(np.int64) * (c.ll_h + 1)))
    for b in (0, shortest):
        one = c.cut(b)
        c1, e1, p1 = loss_on_device(one)
        assert torch.equal(c1[0], costs[b])
        assert torch.equal(e1[0], eg[b]) and torch.equal(p1[0], pg[b])

    # the shortest utterance against the oracle (18 s of one host core)
    one = c.cut(shortest)
    E, P, labels, il, ll = one.host()
    want = oracle.loss_and_grads(E, P, labels, il, ll)
    assert_close(costs[shortest:shortest + 1].cpu().numpy(), want["costs"], what="costs")
    ve, worst_e = violations(eg[shortest].cpu().numpy(), want["egrads"][0])
    vp, worst_p = violations(pg[shortest].cpu().numpy(), want["pgrads"][0])
    print("cfg4 utterance %d (T=%d, U=%d): violations egrads %.4f%%, pgrads %.4f%%; max abs err "
          "%.3g / %.3g" % (shortest, il[0], ll[0], 100 * ve, 100 * vp, worst_e, worst_p))
    # the reference's own fp32 gradients move by more than the tolerance when LN moves in its
    # last bit at this lattice length (both sides round LN, differently); the bar end to end is
    # about three times the fraction measured
    assert ve <= CUT_OUT_BAR[0] and vp <= CUT_OUT_BAR[1]
    # ... and with the SAME log-normaliser on both sides nothing is outside the tolerance: the
    # oracle's recursions and gradient sums, fed the device's LN, against the device's result
    LN = log_norms_on_device(one).cpu().numpy()
    worst = ulp_error(LN, oracle.log_norms_truth(E, P, il, ll), il, ll)
    print("device LN against fp64: %.2f ulp at worst" % worst)
    assert worst <= LN_ULP_BAR
    oc, oe, op = oracle_on_log_norms(E, P, labels, il, ll, LN)
    assert_close(costs[shortest:shortest + 1].cpu().numpy(), oc, what="costs, shared LN")
    assert_close(eg[shortest].cpu().numpy(), oe[0], what="egrads, shared LN")
    assert_close(pg[shortest].cpu().numpy(), op[0], what="pgrads, shared LN")
    # the same for the longest utterance (the whole batch is held to this bar by bench.py, which
    # has the CPU result of every utterance at hand)
    longest = int(np.argmax(c.il_h.astype(np.int64) * (c.ll_h + 1)))
    one = c.cut(longest)
    E, P, labels, il, ll = one.host()
    LN = log_norms_on_device(one).cpu().numpy()
    oc, oe, op = oracle_on_log_norms(E, P, labels, il, ll, LN)
    assert_close(costs[longest:longest + 1].cpu().numpy(), oc, what="costs, shared LN (longest)")
    assert_close(eg[longest].cpu().numpy(), oe[0], what="egrads, shared LN (longest)")
    assert_close(pg[longest].cpu().numpy(), op[0], what="pgrads, shared LN (longest)")


@pytest.mark.parametrize("near_ties,V", [(False, 10000), (True, 10000), (True, 10001)])
def test_headline_viterbi_one_utterance_bit_exact_and_batch_independent(near_ties, V):
    c = DeviceBatch(CONFIGS["cfg5"]._replace(V=V), seed=5, near_ties=near_ties)
    LN = log_norms_on_device(c)
    paths = viterbi_on_device(c, LN)
    U = c.U
    written = torch.arange(U - 1, device="cuda:0")[None, :] < c.ll[:, None]
    assert ((paths >= 1) & (paths < c.V))[written].all()
    assert (paths[~written] == -1).all()  # only the first label_lengths[b] entries are written
    shortest = int(np.argmin(c.il_h.astype(np.int64) * (c.ll_h + 1)))
    one = c.cut(shortest)
    LN1 = LN[shortest:shortest + 1].contiguous()
    alone = viterbi_on_device(one, LN1)
    assert torch.equal(alone[0], paths[shortest])
    E, P, _, il, ll = one.host()
    want = oracle.viterbi(E, P, LN1.cpu().numpy(), il, ll)
    assert np.array_equal(alone.cpu().numpy()[:, :ll[0]], want[:, :ll[0]])

    # The fused entry (criterion.viterbi's: torch_binding.py:130-177) takes another route to the
    # same lattice -- LN and the blank scores go straight into the skewed planes, no row-major
    # LN, no gather -- and must give the same labels for the whole batch, leave the padding
    # alone, and not depend on the batch around an utterance.
    fused = decode_on_device(c)
    assert torch.equal(fused, paths)
    assert torch.equal(decode_on_device(one)[0], fused[shortest])
    longest = int(np.argmax(c.il_h.astype(np.int64) * (c.ll_h + 1)))
    assert torch.equal(decode_on_device(c.cut(longest))[0], fused[longest])


@pytest.mark.parametrize("near_ties,V,dist", [(False, 10000, "normal"), (True, 10000, "normal"),
                                              (False, 10001, "normal"), (False, 10000, "uniform"),
                                              (False, 12000, "bf16")])
def test_headline_table_of_best_labels_is_the_same_however_it_is_built(near_ties, V, dist):
    # every cell of the whole batch: over every column (mode 1), from candidate lists with the
    # sampled go/no-go (default) and from lists unconditionally (mode 2) -- same maxima, same
    # lowest indices.  Uniform scores make the default turn back after its sample; scores
    # rounded to bfloat16 tie in many cells.
    c = DeviceBatch(CONFIGS["cfg5"]._replace(V=V), seed=6, near_ties=near_ties)
    if dist == "uniform":
        c.E.uniform_(0.0, 1.0)
        c.P.uniform_(0.0, 1.0)
    elif dist == "bf16":
        c.E = c.E.to(torch.bfloat16).float()
        c.P = c.P.to(torch.bfloat16).float()
    B, T, U, V = c.dims
    tables = []
    for mode in (1, 0, 2):
        best = torch.full((B, T, U), float("nan"), device="cuda:0")
        arg = torch.full((B, T, U), -7, dtype=torch.int32, device="cuda:0")
        capi.call("rnnt_hip_set_maxplus_mode", mode)
        try:
            capi.call("rnnt_hip_maxplus_table", ptr(c.E), ptr(c.P), ptr(c.il), ptr(c.ll), ptr(best),
                      ptr(arg), B, T, U, V, 0, None)
            torch.cuda.synchronize()
        finally:
            capi.call("rnnt_hip_set_maxplus_mode", 0)
        tables.append((best, arg))
    for best, arg in tables[1:]:
        assert torch.equal(arg, tables[0][1])
        assert torch.equal(best.view(torch.int32), tables[0][0].view(torch.int32))
    # and the all-columns table itself on one frame of one utterance, against numpy
    b, t = 3, 777
    s = (c.E[b, t][None, :] + c.P[b]).cpu().numpy()
    s[:, 0] = -np.inf
    ub = int(c.ll_h[b]) + 1
    assert np.array_equal(tables[0][1][b, t, :ub].cpu().numpy(), s.argmax(axis=1)[:ub])
    assert np.array_equal(tables[0][0][b, t, :ub].cpu().numpy(), s.max(axis=1)[:ub])


def test_table_when_the_sample_passes_and_the_rest_of_the_batch_does_not_suit_lists():
    # The dearest case of the default mode: the two sampled utterances (0 and B/2) have normal
    # scores, so the call goes on with lists, but every other utterance's scores are quantised
    # (five levels: ties everywhere, empty lists, every cell fails its exactness test).  Their
    # tiles are then redone over every column; the list pass gives a tile up once it holds more
    # flagged cells than are redone one by one, a frame or two into each workgroup's eight.
    # Same table as over every column, and at most 1.5 times its time (measured: 1.33; 1.46
    # when the list pass ran over all frames for nothing).
    c = DeviceBatch(CONFIGS["cfg5"], seed=8)
    B, T, U, V = c.dims
    for b in range(B):
        if b not in (0, B // 2):
            c.E[b] = torch.randint(0, 5, (T, V), device="cuda:0").float() * 0.5
            c.P[b] = torch.randint(0, 5, (U, V), device="cuda:0").float() * 0.25
    assert capi.load().rnnt_hip_maxplus_tries_lists(B, T, U, V) == 1
    best = torch.empty((B, T, U), device="cuda:0")
    arg = torch.empty((B, T, U), dtype=torch.int32, device="cuda:0")

    def build(mode, repeats):
        capi.call("rnnt_hip_set_maxplus_mode", mode)
        try:
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ms = []
            for _ in range(repeats):
                best.fill_(float("nan"))
                arg.fill_(-7)
                start.record()
                capi.call("rnnt_hip_maxplus_table", ptr(c.E), ptr(c.P), ptr(c.il), ptr(c.ll),
                          ptr(best), ptr(arg), B, T, U, V, 0, None)
                stop.record()
                torch.cuda.synchronize()
                ms.append(start.elapsed_time(stop))
        finally:
            capi.call("rnnt_hip_set_maxplus_mode", 0)
        return min(ms[1:]), best.clone(), arg.clone()

    every_ms, every_best, every_arg = build(1, 4)
    lists_ms, lists_best, lists_arg = build(0, 4)
    print("table, sample passes but 30 of 32 utterances are quantised: %.2f ms by default, "
          "%.2f ms over every column" % (lists_ms, every_ms))
    assert torch.equal(lists_arg, every_arg)
    assert torch.equal(lists_best.view(torch.int32), every_best.view(torch.int32))
    assert lists_ms <= 1.5 * every_ms


# ------------------------------------------------------------------ the smaller configurations, whole
# Fraction of gradient entries outside rel 1e-4 / abs 1e-5 end to end, each side with its own
# log-normaliser: about three times what was measured, per configuration (egrads, pgrads).
# Measured: cfg2 0.0005 % / 0 (the reference's own spread between two orders of its LN sum: 0 / 0),
# cfg3a 0.038 % / 0.197 % (spread 0.035 % / 0.181 %), cfg3b 0 / 0 (spread 0.030 % / 0.156 %).
# The test takes the larger of this and twice the spread measured on the same inputs.
END_TO_END_BAR = {"cfg2": (2e-5, 2e-5), "cfg3a": (1.2e-3, 6e-3), "cfg3b": (1e-4, 1e-4)}


@pytest.mark.parametrize("name", ["cfg2", "cfg3a", "cfg3b"])
def test_configuration_whole_against_the_oracle(name):
    E, P, labels, il, ll = unpack(make_inputs(CONFIGS[name], seed=0))
    a = oracle.loss_and_grads(E, P, labels, il, ll, lse="naive")
    # How far the reference's own fp32 result moves when only the summation order of ITS
    # normaliser changes: the separable form of torch_binding.py:35-40 with the inner sum in
    # index order against the same with eight partial sums (the reference leaves that order to
    # torch.bmm).  Index order against test.h's sequential sum says little: the two accumulate
    # in the same order and round alike.
    b = oracle.loss_and_grads(E, P, labels, il, ll, lse="sep")
    b8 = oracle.loss_and_grads(E, P, labels, il, ll, lse="sep8")
    floor_e = max(violations(b["egrads"], a["egrads"])[0], violations(b8["egrads"], b["egrads"])[0])
    floor_p = max(violations(b["pgrads"], a["pgrads"])[0], violations(b8["pgrads"], b["pgrads"])[0])
    costs, eg, pg = gpu_loss(DeviceCase(E, P, labels, il, ll))
    assert_close(costs, a["costs"], rtol=RTOL, atol=max(ATOL, 1e-3), what="costs")
    ve, worst_e = violations(eg, a["egrads"])
    vp, worst_p = violations(pg, a["pgrads"])
    print("%s: violations egrads %.4f%% (the reference's own spread between LN orders %.4f%%), "
          "pgrads %.4f%% (spread %.4f%%); max abs err %.3g / %.3g"
          % (name, 100 * ve, 100 * floor_e, 100 * vp, 100 * floor_p, worst_e, worst_p))
    bar_e, bar_p = END_TO_END_BAR[name]
    assert ve <= max(2 * floor_e, bar_e) and vp <= max(2 * floor_p, bar_p)
    # nothing is far off: the reference's own CPU-against-GPU bar (test_cuda.cu:371-373)
    assert violations(eg, a["egrads"], rtol=1e-3, atol=1e-4)[0] <= bar_e / 10
    for i in range(E.shape[0]):
        assert not eg[i, il[i]:].any() and not pg[i, ll[i] + 1:].any()

    # The same with ONE log-normaliser on both sides (the device's, also held against fp64 in
    # units of its own spacing): the oracle's recursions and gradient sums then agree with the
    # device in every entry, which is what says the fraction above comes from the last bit of LN
    # and from nothing else.
    c = DeviceCase(E, P, labels, il, ll)
    LN = gpu_log_norms(c)
    worst = ulp_error(LN, oracle.log_norms_truth(E, P, il, ll), il, ll)
    ref_worst = ulp_error(a["log_norms"], oracle.log_norms_truth(E, P, il, ll), il, ll)
    print("%s: LN against fp64, worst cell: device %.2f ulp, the reference's own fp32 sum %.2f ulp"
          % (name, worst, ref_worst))
    assert worst <= LN_ULP_BAR
    oc, oe, op = oracle_on_log_norms(E, P, labels, il, ll, LN)
    assert_close(costs, oc, what="costs, shared LN")
    assert_close(eg, oe, what="egrads, shared LN")
    assert_close(pg, op, what="pgrads, shared LN")


# ------------------------------------------------------------------ the reference's long shape
def test_long_sequence_shape_of_the_reference_kernel_benchmark():
    """B=8, T=10000, U=400 (transducer/benchmark_cuda.cu:153-158), ragged here and with a
    vocabulary that keeps the oracle to seconds: the label axis takes four slices of the
    egrads contraction and four blocks of 128 rows of the pgrads one, a lane of the lattice
    walks owns eight label positions, and the best path keeps its decision table in global
    memory.  Whole batch against the oracle on the device's log_norms, best path exact."""
    from transducer_amd.synthetic import Config
    cfg = Config("long", 8, 10000, 400, 300, 1.0, (7000, 10000), (300, 400))
    E, P, labels, il, ll = unpack(make_inputs(cfg, seed=2))
    c = DeviceCase(E, P, labels, il, ll)
    costs, eg, pg = gpu_loss(c)
    assert np.isfinite(costs).all() and (costs > 0).all()
    for i in range(cfg.B):
        assert not eg[i, il[i]:].any() and not pg[i, ll[i] + 1:].any()
    LN = gpu_log_norms(c)
    truth = oracle.log_norms_truth(E, P, il, ll)
    worst = ulp_error(LN, truth, il, ll)
    ref_worst = ulp_error(oracle.log_norms_naive(E, P, il, ll), truth, il, ll)
    print("long: LN against fp64, worst of %d cells: device %.2f ulp, the reference's own fp32 "
          "sum %.2f ulp" % (int(np.sum(il * (ll + 1))), worst, ref_worst))
    # (28 million cells with LN in [4, 8), where a spacing is 4.8e-7: the worst cell of so many
    # lies further out than at the benchmark shapes -- measured 3.35 for the device and 3.36
    # for the reference's sequential fp32 sum, test.h:51-80 -- so the bar here is the
    # reference's own worst cell on the same inputs)
    assert worst <= max(LN_ULP_BAR, 1.05 * ref_worst)
    oc, oe, op = oracle_on_log_norms(E, P, labels, il, ll, LN)
    assert_close(costs, oc, what="costs, shared LN")
    for got, ref, name in ((eg, oe, "egrads"), (pg, op, "pgrads")):
        frac, worst = violations(got, ref)
        print("long: %s, shared LN: %.5f%% outside, max abs err %.3g" % (name, 100 * frac, worst))
        # (four slices on the device against one sequential fp32 sum over 401 label positions in
        # the oracle: entries that are small differences of large terms may land just outside)
        assert frac <= 1e-4
        assert violations(got, ref, rtol=1e-3, atol=1e-4)[0] == 0.0
    from util import gpu_viterbi
    assert np.array_equal(gpu_viterbi(c, LN), oracle.viterbi(E, P, LN, il, ll))


# ------------------------------------------------------------------ more than 2^31 score elements
def test_arrays_past_two_to_the_31_elements_index_like_small_ones():
    """B*T*V = 2.3e9 elements (9.2 GB of emissions): element offsets no longer fit 32 bits.  The
    last utterances lie wholly past that point, and an utterance's result does not depend on the
    batch around it, so each must come out with the bits it has as a batch of one (whose offsets
    are small); the size-free properties hold over the whole batch."""
    from transducer_amd.synthetic import small_config
    cfg = small_config(24, 2000, 30, 48000, ragged=True)
    c = DeviceBatch(cfg, seed=11)
    B, T, U, V = c.dims
    assert B * T * V > 2 ** 31 and (B - 1) * T * V > 2 ** 31
    costs, eg, pg = loss_on_device(c)
    assert torch.isfinite(costs).all() and (costs > 0).all()
    tmask = torch.arange(T, device="cuda:0")[None, :] >= c.il[:, None]
    umask = torch.arange(U, device="cuda:0")[None, :] > c.ll[:, None]
    assert not eg[tmask].any() and not pg[umask].any()
    se = eg.sum(-1, dtype=torch.float64).abs()
    ae = eg.abs().sum(-1, dtype=torch.float64)
    assert torch.isfinite(se).all()
    assert float(ae[~tmask].min()) > 1e-3
    assert bool((se <= 1e-5 + 2e-5 * ae).all())
    for b in (0, B - 2, B - 1):
        one = c.cut(b)
        c1, e1, p1 = loss_on_device(one)
        assert torch.equal(c1[0], costs[b]), b
        assert torch.equal(e1[0], eg[b]) and torch.equal(p1[0], pg[b]), b
    del eg, pg

    LN = log_norms_on_device(c)
    paths = viterbi_on_device(c, LN)
    for b in (0, B - 1):
        one = c.cut(b)
        alone = viterbi_on_device(one, LN[b:b + 1].contiguous())
        n = int(c.ll_h[b])
        assert torch.equal(alone[0, :n], paths[b, :n]), b


@pytest.mark.parametrize("T,U", [(16777300, 2), (1060000, 130), (530000, 300)])
def test_planes_that_take_more_than_one_window_carry_the_reference_bits(T, U):
    """The walks address an utterance's planes through windows of a GiB.  Two label positions (64 are the
    least a plane holds) and 16.8 million frames: past 2^32 bytes a plane, five windows on one
    wavefront; 130 positions: two windows, four wavefronts and blocks of two; 300: blocks side by side
    in all three walks."""
    V = 2
    rng = np.random.default_rng(T)
    E = rng.standard_normal((1, T, V), dtype=np.float32)
    P = rng.standard_normal((1, U, V), dtype=np.float32)
    LN = np.empty((1, T, U), np.float32)
    for t in range(0, T, 1 << 17):
        s = E[:, t:t + (1 << 17), None] + P[:, None]
        LN[:, t:t + (1 << 17)] = np.logaddexp(s[..., 0], s[..., 1])
    labels = np.ones((1, U - 1), np.int32)
    il, ll = np.array([T], np.int32), np.array([U - 1], np.int32)
    c = DeviceCase(E, P, labels, il, ll)
    costs, alphas = gpu_forward(c, LN)
    want_costs, want = oracle.forward(E, P, LN, labels, il, ll)
    assert np.array_equal(costs, want_costs) and np.array_equal(alphas, want)
    del alphas
    assert np.array_equal(gpu_viterbi(c, LN), oracle.viterbi(E, P, LN, il, ll))
    got = gpu_backward(c, want, LN)
    for g, w in zip(got, oracle.backward(E, P, want, LN, labels, il, ll)):
        assert np.array_equal(g, w)
