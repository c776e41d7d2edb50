"""The alpha walk runs all but the first and last groups of anti-diagonals without looking at any
bounds.  Where those interior groups begin and end (and whether there are any) depends on the
frames and labels of each utterance and on how the label positions are dealt to wavefronts; the
alphas and costs must carry the oracle's bits in every case."""
import numpy as np
import pytest

import oracle
from util import DeviceCase, assert_same_bits, gpu_backward, gpu_forward, gpu_viterbi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("U", [2, 3, 64, 65, 128, 129, 257, 300])
@pytest.mark.parametrize("T", [31, 66, 97, 164])
def test_alphas_where_the_interior_begins_and_ends(T, U):
    V, il = 6, [T, T, T - 1, T - 2, T - 3, max(T // 2, 1), 17, 1]
    ll = [U - 1, U // 2, max(U - 2, 0), 1, 0, min(63, U - 1), min(64, U - 1), U - 1]
    B = len(il)
    rng = np.random.default_rng(1000 * T + U)
    E = rng.standard_normal((B, T, V), dtype=np.float32)
    P = rng.standard_normal((B, U, V), dtype=np.float32)
    P[1, :, 0] = -np.inf          # no blank anywhere: no path, through interior groups too
    E[2, T // 2, 1:] = -np.inf    # one frame that emits nothing
    labels = rng.integers(1, V, (B, U - 1)).astype(np.int32)
    il, ll = np.array(il, np.int32), np.array(ll, np.int32)
    LN = oracle.log_norms_naive(E, P, il, ll)
    want_costs, want = oracle.forward(E, P, LN, labels, il, ll)
    costs, alphas = gpu_forward(DeviceCase(E, P, labels, il, ll), np.nan_to_num(LN))
    for b in range(B):
        got, ref = alphas[b, :il[b], :ll[b] + 1], want[b, :il[b], :ll[b] + 1]
        assert_same_bits(got, ref, "alphas of utterance %d" % b)
    assert_same_bits(costs, want_costs, "costs")


@pytest.mark.parametrize("U", [65, 128, 193, 256, 520])
@pytest.mark.parametrize("T", [191, 253, 256, 517])
def test_alphas_where_the_hand_over_between_wavefronts_wraps(T, U):
    """What crosses from one wavefront to the next goes through rings of 256 steps: lattices of
    about that many steps and of several times as many, utterances that end in any of the
    wavefronts or blocks, one of them with scores so large that a step's proof never fails and one
    with scores so small that it nearly always does."""
    V = 5
    il = [T, T - 1, T - 2, T - 3, T, max(T - 60, 1)]
    ll = [U - 1, U // 2, min(64, U - 1), 0, U - 1, min(63, U - 1)]
    B = len(il)
    rng = np.random.default_rng(7000 * T + U)
    E = rng.standard_normal((B, T, V), dtype=np.float32)
    P = rng.standard_normal((B, U, V), dtype=np.float32)
    E[1] *= 40.0
    E[4] *= 0.01
    P[4] *= 0.01
    labels = rng.integers(1, V, (B, U - 1)).astype(np.int32)
    il, ll = np.array(il, np.int32), np.array(ll, np.int32)
    LN = oracle.log_norms_naive(E, P, il, ll)
    want_costs, want = oracle.forward(E, P, LN, labels, il, ll)
    costs, alphas = gpu_forward(DeviceCase(E, P, labels, il, ll), np.nan_to_num(LN))
    for b in range(B):
        got, ref = alphas[b, :il[b], :ll[b] + 1], want[b, :il[b], :ll[b] + 1]
        assert_same_bits(got, ref, "alphas of utterance %d" % b)
    assert_same_bits(costs, want_costs, "costs")


@pytest.mark.parametrize("U", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 70])
def test_dalphas_where_groups_of_four_meet_the_lattices_edges(T, U):
    """The transition weights are formed four anti-diagonals at a time: lattices that begin or end
    inside such a group, shorter than one, and utterances of one frame or without labels."""
    V, il, ll = 5, [T, T, max(T - 1, 1), 1], [U - 1, 0, U // 2, U - 1]
    rng = np.random.default_rng(100 * T + U)
    E = rng.standard_normal((4, T, V), dtype=np.float32)
    P = rng.standard_normal((4, U, V), dtype=np.float32)
    labels = rng.integers(1, V, (4, U - 1)).astype(np.int32)
    il, ll = np.array(il, np.int32), np.array(ll, np.int32)
    LN = oracle.log_norms_naive(E, P, il, ll)
    c = DeviceCase(E, P, labels, il, ll)
    _, alphas = gpu_forward(c, np.nan_to_num(LN))
    got = gpu_backward(c, np.nan_to_num(alphas), np.nan_to_num(LN))
    want = oracle.backward(E, P, np.nan_to_num(alphas), LN, labels, il, ll)
    for g, w, what in zip(got, want, ("egrads", "pgrads", "lngrads")):
        assert_same_bits(g, w, what)


@pytest.mark.parametrize("U", [65, 128, 193, 256, 300, 520])
@pytest.mark.parametrize("T", [31, 191, 253, 256, 517])
def test_dalphas_where_the_hand_over_between_wavefronts_wraps(T, U):
    """The same rings, in the other direction: lattices of about 256 steps and of several times as
    many, utterances whose last label lies in any wavefront or block, one whose labels are all the
    blank (one accumulator for both sums)."""
    V = 5
    il = [T, T - 1, T - 2, T - 3, max(T - 60, 1), T]
    ll = [U - 1, U // 2, min(64, U - 1), 0, min(63, U - 1), min(129, U - 1)]
    B = len(il)
    rng = np.random.default_rng(9000 * T + U)
    E = rng.standard_normal((B, T, V), dtype=np.float32)
    P = rng.standard_normal((B, U, V), dtype=np.float32)
    labels = rng.integers(1, V, (B, U - 1)).astype(np.int32)
    labels[1] = 0
    il, ll = np.array(il, np.int32), np.array(ll, np.int32)
    LN = oracle.log_norms_naive(E, P, il, ll)
    _, alphas = oracle.forward(E, P, LN, labels, il, ll)
    alphas, LN = np.nan_to_num(alphas, posinf=0.0, neginf=0.0), np.nan_to_num(LN)
    got = gpu_backward(DeviceCase(E, P, labels, il, ll), alphas, LN)
    want = oracle.backward(E, P, alphas, LN, labels, il, ll)
    for g, w, what in zip(got, want, ("egrads", "pgrads", "lngrads")):
        assert_same_bits(g, w, what)


def check_paths(E, P, il, ll):
    labels = np.ones((E.shape[0], P.shape[1] - 1), np.int32)
    LN = np.nan_to_num(oracle.log_norms_naive(E, P, il, ll))
    got = gpu_viterbi(DeviceCase(E, P, labels, il, ll), LN)
    want = oracle.viterbi(E, P, LN, il, ll)
    for b in range(E.shape[0]):
        assert np.array_equal(got[b, :ll[b]], want[b, :ll[b]]), "path of utterance %d" % b


@pytest.mark.parametrize("U", [2, 64, 65, 129, 256, 300, 520])
@pytest.mark.parametrize("T", [31, 253, 256, 517])
def test_best_paths_where_the_hand_over_between_wavefronts_wraps(T, U):
    """Lattices of about 256 steps and of several times as many, utterances whose last label lies
    in any wavefront or block, with no labels and with one frame."""
    V = 6
    il = np.array([T, T - 1, T - 2, T - 3, max(T - 60, 1), 1], np.int32)
    ll = np.array([U - 1, U // 2, min(64, U - 1), 0, min(63, U - 1), U - 1], np.int32)
    rng = np.random.default_rng(11000 * T + U)
    E = rng.standard_normal((6, T, V), dtype=np.float32)
    P = rng.standard_normal((6, U, V), dtype=np.float32)
    check_paths(E, P, il, ll)


@pytest.mark.parametrize("T,U", [(5200, 4), (2100, 300), (9000, 130), (5200, 60)])
def test_best_paths_with_thousands_of_frames_between_labels(T, U):
    """The backtrace looks at 2048 steps at a time: half of the labels in the first frames, the other
    half in the last ones, blanks only in between; decision columns in LDS and in memory."""
    V = 4
    il, ll = np.array([T, T - 37, T], np.int32), np.array([U - 1, U - 1, U // 2], np.int32)
    rng = np.random.default_rng(T + U)
    E = rng.standard_normal((3, T, V), dtype=np.float32)
    P = rng.standard_normal((3, U, V), dtype=np.float32)
    E[:, U // 2 + 3:T - 40 - U // 2 - 3, 0] += 60.0
    E[:, :U // 2 + 3, 0] -= 60.0
    E[:, T - 40 - U // 2 - 3:, 0] -= 60.0
    check_paths(E, P, il, ll)
