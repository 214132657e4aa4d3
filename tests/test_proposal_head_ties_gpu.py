"""Proposal where only the order of equal scores among the best 512 proposals is open.

mcProposal and mcProposalHead + mcProposalContinue replay the reference's quicksort through the partitions
that hold those scores only; the rows equal the CPU path's bit for bit.  Tables up to the
largest that the head takes, runs of equal scores, scores in an order that makes the quicksort follow the
short or the long side, few candidates, and a result that the head cannot settle after all.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def K(gpu_mode):
    from minicaffe import kernels
    return kernels


def run(K, scores, bbox, im_info, pre, post, steps):
    A, H, W = 9, scores.shape[2], scores.shape[3]
    size = ctypes.c_size_t()
    K.check_mc(K.LIB.mcProposalWorkspaceSize(A * H * W, pre, post, ctypes.byref(size)))
    ws = torch.full((size.value,), 255, dtype=torch.uint8, device="cuda")
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (scores, bbox, im_info, oracle.generate_anchors().astype(np.float32))]
    rois, rs = torch.full((post, 5), float("nan"), device="cuda"), torch.zeros(post, device="cuda")
    cnt = torch.zeros(3, dtype=torch.int32, device="cuda")

    def call(fn):
        K.check_mc(fn(*[x.data_ptr() for x in t], A, H, W, 16, 16.0, pre, post, 0.7, ws.data_ptr(), size.value,
                      rois.data_ptr(), rs.data_ptr(), cnt.data_ptr(), cnt.data_ptr() + 4, None))
        torch.cuda.synchronize()
    if not steps:
        call(K.LIB.mcProposal)
    else:
        call(K.LIB.mcProposalHead)
        if int(cnt[2].item()) == 0:
            call(K.LIB.mcProposalContinue)
            assert int(cnt[2].item()) == 1
    n = int(cnt[0].item())
    return rois[:n].cpu().numpy(), rs[:n].cpu().numpy(), ws


def flags(ws):
    """The call's eight flag words, the last of the workspace (256 bytes with their padding)."""
    return ws[-256:-224].view(torch.int32).tolist()


def inputs(rng, fg, hw, spread=0.2):
    (H, W), A = hw, 9
    scores = rng.random((1, 2 * A, H, W)).astype(np.float32)
    scores[0, A:] = fg.reshape(H, W, A).transpose(2, 0, 1)
    bbox = (rng.standard_normal((1, 4 * A, H, W)) * spread).astype(np.float32)
    return scores, bbox, np.array([H * 16, W * 16, 1.0], np.float32)


@pytest.mark.parametrize("hw,pre,post,order", [
    ((38, 63), 6000, 300, "random"), ((20, 20), 6000, 200, "random"), ((12, 10), 6000, 150, "random"),   # 1080 places
    ((11, 9), 6000, 100, "random"),                         # 891: no long partition at all
    ((6, 5), 300, 100, "random"), ((38, 63), 400, 150, "random"),
    ((40, 63), 6000, 300, "random"),                        # 22 680: the larger selection
    ((64, 64), 6000, 300, "random"),                        # 36 864: the largest table
    ((64, 65), 6000, 300, "random"),                        # beyond it: the full-size path
    ((38, 63), 6000, 300, "worst first"), ((38, 63), 6000, 300, "best first"), ((38, 63), 6000, 300, "waves"),
    ((38, 63), 6000, 511, "random")])                       # hardly settled by 512 candidates
@pytest.mark.parametrize("seed", range(4))
def test_rows_equal_the_reference(K, hw, pre, post, order, seed):
    rng = np.random.default_rng(40 + seed)
    A, (H, W) = 9, hw
    n = A * H * W
    fg = rng.permutation(n).astype(np.float32) / n * 0.9 + 0.05
    if order == "worst first":
        fg[:40] = np.sort(fg[:40])
    elif order == "best first":        # pivots of small rank: short rests before the followed partition
        top = np.argsort(-fg)[:60]
        fg[:60], fg[top] = fg[top].copy(), fg[:60].copy()
    elif order == "waves":
        fg = (0.05 + 0.9 * np.abs(np.sin(np.arange(n) * 0.37 + seed))).astype(np.float32)
    best = np.argsort(-fg, kind="stable")
    head = min(512, n, pre)
    for k in range(1 + 3 * seed):      # pairs and runs, neighbours in order or not, one at the head's end
        at = int(rng.integers(0, head - 6))
        fg[best[at:at + int(rng.integers(2, 6))]] = fg[best[at]]
    if seed == 3:
        fg[rng.choice(best[:head], 2, replace=False)] = fg[best[head // 2]]
    scores = rng.random((1, 2 * A, H, W)).astype(np.float32)
    scores[0, A:] = fg.reshape(H, W, A).transpose(2, 0, 1)
    bbox = (rng.standard_normal((1, 4 * A, H, W)) * 0.2).astype(np.float32)
    im_info = np.array([H * 16, W * 16, 1.0], np.float32)
    want_rois, want_scores = oracle.proposal({"pre_nms_topn": pre, "post_nms_topn": post, "nms_thresh": 0.7}, scores, bbox,
                                             im_info, 2)
    for steps in (False, True):
        rois, rs, _ = run(K, scores, bbox, im_info, pre, post, steps)
        assert np.array_equal(rois, want_rois) and np.array_equal(rs, want_scores), steps


def best_valid(scores, bbox, im_info):
    """Indices by (score descending, index ascending), boxes that are too small last."""
    props = oracle.generate_proposals(scores[0, 9:], bbox[0], oracle.generate_anchors(), float(im_info[0]), float(im_info[1]), 16.0, 16)
    return np.argsort(-props[:, 4], kind="stable")


@pytest.mark.parametrize("hw,post", [((38, 63), 200), ((40, 63), 200), ((64, 64), 200), ((20, 20), 100), ((12, 10), 60),
                                     ((11, 9), 40), ((6, 5), 20)])
@pytest.mark.parametrize("seed", range(2))
def test_the_head_replays_its_equal_scores(K, hw, post, seed):
    """The two best proposals have one score, so their order is open whatever the boxes are: the
    replay that starts from the head settles it (it would not with the general replay forced)."""
    rng = np.random.default_rng(70 + 2 * seed)
    n = 9 * hw[0] * hw[1]
    fg = rng.permutation(n).astype(np.float32) / n * 0.9 + 0.05
    args = scores, bbox, im_info = inputs(rng, fg, hw)
    best = best_valid(*args)
    fg[best[1]] = fg[best[0]]
    fg[best[min(400, n // 2)]] = fg[best[min(401, n // 2 + 1)]]
    scores[0, 9:] = fg.reshape(hw + (9,)).transpose(2, 0, 1)
    want = oracle.proposal({"pre_nms_topn": 6000, "post_nms_topn": post, "nms_thresh": 0.7}, *args, 2)
    for general in (0, 1):
        K.check_mc(K.LIB.mcProposalForceGeneralReplay(general))
        try:
            for steps in (False, True):
                rois, rs, ws = run(K, *args, 6000, post, steps)
                assert np.array_equal(rois, want[0]) and np.array_equal(rs, want[1]), (general, steps)
                f = flags(ws)
                assert (f[3], f[5]) == (0 if general else 2, 1), (f, general, steps)
        finally:
            K.check_mc(K.LIB.mcProposalForceGeneralReplay(0))


@pytest.mark.parametrize("order", ["descending", "ascending", "almost descending", "shuffled by 16", "organ pipe"])
@pytest.mark.parametrize("hw", [(38, 63), (20, 20), (64, 64)])
def test_sorted_tables(K, hw, order):
    """Hundreds of levels with a pivot or two each.  The head's replay follows them where the table is too
    large for the full-size one's LDS, or its front moves along quickly, and else gives up."""
    rng = np.random.default_rng(60)
    n = 9 * hw[0] * hw[1]
    fg = np.arange(n, 0, -1).astype(np.float32) / n * 0.9 + 0.05
    if order == "ascending":
        fg = fg[::-1].copy()
    elif order == "almost descending":
        for i in rng.integers(0, n - 5, n // 50):
            fg[i], fg[i + 4] = fg[i + 4], fg[i]
    elif order == "shuffled by 16":
        fg = rng.permuted(fg[:n // 16 * 16].reshape(-1, 16), axis=1).reshape(-1)
        fg = np.concatenate([fg, np.full(n - fg.size, 0.05, np.float32)])
    elif order == "organ pipe":
        fg = np.concatenate([fg[::2][::-1], fg[1::2]])
    args = scores, bbox, im_info = inputs(rng, fg, hw)
    best = best_valid(*args)
    for at in (0, 7, 100, 101, 300):
        fg[best[at + 1]] = fg[best[at]]
    scores[0, 9:] = fg.reshape(hw + (9,)).transpose(2, 0, 1)
    post = 100
    want = oracle.proposal({"pre_nms_topn": 6000, "post_nms_topn": post, "nms_thresh": 0.7}, *args, 2)
    for steps in (False, True):
        rois, rs, ws = run(K, *args, 6000, post, steps)
        assert np.array_equal(rois, want[0]) and np.array_equal(rs, want[1]), steps
        path = tuple(flags(ws)[k] for k in (3, 5, 7))
        assert path == ((2, 1, 0) if n > 22528 else (0, 1, 1) if order == "descending" else path), steps


@pytest.mark.parametrize("kind", ["crowds", "a pair at the cut", "too many proposals"])
def test_overlaps_beyond_the_best_512_are_left_out_where_these_settle_it(K, kind):
    """Where the head cannot be ordered by itself, the best 512 of the fully ordered table still come
    first: of the 94 x 6000 words of the overlap matrix 8 x 512 are written, the others stay as they were."""
    rng = np.random.default_rng(80)
    hw, pre, post = ((64, 65) if kind == "too many proposals" else (38, 63)), 6000, 200
    n = 9 * hw[0] * hw[1]
    fg = rng.permutation(n).astype(np.float32) / n * 0.9 + 0.05
    if kind == "crowds":
        fg = (np.round(fg * 2000) / 2000).astype(np.float32)
    args = scores, bbox, im_info = inputs(rng, fg, hw)
    if kind == "a pair at the cut":
        best = best_valid(*args)
        fg[best[512]] = fg[best[511]]
        scores[0, 9:] = fg.reshape(hw + (9,)).transpose(2, 0, 1)
    want = oracle.proposal({"pre_nms_topn": pre, "post_nms_topn": post, "nms_thresh": 0.7}, *args, 2)
    for steps in (False, True):
        rois, rs, ws = run(K, *args, pre, post, steps)
        assert np.array_equal(rois, want[0]) and np.array_equal(rs, want[1]), steps
        assert len(rois) == post and flags(ws)[3] == 0
        untouched = int((ws[:ws.numel() // 8 * 8].view(torch.int64) == -1).sum().item())
        assert untouched > 0.95 * pre * 94, steps


def kept_of(boxes, thr):
    """Greedy suppression in order, as the layer's."""
    area = (boxes[:, 2] - boxes[:, 0] + 1) * (boxes[:, 3] - boxes[:, 1] + 1)
    kept = []
    for i, b in enumerate(boxes):
        k = boxes[kept]
        w = np.maximum(0, np.minimum(b[2], k[:, 2]) - np.maximum(b[0], k[:, 0]) + 1)
        h = np.maximum(0, np.minimum(b[3], k[:, 3]) - np.maximum(b[1], k[:, 1]) + 1)
        if not (w * h / (area[i] + area[kept] - w * h) > thr).any():
            kept.append(i)
    return kept


@pytest.mark.parametrize("seed", range(2))
def test_replayed_order_keeps_fewer_than_asked_for(K, seed):
    """Triples of equal scores, neighbours overlap, the outer two do not: in index order two of each
    are kept, with the middle one first just one.  The scan of the best 512 then reaches post_nms_topn in index
    order only, and the full-size path follows the replay."""
    rng = np.random.default_rng(90 + seed)
    hw, A = (38, 63), 9
    H, W = hw
    fg = (rng.permutation(A * H * W).astype(np.float32) / (A * H * W) * 0.9 + 0.05).reshape(H, W, A)
    scores, bbox, im_info = inputs(rng, fg.reshape(-1), hw, 0.0)
    anchors = oracle.generate_anchors()
    square = int(np.argmin(np.abs(anchors[:, 2] - anchors[:, 0] - 127) + np.abs(anchors[:, 3] - anchors[:, 1] - 127)))
    for i, (h, w) in enumerate([(h, w) for h in (10, 20, 28) for w in (10, 25, 40, 50)]):
        scores[0, A:, h - 5:h + 6, w - 5:w + 8] *= 0.1    # (nothing else that the triple's members would suppress)
        scores[0, A + square, h, w:w + 3] = 0.99 - 0.001 * i
    props = oracle.generate_proposals(scores[0, A:], bbox[0], anchors, float(im_info[0]), float(im_info[1]), 16.0, 16)
    first = props[np.argsort(-props[:, 4], kind="stable")[:512]]
    post = len(kept_of(first[:, :4], 0.7))
    want = oracle.proposal({"pre_nms_topn": 6000, "post_nms_topn": post, "nms_thresh": 0.7}, scores, bbox, im_info, 2)
    for steps in (False, True):
        rois, rs, ws = run(K, scores, bbox, im_info, 6000, post, steps)
        assert np.array_equal(rois, want[0]) and np.array_equal(rs, want[1]), steps
        f = flags(ws)
        assert (f[3], f[5], f[6], f[7]) == (0, 1, 1, 0), f
