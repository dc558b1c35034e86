"""Exact ReLU zeros of the FP8 index scorer.

The reference's logit sum_h w_h * ReLU(q_h . k) * s_k is exactly 0 for a key
whose every head dot is <= 0 (sglang/srt/layers/attention/v1_deepseek/
kernels.py:310-313), and Top-K breaks the ties of that zero plateau by lower
index.  The shapes below are the reference probe's query packing
(qwen_gqa_probe_kernels.py:14-20: 4 live heads of 32, w = s_q * SCALE / 4,
zero queries and weights past them) and a single head with w = s_q * SCALE:
non-power-of-two weights, about 1/16 (resp. 1/2) of the keys exact zeros, and
rows of ~2100 keys so that the Top-2048 boundary falls inside the plateau.
Both the shared-table kernel (one page table for the whole chunk) and the
per-row kernel are checked, and the selected indices are compared with a
Top-2048 over the fp64 reference scores themselves."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import pkg
from oracle import v1 as O
from test_gpu_kernels import H, T, assert_scores_close, assert_scores_rel

pytestmark = pytest.mark.gpu

SC = pkg("scoring")
TK = pkg("topk")
W = pkg("workloads")

SOFTMAX_SCALE = 128 ** -0.5


def _probe_case(g, rows, heads, live, ctx, pool_pages, signed):
    q8l, sq = W.quantize_rows(g.standard_normal((rows * live, 128), dtype=np.float32))
    q8 = np.zeros((rows, heads, 128), np.uint8)
    q8[:, :live] = q8l.reshape(rows, live, 128)
    w = np.zeros((rows, heads), np.float32)
    w[:, :live] = (sq.reshape(rows, live) * np.float32(SOFTMAX_SCALE / live)).astype(np.float32)
    if signed:
        w[:, :live] *= np.where(g.random((rows, live)) < 0.5, -1, 1).astype(np.float32)
    k8, ks = W.quantize_rows(g.standard_normal((pool_pages * 64, 128), dtype=np.float32))
    native = W.pack_pages(k8, ks)
    blocks = -(-ctx // 64)
    table = g.permutation(pool_pages)[:blocks].astype(np.int32)
    lens = (ctx - rows + 1 + np.arange(rows)).astype(np.int32)
    return q8, w, native, table, lens


def _top_fp64(ref, lens, topk):
    """Top-`topk` per row over fp64 scores: value descending, ties by lower
    index, returned ascending (the order the Top-K kernels emit)."""
    out = np.full((ref.shape[0], topk), -1, np.int64)
    for b in range(ref.shape[0]):
        L = int(lens[b])
        order = np.lexsort((np.arange(L), -ref[b, :L]))[:topk]
        out[b, :min(L, topk)] = np.sort(order)
    return out


@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("heads,live,signed", [(1, 1, False), (32, 4, False), (32, 4, True), (64, 8, False)])
def test_relu_zeros_exact_and_topk_on_fp64_scores(dev, shared, heads, live, signed):
    g = np.random.default_rng(100 * heads + 10 * live + int(signed) + 2 * int(shared))
    rows, ctx = 40, 2120
    q8, w, native, table, lens = _probe_case(g, rows, heads, live, ctx, 96, signed)
    full = np.broadcast_to(table, (rows, table.size))
    bt = T(table, dev)[None].expand(rows, -1) if shared else T(np.ascontiguousarray(full), dev)
    out = SC.fp8_paged_mqa_logits(T(q8, dev).view(torch.float8_e4m3fn), T(native, dev), T(w, dev), T(lens, dev), bt,
                                  None, ctx, clean_logits=True)
    got = H(out)
    ref = O.paged_logits(q8, w, native, full, lens, ctx)
    bound = O.paged_logits(q8, w, native, full, lens, ctx, magnitude=True)
    assert_scores_close(got.astype(np.float64), ref, bound)
    fin = np.isfinite(ref)
    zero = fin & (ref == 0)
    # the plateau is there (about 2^-live of the keys), its scores are +0.0 bit
    # for bit, and no key with a positive head dot lands on it
    assert zero.sum() > 0.5 * fin.sum() * 2.0 ** -live
    assert (got[zero].view(np.uint32) == 0).all(), f"{int((got[zero] != 0).sum())} reference zeros scored nonzero"
    assert (got[fin & (ref != 0)] != 0).all()
    if signed or live > 4:
        return
    # Top-2048 on the GPU logits equals Top-2048 on the fp64 reference scores
    # for rows whose boundary falls inside the zero plateau
    positive = (fin & (ref > 0)).sum(axis=1)
    plateau_rows = (positive < 2048) & (positive + zero.sum(axis=1) > 2048)
    assert plateau_rows.all()
    slots = torch.empty((rows, 2048), device=dev, dtype=torch.int32)
    raw = torch.empty_like(slots)
    ident = np.arange(-(-ctx // 64), dtype=np.int32)[None].repeat(rows, 0)
    TK.topk_transform_512_v2(out, T(lens, dev), T(ident, dev), slots, 64, None, raw)
    assert np.array_equal(H(raw), _top_fp64(ref, lens, 2048))


@pytest.mark.parametrize("rows,heads,longest,capacity", [
    (600, 32, 5003, 5003),     # fewer 16-page chunks than work-groups: 14 pages
    (9, 64, 1100, 16384),      # two groups, 4-page chunks, most of them past every row
    (1030, 64, 8064, 16384),   # ranges of two chunks by the longest context, not by the capacity
    (2000, 17, 8000, 8000),    # ranges of three chunks and a halving tail
    (520, 16, 70, 40000),      # ranges of one chunk, all but the first empty
    (40, 32, 0, 300),          # no row has a key
])
def test_shared_table_ranges(dev, rows, heads, longest, capacity):
    """Shared-table scores over the ranges that the longest context and the
    count of work-groups give, against the row-by-row kernel (each row its own
    copy of the table, at most 512 rows a call).  4 live heads put keys on the
    zero plateau, so marked pages cross the ranges too."""
    g = np.random.default_rng(rows + heads)
    live = 4
    pages = -(-max(longest, 64) // 64)
    q8, w, native, table = _probe_case(g, rows, heads, live, pages * 64, pages, False)[:4]
    lens = g.integers(0, longest + 1, rows).astype(np.int32)
    lens[rows // 2] = longest
    tq, tn, tw, tl = T(q8, dev).view(torch.float8_e4m3fn), T(native, dev), T(w, dev), T(lens, dev)
    tt = T(table, dev)[None]
    out = torch.full((rows, capacity), 7.0, device=dev)
    ref = torch.full((rows, capacity), 7.0, device=dev)
    SC.fp8_paged_mqa_logits(tq, tn, tw, tl, tt.expand(rows, -1), None, capacity, clean_logits=True, out=out)
    for r in range(0, rows, 512):
        n = min(512, rows - r)
        SC.fp8_paged_mqa_logits(tq[r:r + n], tn, tw[r:r + n], tl[r:r + n], tt.expand(n, -1).contiguous(), None, capacity,
                                clean_logits=True, out=ref[r:r + n])
    assert_scores_rel(H(out).astype(np.float64), H(ref).astype(np.float64))


@pytest.mark.parametrize("clean", [False, True])
@pytest.mark.parametrize("rows,heads,longest,capacity", [
    (4096, 16, 1024, 131072),   # one live chunk of 128
    (1024, 32, 4096, 131072),
    (259, 64, 500, 131000),     # ranges of one chunk, a last row group of three, a last page of 56 columns
    (520, 64, 0, 33001),        # no live chunk, rows off 16-byte alignment
])
def test_shared_table_capacity_past_the_longest_context(dev, rows, heads, longest, capacity, clean):
    """A capacity far above every context: the work items that work-groups draw
    follow the longest context (the drawn count is the first word behind the
    rows' records in the workspace), and the columns past it are -inf with
    clean_logits and left alone without it."""
    L = pkg("_lib")
    g = np.random.default_rng(rows + longest)
    pages = -(-max(longest, 64) // 64)
    q8, w, native, table = _probe_case(g, rows, heads, 4, pages * 64, pages, False)[:4]
    lens = g.integers(0, longest + 1, rows).astype(np.int32)
    lens[rows // 2] = longest
    tq, tn, tw, tl = T(q8, dev).view(torch.float8_e4m3fn), T(native, dev), T(w, dev), T(lens, dev)
    tt = T(np.pad(table, (0, -(-capacity // 64) - pages)), dev)
    lib = L.lib()
    ws = torch.empty(lib.v1_score_workspace(rows, capacity), device=dev, dtype=torch.uint8)

    def run(cap):
        out = torch.full((rows, cap), 7.0, device=dev)
        a = L.ScoreArgs(tq.data_ptr(), tn.data_ptr(), tn.shape[0], tw.data_ptr(), tl.data_ptr(), tt.data_ptr(), 0,
                        tt.numel(), out.data_ptr(), out.stride(0), cap, rows, heads, 1, int(clean), ws.data_ptr(),
                        ws.numel())
        L.call("v1_score", ctypes.byref(a), torch.cuda.current_stream().cuda_stream)
        at = lib.v1_score_workspace(rows, 0) - 256
        return out, int(ws[at:at + 4].view(torch.int32).item())

    out, drawn = run(capacity)
    groups, chunks = -(-rows // 8), -(-longest // 1024)
    work_groups = 2 * torch.cuda.get_device_properties(dev).multi_processor_count
    filled = groups * (capacity // 8192 + 1) + work_groups if clean else 0  # (ranges of 8 chunks, or one a work-group)
    assert drawn <= groups * chunks + filled + work_groups  # (each work-group's last draw finds none)
    tight = run(max(longest, 1))[0]
    assert_scores_rel(H(out[:, :longest]).astype(np.float64), H(tight[:, :longest]).astype(np.float64))
    at = torch.arange(capacity, device=dev)[None] >= tl[:, None]
    assert (out[at] == (-np.inf if clean else 7.0)).all()
    assert torch.isfinite(out[~at]).all()
