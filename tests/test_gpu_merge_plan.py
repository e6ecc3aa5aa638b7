"""The merge's bookkeeping kernels (gpa::merge_order, gpa::merge_plan) against
torch's stable sorts: exact, every output.  Row counts sit at the edges of the
counting path (16 rows a workgroup, 4,096 keys staged at a time) and of the
radix sort's blocks (4,096 rows), and on both sides of the line between them;
maxima with ties, NaN, both zeros and infinities; all rows of a batch element
in one slot; destination counts of one to three key bytes."""
import pytest
import torch

from merging import _native  # noqa: F401  (registers the ops)
from merging.merge import dst_mask, num_dst_tokens, token_merge_bipartite2d, window_cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frames,w,h,sx,sy,ns,no_rand", [
    (1, 37, 37, 2, 2, 5, False), (3, 37, 37, 2, 2, 5, False), (9, 37, 28, 2, 3, 5, False),
    (4, 5, 7, 3, 2, 0, False), (4, 6, 6, 2, 2, 5, True), (2, 3, 3, 4, 4, 1, False),
    (2, 45, 45, 1, 1, 7, False)])
def test_order_and_mask(dev, frames, w, h, sx, sy, ns, no_rand):
    def gen():
        return torch.Generator(device=dev).manual_seed(frames)

    mask = dst_mask(frames, w, h, sx, sy, ns, no_rand, gen(), dev)
    cell = None if no_rand or frames == 1 else window_cells(frames, w, h, sx, sy, gen(), dev)
    got_mask, got = torch.ops.gpa.merge_order(cell, frames, w, h, sx, sy, ns, dev)
    assert torch.equal(got_mask, mask)
    assert torch.equal(got, torch.argsort(mask, stable=True))
    assert int((mask == -1).sum()) == num_dst_tokens(frames, w, h, sx, sy, ns, no_rand)


@pytest.mark.parametrize("frames,w,h,sx,sy,ns,no_rand", [
    (1, 6, 6, 0, 0, 5, False), (1, 6, 6, -1, 2, 5, False), (3, 6, 6, 0, 0, 5, True),
    (3, 5, 7, 2, -3, 0, True), (1, 6, 6, 2, 2, -2, False), (1, -6, -6, 2, 2, 5, False),
    (2, -6, -6, 2, 2, 5, True)])
def test_sizes_that_no_window_uses(dev, frames, w, h, sx, sy, ns, no_rand):
    """One frame, or no drawn patch: the windows are not looked at."""
    mask = dst_mask(frames, w, h, sx, sy, ns, no_rand, None, dev)
    got_mask, got = torch.ops.gpa.merge_order(None, frames, w, h, sx, sy, ns, dev)
    assert torch.equal(got_mask, mask) and torch.equal(got, torch.argsort(mask, stable=True))
    n = frames * (w * h + ns)
    x = torch.randn(1, n, 256, device=dev)
    m = token_merge_bipartite2d(x, w, h, sx, sy, 10, no_rand, num_special=ns)
    assert torch.equal(m.index.mask, mask) and m.size.sum() == n


def test_sizes_that_are_refused(dev):
    cell = torch.zeros(2, 3, 3, device=dev, dtype=torch.int64)
    mask = torch.empty(1, device=dev, dtype=torch.int64)
    L = _native.lib()
    for frames, w, h, sx, sy, ns, p, code in [
            (-1, 6, 6, 2, 2, 5, 0, _native.GPA_E_INVALID), (3, 6, 6, 0, 2, 5, 1, _native.GPA_E_INVALID),
            (3, -6, -6, 2, 2, 5, 1, _native.GPA_E_INVALID), (3, 6, 6, 2, 2, -1, 0, _native.GPA_E_INVALID),
            (1, 6, -6, 2, 2, 5, 0, _native.GPA_E_INVALID),
            (1, 2 ** 40, 2 ** 40, 2, 2, 5, 0, _native.GPA_E_UNSUPPORTED),
            (1, 2 ** 16, 2 ** 16, 2, 2, 5, 0, _native.GPA_E_UNSUPPORTED)]:
        assert L.gpa_merge_order(cell.data_ptr() if p else None, frames, w, h, sx, sy, ns,
                                 mask.data_ptr(), mask.data_ptr(), None) == code


@pytest.mark.parametrize("bad", [-1, 6, -2 ** 40, 2 ** 40])
@pytest.mark.parametrize("every", [1, 3])
def test_cells_outside_their_window(dev, bad, every):
    """They count as the nearest cell inside, and nothing is written past the
    mask and the order (a mask without a destination in a window would shift
    the sources' ranks past the end)."""
    frames, w, h, sx, sy, ns = 3, 13, 8, 2, 3, 5
    n, pad = frames * (w * h + ns), 256
    cell = torch.randint(0, 6, (frames - 1, h // sy, w // sx),
                         generator=torch.Generator().manual_seed(5))
    cell.view(-1)[::every] = bad
    want_mask, want = torch.ops.gpa.merge_order(cell.clamp(0, 5).to(dev), frames, w, h, sx, sy, ns,
                                                dev)
    mask, order = (torch.full((n + pad,), -7, device=dev, dtype=torch.int64) for _ in range(2))
    cell = cell.to(dev)
    rc = _native.lib().gpa_merge_order(cell.data_ptr(), frames, w, h, sx, sy, ns, mask.data_ptr(),
                                       order.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == _native.GPA_OK
    assert torch.equal(mask[:n], want_mask) and torch.equal(order[:n], want)
    assert (mask[n:] == -7).all() and (order[n:] == -7).all()
    assert torch.equal(want, torch.argsort(want_mask, stable=True))


def _expected(node_max, node_idx, order, num_dst, r):
    """The same lists from torch's stable sorts, on the CPU."""
    B, ns = node_max.shape
    N = num_dst + ns
    b_pos, a_pos = order[:num_dst], order[num_dst:]
    edge = torch.argsort(node_max.float(), dim=-1, descending=True, stable=True)
    dst_slot = torch.gather(node_idx, 1, edge[:, :r])
    unm_abs, src_abs = a_pos[edge[:, r:]], a_pos[edge[:, :r]]
    unm = ns - r
    size = torch.ones(B, unm + num_dst)
    size[:, unm:].scatter_add_(1, dst_slot, torch.ones(B, r))
    key = torch.cat([torch.arange(unm + num_dst).expand(B, -1), unm + dst_slot], 1)
    tok = torch.cat([unm_abs, b_pos.expand(B, num_dst), src_abs], 1)
    sub = torch.cat([torch.zeros(B, unm + num_dst, dtype=torch.int64), src_abs + 1], 1)
    tokens = torch.gather(tok, 1, torch.argsort(key * (N + 1) + sub, dim=1)).reshape(-1)
    offsets = torch.zeros(B * (unm + num_dst) + 1, dtype=torch.int64)
    offsets[1:] = torch.cumsum(size.reshape(-1).to(torch.int64), 0)
    return edge, dst_slot, unm_abs, src_abs, size, offsets, tokens


@pytest.mark.parametrize("ns", [0, 1, 15, 64, 1023, 1045, 4096, 4097, 8193, 15360, 15361,
                                20481])
@pytest.mark.parametrize("num_dst,share,dtype,kind", [
    (1, 1.0, torch.float32, "plain"), (255, 0.2, torch.float32, "ties"),
    (256, 1.0, torch.bfloat16, "special"), (300, 0.0, torch.float16, "ties"),
    (70_000, 0.5, torch.float32, "special")])
def test_plan(dev, ns, num_dst, share, dtype, kind):
    g = torch.Generator().manual_seed(ns + num_dst)
    B = 1 if ns == 1045 else 2
    node_max = torch.randn(B, ns, generator=g)
    if kind == "ties":
        node_max = (node_max * 4).round() / 4
    elif kind == "special" and ns > 0:
        pool = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), 1.0, -1.0])
        pick = torch.randint(0, 14, (B, ns), generator=g)
        node_max = torch.where(pick < 7, pool[pick.clamp_max(6)], node_max)
    node_max = node_max.to(dtype)
    node_idx = torch.randint(0, num_dst, (B, ns), generator=g)
    node_idx[B - 1, ns // 3:] = num_dst - 1                 # most rows in one slot
    order = torch.randperm(num_dst + ns, generator=g)
    order = torch.cat([order[:num_dst].sort().values, order[num_dst:].sort().values])
    r = int(ns * share)
    want = _expected(node_max, node_idx, order, num_dst, r)
    got = torch.ops.gpa.merge_plan(node_max.to(dev), node_idx.to(dev), order.to(dev), num_dst, r)
    for name, x, y in zip(("edge", "dst_slot", "unm_abs", "src_abs", "size", "offsets", "tokens"),
                          got, want):
        assert x.dtype == y.dtype and torch.equal(x.cpu(), y), name


@pytest.mark.parametrize("B,ns,num_dst", [
    (1, 15_360, 6234), (1, 16_500, 6234), (4, 7280, 3677), (4, 7900, 3900), (32, 2080, 2032),
    (32, 2500, 2032), (128, 900, 1500), (128, 1040, 1703), (59, 17, 20_001), (60, 17, 20_002),
    (300, 1, 5000), (40, 0, 40_000)])
def test_both_sides_of_the_line_in_batches(dev, B, ns, num_dst):
    """Counting on one side, radix passes on the other, down to one row each;
    the workspace the entry point asks for is enough and no less is taken
    than it needs."""
    g = torch.Generator().manual_seed(B + ns)
    node_max = (torch.randn(B, ns, generator=g) * 64).round() / 64          # ties
    node_idx = torch.randint(0, num_dst, (B, ns), generator=g)
    order = torch.randperm(num_dst + ns, generator=g)
    order = torch.cat([order[:num_dst].sort().values, order[num_dst:].sort().values])
    r = int(0.9 * ns + 0.5)
    want = _expected(node_max, node_idx, order, num_dst, r)
    got = torch.ops.gpa.merge_plan(node_max.to(dev), node_idx.to(dev), order.to(dev), num_dst, r)
    for name, x, y in zip(("edge", "dst_slot", "unm_abs", "src_abs", "size", "offsets", "tokens"),
                          got, want):
        assert x.dtype == y.dtype and torch.equal(x.cpu(), y), name
    if ns > 0:
        L = _native.lib()
        p = [x.data_ptr() for x in got]
        x, i, o = node_max.to(dev), node_idx.to(dev), order.to(dev)
        ws = torch.empty(B * ns * 4, device=dev, dtype=torch.uint8)
        assert L.gpa_merge_plan_workspace_bytes(B, ns) >= ws.numel()
        assert L.gpa_merge_plan(x.data_ptr(), _native.GPA_DTYPE_F32, i.data_ptr(), o.data_ptr(), B,
                                num_dst + ns, num_dst, r, *p, ws.data_ptr(), ws.numel() - 4,
                                None) == _native.GPA_E_WORKSPACE


@pytest.mark.parametrize("metric_dim", [0, 128])
def test_a_metric_of_another_type_without_sources(dev, metric_dim):
    """One frame has no source: its maxima are an empty row of the metric's
    type, which nothing reads; with sources the similarity refuses the type."""
    x = torch.randn(2, 41, 256, device=dev, dtype=torch.float64)
    m = token_merge_bipartite2d(x, 6, 6, 2, 2, 10, metric_dim=metric_dim)
    assert torch.equal(m(x), x) and m.index.node_max.dtype == torch.float64
    assert torch.equal(m.index.slot_tokens, torch.arange(41, device=dev).repeat(2))
    with pytest.raises(ValueError):
        token_merge_bipartite2d(x.view(1, 82, 256), 6, 6, 2, 2, 10, metric_dim=metric_dim)
