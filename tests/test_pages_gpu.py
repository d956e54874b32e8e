"""The decode kernels for pages of exactly one pass (hidden 4096, 5120, 6144 or 8192): planned shrink and expand, and
both in one launch, bit for bit against the calls without a plan (kernels of their own) over the forms the launches
accept: run lengths 1 to 4, ranks on and off the vector path, grouped-query outputs, pages that do not exist, delta
narrower than the rank, an output that is not 16-byte aligned, launches with and without an item count."""
import numpy as np
import pytest
import torch

from lora_cases import make_case
from test_bgmv_gpu import GpuCase

pytestmark = pytest.mark.gpu


def _outputs(c, g, gpu, aligned):
    gen = torch.Generator(device=gpu)
    gen.manual_seed(7)
    out = []
    for h in c.h_out:
        flat = torch.empty(c.batch * h + 8, dtype=g.tdt, device=gpu).normal_(generator=gen)
        out.append(flat[0 if aligned else 4:][: c.batch * h].view(c.batch, h))
    return out


def _fresh(c, g, gpu, y0, R, aligned):
    y = _outputs(c, g, gpu, aligned)
    for a, b in zip(y, y0):
        a.copy_(b)
    return y, [torch.full((c.batch, R), 0.5, dtype=g.tdt, device=gpu) for _ in range(4)]


def _hand_over_area(batch, R):
    """Where a plan's hand-over area starts (behind header, records and scratch) and its items: a plan is 16 words, 48 per item
    and 6 per token; 16 words of launch counts per item follow."""
    per_run = (R + 7) // 8
    items = (batch * per_run + 7) // 8 * 8 + 8 * (per_run + 1)
    return (16 + items * 48 + batch * 6 + 3) // 4 * 4, items


def _launches_counted(plan, batch, R, first=0, proj=slice(0, 4)):
    """Sum of the launch counts of a plan's items from `first` on: 0 unless a call took the one launch."""
    area, items = _hand_over_area(batch, R)
    return int(plan.buf[area + 16 * first:area + 16 * items].view(-1, 16)[:, :12].view(-1, 4, 3)[:, proj].sum())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("hidden,ranks,batch,h_out,R,aligned", [
    (4096, [64, 8, 16, 32, 128], 11, None, 128, True),
    (4096, [8], 4, None, 8, True),                             # one run of four tokens, one item
    (4096, [16, 8], 41, [4096, 512, 512, 4096], 16, True),     # one launch at any size; k and v an eighth of a page
    (4096, [64, 24, 4, 12, 8], 9, None, 64, True),             # ranks off the vector path
    (4096, [64, 32, 8], 9, None, 16, True),                    # delta narrower than the rank
    (4096, [64, 8], 7, None, 64, False),
    (5120, [64, 8, 16], 7, None, 64, True),
    (6144, [8, 16], 13, None, 16, True),
    (8192, [64, 8, 32], 10, [8192, 1024, 1024, 8192], 64, True),
    (8192, [16, 8], 130, None, 16, True),
])
def test_whole_page_launches_equal_the_calls_without_a_plan(gpu, dtype, hidden, ranks, batch, h_out, R, aligned):
    import slora_hip
    from slora_hip import (dispatch_bgmv, dispatch_bgmv_lora, dispatch_bgmv_qkv_expand, dispatch_bgmv_qkv_lora,
                           dispatch_bgmv_qkv_shrink)
    c = make_case(500 + hidden + batch + R, hidden, ranks, batch, dtype=dtype, h_out=h_out, zipf_alpha=1.0)
    c.bins[batch // 2] = -1                                     # a token without an adapter
    c.a_loc[int(c.a_start[0]) + 1] = c.n_pages + 3              # a page outside the pool
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    y0 = [v.clone() for v in _outputs(c, g, gpu, True)]
    y_s, d_s = _fresh(c, g, gpu, y0, R, aligned)
    for p in range(4):
        dispatch_bgmv(d_s[p], g.x, g.key, *t, p, g.scales, plan=False)
        dispatch_bgmv(y_s[p], d_s[p], g.value, *t, p, g.scales, plan=False)
    for readback in (True, False):
        plan = slora_hip.make_plan(*t, R, c.n_pages, readback=readback)
        for rep in range(3):
            print(f"{dtype} hidden {hidden} batch {batch} R {R} readback {readback} rep {rep}", flush=True)
            y, d = _fresh(c, g, gpu, y0, R, aligned)
            dispatch_bgmv_qkv_shrink(*d[:3], g.x, g.key, *t, plan=plan)
            dispatch_bgmv_qkv_expand(*y[:3], *d[:3], g.value, *t, g.scales, plan=plan)
            dispatch_bgmv(d[3], g.x, g.key, *t, 3, g.scales, plan=plan)
            dispatch_bgmv(y[3], d[3], g.value, *t, 3, g.scales, plan=plan)
            for p in range(4):
                assert torch.equal(d[p], d_s[p]) and torch.equal(y[p], y_s[p]), (p, "two launches")
            y, d = _fresh(c, g, gpu, y0, R, aligned)
            dispatch_bgmv_qkv_lora(*y[:3], *d[:3], g.x, g.key, g.value, *t, g.scales, plan=plan)
            dispatch_bgmv_lora(y[3], d[3], g.x, g.key, g.value, *t, 3, g.scales, plan=plan)
            for p in range(4):
                assert torch.equal(d[p], d_s[p]) and torch.equal(y[p], y_s[p]), (p, "one launch")
        assert plan.status() == 0


@pytest.mark.parametrize("ranks,R,aligned", [
    ([16, 8], 16, True),
    ([24, 8], 24, True),        # a rank off the vector path: delta itself is read
    ([16, 8], 16, False),       # an output that is not 16-byte aligned: the same
])
def test_a_hand_over_that_never_comes_is_computed(gpu, ranks, R, aligned):
    """The word that counts a shrink workgroup's launches is changed in the plan, so that its rows name a launch nobody
    waits for: the readers give up after their poll limit, compute the rows themselves and mark the plan."""
    import slora_hip
    from slora_hip import dispatch_bgmv, dispatch_bgmv_lora
    c = make_case(9, 4096, ranks, 6, dtype="f16", bins=[0, 0, 1, 0, 0, 0])
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    y0 = _outputs(c, g, gpu, True)
    y_s, d_s = _fresh(c, g, gpu, y0, R, aligned)
    dispatch_bgmv(d_s[3], g.x, g.key, *t, 3, g.scales, plan=False)
    dispatch_bgmv(y_s[3], d_s[3], g.value, *t, 3, g.scales, plan=False)
    plan = slora_hip.make_plan(*t, R, c.n_pages)
    area, _ = _hand_over_area(c.batch, R)
    words = plan.buf.cpu().numpy()
    unit = next(u for u in range(plan.n_items) if words[16 + u * 48 + 2] > 0 and words[16 + u * 48 + 1] == ranks[0])
    plan.buf[area + unit * 16 + 3 * 3] = 7                      # projection o, workgroup of the shrink
    y, d = _fresh(c, g, gpu, y0, R, aligned)
    dispatch_bgmv_lora(y[3], d[3], g.x, g.key, g.value, *t, 3, g.scales, plan=plan)
    torch.cuda.synchronize()
    assert torch.equal(y[3], y_s[3]) and torch.equal(d[3], d_s[3])
    assert plan.status() == 2


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("hidden,kv,ranks,adapters,batch,R,qkv,o", [
    (4096, 4096, [16], 100, 245, 16, True, True),
    (4096, 1024, [16, 24, 8], 90, 200, 24, True, True),     # the one-dimensional grid; ranks off the vector path
    (5120, 5120, [16], 80, 245, 16, True, True),
    (6144, 6144, [16], 80, 245, 16, True, True),
    (8192, 1024, [16], 60, 245, 16, True, True),
    (4096, 4096, [32, 64], 64, 64, 64, False, False),
    (8192, 1024, [32], 60, 64, 64, True, False),
])
def test_workgroups_that_walk_several_items(gpu, dtype, hidden, kv, ranks, adapters, batch, R, qkv, o):
    """A plan without an item count, a capacity above 512 (launches get a quarter of it) and a batch of more items than that, so
    that workgroups take a second turn: two launches and, where it is one, one launch, three times on one plan, bit for bit
    the calls without a plan."""
    import slora_hip
    from slora_hip import (dispatch_bgmv, dispatch_bgmv_lora, dispatch_bgmv_qkv_expand, dispatch_bgmv_qkv_lora,
                           dispatch_bgmv_qkv_shrink)
    rng = np.random.default_rng(batch + hidden)
    mix = [ranks[i % len(ranks)] for i in range(adapters)]
    bins = rng.permutation(np.concatenate([np.arange(adapters), rng.integers(0, adapters, size=batch)])[:batch])
    need = 4 * sum(mix)
    c = make_case(700 + hidden + R, hidden, mix, batch, dtype=dtype, h_out=[hidden, kv, kv, hidden], bins=bins, n_pages=need + 9)
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    y0 = _outputs(c, g, gpu, True)
    want_y, want_d = _fresh(c, g, gpu, y0, R, True)
    for p in range(4):
        dispatch_bgmv(want_d[p], g.x, g.key, *t, p, g.scales, plan=False)
        dispatch_bgmv(want_y[p], want_d[p], g.value, *t, p, g.scales, plan=False)
    plan = slora_hip.make_plan(*t, R, c.n_pages, readback=False)
    _, capacity = _hand_over_area(batch, R)
    grid = (capacity // 4 + 7) // 8 * 8
    assert capacity > 512 and int(plan.buf[1]) > grid, (capacity, int(plan.buf[1]))
    for rep in range(3):
        print(f"walk {dtype} hidden {hidden} kv {kv} batch {batch} R {R} rep {rep}", flush=True)
        y, d = _fresh(c, g, gpu, y0, R, True)
        dispatch_bgmv_qkv_shrink(*d[:3], g.x, g.key, *t, plan=plan)
        dispatch_bgmv_qkv_expand(*y[:3], *d[:3], g.value, *t, g.scales, plan=plan)
        dispatch_bgmv(d[3], g.x, g.key, *t, 3, g.scales, plan=plan)
        dispatch_bgmv(y[3], d[3], g.value, *t, 3, g.scales, plan=plan)
        assert all(torch.equal(a, b) for a, b in zip(y + d, want_y + want_d)), (rep, "two launches")
        y, d = _fresh(c, g, gpu, y0, R, True)
        dispatch_bgmv_qkv_lora(*y[:3], *d[:3], g.x, g.key, g.value, *t, g.scales, plan=plan)
        dispatch_bgmv_lora(y[3], d[3], g.x, g.key, g.value, *t, 3, g.scales, plan=plan)
        assert all(torch.equal(a, b) for a, b in zip(y + d, want_y + want_d)), (rep, "one call")
    # items behind the grid have been taken, and counted, by workgroups on their second turn
    counted = [_launches_counted(plan, batch, R, first=grid, proj=p) > 0 for p in (slice(0, 3), slice(3, 4))]
    assert counted == [qkv, o] and plan.status() == 0


def test_one_plan_takes_deltas_of_different_widths(gpu):
    """Narrow and wide deltas in turn on one plan, each right and none late: a launch that skips the rows behind a narrow
    delta must not leave readers of a later one waiting for them."""
    import slora_hip
    from slora_hip import dispatch_bgmv, dispatch_bgmv_lora, dispatch_bgmv_qkv_lora
    c = make_case(21, 4096, [64, 32, 8, 64], 9, dtype="f16", zipf_alpha=1.0)
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    y0 = _outputs(c, g, gpu, True)
    want = {}
    for R in (16, 64):
        y, d = _fresh(c, g, gpu, y0, R, True)
        for p in range(4):
            dispatch_bgmv(d[p], g.x, g.key, *t, p, g.scales, plan=False)
            dispatch_bgmv(y[p], d[p], g.value, *t, p, g.scales, plan=False)
        want[R] = (y, d)
    plan = slora_hip.make_plan(*t, 64, c.n_pages)
    for i, R in enumerate((64, 16, 64, 16, 16, 64)):
        y, d = _fresh(c, g, gpu, y0, R, True)
        dispatch_bgmv_qkv_lora(*y[:3], *d[:3], g.x, g.key, g.value, *t, g.scales, plan=plan)
        dispatch_bgmv_lora(y[3], d[3], g.x, g.key, g.value, *t, 3, g.scales, plan=plan)
        for p in range(4):
            assert torch.equal(d[p], want[R][1][p]) and torch.equal(y[p], want[R][0][p]), (i, R, p)
        assert plan.status() == 0, (i, R)


@pytest.mark.parametrize("shift", [0, 1])
def test_outputs_that_share_memory_with_the_activations(gpu, shift):
    """The o projection added in place to its own activations, and k written over those of q, k and v (whole, and one row
    further down): every row of x is read before the first output is written, as with two calls."""
    import slora_hip
    from slora_hip import (dispatch_bgmv, dispatch_bgmv_lora, dispatch_bgmv_qkv_expand, dispatch_bgmv_qkv_lora,
                           dispatch_bgmv_qkv_shrink)
    c = make_case(33, 4096, [8, 16, 8], 40, dtype="bf16", zipf_alpha=1.0)
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    plan = slora_hip.make_plan(*t, 16, c.n_pages)

    def tensors():
        rows = torch.zeros((c.batch + shift, 4096), dtype=g.tdt, device=gpu)
        rows[:c.batch].copy_(g.x)
        y, d = _fresh(c, g, gpu, _outputs(c, g, gpu, True), 16, True)
        return rows[:c.batch], rows[shift:], y, d

    x, over, y, d = tensors()
    dispatch_bgmv_qkv_shrink(*d[:3], x, g.key, *t, plan=False)
    dispatch_bgmv_qkv_expand(y[0], over, y[2], *d[:3], g.value, *t, g.scales, plan=False)
    want = [over.clone(), y[0], y[2], *d[:3]]
    x, over, y, d = tensors()
    dispatch_bgmv_qkv_lora(y[0], over, y[2], *d[:3], x, g.key, g.value, *t, g.scales, plan=plan)
    assert all(torch.equal(a, b) for a, b in zip([over, y[0], y[2], *d[:3]], want))
    x, over, y, d = tensors()
    dispatch_bgmv(d[3], x, g.key, *t, 3, g.scales, plan=False)
    dispatch_bgmv(over, d[3], g.value, *t, 3, g.scales, plan=False)
    want = [over.clone(), d[3]]
    x, over, y, d = tensors()
    dispatch_bgmv_lora(over, d[3], x, g.key, g.value, *t, 3, g.scales, plan=plan)
    assert torch.equal(over, want[0]) and torch.equal(d[3], want[1])
    # (the calls above had to take two launches to be right; others on this plan take one)
    assert _launches_counted(plan, c.batch, 16) == 0
    dispatch_bgmv_lora(y[3], d[3], x, g.key, g.value, *t, 3, g.scales, plan=plan)
    assert _launches_counted(plan, c.batch, 16) > 0 and plan.status() == 0


@pytest.mark.parametrize("hidden,kv,ranks,batch,R,counted,qkv,o", [
    (4096, 4096, [8], 1, 64, True, True, True),                     # 8 items
    (4096, 4096, [64], 1, 64, True, False, True),                   # 8 items of one queue: 64
    (4096, 4096, [64, 32, 64, 32], 23, 64, True, False, True),      # forty to 256 items
    (4096, 4096, [64, 64, 64], 160, 64, True, False, False),        # more than 256
    (4096, 4096, [64, 32, 16, 8], 4, 64, False, True, True),        # not counted: what the capacity can hold decides
    (4096, 4096, [64, 32, 16, 8], 6, 64, False, False, True),
    (4096, 4096, [8], 23, 64, False, False, True),
    (4096, 4096, [8], 33, 64, False, False, False),
    (4096, 4096, [16, 8], 150, 16, False, True, True),              # 3 * 328 shrink workgroups
    (4096, 4096, [16, 8], 160, 16, False, False, True),             # 3 * 344
    (4096, 1024, [64, 32, 16, 8], 23, 64, False, True, True),       # narrow k and v
    (4096, 2048, [64, 32, 16, 8], 23, 64, False, False, True),
    (8192, 8192, [16, 8], 64, 16, False, True, True),               # 3 * 152
    (8192, 8192, [16, 8], 80, 16, False, False, True),              # 3 * 184
])
def test_one_launch_or_two(gpu, hidden, kv, ranks, batch, R, counted, qkv, o):
    """On both sides of the lines between one launch and two, with the item count and without: which one a call took, and
    the bits of the calls without a plan."""
    import slora_hip
    from slora_hip import dispatch_bgmv, dispatch_bgmv_lora, dispatch_bgmv_qkv_lora
    c = make_case(600 + batch + R, hidden, ranks, batch, dtype="f16", h_out=[hidden, kv, kv, hidden])
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    y0 = _outputs(c, g, gpu, True)
    want_y, want_d = _fresh(c, g, gpu, y0, R, True)
    for p in range(4):
        dispatch_bgmv(want_d[p], g.x, g.key, *t, p, g.scales, plan=False)
        dispatch_bgmv(want_y[p], want_d[p], g.value, *t, p, g.scales, plan=False)
    plan = slora_hip.make_plan(*t, R, c.n_pages, readback=counted)
    y, d = _fresh(c, g, gpu, y0, R, True)
    dispatch_bgmv_qkv_lora(*y[:3], *d[:3], g.x, g.key, g.value, *t, g.scales, plan=plan)
    dispatch_bgmv_lora(y[3], d[3], g.x, g.key, g.value, *t, 3, g.scales, plan=plan)
    assert all(torch.equal(a, b) for a, b in zip(y + d, want_y + want_d))
    got = [_launches_counted(plan, batch, R, proj=p) > 0 for p in (slice(0, 3), slice(3, 4))]
    assert got == [qkv, o] and plan.status() == 0, (got, plan.n_items)


def test_launch_numbers_wrap(gpu):
    """Launches are numbered in 16 bits: the four around the wrap, each on activations of its own, take no row of another."""
    import slora_hip
    from slora_hip import dispatch_bgmv, dispatch_bgmv_lora
    c = make_case(44, 4096, [16, 12, 8], 11, dtype="f16")
    g = GpuCase(c, gpu)
    t = (g.a_start, g.a_len, g.a_loc, g.bins)
    plan = slora_hip.make_plan(*t, 16, c.n_pages)
    area, items = _hand_over_area(c.batch, 16)
    plan.buf[area:area + 16 * items] = 65533
    y0 = _outputs(c, g, gpu, True)
    for rep in range(5):
        x = torch.roll(g.x, rep, 1)
        want_y, want_d = _fresh(c, g, gpu, y0, 16, True)
        dispatch_bgmv(want_d[3], x, g.key, *t, 3, g.scales, plan=False)
        dispatch_bgmv(want_y[3], want_d[3], g.value, *t, 3, g.scales, plan=False)
        y, d = _fresh(c, g, gpu, y0, 16, True)
        dispatch_bgmv_lora(y[3], d[3], x, g.key, g.value, *t, 3, g.scales, plan=plan)
        assert torch.equal(y[3], want_y[3]) and torch.equal(d[3], want_d[3]), rep
    assert plan.status() == 0 and int(plan.buf[area:area + 16 * items].max()) == 65538
