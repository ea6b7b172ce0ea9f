"""What the experts' kernels of few-row steps do on their way, against the kernels of its own that each replaces: the
pairs' order from the router's launch, the gate inside the first product, a shared expert's gate inside the sum."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,E,top,groups,keep", [(1, 8, 1, 1, 1), (3, 32, 4, 4, 2), (16, 32, 4, 1, 1), (16, 65, 7, 5, 3),
                                                 (5, 256, 8, 8, 4), (16, 128, 64, 1, 1)])
@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
def test_order_from_the_routers_launch(n, E, top, groups, keep, scoring):
    from gpt_fast_amd.ops import routed_experts as RE
    torch.manual_seed(n * 1000 + E)
    z = torch.randn(n, E + 3, device=DEV)[:, :E + 1]
    correction = torch.randn(E, device=DEV) * 0.1
    args = dict(scoring=scoring, correction=correction, group_top=2)
    assert RE.orders_with_route(n, E, groups)
    want_c, want_w = RE.route(z, E, top, groups, keep, 1e-20, **args)
    chosen, weights, (offsets, order, place) = RE.route(z, E, top, groups, keep, 1e-20, ordered=True, **args)
    assert torch.equal(chosen, want_c) and torch.equal(weights, want_w)
    counts = torch.bincount(chosen.flatten().long(), minlength=E)
    assert offsets.tolist() == [0] + counts.cumsum(0).tolist()
    # every pair once, among its expert's places; the order inside an expert is free
    assert sorted(order.tolist()) == list(range(n * top))
    assert torch.equal(place[order.long()], torch.arange(n * top, dtype=torch.int32, device=DEV))
    experts = chosen.flatten()[order.long()]
    assert torch.equal(experts, experts.sort().values)


def test_what_does_not_fit_one_workgroup_is_refused():
    from gpt_fast_amd.ops import routed_experts as RE
    from gpt_fast_amd.ops.library import KernelError
    assert not RE.orders_with_route(17, 8, 1) and not RE.orders_with_route(16, 1024, 1)
    with pytest.raises(KernelError):
        RE.route(torch.zeros(17, 8, device=DEV), 8, 2, 1, 1, 0.0, ordered=True)


@pytest.mark.parametrize("activation,limit", [("silu", None), ("gelu_tanh", None), ("clamped_swish", 1.5)])
@pytest.mark.parametrize("n,E,top,F,K", [(1, 4, 2, 8, 64), (2, 6, 2, 40, 136), (7, 3, 2, 100, 520), (16, 5, 3, 72, 1032),
                                         (30, 4, 2, 64, 256), (60, 3, 1, 136, 264)])
def test_gate_inside_the_grouped_product(n, E, top, F, K, activation, limit):
    from gpt_fast_amd.ops import kernels, routed_experts as RE
    torch.manual_seed(n * 100 + F)
    x = torch.randn(n, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, 2 * F, K, device=DEV) * K ** -0.5).to(torch.bfloat16)
    chosen = torch.stack([torch.randperm(E)[:top] for _ in range(n)]).to(torch.int32).to(DEV)
    offsets, order, _ = RE.expert_order(chosen, E)
    sums = RE.grouped_rows(x, order, top, w, offsets, None, n)
    want = kernels.gate_mul_sums(sums, activation, limit)
    got = RE.grouped_rows(x, order, top, w, offsets, activation, n, True, limit)
    assert got.shape == want.shape and got.dtype == torch.bfloat16
    # the same sums at these sizes, and the gate's own arithmetic in either kernel, one rounding apart: now and then the
    # neighbouring bfloat16 (2^-8)
    assert rel_err(got, want) <= 2.0 ** -8


def _pairs(n, E, top, K, N, seed):
    torch.manual_seed(seed)
    x = torch.randn(n, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, N, K, device=DEV) * K ** -0.5).to(torch.bfloat16)
    return x, w, torch.stack([torch.randperm(E)[:top] for _ in range(n)]).to(torch.int32).to(DEV)


# up to 16 rows a wave takes a quarter of K in pieces of 128: quarters without, with unequal and with cut pieces, one
# piece ahead and two (which of them by the workgroups that a unit gets: few columns and many).  More rows: K whose
# pieces are walked from the workgroup's own place on (multiples of 2,048), several of these, and others.
WALKS = [(1, 3, 2, 40, 1032), (2, 8, 4, 24, 136), (4, 24, 4, 1024, 3584), (5, 4, 2, 24, 4096), (9, 16, 6, 2048, 640),
         (16, 5, 3, 72, 4104), (17, 5, 3, 328, 2048), (30, 6, 2, 200, 4096), (33, 6, 2, 136, 2056), (60, 4, 3, 520, 6144)]


@pytest.mark.parametrize("n,E,top,F,K", WALKS)
def test_grouped_product_from_every_place_of_the_walk(n, E, top, F, K):
    from gpt_fast_amd.ops import routed_experts as RE
    x, w, chosen = _pairs(n, E, top, K, 2 * F, n + K)
    offsets, order, _ = RE.expert_order(chosen, E)
    sums = RE.grouped_rows(x, order, top, w, offsets, None, n).double()
    gated = RE.grouped_rows(x, order, top, w, offsets, "silu", n, True)
    for e in range(E):
        a, b = int(offsets[e]), int(offsets[e + 1])
        xs = x[(order[a:b] // top).long()].double()
        want, size = xs @ w[e].double().t(), xs.abs() @ w[e].double().abs().t()
        # K / 32 matrix instructions one after the other, of 32 products each: as many float32 roundings of at most the
        # sum of the products' sizes, and four partial sums
        assert ((sums[a:b] - want).abs() <= (K / 32 + 36) * 2.0 ** -23 * size).all(), e
        if b > a:                                        # one rounding to bfloat16 more
            assert rel_err(gated[a:b], torch.nn.functional.silu(want[:, :F]) * want[:, F:]) < 2.0 ** -8, e


@pytest.mark.parametrize("counts", [(16, 1, 3, 4, 9), (60, 17, 32, 33)])
@pytest.mark.parametrize("K", [1032, 4096])
def test_a_pairs_sums_are_the_same_among_steps_of_one_form(counts, K):
    """Up to 16 rows, and more: whatever else the step holds."""
    from gpt_fast_amd.ops import routed_experts as RE
    E, top, N = 6, 2, 200
    x, w, chosen = _pairs(counts[0], E, top, K, N, K)
    rows = []
    for n in counts:
        offsets, order, place = RE.expert_order(chosen[:n], E)
        rows.append(RE.grouped_rows(x[:n], order, top, w, offsets, None, n)[place.long()])
        assert torch.equal(rows[-1], rows[0][:n * top]), n


@pytest.mark.parametrize("n,top,D,dtype", [(1, 1, 8, torch.float32), (3, 4, 136, torch.bfloat16), (16, 2, 100, torch.float32),
                                           (1100, 3, 264, torch.bfloat16)])
def test_sum_of_the_pairs_with_a_gate_on_what_is_there(n, top, D, dtype):
    from gpt_fast_amd.ops import kernels, routed_experts as RE
    torch.manual_seed(n + D)
    ys = torch.randn(n * top, D, device=DEV).to(dtype)
    place = torch.randperm(n * top, device=DEV).to(torch.int32)
    weights = torch.rand(n, top, device=DEV)
    gate = torch.randn(n, 5, device=DEV)[:, 2:]
    start = torch.randn(n, D, device=DEV)
    want = start.double() * torch.sigmoid(gate[:, :1].double()) + \
        (ys.double()[place.long()].view(n, top, D) * weights.double()[:, :, None]).sum(1)
    got = RE.combine_pairs(ys, place, weights, out=start.clone(), gate=gate)
    assert rel_err(got, want) < 1e-6                     # top + 2 float32 roundings of 6e-8 each
    scaled = start.clone()
    kernels.scale_rows_sigmoid(scaled, gate)
    assert rel_err(RE.combine_pairs(ys, place, weights, out=scaled), want) < 1e-6


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("rows", [[1, 64, 65, 0, 128], [129, 192, 193, 255], [256, 257, 300], [513, 0, 2, 1030]])
def test_tall_tiles_of_every_height(rows, gated, monkeypatch):
    """Tiles of 64, 128, 192 and 256 rows: an expert's rows in equal parts, remainders on either side of a step."""
    from gpt_fast_amd.ops import routed_experts as RE
    monkeypatch.setattr(RE, "tall_tiles_win", lambda *a: True)
    torch.manual_seed(sum(rows))
    E, F, K, n = len(rows), 328, 192, sum(rows)
    x = torch.randn(n, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, (2 if gated else 1) * F, K, device=DEV) * K ** -0.5).to(torch.bfloat16)
    offsets = torch.tensor([0] + list(torch.tensor(rows).cumsum(0)), dtype=torch.int32, device=DEV)
    order = torch.randperm(n, device=DEV).to(torch.int32)
    got = RE.expert_tile_product(x, order, 1, w, offsets, None, n, "silu" if gated else None, gated)
    assert got.shape == (n, F)
    for e in range(E):
        a, b = int(offsets[e]), int(offsets[e + 1])
        if a == b:
            continue
        want = x[order[a:b].long()].double() @ w[e].double().t()
        if gated:
            want = torch.nn.functional.silu(want[:, :F]) * want[:, F:]
        # one rounding to bfloat16 (2^-9 of a value) and float32 sums
        assert rel_err(got[a:b], want) < 2.0 ** -8, (e, rows[e])
