"""Each new mechanism's kernels alone against the plain functions of ``plain_fezupel``, in
32-bit and in bfloat16: norms that store or add, embedding plus position row, the router, the
experts, and the attention whose values are its keys (keys spread over shuffled pages; windows
of one token, less than a page, a page, more; with and without the silent soft-max term and
the gate; a key that would dominate planted just inside and just outside the window)."""
import math

import pytest
import torch

import plain_fezupel as P
from gpu_util import DEV, rel_err, tol
from zinfer_amd import ops

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


def _rand(shape, seed, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


# ------------------------------------------------------------------------------ norms
@pytest.mark.parametrize("T, W", [(1, 48), (5, 77), (33, 336), (3, 4096), (2, 9000)])
@pytest.mark.parametrize("centred, bias", [(True, True), (True, False), (False, True)])
def test_norm_rows_store_and_add(T, W, centred, bias):
    x = _rand((T, W), 1, 3.0) + 1.5
    w = 1 + _rand((W,), 2, 0.2)
    b = _rand((W,), 3, 0.5) if bias else None
    eps = 1e-5
    if centred:
        ref = P.layer_norm(x, w, b if bias else torch.zeros(W), eps)
    else:
        x64 = x.double()
        ref = x64 / torch.sqrt((x64 * x64).mean(-1, keepdim=True) + eps) * w.double() \
            + (b.double() if bias else 0.0)
    xd, wd = x.to(DEV), w.to(DEV)
    bd = b.to(DEV) if bias else None
    for dt in DTYPES:
        out = torch.empty((T, W), dtype=dt, device=DEV)
        ops.norm_rows(xd, wd, bd, eps, out, centred)
        assert rel_err(out, ref) < tol(dt)
    base = _rand((T, W), 4)
    acc = base.to(DEV)
    ops.norm_rows(xd, wd, bd, eps, acc, centred, add=True)
    assert rel_err(acc, base.double() + ref) < tol(torch.float32)


@pytest.mark.parametrize("T, W", [(1, 48), (7, 336), (3, 4096), (2, 8192)])
@pytest.mark.parametrize("dt", DTYPES)
def test_norm_add_norm_is_the_two_norms_one_after_the_other(T, W, dt):
    y, x = _rand((T, W), 81, 2.0) + 0.5, _rand((T, W), 82)
    wa, ba = 1 + _rand((W,), 83, 0.2), _rand((W,), 84, 0.5)
    wb, bb = 1 + _rand((W,), 85, 0.2), _rand((W,), 86, 0.5)
    dev = lambda t: t.to(DEV)
    x1, out1 = dev(x), torch.empty((T, W), dtype=dt, device=DEV)
    ops.norm_add_norm(dev(y), dev(wa), dev(ba), 1e-5, True, x1, dev(wb), dev(bb), 1e-6, True, out1)
    x2, out2 = dev(x), torch.empty((T, W), dtype=dt, device=DEV)
    ops.norm_rows(dev(y), dev(wa), dev(ba), 1e-5, x2, True, add=True)
    ops.norm_rows(x2, dev(wb), dev(bb), 1e-6, out2, True)
    assert rel_err(x1, x2) < 1e-6 and rel_err(out1, out2.double()) < (1e-6 if dt == torch.float32 else 2.0 ** -8)
    ref_x = x.double() + P.layer_norm(y, wa, ba, 1e-5)
    assert rel_err(x1, ref_x) < 2e-5
    assert rel_err(out1, P.layer_norm(ref_x, wb, bb, 1e-6)) < tol(dt)


def test_layer_norm_of_a_row_with_a_large_mean():
    """The variance comes from the deviations: a mean a thousand times the spread leaves it."""
    x = 1000.0 + _rand((4, 256), 5, 1.0)
    ref = P.layer_norm(x, torch.ones(256), torch.zeros(256), 1e-6)
    out = torch.empty((4, 256), dtype=torch.float32, device=DEV)
    ops.norm_rows(x.to(DEV), torch.ones(256, device=DEV), None, 1e-6, out, True)
    assert float((out.cpu().double() - ref).abs().max()) < 1e-3


@pytest.mark.parametrize("dt", DTYPES)
def test_embed_position(dt):
    E, Pt = _rand((50, 72), 6, dtype=dt), _rand((40, 72), 7, dtype=dt)
    ids = torch.tensor([3, 49, 0, 3], dtype=torch.int32)
    pos = torch.tensor([0, 39, 17, 1], dtype=torch.int32)
    out = torch.empty((4, 72), dtype=torch.float32, device=DEV)
    ops.embed_position(E.to(DEV), ids.to(DEV), Pt.to(DEV), pos.to(DEV), out)
    ref = E.double()[ids.long()] + Pt.double()[pos.long()]
    assert rel_err(out, ref) < 1e-6


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("H,off", [(2048, 0), (8, 0), (50, 0), (2056, 1), (4104, 0)])
def test_embed_position_in_wide_loads_and_in_copies(H, off, dt):
    """Rows whose width or place keeps 8 columns a thread out, and every copy of a stream kept several times:
    the same bits everywhere."""
    E, Pt = _rand((9, H), 6, dtype=dt), _rand((7, H), 7, dtype=dt)
    ids, pos = torch.tensor([8, 0, 3], dtype=torch.int32), torch.tensor([6, 0, 5], dtype=torch.int32)
    flat = torch.empty((9 * H + off,), dtype=dt, device=DEV)
    table = flat[off:].view(9, H)
    table.copy_(E)
    out = torch.full((4, 3, H), float("nan"), device=DEV)
    ops.embed_position(table, ids.to(DEV), Pt.to(DEV), pos.to(DEV), out, 1.5)
    one = torch.full((3, H), float("nan"), device=DEV)
    ops.embed_position(table, ids.to(DEV), Pt.to(DEV), pos.to(DEV), one, 1.5)
    ref = E.double()[ids.long()] * 1.5 + Pt.double()[pos.long()]
    assert rel_err(one, ref) < 1e-6
    assert all(torch.equal(out[c], one) for c in range(4))


# ------------------------------------------------------------------------------ experts
@pytest.mark.parametrize("T, W, E, top", [(7, 48, 6, 2), (3, 50, 1, 1), (5, 72, 9, 9),
                                           (4, 64, 130, 70), (2, 384, 12, 5)])
@pytest.mark.parametrize("dt", DTYPES)
def test_router(T, W, E, top, dt):
    h = _rand((T, W), 8, dtype=dt)
    R = _rand((E, W), 9, 0.5).to(torch.bfloat16).float()
    b = _rand((E,), 10, 0.5)
    ids = torch.empty((T, top), dtype=torch.int32, device=DEV)
    wts = torch.empty((T, top), dtype=torch.float32, device=DEV)
    ops.moe_route(h.to(DEV), R.to(DEV), b.to(DEV), ids, wts)
    ref_ids, ref_w = P.route(h, R, b, top)
    assert torch.equal(ids.cpu().long(), ref_ids)       # in the order of their logits
    assert rel_err(wts, ref_w) < 1e-5
    assert torch.allclose(wts.sum(-1).cpu(), torch.ones(T), atol=1e-5)


def test_router_bias_decides():
    h = torch.zeros((1, 16))
    b = torch.tensor([0.0, 3.0, -1.0, 2.0])
    ids = torch.empty((1, 2), dtype=torch.int32, device=DEV)
    wts = torch.empty((1, 2), dtype=torch.float32, device=DEV)
    ops.moe_route(h.to(DEV), torch.zeros((4, 16), device=DEV), b.to(DEV), ids, wts)
    assert ids.cpu().tolist() == [[1, 3]]
    e = math.exp(-1.0)
    assert torch.allclose(wts.cpu(), torch.tensor([[1 / (1 + e), e / (1 + e)]]), atol=1e-6)


@pytest.mark.parametrize("T, W, ff, E, top", [(6, 48, 20, 6, 2), (3, 50, 30, 1, 1),
                                               (9, 72, 17, 5, 5), (4, 128, 64, 8, 3)])
@pytest.mark.parametrize("dt", DTYPES)
def test_experts(T, W, ff, E, top, dt):
    limit, alpha, shift = 0.5, 1.702, 1.0
    h = _rand((T, W), 11, dtype=dt)
    w = {}
    for e in range(E):
        w[f"e{e}.gate"] = _rand((ff, W), 20 + e, 2 / W ** 0.5, dt)
        w[f"e{e}.up"] = _rand((ff, W), 40 + e, 2 / W ** 0.5, dt)
        w[f"e{e}.down"] = _rand((W, ff), 60 + e, 2 / ff ** 0.5, dt)
    g = torch.Generator().manual_seed(12)
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32)
    share = torch.rand((T, top), generator=g)
    gate_up = torch.stack([torch.cat([w[f"e{e}.gate"], w[f"e{e}.up"]]) for e in range(E)]).to(DEV)
    down = torch.stack([w[f"e{e}.down"] for e in range(E)]).to(DEV)
    y = torch.empty((T, top, ff), dtype=dt, device=DEV)
    ops.moe_gate_up(h.to(DEV), gate_up, ids.to(DEV), y, limit, alpha, shift)
    base = _rand((T, W), 13)
    for add in (False, True):
        out = base.to(DEV)
        ops.moe_down(y, down, ids.to(DEV), share.to(DEV), out, add=add)
        ref = base.double() if add else torch.zeros((T, W), dtype=torch.float64)
        for t in range(T):
            for s in range(top):
                ref[t] += share[t, s].double() * P.clamped_expert(h[t:t + 1], w, f"e{int(ids[t, s])}.", limit)[0]
        assert rel_err(out, ref) < (2e-5 if dt == torch.float32 else 2e-2)
    # the limits bite: some products lie beyond them
    gates = h.double() @ w["e0.gate"].double().T
    assert float(gates.max()) > limit


@pytest.mark.parametrize("T, W, ff, E, top", [(1, 64, 64, 3, 2), (16, 128, 192, 5, 4),
                                               (7, 320, 64, 40, 6), (16, 64, 576, 2, 16),
                                               (9, 64, 1088, 1, 3)])
@pytest.mark.parametrize("kind", ["gated", "plain", "shared", "shared gate"])
def test_experts_of_a_few_tokens_against_plain(T, W, ff, E, top, kind):
    """bfloat16, up to 16 tokens: every used expert once for all its pairs.  Ids name experts,
    some of them twice a token (up to 3 units of 16 pairs an expert) and some none; with an expert
    that all tokens share; a token's result is the same bits alone."""
    dt = torch.bfloat16
    limit, alpha, shift, sff = 0.6, 1.702, 1.0, 128
    plain, shared = kind == "plain", kind.startswith("shared")
    h = _rand((T, W), 14, dtype=dt)
    gate_up = _rand((E, ff if plain else 2 * ff, W), 15, 2 / W ** 0.5, dt)
    down = _rand((E, W, ff), 16, 2 / ff ** 0.5, dt)
    s_gu, s_down = _rand((2 * sff, W), 17, 2 / W ** 0.5, dt), _rand((W, sff), 18, 2 / sff ** 0.5, dt)
    g = torch.Generator().manual_seed(19)
    ids = torch.randint(0, E + 1, (T, top), generator=g).to(torch.int32)      # E: no expert
    share = torch.rand((T, top), generator=g)
    factor = torch.rand((T, 2), generator=g) if kind == "shared gate" else None
    base = _rand((T, W), 20)
    act = "relu2" if plain else None
    tiled = [torch.stack([ops.pretile_weight(m) for m in w.to(DEV)]) for w in (gate_up, down)]
    assert ops.moe_few_covers(h.to(DEV), top) and ops.moe_can_pretile(*tiled)

    def run(rows, add):
        n = len(rows)
        y = torch.full((n, top, ff), float("nan"), dtype=dt, device=DEV)
        ys = torch.full((n, sff), float("nan"), dtype=dt, device=DEV)
        out = base[rows].to(DEV)
        f = None if factor is None else factor[rows].to(DEV)[:, 1]
        more = (ops.pretile_weight(s_gu.to(DEV)), ops.pretile_weight(s_down.to(DEV)), ys, 0.7,
                1.0, 0.0, f) if shared else None
        ops.moe_experts(h[rows].contiguous().to(DEV), *tiled, ids[rows].contiguous().to(DEV),
                        share[rows].contiguous().to(DEV), y, out, limit, alpha, shift, add=add,
                        act=act, n_identity=1, w_tiled=True, shared=more)
        return out

    def unit(z, lim, a, b, ff):
        gate, up = torch.clamp(z[:ff], max=lim), torch.clamp(z[ff:], -lim, lim)
        return gate * torch.sigmoid(a * gate) * (up + b)

    want = torch.zeros((T, W), dtype=torch.float64)
    for t in range(T):
        x = h[t].double()
        for s_ in range(top):
            e, c = int(ids[t, s_]), share[t, s_].double()
            if e == E:
                want[t] += c * x
                continue
            z = gate_up[e].double() @ x
            z = torch.clamp(z, min=0.0) ** 2 if plain else unit(z, limit, alpha, shift, ff)
            want[t] += c * (down[e].double() @ z.to(dt).double())
        if shared:
            z = unit(s_gu.double() @ x, 0.7, 1.0, 0.0, sff)
            z = z * (1.0 if factor is None else factor[t, 1].double())
            want[t] += s_down.double() @ z.to(dt).double()
    everyone = list(range(T))
    # (the activations round to bfloat16 from sums of another order: half a last place of each)
    got = run(everyone, False)
    assert rel_err(got, want) < 1e-2
    assert rel_err(run(everyone, True), want + base.double()) < 1e-2
    for t in (0, T - 1):
        assert torch.equal(run([t], False)[0], got[t])
    if not shared:
        # more tokens, sorted by expert: the same bits from pre-tiled matrices as from rows
        many = [t % T for t in range(40)]
        outs = []
        for w_tiled, (gu, dn) in ((True, tiled), (False, (gate_up.to(DEV), down.to(DEV)))):
            y = torch.empty((40, top, ff), dtype=dt, device=DEV)
            outs.append(torch.empty((40, W), device=DEV))
            ops.moe_experts(h[many].to(DEV), gu, dn, ids[many].to(DEV), share[many].to(DEV), y,
                            outs[-1], limit, alpha, shift, act=act, n_identity=1, w_tiled=w_tiled)
        assert torch.equal(*outs) and rel_err(outs[0][:T], want) < 1e-2


@pytest.mark.parametrize("E, top, extra", [(5, 5, 0), (31, 4, 2), (64, 6, 1), (128, 9, 0), (129, 9, 0)])
@pytest.mark.parametrize("T", [1, 16, 35])
@pytest.mark.parametrize("scoring", ["softmax", "sigmoid", "softmax_all"])
def test_router_ties_and_what_cannot_be_chosen(E, top, extra, T, scoring):
    """Equal logits go to the lower index, NaN and -inf are never chosen (expert 0 stands in),
    around the number of rows where the kernel changes, at an odd width."""
    W, extra = 33, 0 if scoring == "softmax" else extra
    g = torch.Generator().manual_seed(3)
    h = torch.zeros((T, W))
    h[:, 0] = 1.0
    router = torch.zeros((E + extra, W))
    router[:, 0] = torch.randint(-2, 3, (E + extra,), generator=g).float()
    router[min(3, E - 1), 0] = float("nan")
    if scoring == "softmax":
        router[min(4, E - 1), 0] = -float("inf")
    ids = torch.empty((T, top), dtype=torch.int32, device=DEV)
    wts = torch.empty((T, top), dtype=torch.float32, device=DEV)
    more = torch.empty((T, extra), device=DEV) if extra else None
    correction = None
    if scoring != "softmax":
        # (a soft-max over all with a NaN among them is NaN: bring it in behind the scores)
        router[min(3, E - 1), 0] = 1.0
        correction = torch.zeros(E)
        correction[min(3, E - 1)] = float("nan")
        correction[min(4, E - 1)] = -float("inf")
    ops.moe_route(h.to(DEV), router.to(DEV), None, ids, wts, scoring=scoring, extra=more,
                  correction=None if correction is None else correction.to(DEV), normalize=True)
    z = router[:E, 0].double()
    s = z if scoring == "softmax" else torch.sigmoid(z) if scoring == "sigmoid" else torch.softmax(z, 0)
    choice = s if correction is None else s + correction.double()
    order = sorted((e for e in range(E) if float(choice[e]) > -float("inf")),
                   key=lambda e: (-float(choice[e]), e))[:top]
    stand_in = [0] * (top - len(order))
    assert ids.cpu().tolist() == [order + stand_in] * T
    if scoring == "softmax":
        w = torch.cat([torch.softmax(s[order], 0), torch.zeros(len(stand_in), dtype=torch.float64)])
    else:
        w = s[order + stand_in]
        w = w / (w.sum() + 1e-20)
    assert torch.allclose(wts.cpu().double(), w.expand(T, top), atol=1e-6)
    if extra:
        assert torch.allclose(more.cpu(), torch.sigmoid(router[E:, 0]).expand(T, extra), atol=1e-6)


@pytest.mark.parametrize("T, W, E, extra", [(1, 2048, 32, 0), (16, 2048, 32, 1), (17, 100, 128, 0),
                                            (64, 4104, 96, 3), (65, 64, 5, 0)])
def test_router_over_workgroups_gives_the_same_bits(T, W, E, extra):
    """With work space of its own a router of up to 64 tokens is spread over workgroups; used again
    and again the space serves other sizes too."""
    work, got = ops.moe_route_work(DEV), []
    h, router = _rand((T, W), 1).to(DEV), _rand((E + extra, W), 2, W ** -0.5).to(DEV)
    for w in (None, work, work):
        ids = torch.empty((T, 4), dtype=torch.int32, device=DEV)
        wts = torch.empty((T, 4), dtype=torch.float32, device=DEV)
        more = torch.empty((T, extra), device=DEV) if extra else None
        ops.moe_route(h, router, None, ids, wts, scoring="sigmoid", extra=more, work=w)
        got.append((ids, wts.view(torch.int32), more if extra else ids))
    assert all(torch.equal(x, y) for other in got[1:] for x, y in zip(got[0], other))
    assert not work[-4:].any()
    with pytest.raises(ops.KernelUnavailable):
        ops.moe_route(h, router, None, ids, wts, scoring="sigmoid", extra=more, work=work[:-4])


@pytest.mark.parametrize("W, T, dt", [(512, 1040, torch.bfloat16), (1024, 64, torch.float32),
                                      (1100, 64, torch.float32), (2048, 64, torch.float32),
                                      (2048, 16, torch.bfloat16), (4096, 64, torch.float32)])
def test_router_logits_are_as_close_as_those_of_more_rows(W, T, dt):
    """The sums of up to 128 router rows against the kernel that takes more of them (a wave a row, a
    tree over its lanes), on rows whose exact logits are 0: no further off in the mean."""
    E = 60
    g = torch.Generator().manual_seed(W)
    mix = torch.randperm(W, generator=g)
    x, r = 64 * torch.randn((T, W // 2), generator=g), 64 * torch.randn((E + 69, W // 2), generator=g)
    h = torch.cat([x, x], 1)[:, mix].to(dt).to(DEV)
    router = torch.cat([r, -r], 1)[:, mix].contiguous().to(DEV)
    off = []
    for extra in (0, 69):                  # (69 more rows: 129, the other kernel)
        ids = torch.empty((T, E), dtype=torch.int32, device=DEV)
        wts = torch.empty((T, E), dtype=torch.float32, device=DEV)
        more = torch.empty((T, extra), device=DEV) if extra else None
        ops.moe_route(h, router[:E + extra].contiguous(), None, ids, wts, scoring="sigmoid",
                      normalize=False, extra=more, work=ops.moe_route_work(DEV))
        z = torch.logit(wts.cpu().double())
        off.append(float((z ** 2).mean().sqrt()))
    # (960 sums and more: their root mean square is known to about 2 %)
    assert off[0] <= 1.04 * off[1], f"root mean square off: {off[0]:.3e}, {off[1]:.3e}"


@pytest.mark.parametrize("T, W, E", [(64, 2048, 8), (65, 2048, 8), (256, 1024, 32), (257, 1024, 32),
                                     (16, 1023, 40), (512, 3072, 20), (513, 3072, 20),
                                     (1024, 2048, 128), (1025, 520, 128), (1030, 504, 65)])
@pytest.mark.parametrize("dt", DTYPES)
def test_router_where_the_kernel_changes(T, W, E, dt):
    """On both sides of every line at which the router's kernel changes, against 64-bit: the chosen
    and their weights, twice on the same work space."""
    h, router = _rand((T, W), 5, dtype=dt), _rand((E, W), 6, W ** -0.5)
    z = h.double() @ router.double().T
    work = ops.moe_route_work(DEV)
    for _ in range(2):
        ids = torch.empty((T, E), dtype=torch.int32, device=DEV)
        wts = torch.empty((T, E), dtype=torch.float32, device=DEV)
        ops.moe_route(h.to(DEV), router.to(DEV), None, ids, wts, work=work)
        at = ids.cpu().long()
        assert torch.equal(at.sort(1).values, torch.arange(E).expand(T, E))
        # logits of about 1 formed from W terms in 32-bit: off by a few 2^-24 of their scale
        ordered = z.gather(1, at)
        assert bool((ordered[:, 1:] <= ordered[:, :-1] + 4e-6).all())
        assert torch.allclose(wts.cpu().double(), torch.softmax(ordered, 1), rtol=8e-6, atol=0)
        assert not work[-64:].any()


def test_router_in_float32_does_not_depend_on_the_number_of_tokens():
    """A token's bits with 1, 300 and 1100 tokens beside it, in one workgroup and over several."""
    W, E = 2048, 40
    h, router = _rand((1100, W), 7).to(DEV), _rand((E, W), 8, W ** -0.5).to(DEV)
    got = []
    for T, work in ((1100, None), (1100, ops.moe_route_work(DEV)), (300, ops.moe_route_work(DEV)),
                    (1, ops.moe_route_work(DEV))):
        ids = torch.empty((T, 6), dtype=torch.int32, device=DEV)
        wts = torch.empty((T, 6), dtype=torch.float32, device=DEV)
        ops.moe_route(h[:T], router, None, ids, wts, work=work)
        got.append((T, ids, wts))
    for T, ids, wts in got[1:]:
        assert torch.equal(ids, got[0][1][:T]) and torch.equal(wts, got[0][2][:T])


@pytest.mark.parametrize("T, W", [(16, 64), (256, 256), (1024, 2048)])
def test_router_of_128_rows_takes_no_longer_than_one_of_129(T, W):
    """Where the kernel for sixteen tokens a workgroup is the slower one (narrow rows, some hundred
    tokens; by a third to twice the time) it is not taken."""
    h, router = _rand((T, W), 9, dtype=torch.bfloat16).to(DEV), _rand((129, W), 10, W ** -0.5).to(DEV)
    ids = torch.empty((T, 4), dtype=torch.int32, device=DEV)
    wts = torch.empty((T, 4), dtype=torch.float32, device=DEV)
    work, best = ops.moe_route_work(DEV), []
    for rows in (128, 129):
        r = router[:rows].contiguous()
        ops.moe_route(h, r, None, ids, wts, work=work)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                ops.moe_route(h, r, None, ids, wts, work=work)
        times = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        best.append(min(times))
    assert best[0] <= 1.2 * best[1], f"{best[0] * 50:.1f} us, {best[1] * 50:.1f} us"


@pytest.mark.parametrize("T, W, ff, E, top", [(16, 64, 64, 20, 16), (16, 128, 64, 20, 17),
                                               (9, 64, 128, 64, 32), (1, 64, 64, 300, 257)])
@pytest.mark.parametrize("act", [None, "relu2"])
def test_pre_tiled_experts_of_a_few_tokens_with_many_pairs(T, W, ff, E, top, act):
    """Up to 16 tokens whose pairs are 256 or more: beyond 256 pre-tiled matrices go through the tiles
    sorted by expert.  Against the same matrices row by row."""
    dt = torch.bfloat16
    h = _rand((T, W), 24, dtype=dt).to(DEV)
    gate_up = _rand((E, ff if act else 2 * ff, W), 25, 2 / W ** 0.5, dt).to(DEV)
    down = _rand((E, W, ff), 26, 2 / ff ** 0.5, dt).to(DEV)
    g = torch.Generator().manual_seed(27)
    ids = torch.stack([torch.randperm(E + 1, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    share = (torch.rand((T, top), generator=g) / top).to(DEV)
    tiled = [torch.stack([ops.pretile_weight(m) for m in w]) for w in (gate_up, down)]
    assert (T * top > 256) == (not ops.moe_few_covers(h, top))
    base, outs = _rand((T, W), 28).to(DEV), []
    for w_tiled, (gu, dn) in ((False, (gate_up, down)), (True, tiled)):
        y = torch.empty((T, top, ff), dtype=dt, device=DEV)
        outs.append(base.clone())
        ops.moe_experts(h, gu, dn, ids, share, y, outs[-1], 0.6, 1.702, 1.0, add=True, act=act,
                        n_identity=1, w_tiled=w_tiled)
    # (activations rounded to bfloat16 from sums of another order)
    assert rel_err(outs[1], outs[0]) < 1e-2


@pytest.mark.parametrize("W, ff, top", [(4096, 1024, 8), (1024, 4096, 4)])
def test_experts_of_a_few_tokens_are_as_close_pre_tiled(W, ff, top):
    """Pre-tiled against row by row, both against 64 bits: the outputs from the activations that either
    left, and how many of the activations are not the rounding of the 64-bit ones."""
    E, T, dt = 8, 16, torch.bfloat16
    h = _rand((T, W), 41, dtype=dt).to(DEV)
    gate_up = _rand((E, 2 * ff, W), 42, W ** -0.5, dt).to(DEV)
    down = _rand((E, W, ff), 43, ff ** -0.5, dt).to(DEV)
    g = torch.Generator().manual_seed(44)
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    share = torch.rand((T, top), generator=g).to(DEV)
    tiled = [torch.stack([ops.pretile_weight(m) for m in w]) for w in (gate_up, down)]
    off, other = [], []
    for w_tiled, (gu, dn) in ((False, (gate_up, down)), (True, tiled)):
        y = torch.empty((T, top, ff), dtype=dt, device=DEV)
        out = torch.empty((T, W), device=DEV)
        ops.moe_experts(h, gu, dn, ids, share, y, out, 0.0, 1.0, 0.0, w_tiled=w_tiled)
        want, wrong = torch.zeros((T, W), dtype=torch.float64, device=DEV), 0
        for t in range(T):
            for s_ in range(top):
                e = int(ids[t, s_])
                z = gate_up[e].double() @ h[t].double()
                z = z[:ff] * torch.sigmoid(z[:ff]) * z[ff:]
                wrong += int((z.to(dt) != y[t, s_]).sum())
                want[t] += share[t, s_].double() * (down[e].double() @ y[t, s_].double())
        off.append(float((out.double() - want).norm() / want.norm()))
        other.append(wrong)
    # (16384 outputs and more; some 20 of 131072 activations lie that close to a tie)
    assert off[1] <= 1.04 * off[0], off
    assert other[1] <= 1.5 * other[0] + 8, other


@pytest.mark.parametrize("rows", [17, 96, 97, 200])
@pytest.mark.parametrize("act", [None, "relu2"])
def test_pre_tiled_experts_of_some_rows_each(rows, act):
    """Experts with up to 96 rows in the mean take their matrices past the caches, the others not: the
    same bits as from matrices in rows, spread over the experts and all on one."""
    W, ff, E, top, dt = 128, 192, 6, 2, torch.bfloat16
    T = rows * E // top
    h = _rand((T, W), 34, dtype=dt).to(DEV)
    gate_up = _rand((E, ff if act else 2 * ff, W), 35, 2 / W ** 0.5, dt).to(DEV)
    down = _rand((E, W, ff), 36, 2 / ff ** 0.5, dt).to(DEV)
    tiled = [torch.stack([ops.pretile_weight(m) for m in w]) for w in (gate_up, down)]
    g = torch.Generator().manual_seed(37)
    spread = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32)
    share = torch.rand((T, top), generator=g).to(DEV)
    for ids in (spread.to(DEV), torch.full((T, top), 3, dtype=torch.int32, device=DEV)):
        outs = []
        for w_tiled, (gu, dn) in ((False, (gate_up, down)), (True, tiled)):
            y = torch.empty((T, top, ff), dtype=dt, device=DEV)
            outs.append(torch.empty((T, W), device=DEV))
            ops.moe_experts(h, gu, dn, ids, share, y, outs[-1], 0.6, 1.702, 1.0, act=act,
                            w_tiled=w_tiled)
        assert torch.equal(*outs)


@pytest.mark.parametrize("T, W, ff, E, top", [(40, 64, 24, 6, 2), (300, 128, 64, 8, 3),
                                               (17, 72, 136, 1, 1), (150, 352, 104, 40, 4),
                                               (260, 64, 8, 3, 3)])
def test_experts_of_many_tokens_sorted_by_expert(T, W, ff, E, top):
    """bfloat16, more tokens than stream their experts one by one: the tokens sorted by expert
    through MFMA tiles against the plain expert, and against the streaming kernels."""
    dt = torch.bfloat16
    limit, alpha, shift = 0.6, 1.702, 1.0
    h = _rand((T, W), 14, dtype=dt)
    w = {}
    for e in range(E):
        w[f"e{e}.gate"] = _rand((ff, W), 120 + e, 2 / W ** 0.5, dt)
        w[f"e{e}.up"] = _rand((ff, W), 220 + e, 2 / W ** 0.5, dt)
        w[f"e{e}.down"] = _rand((W, ff), 320 + e, 2 / ff ** 0.5, dt)
    g = torch.Generator().manual_seed(15)
    # an expert nobody uses where there are experts to spare; a token names an expert once
    allowed = [e for e in range(E) if e != 1 or E <= top + 1]
    ids = torch.stack([torch.tensor(allowed)[torch.randperm(len(allowed), generator=g)[:top]]
                       for _ in range(T)]).to(torch.int32)
    share = torch.rand((T, top), generator=g)
    gate_up = torch.stack([torch.cat([w[f"e{e}.gate"], w[f"e{e}.up"]]) for e in range(E)]).to(DEV)
    down = torch.stack([w[f"e{e}.down"] for e in range(E)]).to(DEV)
    assert ops.moe_grouped_covers(h.to(DEV), gate_up) and T > ops.MOE_STREAM_MAX_TOKENS
    base = _rand((T, W), 16)
    for add in (False, True):
        y = torch.empty((T, top, ff), dtype=dt, device=DEV)
        out = base.to(DEV)
        ops.moe_experts(h.to(DEV), gate_up, down, ids.to(DEV), share.to(DEV), y, out, limit, alpha,
                        shift, add=add)
        y2 = torch.empty((T, top, ff), dtype=dt, device=DEV)
        out2 = base.to(DEV)
        ops.moe_gate_up(h.to(DEV), gate_up, ids.to(DEV), y2, limit, alpha, shift)
        ops.moe_down(y2, down, ids.to(DEV), share.to(DEV), out2, add=add)
        assert rel_err(out, out2) < 2e-2
        if T <= 150:
            ref = base.double() if add else torch.zeros((T, W), dtype=torch.float64)
            for t in range(T):
                for s_ in range(top):
                    ref[t] += share[t, s_].double() * P.clamped_expert(
                        h[t:t + 1], w, f"e{int(ids[t, s_])}.", limit)[0]
            assert rel_err(out, ref) < 2e-2
    # a token's result does not depend on the tokens beside it: the first 20 alone, the same bits
    if T >= 20:
        y3 = torch.empty((20, top, ff), dtype=dt, device=DEV)
        out3 = torch.empty((20, W), dtype=torch.float32, device=DEV)
        ops.moe_experts(h[:20].to(DEV), gate_up, down, ids[:20].contiguous().to(DEV),
                        share[:20].contiguous().to(DEV), y3, out3, limit, alpha, shift)
        out4 = torch.empty((T, W), dtype=torch.float32, device=DEV)
        ops.moe_experts(h.to(DEV), gate_up, down, ids.to(DEV), share.to(DEV), y, out4, limit,
                        alpha, shift)
        assert torch.equal(out3, out4[:20])


@pytest.mark.parametrize("dt", DTYPES)
def test_gated_act(dt):
    gu = _rand((7, 2 * 24), 17, 2.0, dtype=dt)
    out = torch.empty((7, 24), dtype=dt, device=DEV)
    ops.gated_act(gu.to(DEV), out, 1.5, 1.702, 1.0)
    g = gu[:, :24].double().clamp(max=1.5)
    u = gu[:, 24:].double().clamp(-1.5, 1.5)
    assert rel_err(out, g * torch.sigmoid(1.702 * g) * (u + 1)) < tol(dt)


# ------------------------------------------------------------------------------ attention
def _paged(k, n_kv, hd, page_size, seed):
    """Keys [n, n_kv * hd] of one sequence put into a pool through shuffled pages; returns the
    pool, the sequence's block table and the slots."""
    n = k.shape[0]
    pages = (n + page_size - 1) // page_size
    total = pages + 5
    g = torch.Generator().manual_seed(seed)
    table = torch.randperm(total, generator=g)[:pages].to(torch.int32)
    pool = torch.full((total, n_kv * page_size * hd), float("nan"), dtype=k.dtype, device=DEV)
    slots = torch.tensor([int(table[p // page_size]) * page_size + p % page_size for p in range(n)],
                         dtype=torch.int32)
    ops.kv_rows_write(k.to(DEV), slots.to(DEV), pool, n_kv, hd, page_size)
    return pool, table, slots


def _attend(q, gate, pool, table, n_ctx, n_q, nH, nKV, hd, page_size, scale, window, sink,
            mfma=False, n_splits=None, shared_tiles=None):
    """The last ``n_q`` positions of a sequence of ``n_ctx`` keys."""
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    out = torch.empty((n_q, nH * hd), dtype=q.dtype, device=DEV)
    if mfma:
        ops.tied_attention_mfma(q.to(DEV), None if gate is None else gate.to(DEV), pool,
                                table.view(1, -1).to(DEV), dev([0, n_q]), dev([n_ctx]), out, scale,
                                window, sink, nH, nKV, hd, page_size, n_q, n_ctx, n_splits=n_splits,
                                shared_tiles=shared_tiles)
        return out
    ops.shared_kv_attention(q.to(DEV), None if gate is None else gate.to(DEV), pool,
                            table.view(1, -1).to(DEV), dev([0, n_q]), dev([n_ctx]),
                            dev([0] * n_q), out, scale, window, sink, nH, nKV, hd, page_size,
                            n_ctx)
    return out


@pytest.mark.parametrize("nH, nKV, hd, page", [(4, 2, 32, 16), (9, 3, 96, 8), (16, 4, 128, 16)])
@pytest.mark.parametrize("window", [0, 1, 33, 100])
def test_decode_attention_stores_the_tokens_own_rows(nH, nKV, hd, page, window):
    """Single tokens whose rows are not in the pool yet, at the edges of a page, a chunk and a wave's
    keys: the output and the pool of the two kernels, bit for bit."""
    ctx = [1, 2, 16, 17, 32, 33, 64, 65, 129, 300]
    n, most = len(ctx), (max(ctx) + page - 1) // page
    perm = torch.randperm(n * most, generator=torch.Generator().manual_seed(5)).to(torch.int32)
    table = perm.view(n, most)
    slots = torch.tensor([int(table[i, (c - 1) // page]) * page + (c - 1) % page
                          for i, c in enumerate(ctx)], dtype=torch.int32, device=DEV)
    pool = _rand((n * most, nKV * page * hd), 150, dtype=torch.bfloat16).to(DEV)
    wide = _rand((n, (2 * nH + nKV) * hd), 151, dtype=torch.bfloat16).to(DEV)
    q, k, gate = wide[:, :nH * hd], wide[:, nH * hd:(nH + nKV) * hd], wide[:, (nH + nKV) * hd:]
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    args = (table.to(DEV), dev(list(range(n + 1))), dev(ctx), dev(list(range(n))))
    tail = (0.7 / hd ** 0.5, window, True, nH, nKV, hd, page, 1, max(ctx))
    pools, outs = [pool.clone(), pool.clone()], [torch.empty((n, nH * hd), dtype=torch.bfloat16,
                                                             device=DEV) for _ in range(2)]
    ops.kv_rows_write(k, slots, pools[0], nKV, hd, page)
    ops.tied_attention(q, gate, pools[0], *args, outs[0], *tail)
    at = ops.launch_count()
    ops.tied_attention(q, gate, pools[1], *args, outs[1], *tail, new=(k, slots))
    assert ops.launch_count() == at + 1
    assert torch.equal(pools[1], pools[0]) and torch.equal(outs[1], outs[0])
    # what the decode kernel does not take is stored by the kernel for it
    big = _rand((n, nH * 192), 152, dtype=torch.bfloat16).to(DEV)
    rows = _rand((n, nKV * 192), 153, dtype=torch.bfloat16).to(DEV)
    pools = [torch.zeros((n * most, nKV * page * 192), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    outs = [torch.empty_like(big) for _ in range(2)]
    tail = (0.05, window, True, nH, nKV, 192, page, 1, max(ctx))
    ops.kv_rows_write(rows, slots, pools[0], nKV, 192, page)
    ops.tied_attention(big, None, pools[0], *args, outs[0], *tail)
    ops.tied_attention(big, None, pools[1], *args, outs[1], *tail, new=(rows, slots))
    assert torch.equal(pools[1], pools[0]) and torch.equal(outs[1], outs[0])


@pytest.mark.parametrize("nH, nKV, hd, page", [(4, 2, 32, 16), (9, 3, 96, 16), (5, 1, 64, 8),
                                               (2, 2, 128, 16), (3, 1, 192, 4), (2, 1, 256, 16),
                                               (40, 2, 32, 16)])
@pytest.mark.parametrize("window", [0, 1, 5, 32, 33, 100])
def test_mfma_attention_against_plain(nH, nKV, hd, page, window):
    """The bfloat16 MFMA kernel: a whole prompt of several tiles, a portion behind a context,
    single tokens with the context unsplit and split over 2 and 5 workgroups."""
    dt = torch.bfloat16
    n = 171
    q = _rand((n, nH * hd), 130, dtype=dt)
    k = _rand((n, nKV * hd), 131, dtype=dt)
    gate = _rand((n, nH * hd), 132, 2.0, dtype=dt)
    pool, table, _ = _paged(k, nKV, hd, page, 133)
    scale = 0.7 / hd ** 0.5
    ref = P.sink_window_attention(q, k, nH, nKV, hd, scale, window if window else 10 ** 6)
    gated = ref * torch.sigmoid(gate.double())
    tolerance = 2.0 ** -7
    for tiles in (None, True):          # waves on their own where the shape allows; shared tiles
        out = _attend(q, gate, pool, table, n, n, nH, nKV, hd, page, scale, window, True, mfma=True,
                      shared_tiles=tiles)
        assert rel_err(out, gated) < tolerance
        tail = _attend(q[-50:], gate[-50:], pool, table, n, 50, nH, nKV, hd, page, scale, window,
                       True, mfma=True, shared_tiles=tiles)
        assert rel_err(tail, gated[-50:]) < tolerance
        one = _attend(q[-1:], gate[-1:], pool, table, n, 1, nH, nKV, hd, page, scale, window, True,
                      mfma=True, n_splits=2, shared_tiles=tiles)
        assert rel_err(one, gated[-1:]) < tolerance
    for splits in (1, 2, 5):
        last = _attend(q[-1:], None, pool, table, n, 1, nH, nKV, hd, page, scale, window, True,
                       mfma=True, n_splits=splits)
        assert rel_err(last, ref[-1:]) < tolerance
    nosink = _attend(q[-1:], gate[-1:], pool, table, n, 1, nH, nKV, hd, page, scale, window, False,
                     mfma=True, n_splits=3)
    exact = _attend(q[-1:], gate[-1:], pool, table, n, 1, nH, nKV, hd, page, scale, window, False)
    assert rel_err(nosink, exact.double()) < tolerance


@pytest.mark.parametrize("nH, nKV, hd, page", [(4, 2, 12, 16), (6, 2, 96, 16), (20, 1, 10, 4),
                                               (3, 3, 200, 8), (2, 1, 64, 16), (34, 2, 8, 16)])
@pytest.mark.parametrize("window", [0, 1, 5, 16, 17, 40])
@pytest.mark.parametrize("dt", DTYPES)
def test_attention_against_plain(nH, nKV, hd, page, window, dt):
    n = 45
    q = _rand((n, nH * hd), 30, dtype=dt)
    k = _rand((n, nKV * hd), 31, dtype=dt)
    gate = _rand((n, nH * hd), 32, 2.0, dtype=dt)
    pool, table, _ = _paged(k, nKV, hd, page, 33)
    scale = 0.7 / hd ** 0.5
    w = window if window else 10 ** 6
    ref = P.sink_window_attention(q, k, nH, nKV, hd, scale, w)
    tolerance = 2e-5 if dt == torch.float32 else 2.0 ** -7
    # the whole sequence as one portion, with the silent term and the gate
    out = _attend(q, gate, pool, table, n, n, nH, nKV, hd, page, scale, window, True)
    assert rel_err(out, ref * torch.sigmoid(gate.double())) < tolerance
    # its last 3 tokens as a portion, and its last token alone: the same rows, bit for bit
    tail = _attend(q[-3:], gate[-3:], pool, table, n, 3, nH, nKV, hd, page, scale, window, True)
    assert torch.equal(tail, out[-3:])
    last = _attend(q[-1:], gate[-1:], pool, table, n, 1, nH, nKV, hd, page, scale, window, True)
    assert torch.equal(last, out[-1:])
    # without the gate
    plain_out = _attend(q, None, pool, table, n, n, nH, nKV, hd, page, scale, window, True)
    assert rel_err(plain_out, ref) < tolerance


def test_attention_without_the_silent_term_is_a_plain_softmax():
    nH, nKV, hd, page, n = 2, 1, 16, 8, 20
    q, k = _rand((n, nH * hd), 34), _rand((n, nKV * hd), 35)
    pool, table, _ = _paged(k, nKV, hd, page, 36)
    out = _attend(q, None, pool, table, n, n, nH, nKV, hd, page, 0.25, 6, False)
    ref = torch.zeros((n, nH, hd), dtype=torch.float64)
    for i in range(n):
        lo = max(0, i - 5)
        for h in range(nH):
            a = torch.softmax((k[lo:i + 1].double() @ q[i].view(nH, hd)[h].double()) * 0.25, 0)
            ref[i, h] = a @ k[lo:i + 1].double()
    assert rel_err(out, ref.view(n, -1)) < 2e-5
    with_sink = _attend(q, None, pool, table, n, n, nH, nKV, hd, page, 0.25, 6, True)
    assert rel_err(with_sink, ref.view(n, -1)) > 1e-2       # the term is not nothing


@pytest.mark.parametrize("window, page", [(7, 16), (16, 16), (33, 8), (64, 16), (65, 16)])
@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("mfma", [False, True])
def test_a_loud_key_just_inside_and_just_outside_the_window(window, page, decode, mfma):
    """Among hundreds of quiet keys one key answers the last query loudly.  Planted at the
    oldest position the window still holds it takes the output; one position earlier it
    must not be seen at all."""
    nH, nKV, hd, n = 2, 1, 32, 300
    for planted, seen in ((n - window, True), (n - window - 1, False)):
        dt = torch.bfloat16 if mfma else torch.float32
        k = _rand((n, nKV * hd), 37, 0.05, dt)
        q = _rand((n, nH * hd), 38, 0.05, dt)
        loud = torch.zeros(hd, dtype=dt)
        loud[3] = 6.0
        k[planted] = loud
        q[n - 1] = torch.cat([loud, loud]) * 2.0
        pool, table, _ = _paged(k, nKV, hd, page, 39)
        n_q = 1 if decode else 9
        out = _attend(q[-n_q:], None, pool, table, n, n_q, nH, nKV, hd, page, 1.0, window, True,
                      mfma=mfma)
        got = out[-1].view(nH, hd).float().cpu()
        if seen:
            assert float(got[0, 3]) > 5.9 and float(got[1, 3]) > 5.9
        else:
            assert float(got.abs().max()) < 0.5
        ref = P.sink_window_attention(q, k, nH, nKV, hd, 1.0, window)[-1]
        assert rel_err(out[-1], ref) < (2.0 ** -7 if mfma else 2e-5)


@pytest.mark.parametrize("mfma", [False, True])
def test_pages_before_the_window_are_not_touched(mfma):
    """The block-table entries of pages that lie wholly before the window are -1 (the pages
    have gone back): no kernel may look them up."""
    dt = torch.bfloat16 if mfma else torch.float32
    nH, nKV, hd, page, n, window = 4, 2, 32, 4, 200, 21
    q, k = _rand((n, nH * hd), 70, dtype=dt), _rand((n, nKV * hd), 71, dtype=dt)
    pool, table, _ = _paged(k, nKV, hd, page, 72)
    ref = P.sink_window_attention(q, k, nH, nKV, hd, 0.2, window)
    for n_q in (1, 7):
        gone = table.clone()
        gone[:(n - n_q + 1 - window) // page] = -1         # wholly before the first query's window
        out = _attend(q[-n_q:], None, pool, gone, n, n_q, nH, nKV, hd, page, 0.2, window, True,
                      mfma=mfma)
        assert rel_err(out, ref[-n_q:]) < (2.0 ** -7 if mfma else 2e-5)


def test_first_tokens_and_a_far_key_without_a_window():
    """Position 0 sees itself and the silent term only; with no window the first key of a long
    context still counts."""
    nH, nKV, hd, n, page = 2, 2, 16, 700, 16
    k = _rand((n, nKV * hd), 40, 0.05)
    q = _rand((n, nH * hd), 41, 0.05)
    k[0, :hd] = 0.0
    k[0, 5] = 5.0
    q[n - 1, :hd] = 0.0
    q[n - 1, 5] = 4.0
    pool, table, _ = _paged(k, nKV, hd, page, 42)
    out = _attend(q[-1:], None, pool, table, n, 1, nH, nKV, hd, page, 1.0, 0, True)
    assert float(out[0, 5]) > 4.9
    first = _attend(q[:1], None, pool, table, 1, 1, nH, nKV, hd, page, 1.0, 0, True)
    s = (q[0].view(nH, hd).double() * k[0].view(nKV, hd).double()).sum(-1)
    ref = (torch.exp(s) / (1 + torch.exp(s))).unsqueeze(-1) * k[0].view(nKV, hd).double()
    assert rel_err(first, ref.view(1, -1)) < 2e-5


def test_sequences_of_a_batch_read_their_own_pages():
    """Three sequences in one launch (a portion, a single token, a whole prompt) against each
    alone: the same bits."""
    nH, nKV, hd, page = 4, 2, 24, 8
    lens, q_lens = (50, 31, 12), (6, 1, 12)
    total_pages = sum((n + page - 1) // page for n in lens) + 3
    g = torch.Generator().manual_seed(43)
    perm = torch.randperm(total_pages, generator=g).tolist()
    pool = torch.zeros((total_pages, nKV * page * hd), dtype=torch.float32, device=DEV)
    tables, qs, alone = [], [], []
    max_pages = max((n + page - 1) // page for n in lens)
    for i, (n, nq) in enumerate(zip(lens, q_lens)):
        k = _rand((n, nKV * hd), 50 + i)
        pages = [perm.pop() for _ in range((n + page - 1) // page)]
        slots = torch.tensor([pages[p // page] * page + p % page for p in range(n)], dtype=torch.int32)
        ops.kv_rows_write(k.to(DEV), slots.to(DEV), pool, nKV, hd, page)
        tables.append(pages + [-1] * (max_pages - len(pages)))
        qs.append(_rand((nq, nH * hd), 60 + i))
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    table = dev(tables)
    for i, (n, nq) in enumerate(zip(lens, q_lens)):
        out = torch.empty((nq, nH * hd), dtype=torch.float32, device=DEV)
        ops.shared_kv_attention(qs[i].to(DEV), None, pool, table[i:i + 1].contiguous(), dev([0, nq]),
                                dev([n]), dev([0] * nq), out, 0.2, 9, True, nH, nKV, hd, page, n)
        alone.append(out)
    T = sum(q_lens)
    out = torch.empty((T, nH * hd), dtype=torch.float32, device=DEV)
    starts = [0, 6, 7, 19]
    seq_index = [0] * 6 + [1] + [2] * 12
    ops.shared_kv_attention(torch.cat(qs).to(DEV), None, pool, table, dev(starts), dev(list(lens)),
                            dev(seq_index), out, 0.2, 9, True, nH, nKV, hd, page, max(lens))
    assert torch.equal(out, torch.cat(alone))
