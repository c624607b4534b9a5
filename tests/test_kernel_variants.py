"""Variants a dispatch chooses by size, type or layout, at the sizes where each can go wrong,
against the path they stand in for or the float64 oracle."""

import numpy as np
import pytest
import torch


@pytest.fixture(scope="module")
def m(cuda):
    import mlx_cce_amd
    mlx_cce_amd._ext.lib()
    return mlx_cce_amd


def _case(N, D, V, dtype, dev, seed, std=0.1):
    g = torch.Generator(device=dev).manual_seed(seed)
    e = torch.randn((N, D), generator=g, device=dev).to(dtype)
    c = (torch.randn((V, D), generator=g, device=dev) * std).to(dtype)
    t = torch.randint(0, V, (N,), generator=g, device=dev)
    return e, c, t


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["input", "sorted"])
@pytest.mark.parametrize("N,V", [(1, 100), (127, 4097), (129, 8191), (300, 9000), (260, 20000)])
def test_filter_of_reference_layout_statistics(m, cuda, N, V, order):
    """The filter over the reference's [N][ceil(V/32)] statistics keeps the tiles that it keeps
    over the [ceil(V/128)][N] ones (the same maxima), so every gradient agrees bit for bit."""
    e, c, t = _case(N, 64, V, torch.bfloat16, cuda, seed=N)
    t[::7] = -100
    tm, _, _, lse = m.cce_forward_raw(e, c, t, ignore_index=-100)
    tm128, _, _, _ = m.cce_forward_raw(e, c, t, ignore_index=-100, layout="tiles128")
    d = torch.linspace(0.0, 1.5, N, device=cuda)  # the first row has no cotangent
    out = []
    with m._ext.backward_options(token_order=order):
        for stats in (tm, tm128):
            kept = torch.empty(3, dtype=torch.int64, device=cuda)
            g = m._ext.backward(e, c, t, lse, stats, d, ignore_index=-100, tile_stats=kept)
            out.append((kept, g[0], g[1]))
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a, b)


def tile_order(ntb, nvb):
    """The persistent kernels' tile order (TileWalk::at, csrc/cce_device.h): number -> (token block, vocabulary block)."""
    ng = (ntb + 3) // 4
    b = ntb // ng
    big = ntb - b * ng
    split = big * (b + 1) * nvb
    out = []
    for r in range(ntb * nvb):
        gs, q = (b + 1, r) if r < split else (b, r - split)
        g, w = divmod(q, gs * nvb)
        vb, i = divmod(w, gs)
        out.append(((g * (b + 1) if r < split else big * (b + 1) + g * b) + i, vb))
    return out


def tile_walk(ntb, nvb, r, step):
    """TileWalk::next restated: the tiles r, r + step, ... by additions inside a token group."""
    order = tile_order(ntb, nvb)
    ng = (ntb + 3) // 4
    b = ntb // ng
    big = ntb - b * ng
    out = []

    def at(r):
        gs = b + 1 if r < big * (b + 1) * nvb else b
        tb, vb = order[r]
        return tb, vb, gs, (tb % gs if r < big * (b + 1) * nvb else (tb - big * (b + 1)) % gs)

    tb, vb, gs, i = at(r)
    while True:
        out.append((tb, vb))
        r += step
        if r >= ntb * nvb:
            return out
        vb, i, tb = vb + step // gs, i + step % gs, tb + step % gs
        if i >= gs:
            i, tb, vb = i - gs, tb - gs, vb + 1
        if vb >= nvb:
            tb, vb, gs, i = at(r)


@pytest.mark.parametrize("ntb", [1, 2, 3, 4, 5, 6, 7, 9, 11, 16, 33])
@pytest.mark.parametrize("nvb", [1, 2, 7, 63])
def test_tile_order_covers_every_tile_once(ntb, nvb):
    """Every tile has one number, token groups hold at most 4 blocks and differ by at most one,
    and no XCD's share takes more rounds than an eighth of the tiles."""
    order = tile_order(ntb, nvb)
    assert sorted(order) == [(t, v) for t in range(ntb) for v in range(nvb)]
    T = ntb * nvb
    al = 4 if ntb % 4 == 0 else 2 if ntb == 2 else 1
    begins = [x * T // 8 // al * al for x in range(9)]
    shares = [b - a for a, b in zip(begins, begins[1:])]
    assert begins[8] == T and max(-(-s // 32) for s in shares) == -(-(-(-T // 8)) // 32)  # rounds of 32 workgroups
    sizes = []
    for tb, _ in [o for o in order if o[1] == 0]:
        if not sizes or tb != sizes[-1][-1] + 1 or order.index((tb, 0)) != order.index((sizes[-1][-1], 0)) + 1:
            sizes.append([tb])
        else:
            sizes[-1].append(tb)
    for r in range(min(T, 5)):
        assert tile_walk(ntb, nvb, r, 32) == order[r::32]
    if nvb > 1:
        n = [len(s) for s in sizes]
        assert max(n) <= 4 and max(n) - min(n) <= 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,V", [(1, 257), (65, 129), (300, 385), (1100, 2000), (1281, 1500), (1537, 300)])
def test_ragged_token_blocks(m, cuda, N, V, dtype):
    """Token counts whose last blocks leave waves without tokens, and 5 to 7 token blocks: loss and
    unfiltered gradients against float64 (16-bit: the outputs' own rounding, 2^-9 and fp32 sums)."""
    e, c, t = _case(N, 72, V, dtype, cuda, seed=N)
    b = (torch.randn(V, device=cuda) * 0.3).to(dtype)
    t[::9] = -100
    leaves = [x.detach().requires_grad_() for x in (e, c, b)]
    loss = m.linear_cross_entropy(*leaves[:2], t, leaves[2], reduction="sum", filter_eps=None)
    got = torch.autograd.grad(loss, leaves)
    ref = [x.detach().double().requires_grad_() for x in (e, c, b)]
    want = torch.nn.functional.cross_entropy(ref[0] @ ref[1].T + ref[2], t, reduction="sum", ignore_index=-100)
    grads = torch.autograd.grad(want, ref)
    assert abs(loss.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -8
    for g, w in zip(got, grads):
        assert (g.double() - w).norm() <= tol * w.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("N", [1, 15, 16, 1024, 1025, 8192, 8193])
@pytest.mark.parametrize("V", [1, 130, 8000, 70000])
def test_lse_of_every_row_width(m, cuda, N, V):
    """The lse merge with 16, 32 and 64 tokens a workgroup, ragged in both, a column of -inf bias
    and rows of large logits: against float64 (fp32 logits of a 16-term product and fp32 exps, 1e-5)."""
    e, c, t = _case(N, 16, V, torch.float32, cuda, seed=V, std=1.0)
    e[::3] *= 20
    b = torch.zeros(V, device=cuda)
    b[V // 2 + 1:V // 2 + 200] = -float("inf")
    t[:] = V // 2
    _, _, _, lse, nll = m._ext.forward(e, c, t, b)
    x = e.double() @ c.double().T + b.double()
    want = torch.logsumexp(x, 1)
    assert ((lse.double() - want).abs() <= 1e-5 * want.abs().clamp(min=1)).all()
    assert ((nll.double() - (want - x[:, V // 2])).abs() <= 1e-5 * x.abs().nan_to_num(0, 0, 0).amax(1).clamp(min=1)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("N,D,V", [(1, 64, 100), (100, 512, 900), (128, 200, 40000), (129, 64, 300)])
def test_one_token_block_and_short_tasks(m, cuda, N, D, V):
    """One token block (no row sort) and dE tasks of fewer kept tiles than pieces: the host-driven and
    the device-skipped launches, and cut and whole tasks, agree with float64 and each other."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=D)
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    d = torch.linspace(0.5, 1.5, N, device=cuda)
    args = (e, c, t, lse, tm, d)
    base = m._ext.backward(*args, filter_eps=None)
    with m._ext.backward_options(passes="device"):
        dev = m._ext.backward(*args, filter_eps=None)
    with m._ext.backward_options(de_tasks="whole"):
        whole = m._ext.backward(*args, filter_eps=None)
    G = torch.softmax(e.double() @ c.double().T, 1)
    G[torch.arange(N, device=cuda), t] -= 1
    G *= d.double().unsqueeze(1)
    assert torch.equal(base[0], dev[0]) and torch.equal(base[1], dev[1])
    for got in (base, whole):
        for g, w in zip(got, (G @ c.double(), G.T @ e.double())):
            assert (g.double() - w).norm() <= 1e-5 * w.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 1e-15, 1e15])
@pytest.mark.parametrize("N,D,V", [(3, 4, 5), (130, 20, 300), (257, 68, 513), (512, 1024, 1000)])
def test_fp32_products_on_bf16_mfma(m, cuda, N, D, V, scale):
    """The fp32 logits from three bf16 cuts, against float64, at three magnitudes of e: no further off
    than fp32 sums of two products at a time (the fp32 MFMA's order) by more than one rounding
    of the result (the six products of a slice are added to the accumulator one after another)."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=D, std=1.0)
    e, c = e * scale, c / scale  # logits of one magnitude
    tm, _, _, lse = m.cce_forward_raw(e, c, t)
    x = e.double() @ c.double().T
    acc = torch.zeros(N, V, device=cuda)
    for k in range(0, D, 2):
        acc = (acc.double() + e[:, k:k + 2].double() @ c[:, k:k + 2].double().T).float()
    pad = torch.full((N, -V % 32), -float("inf"), device=cuda, dtype=torch.float64)
    top = torch.cat([x, pad], 1).view(N, -1, 32)
    want, at = top.max(2)
    err = (tm.view(N, -1).double() - want).norm()
    ref = torch.cat([acc.double(), pad], 1).view(N, -1, 32).gather(2, at.unsqueeze(2)).squeeze(2)
    assert err <= (ref - want).norm() + 2.0 ** -23 * want.norm()
    assert (lse.double() - torch.logsumexp(x, 1)).norm() <= 1e-6 * torch.logsumexp(x, 1).norm()


@pytest.mark.gpu
@pytest.mark.parametrize("filter_eps", [None, -8.3177661667])
@pytest.mark.parametrize("N,D,V", [(40, 16, 300), (600, 36, 700)])
def test_fp32_infinite_operands(m, cuda, N, D, V, filter_eps):
    """An infinite classifier entry makes its column's logits infinite as fp32 products are, not NaN:
    a column of -inf logits drops out of the loss and of every other gradient."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=3, std=0.5)
    e[:, 0] = e[:, 0].abs() + 0.5
    c[7, 0] = -float("inf")
    t[t == 7] = 8
    e.requires_grad_()
    loss = m.linear_cross_entropy(e, c, t, reduction="sum", filter_eps=filter_eps)
    keep = torch.arange(V, device=cuda) != 7
    x = e.detach().double() @ c[keep].double().T
    tk = torch.where(t > 7, t - 1, t)
    want = torch.nn.functional.cross_entropy(x, tk, reduction="sum")
    assert abs(loss.item() - want.item()) <= 1e-5 * abs(want.item())
    dE, = torch.autograd.grad(loss, e)
    assert torch.isfinite(dE[:, 1:]).all()  # (column 0 holds 0 * -inf where column 7's tile is kept)
    if filter_eps is None:
        G = torch.softmax(x, 1)
        G[torch.arange(N, device=cuda), tk] -= 1
        ref = (G @ c[keep].double())[:, 1:]
        assert (dE[:, 1:].double() - ref).norm() <= 1e-5 * ref.norm()
    c[9, 1] = float("nan")
    assert torch.isnan(m.linear_cross_entropy(e.detach(), c, t))


@pytest.mark.gpu
@pytest.mark.parametrize("N,D,V", [(40, 16, 300), (300, 36, 701), (600, 512, 704)])
def test_fp32_infinite_hidden_row(m, cuda, N, D, V):
    """An infinite entry in an ignored row of e: the forward tiles that hold it are computed again, the bias
    included (in LDS or, for V not a multiple of 4, from memory); every other row's loss is float64's
    (1e-5: fp32 sums) and the row itself is masked."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=5, std=0.5)
    b = torch.randn(V, device=cuda)
    e[3, 1] = float("inf")
    t[3] = -100
    nll = m._ext.forward(e, c, t, b)[4]
    keep = torch.arange(N, device=cuda) != 3
    want = torch.nn.functional.cross_entropy(e[keep].double() @ c.double().T + b.double(), t[keep], reduction="none")
    assert nll[3] == 0 and ((nll[keep].double() - want).abs() <= 1e-5 * want.abs().clamp(min=1)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("g_tasks", [None, "blocks"])
@pytest.mark.parametrize("what", ["infinite", "tiny"])
@pytest.mark.parametrize("N,D,V", [(40, 16, 300), (2100, 36, 3999), (2300, 64, 4000)])
def test_fp32_gradients_beside_the_cut(m, cuda, N, D, V, what, g_tasks):
    """Filtered gradients of all three operands where G tiles and dC / dE tasks are computed on the fp32 path, in
    the G kernel's pair tasks (the first size) and its tasks of up to 4 vocabulary tiles or token blocks
    (over 512 kept pairs, last blocks partial): against float64 (2e-6, logits near zero and V < 4096
    keep every tile).  An infinite classifier entry makes its column's logits -inf; dE's own column
    of it holds 0 * inf and is left out."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=N, std=0.02)
    b = torch.randn(V, device=cuda) * 0.01
    keep = torch.ones(V, dtype=torch.bool, device=cuda)
    if what == "infinite":
        e[:, 0] = e[:, 0].abs() + 0.5
        c[7, 0] = -float("inf")
        keep[7] = False
        t[t == 7] = 8
    else:
        e, c = e * 1e-35, c * 1e34
    t[::8] = -100
    tm, _, _, lse, _ = m._ext.forward(e, c, t, b)
    d = torch.linspace(0.5, 1.5, N, device=cuda)
    kept = torch.empty(3, dtype=torch.int64, device=cuda)
    with m._ext.backward_options(g_tasks=g_tasks, token_order="input"):  # (sorted, the ignored rows leave blocks empty)
        dE, dC, dB = m._ext.backward(e, c, t, lse, tm, d, b, tile_stats=kept)
    assert kept[0] == kept[1] and (kept[0] > 512) == (N > 2000)
    G = torch.zeros((N, V), dtype=torch.float64, device=cuda)
    G[:, keep] = torch.softmax(e.double() @ c[keep].double().T + b[keep].double(), 1)
    rows = t >= 0
    G[rows.nonzero().flatten(), t[rows]] -= 1
    G *= (d.double() * rows).unsqueeze(1)
    skip = 1 if what == "infinite" else 0
    for g, w in ((dE[:, skip:], G[:, keep] @ c[keep, skip:].double()), (dC, G.T @ e.double()), (dB, G.sum(0))):
        assert (g.double() - w).norm() <= 2e-6 * w.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("N,D,V", [(300, 512, 1000), (700, 4096, 1000), (700, 4096, 1002), (2500, 2048, 5000)])
def test_fp32_confident_rows_with_a_bias(m, cuda, N, D, V):
    """softmax - 1 of confident rows is what is left of exp(logit - lse): the logit's own rounding cancels
    when the dense G kernel forms the bits the forward formed, the bias included (in LDS or from
    memory).  What stays is the rounding of lse and of its product with log2(e), half an ulp each: the
    error of G at the target, from dE along c_t, is below 2^-24 of lse (2-norm over the rows)."""
    g = torch.Generator(device=cuda).manual_seed(D)
    c = torch.randn((V, D), generator=g, device=cuda) * 0.02
    b = torch.randn(V, generator=g, device=cuda) * 0.1
    t = torch.randint(0, V, (N,), generator=g, device=cuda)
    ct = c[t]
    e = ct * (14 / ct.pow(2).sum(1, keepdim=True)) + 0.5 * torch.randn((N, D), generator=g, device=cuda)
    tm, _, _, lse, _ = m._ext.forward(e, c, t, b)
    dE = m._ext.backward(e, c, t, lse, tm, torch.ones(N, device=cuda), b, filter_eps=None, want_dc=False)[0]
    x = e.double() @ c.double().T + b.double()
    l = torch.logsumexp(x, 1)
    G = torch.exp(x - l.unsqueeze(1))
    G[torch.arange(N, device=cuda), t] -= 1
    err = ((dE.double() - G @ c.double()) * ct.double()).sum(1) / ct.double().pow(2).sum(1)
    assert err.pow(2).mean().sqrt() <= 2.0 ** -24 * l.mean()


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(512, 1), (4096, 1), (4096, 300), (4100, 1)])
def test_fp32_logits_do_not_lean(m, cuda, D, V):
    """The mean error of 16384 fp32 logits per column: bf16 MFMA sums lean towards -inf (3e-7 of the rms logit
    at D = 4096 as they are), which moves every lse the same way.  The random errors' mean is
    1e-6 / 128; a third of the lean is allowed."""
    e, c, t = _case(16384, D, V, torch.float32, cuda, seed=D, std=1.0)
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    x = e.double() @ c.double().T
    want = torch.nn.functional.pad(x, (0, -V % 128), value=-float("inf")).view(16384, -1, 128).amax(2).T
    assert abs(float((tm.double() - want).mean())) <= 1e-7 * float(x.pow(2).mean().sqrt())


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-34, 1e-36, 1e34])
@pytest.mark.parametrize("N,D,V", [(3, 4, 5), (257, 68, 513), (700, 512, 9000)])
def test_fp32_products_of_tiny_values(m, cuda, N, D, V, scale):
    """Operands below 2^-110 (e or c), which three bf16 values do not hold: the logits are as close to
    float64 as fp32 sums (each of the D products and sums rounds by 2^-24; 2e-6 is far above their
    2-norm).  e stays above 2^-126, where fp32 itself has no fewer bits."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=D, std=1.0)
    e = torch.where(e.abs() < 0.05, torch.full_like(e, 0.05), e) * scale
    c = torch.where(c.abs() < 0.05, torch.full_like(c, 0.05), c) / scale
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    x = e.double() @ c.double().T
    want = torch.nn.functional.pad(x, (0, -V % 128), value=-float("inf")).view(N, -1, 128).amax(2).T
    assert (tm.double() - want).norm() <= 2e-6 * want.norm()
    assert (lse.double() - torch.logsumexp(x, 1)).norm() <= 2e-6 * torch.logsumexp(x, 1).norm()


@pytest.mark.gpu
@pytest.mark.parametrize("cot,es,cs", [(1e-33, 1, 1), (1e-36, 1, 1), (1e30, 1, 1), (1, 1e-35, 1e34), (1, 1e34, 1e-35), (1e25, 1e-10, 1)])
@pytest.mark.parametrize("N,D,V,eps", [(5, 4, 100, None), (5, 4, 100, -8.3177661667), (384, 260, 2000, None),
                                       (384, 260, 2000, -8.3177661667), (130, 64, 40000, None)])
def test_fp32_gradients_of_tiny_values(m, cuda, N, D, V, cot, es, cs, eps):
    """fp32 gradients with cotangents, or classifier or hidden rows, whose magnitudes three bf16 values
    do not hold, or larger than the sums' scaled range: against float64 as at ordinary magnitudes (2e-6,
    and half of fp32's last subnormal bit for each value).  With the filter on, logits near zero and
    V < 4096 keep every tile."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=N + D, std=0.02)
    e, c = e * es, c * cs
    t[::8] = -100
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    d = torch.linspace(0.5, 1.5, N, device=cuda) * cot
    dE, dC, _ = m._ext.backward(e, c, t, lse, tm, d, filter_eps=eps)
    G = torch.softmax(e.double() @ c.double().T, 1)
    rows = t >= 0
    G[rows.nonzero().flatten(), t[rows]] -= 1
    G *= (d.double() * rows).unsqueeze(1)
    for g, w in ((dE, G @ c.double()), (dC, G.T @ e.double())):
        assert (g.double() - w).norm() <= 2e-6 * w.norm() + 2.0 ** -150 * w.numel() ** 0.5


@pytest.mark.gpu
def test_fp32_infinite_operand_stays_with_its_tasks(m, cuda):
    """An infinite classifier entry has the dE tasks of its 256 columns computed on the fp32 path, and not
    later tasks of the same workgroup: 600 tasks on 256 workgroups here, where a third of them take a
    task of the last 256 columns after one of the first.  The last columns are the same bits as with a
    finite entry of the same effect.  (Whole-number operands: exact logits either way, so G is the
    same; dE's sums depend on the path in their last bits.)"""
    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the tasks are laid out for a 256-workgroup grid")
    N, D, V = 200 * 128, 768, 256
    g = torch.Generator(device=cuda).manual_seed(5)
    e = torch.randint(-1, 2, (N, D), generator=g, device=cuda).float()
    c = torch.randint(-8, 9, (V, D), generator=g, device=cuda).float() / 64
    e[:, 0] = 1.0
    t = torch.randint(8, V, (N,), generator=g, device=cuda)
    out = []
    for entry in (-1e4, -float("inf")):
        c[7, 0] = entry
        tm, _, _, lse, _ = m._ext.forward(e, c, t)
        dE = m._ext.backward(e, c, t, lse, tm, torch.ones(N, device=cuda), filter_eps=None, want_dc=False)[0]
        out.append((lse, dE[:, 512:]))
    assert torch.equal(out[0][0], out[1][0])
    assert torch.isfinite(out[0][1]).all() and torch.equal(out[0][1], out[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("reduction", ["none", "sum", "mean"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_native_host_calls_match_the_general_path(m, cuda, dtype, reduction):
    """The native calls and the general path (taken for operands that are not plain: here a
    strided e, int32 targets, an expanded cotangent) give the same loss and gradients bit for bit."""
    N, D, V = 150, 40, 500
    e, c, t = _case(N, D, V, dtype, cuda, seed=1)
    b = torch.randn(V, device=cuda).to(dtype)
    t[::5] = -100
    wide = torch.zeros((N, 2 * D), dtype=dtype, device=cuda)
    wide[:, ::2] = e
    forms = [(e, t, True), (wide[:, ::2], t, False), (e, t.to(torch.int32), False)]
    out = []
    for ee, tt, plain in forms:
        leaves = [ee.detach().requires_grad_(), c.detach().requires_grad_(), b.detach().requires_grad_()]
        r = m._ext.forward_loss(leaves[0], leaves[1], tt, leaves[2], -100, reduction)
        assert (r is not None) == plain
        loss, lse = m.linear_cross_entropy(*leaves[:2], tt, leaves[2], reduction=reduction, return_lse=True)
        cot = torch.ones((), device=cuda).expand(N) if reduction == "none" and not plain else torch.ones_like(loss)
        out.append((loss.detach(), lse, *torch.autograd.grad(loss, leaves, cot)))
    for other in out[1:]:
        for x, y in zip(out[0], other):
            assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("ignore", [-100.0, np.float32(-100), np.int32(-100), torch.tensor(-100), "-100", 2 ** 64 - 100])
def test_native_host_calls_take_any_ignore_index(m, cuda, ignore):
    """ignore_index goes through int() whatever the operands' layout: the native call and the general
    path (int32 targets) take the same values, and refuse the same."""
    e, c, t = _case(60, 24, 300, torch.bfloat16, cuda, seed=4)
    t[::4] = -100
    want = m.linear_cross_entropy(e, c, t)
    for tt in (t, t.to(torch.int32)):
        x = e.detach().requires_grad_()
        loss = m.linear_cross_entropy(x, c, tt, ignore_index=ignore)
        dE, = torch.autograd.grad(loss, x)
        assert torch.equal(loss, want) and (dE[::4] == 0).all()
        with pytest.raises(ValueError):
            m.linear_cross_entropy(e, c, tt, ignore_index="none")


@pytest.mark.gpu
def test_native_host_calls_refuse_what_the_library_refuses(m, cuda):
    """Sizes the library refuses raise the library's error from the native call too, and operands that
    do not fit each other raise the general path's."""
    e, c, t = _case(8, 12, 50, torch.bfloat16, cuda, seed=2)  # D = 12: not a multiple of 8
    with pytest.raises(ValueError, match="D must be a multiple of 8"):
        m.linear_cross_entropy(e, c, t)
    with pytest.raises(ValueError, match="must equal"):
        m.linear_cross_entropy(e, c[:, :8].contiguous(), t)
    with pytest.raises(ValueError, match="targets"):
        m.cce_loss(e, c, t[:4])
    with pytest.raises(TypeError, match="share one dtype"):
        m.linear_cross_entropy(e, c.float(), t)
    with pytest.raises(RuntimeError):
        m.linear_cross_entropy(e.cpu(), c.cpu(), t.cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [None, "pair"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N,D,V", [(5, 8, 50), (130, 72, 1000), (300, 264, 3000), (700, 128, 9000)])
def test_pair_tasks_match_block_tasks(m, cuda, N, D, V, dtype, precision):
    """The G kernel's tasks of one pair spread over the workgroup against runs of a block's tiles:
    the same sums with the contraction's slices rotated differently (fp32 1e-5; 16-bit: a
    rounded G entry moves by its last bit now and then, 2e-3)."""
    e, c, t = _case(N, D, V, dtype, cuda, seed=D, std=0.3)
    b = (torch.randn(V, device=cuda) * 0.5).to(dtype)
    t[::6] = -100
    tm, _, _, lse, _ = m._ext.forward(e, c, t, b)
    d = torch.linspace(-0.5, 1.5, N, device=cuda)
    got = []
    for kw in (dict(), dict(g_tasks="blocks")):
        kept = torch.empty(3, dtype=torch.int64, device=cuda)
        with m._ext.backward_options(g_precision=precision, **kw):
            got.append((kept, *m._ext.backward(e, c, t, lse, tm, d, b, tile_stats=kept)))
    assert torch.equal(got[0][0], got[1][0]) and got[0][0][0] <= 2 * 256
    tol = 1e-5 if dtype == torch.float32 else 2e-3
    for x, y in zip(got[0][1:], got[1][1:]):
        assert (x.double() - y.double()).norm() <= tol * y.double().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("dc", [None, "wide", "narrow"])
@pytest.mark.parametrize("eps", [None, -8.3177661667])
@pytest.mark.parametrize("N,D,V", [(1, 4, 3), (100, 60, 129), (129, 256, 127), (384, 260, 2000), (1500, 516, 900)])
def test_fp32_sums_on_bf16_mfma(m, cuda, N, D, V, eps, dc):
    """The fp32 dE and dC sums from three bf16 cuts (last rows and columns partial, one and several
    tasks and pieces, both ways of dealing dC) against float64 over the kernel's own kept tiles: all
    of them here (near-uniform logits over V < 4096 keep every tile)."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=N + D, std=0.02)
    t[::8] = -100
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    d = torch.linspace(0.5, 1.5, N, device=cuda)
    kept = torch.empty(3, dtype=torch.int64, device=cuda)
    with m._ext.backward_options(dc_sums=dc):
        dE, dC, _ = m._ext.backward(e, c, t, lse, tm, d, filter_eps=eps, tile_stats=kept)
    G = torch.softmax(e.double() @ c.double().T, 1)
    rows = t >= 0
    G[rows.nonzero().flatten(), t[rows]] -= 1
    G *= (d.double() * rows).unsqueeze(1)
    blocks = torch.nn.functional.pad(rows, (0, -N % 128)).view(-1, 128).any(1)
    assert kept[0] == blocks.sum() * ((V + 127) // 128)
    for g, w in ((dE, G @ c.double()), (dC, G.T @ e.double())):
        assert (g.double() - w).norm() <= 2e-6 * w.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("skewed", [False, True])
@pytest.mark.parametrize("passes", [None, "device"])
@pytest.mark.parametrize("N,D,V,max_g", [(300, 260, 3000, 0), (2000, 64, 9000, 0), (2000, 64, 9000, 1)])
def test_fp32_dc_dealt_as_picked(m, cuda, N, D, V, max_g, passes, skewed):
    """The filtered fp32 dC sums deal their owners as the compaction picked, in one launch: the same
    bits as with either way of dealing forced (an owner's sum does not depend on who runs it), with
    evenly shared tiles and with most targets in one, in one pass and several."""
    e, c, t = _case(N, D, V, torch.float32, cuda, seed=N, std=0.3)
    if skewed:
        t[: N * 3 // 4] = 5
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    d = torch.linspace(0.5, 1.5, N, device=cuda)
    out = []
    for dc in (None, "wide", "narrow"):
        with m._ext.backward_options(dc_sums=dc, passes=passes, max_g_tiles=max_g):
            out.append(m._ext.backward(e, c, t, lse, tm, d))
    for other in out[1:]:
        assert torch.equal(out[0][0], other[0]) and torch.equal(out[0][1], other[1])


@pytest.mark.parametrize("V,D,dtype,rows", [
    (128256, 4096, torch.bfloat16, 65536), (128256, 4096, torch.float32, 32768), (32000, 16384, torch.bfloat16, 32768),
    (245631, 128, torch.float32, 1048576), (100000, 768, torch.bfloat16, 348160)])
def test_quantized_rows_per_chunk(V, D, dtype, rows):
    """The autograd op's chunks: what 512 MiB hold in whole 4096-row steps, at least 32768 rows."""
    import mlx_cce_amd as cce

    qw = cce.QuantizedWeight(torch.empty((V, D * 4 // 32), dtype=torch.int32, device="meta"),
                             torch.empty((V, D // 64), dtype=dtype, device="meta"),
                             torch.empty((V, D // 64), dtype=dtype, device="meta"))
    got = cce._ext.quant_chunk_rows(qw)
    assert got == rows and got % 4096 == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_quantized_step_across_chunk_sizes(m, cuda, dtype, monkeypatch):
    """A quantized step in one chunk and in several (the scratch budget lowered to the least rows): the
    same loss and dE up to the slices' rotation (fp32 1e-5; bf16 a rounded G entry, 2e-3)."""
    V, D, N = 40000, 64, 200
    e, c, t = _case(N, D, V, dtype, cuda, seed=11, std=0.3)
    qw = m.quantize(c, group_size=64, bits=4)
    out = []
    for budget in (m._ext.QUANT_SCRATCH_BYTES, 0):
        monkeypatch.setattr(m._ext, "QUANT_SCRATCH_BYTES", budget)
        x = e.detach().requires_grad_()
        loss = m.linear_cross_entropy(x, qw, t)
        out.append((loss.detach(), torch.autograd.grad(loss, x)[0]))
    assert abs(out[0][0] - out[1][0]) <= 1e-6 * abs(out[1][0])
    d = (out[0][1].double() - out[1][1].double()).norm() / out[1][1].double().norm()
    assert d <= (1e-5 if dtype == torch.float32 else 2e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("layout_ref", [False, True])
def test_loss_of_confident_rows(m, cuda, layout_ref):
    """Rows whose target has nearly all the mass, logits whole numbers (exact sums): the loss is log(1 +
    sum exp) to the hardware exp2's and log2's last bits (2^-18 absolute covers the log near 1, 1.8e-5 of
    the loss the 299 exps and their sum), whatever the logit's size, up to 66 here."""
    V, D = 300, 8
    c = torch.zeros((V, D), device=cuda)
    c[5, 0] = 1.0
    e = torch.zeros((40, D), device=cuda)
    e[:, 0] = torch.arange(5, 45, device=cuda) * 1.5
    t = torch.full((40,), 5, device=cuda)
    nll = m._ext.forward(e, c, t, ref_stats=layout_ref)[4]
    want = torch.log1p((V - 1) * torch.exp(-e[:, 0].double()))
    assert ((nll.double() - want).abs() <= 2e-5 * want + 2.0 ** -18).all()


@pytest.mark.gpu
@pytest.mark.parametrize("split", [dict(), dict(max_g_tiles=1), dict(max_chunk_tiles=32)])
@pytest.mark.parametrize("order", ["input", "sorted"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,D,masked", [(2176, 4096, 1152), (4096, 2304, 2304), (2176, 4096, 2000)])
def test_de_pieces_of_masked_token_blocks(m, cuda, N, D, masked, dtype, order, split):
    """More than 256 dE tasks by the sizes, but over half of the token blocks hold only ignored rows:
    the tasks that are left are cut into pieces, and every one of them is finished (dE starts from
    memory that holds NaN).  Against whole tasks: fp32 sums in another order (1e-5), 16-bit outputs
    rounded from them (2e-3), as without masked rows."""
    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the task counts are laid out for a 256-workgroup grid")
    e, c, t = _case(N, D, 9000, dtype, cuda, seed=37, std=0.05)
    t[N - masked:] = -100
    tm, _, _, lse, _ = m._ext.forward(e, c, t)
    d = torch.linspace(0.5, 1.5, N, device=cuda)
    out = []
    for tasks in (None, "whole"):
        used = torch.full_like(e, float("nan"))  # the next tensor of this size takes its memory
        del used
        with m._ext.backward_options(token_order=order, de_tasks=tasks, **split):
            out.append(m._ext.backward(e, c, t, lse, tm, d, want_dc=False)[0])
    assert torch.isfinite(out[0]).all()
    err = (out[0].double() - out[1].double()).norm() / out[1].double().norm()
    assert err <= (1e-5 if dtype == torch.float32 else 2e-3)
