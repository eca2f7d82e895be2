"""The linear cross-entropy's references of a row's exponentials: its label's logit, and for blocks of 256 rows with a row
whose sum that does not suit, the log-sum-exp, found against the maxima over half vocabulary tiles."""
import pytest
import torch

DEV = "cuda:0"


def _case(N, D, V, seed, one_label=False):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(N, D, generator=gen).to(torch.bfloat16).to(DEV)
    w = (0.7 / D ** 0.5 * torch.randn(V, D, generator=gen)).to(torch.bfloat16).to(DEV)
    lab = torch.full((N,), V - 1) if one_label else torch.randint(0, V, (N,), generator=gen)
    lab[0], lab[N // 2], lab[N // 3] = 0, V - 1, -100
    return x, w, lab.to(DEV)


def _poison(x, w, lab):
    """One more row that no single reference fits: its logits spread over hundreds, and its label has the lowest."""
    row = (w[1] - w[0]).float()
    row = (row * (300.0 / row.norm() ** 2)).to(torch.bfloat16)
    return torch.cat([x, row[None]]), w, torch.cat([lab, lab.new_tensor([0])])


def _run(x, w, lab, **kw):
    from sisa_amd.kernels.linear_ce import linear_cross_entropy
    x, w = x.clone().requires_grad_(True), w.float().requires_grad_(True)
    loss = linear_cross_entropy(x, w, lab, **kw)
    dx, dw = torch.autograd.grad(loss, (x, w))
    return loss.detach(), dx, dw


def _truth(x, w, lab):
    x, w = x.double().requires_grad_(True), w.double().requires_grad_(True)
    loss = torch.nn.functional.cross_entropy(x @ w.t(), lab, ignore_index=-100)
    return (loss.detach(), *torch.autograd.grad(loss, (x, w)))


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


# ragged rows and vocabularies; the hidden sizes' tile remainders (64, 768, 1024 of 256-wide tiles); one, several and many
# vocabulary splits of dx; 5,000 rows with one label (a label list longer than the kernel's batch)
@pytest.mark.gpu
@pytest.mark.parametrize("N,D,V,one_label", [(1, 64, 65, False), (300, 512, 1003, False), (257, 768, 50277, False),
                                             (5000, 64, 130, True), (4500, 320, 1000, False), (70, 1024, 8191, False)])
def test_row_references_match_tile_maxima(N, D, V, one_label):
    x, w, lab = _case(N, D, V, N + D, one_label)
    if N == 1:
        lab[0] = 3
    for case in ((x, w, lab), _poison(x, w, lab)):
        ref, got = _truth(*case), _run(*case)
        # logits rounded to 8 bits shift the loss by the mean of their errors; gradients: three 8-bit roundings
        assert abs(float(got[0] - ref[0])) <= 2 ** -8 * (1 + abs(float(ref[0])))
        assert _rel(got[1], ref[1]) <= 3 * 2 ** -8 and _rel(got[2], ref[2]) <= 3 * 2 ** -8
        assert _rel(got[1][:N], ref[1][:N]) <= 3 * 2 ** -8      # the poison row's gradient outweighs the others'
        again = _run(*case)
        assert all(torch.equal(a, b) for a, b in zip(got, again))
        with torch.no_grad():
            from sisa_amd.kernels.linear_ce import linear_cross_entropy
            assert torch.equal(linear_cross_entropy(case[0], case[1].float(), case[2]), got[0])


@pytest.mark.gpu
@pytest.mark.parametrize("top", [6.0, 12.0])
def test_confident_rows(top):
    """Rows whose label holds nearly all the probability: G at the label is p - 1, far below p, and keeps its relative
    precision. The truth takes the logits as the kernels round them; then three 8-bit roundings, as above."""
    _, w, lab = _case(300, 256, 1003, 5)
    lab = lab.clamp_min(0)
    wl = w[lab].double()
    x = (top * wl / (wl * wl).sum(1, keepdim=True)).to(torch.bfloat16)
    logits = (x.double() @ w.double().t()).to(torch.bfloat16).double()
    G = torch.softmax(logits, 1)
    rest = G.scatter(1, lab[:, None], 0.0)
    G = rest.scatter(1, lab[:, None], -rest.sum(1, keepdim=True))
    _, dx, dw = _run(x, w, lab)
    assert _rel(dx, G / 300 @ w.double()) <= 3 * 2 ** -8
    assert _rel(dw, G.t() / 300 @ x.double()) <= 3 * 2 ** -8
    px, _, plab = _poison(x, w, lab)
    _, dx, dw = _run(px, w, plab)
    assert _rel(dx[:300], G / 301 @ w.double()) <= 3 * 2 ** -8
    assert _rel(dw[2:], G.t()[2:] / 301 @ x.double()) <= 3 * 2 ** -8     # the poison row reaches rows 0 and 1 only


@pytest.mark.gpu
def test_chunks_of_both_kinds_and_a_hopeless_label():
    """Chunks decide for themselves (dW accumulates over both kinds); a valid row whose label lies 200 below its
    largest logit is exact in the second way."""
    x, w, lab = _poison(*_case(500, 256, 2000, 9))
    order = torch.randperm(501, generator=torch.Generator().manual_seed(1)).to(DEV)
    x, lab = x[order], lab[order]
    rest = order != 500
    ref = _truth(x, w, lab)
    for kw in (dict(chunk_tokens=128), {}):
        got = _run(x, w, lab, **kw)
        assert float(ref[0]) > 0.25 and abs(float(got[0] - ref[0])) <= 2 ** -8 * float(ref[0])
        assert _rel(got[1], ref[1]) <= 3 * 2 ** -8 and _rel(got[2], ref[2]) <= 3 * 2 ** -8
        assert _rel(got[1][rest], ref[1][rest]) <= 3 * 2 ** -8
    bad = lab.clone()
    bad[7] = 2000                                           # outside the vocabulary: NaN loss, as without it
    assert not bool(torch.isfinite(_run(x, w, bad)[0]))


@pytest.mark.gpu
@pytest.mark.parametrize("N", [0, 1, 63, 1024, 8191, 8193, 100001])
def test_scalars(N):
    """The valid-row count, its reciprocal and the mean loss over remainders of the workgroup's 1,024 and 8,192."""
    from sisa_amd.kernels import _lib
    gen = torch.Generator().manual_seed(N)
    lab = torch.randint(-1, 3, (N,), generator=gen).to(DEV)
    rows = (10 + torch.randn(N, generator=gen)).to(DEV)
    n, inv, mean = torch.empty(3, device=DEV).split(1)
    _lib.call_values("sisa_ce_count", n, lab.data_ptr(), N, -1, n.data_ptr(), inv.data_ptr())
    _lib.call_values("sisa_ce_mean", n, rows.data_ptr(), N, n.data_ptr(), mean.data_ptr())
    count = int((lab != -1).sum())
    assert float(n) == count and torch.equal(inv, torch.reciprocal(n))
    want = rows.double().sum() / count
    if count:       # one rounding of the sum, one of the quotient
        assert abs(float(mean) - float(want)) <= 2 * 2.0 ** -24 * abs(float(want))
    else:
        assert not bool(torch.isfinite(mean))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fill", [0x45, 0xff, 0x7f])          # large finite numbers, NaNs, and the largest finite ones
def test_ignored_label_inside_the_vocabulary(dtype, fill):
    """A padding id as ignore_index: its rows have no label term at all, whatever the workspace held before."""
    from sisa_amd.kernels import linear_ce as LC
    x, w, lab = _case(300, 256, 1003, 11)
    x, w = x.to(dtype), w.to(dtype)
    lab[lab < 0] = 0
    lab[::3] = 0
    valid = lab != 0
    wpad = LC.padded_weight(w, dtype)
    inv_n = torch.reciprocal(valid.sum().float()).reshape(1)
    ws = LC.train_workspace([300], wpad.shape[0], 256, DEV)
    ws.fill_(fill)
    rows, dx = torch.empty(300, device=DEV), torch.empty(300, 256, device=DEV)
    dw = torch.empty(wpad.shape[0], 256, device=DEV)
    LC.lmce_train_chunk(x, wpad, lab, 1003, 0, inv_n, 256.0, rows, dx, dw, False, ws)   # 256: G above fp16's subnormals
    assert torch.equal(rows[~valid], torch.zeros_like(rows[~valid]))
    assert torch.equal(dx[~valid], torch.zeros_like(dx[~valid]))
    ref = _truth(x, w, torch.where(valid, lab, -100))
    assert _rel(dx, 256 * ref[1]) <= 3 * 2 ** -8 and _rel(dw[:1003], 256 * ref[2]) <= 3 * 2 ** -8


@pytest.mark.gpu
def test_ignored_label_inside_the_vocabulary_over_short_chunks():
    """The same through the public call, the last chunk shorter, so that its slots hold the previous one's exponentials.
    Logits spread over 35 make those large; the truth takes the logits as the kernels round them."""
    x, w, lab = _case(500, 256, 1003, 12)
    w = (8 * w.float()).to(torch.bfloat16)
    lab[lab < 0] = 0
    lab[::3] = 0
    valid = lab != 0
    logits = (x.double() @ w.double().t()).to(torch.bfloat16).double()
    G = torch.softmax(logits, 1).scatter_add(1, lab[:, None], -torch.ones(500, 1, dtype=torch.float64, device=DEV))
    G = G * valid[:, None] / valid.sum()
    got = _run(x, w, lab, ignore_index=0, chunk_tokens=192)
    assert _rel(got[1], G @ w.double()) <= 3 * 2 ** -8 and _rel(got[2], G.t() @ x.double()) <= 3 * 2 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("N", [300, 1500])
def test_ignored_rows_are_never_outliers(N):
    """Masked rows whose logits no column's logit represents leave the other rows on the fast way: the same bits as with
    ordinary masked rows, in both passes, and their own gradient is zero. Asked for, their log-sum-exp is exact."""
    from sisa_amd.kernels import linear_ce as LC
    x, w, lab = _case(N, 256, 1003, N)
    far = (w[1] - w[0]).float()
    far = (far * (300.0 / far.norm() ** 2)).to(torch.bfloat16)
    masked = torch.arange(N, device=DEV) % 7 == 0
    lab[masked] = -100
    for sign in (1, -1):                                    # column 0 far below the row's largest logit, and above all
        xo = torch.where(masked[:, None], sign * far, x)
        (loss, dx, dw), (lo, dxo, dwo) = _run(x, w, lab), _run(xo, w, lab)
        assert torch.equal(loss, lo) and torch.equal(dx, dxo) and torch.equal(dw, dwo)
        assert not dx[masked].any()
        with torch.no_grad():
            assert torch.equal(LC.linear_cross_entropy(xo, w, lab), loss)
        lse = torch.empty(N, device=DEV)
        LC.lmce_fused_loss_rows(xo, LC.padded_weight(w, torch.bfloat16), lab, 1003, -100, lse)
        logits = (xo.double() @ w.double().t()).to(torch.bfloat16).double()
        assert float((lse.double() - torch.logsumexp(logits, 1)).abs().max()) <= 1e-4


def _outliers(x, w, lab, gaps):
    """``gaps``: row -> how far the row's label lies below its largest logit."""
    x, lab = x.clone(), lab.clone()
    d = (w[1] - w[0]).double()
    for n, gap in gaps.items():
        x[n], lab[n] = (d * (gap / d.norm() ** 2)).to(torch.bfloat16), 0
    return x, w, lab


# a label's logit up to 62 below the largest suits; 63 is the first that does not, from 89 the exponentials overflow; blocks 0,
# 1, the last and a partial one, past the 64 blocks that a wave looks at together, every block, and fewer splits than tiles
@pytest.mark.gpu
@pytest.mark.parametrize("N,D,V,gaps", [(700, 128, 1003, {3: 64.0}), (700, 128, 1003, {300: 100.0}),
                                        (700, 128, 1003, {3: 61.0, 300: 64.0}),
                                        (700, 128, 50277, {0: 70.0, 699: 100.0}), (513, 64, 1003, {512: 300.0}),
                                        (16900, 64, 130, {100: 70.0, 16400: 64.0, 16899: 100.0}),
                                        (16900, 64, 130, {256 * i + 7: 64.0 + i for i in range(66)})])
def test_outliers_reach_their_row_block_alone(N, D, V, gaps):
    x, w, lab = _case(N, D, V, N + V)
    lab[list(gaps)] = 0
    case = _outliers(x, w, lab, gaps)
    base, got, ref = _run(x, w, lab), _run(*case), _truth(*case)
    block = torch.arange(N, device=DEV) // 256
    hit = torch.isin(block, torch.tensor([n // 256 for n, gap in gaps.items() if gap > 62], device=DEV))
    same = ~hit & ~torch.isin(torch.arange(N, device=DEV), torch.tensor(list(gaps), device=DEV))
    assert torch.equal(got[1][same], base[1][same])
    rest = torch.ones(N, dtype=torch.bool, device=DEV)
    rest[list(gaps)] = False
    assert abs(float(got[0] - ref[0])) <= 2 ** -8 * (1 + abs(float(ref[0])))
    assert _rel(got[1], ref[1]) <= 3 * 2 ** -8 and _rel(got[1][rest], ref[1][rest]) <= 3 * 2 ** -8
    assert _rel(got[2], ref[2]) <= 3 * 2 ** -8 and _rel(got[2][2:], ref[2][2:]) <= 3 * 2 ** -8
    with torch.no_grad():
        from sisa_amd.kernels.linear_ce import linear_cross_entropy
        assert torch.equal(linear_cross_entropy(*case), got[0])


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_row_that_is_not_finite(bad):
    x, w, lab = _case(700, 128, 1003, 21)
    x2 = x.clone()
    x2[300, 5] = bad
    base, got = _run(x, w, lab), _run(x2, w, lab)
    assert not torch.isfinite(got[0]) and torch.isnan(got[1][300]).all() and torch.isnan(got[2]).any()
    keep = torch.arange(700, device=DEV) // 256 != 1
    assert torch.equal(got[1][keep], base[1][keep]) and torch.isfinite(got[1][torch.arange(700) != 300]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("N", [1, 63, 8192, 8193, 65537, 131071, 8192 * 256, 8192 * 256 + 1, 5000001])
def test_wide_scalars(N):
    """Remainders of the workgroups' 8,192 rows, as many workgroups as there may be, and two batches each."""
    from sisa_amd.kernels import _lib
    gen = torch.Generator().manual_seed(N)
    lab = torch.randint(-1, 3, (N,), generator=gen).to(DEV)
    rows = (10 + torch.randn(N, generator=gen)).to(DEV)
    n, inv, mean, one = torch.empty(4, device=DEV).split(1)
    size = _lib.workspace_bytes("sisa_ce_workspace_bytes", N)
    assert 8 <= size <= 8 * 256
    ws = torch.full((size // 8 + 1,), -7, dtype=torch.int64, device=DEV)
    _lib.call_values("sisa_ce_count_wide", n, lab.data_ptr(), N, -1, n.data_ptr(), inv.data_ptr(), ws.data_ptr())
    _lib.call_values("sisa_ce_mean_wide", n, rows.data_ptr(), N, n.data_ptr(), mean.data_ptr(), ws.data_ptr())
    _lib.call_values("sisa_ce_mean", n, rows.data_ptr(), N, n.data_ptr(), one.data_ptr())
    assert int(ws[-1]) == -7
    count = int((lab != -1).sum())
    assert float(n) == count and torch.equal(inv, torch.reciprocal(n))
    want = rows.double().sum() / count
    if count:       # one rounding of the sum, one of the quotient
        assert abs(float(mean) - float(want)) <= 2 * 2.0 ** -24 * abs(float(want))
        assert torch.equal(mean, one)               # fp64 sums round to fp32 alike in any order


@pytest.mark.gpu
def test_scalars_in_a_captured_call():
    """Training and evaluation of more rows than one workgroup counts, replayed between eager work, give the eager bits."""
    from sisa_amd.kernels.linear_ce import linear_cross_entropy
    x, w, lab = _case((1 << 16) + 77, 64, 130, 5)
    w, other = w.float(), lab.roll(1)

    def both(labels):
        xg, wg = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
        loss = linear_cross_entropy(xg, wg, labels)
        dx, dw = torch.autograd.grad(loss, (xg, wg))
        with torch.no_grad():
            return loss.detach(), dx, dw, linear_cross_entropy(x, w, labels)
    eager = [t.clone() for t in both(lab)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        both(lab)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = both(lab)
    for _ in range(4):
        both(other)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, eager))


@pytest.mark.gpu
@pytest.mark.parametrize("N", [1 << 15, (1 << 15) + 1])
def test_rows_at_the_line_of_the_scalar_kernels(N):
    """One workgroup counts and averages up to 32,768 rows, several beyond. Both against float64."""
    from sisa_amd.kernels.linear_ce import linear_cross_entropy
    x, w, lab = _case(N, 64, 130, 3)
    got, ref = _run(x, w, lab), _truth(x, w, lab)
    # logits rounded to 8 bits shift the loss by the mean of their errors; gradients: three 8-bit roundings
    assert abs(float(got[0] - ref[0])) <= 2 ** -8 * (1 + abs(float(ref[0])))
    assert _rel(got[1], ref[1]) <= 3 * 2 ** -8 and _rel(got[2], ref[2]) <= 3 * 2 ** -8
    with torch.no_grad():
        assert torch.equal(linear_cross_entropy(x, w.float(), lab), got[0])
