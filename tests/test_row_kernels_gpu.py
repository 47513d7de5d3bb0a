"""The kernels of a decode step that have a row or a few to work on, at the edges of what a thread and a workgroup take."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from llm_infer_amd.kernels import ops
    return ops


# rows of whole quads and not, shared by one workgroup and by several, of a table that is 16-byte aligned and not
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,d,shift", [(1, 1, 0), (1, 7, 0), (3, 1024, 0), (2, 1028, 0), (5, 4100, 0), (255, 260, 0), (256, 260, 0), (300, 2049, 0),
                                       (2, 64, 4), (2, 66, 1)])
def test_gathered_rows(ops, dtype, n, d, shift):
    table = torch.randn(50 * d + shift, device=DEV, dtype=dtype)[shift:].view(50, d)
    ids = torch.randint(0, 50, (n,), device=DEV, dtype=torch.int32)
    assert torch.equal(ops.embed(table, ids), table[ids.long()].float())
    if d % 2:
        return
    pos = torch.randint(0, 5000, (n,), device=DEV, dtype=torch.int32)
    freq = 10000.0 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    got = ops.embed_positions(table, ids, pos, freq, 1.5).double()
    angle = pos.double()[:, None] * freq.double()
    want = table[ids.long()].double() * 1.5
    want[:, 0::2] += angle.sin()
    want[:, 1::2] += angle.cos()
    # the angle rounds to float32 once (half an ulp of it), sine, product and sum to some ulps of their size
    bound = angle.repeat_interleave(2, 1) * 2.0 ** -24 + 4 * 2.0 ** -23 * (1 + want.abs())
    assert ((got - want).abs() <= bound).all()


# index arrays one behind the other while the device is busy, of one row, two rows and none: every one keeps its own values
def test_uploads_behind_queued_work(ops):
    a = torch.randn(4096, 4096, device=DEV)
    torch.cuda.synchronize()
    for _ in range(20):
        a = (a @ a).clamp_(-1, 1)
    values = [[[i * 1000 + j for j in range(1 + i * 37 % 5000)]] * (1 + i % 2) for i in range(200)] + [[], [[], []]]
    there = [ops.upload(v if len(v) != 1 else v[0], DEV) for v in values]
    for v, t in zip(values, there):
        assert t.dtype == torch.int32 and t.tolist() == (v if len(v) != 1 else v[0])


# also where the page-locked memory is there already and nothing else would refuse
def test_no_upload_into_a_graph(ops):
    from llm_infer_amd.kernels.ops import KernelError
    x = torch.zeros(4, device=DEV)
    for _ in range(4):
        ops.upload([7, 7, 7], DEV)
        torch.cuda.synchronize()
    free = [torch.empty(3, dtype=torch.int32, pin_memory=True) for _ in range(4)]
    del free
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        x.add_(1.0)
        with pytest.raises(KernelError):
            ops.upload([1, 2, 3], DEV)
    for n in (1, 2, 3):
        graph.replay()
        assert x.tolist() == [float(n)] * 4


# one chunk, the edges between chunks and between a thread's elements, ties: the first of the largest
@pytest.mark.parametrize("v", [1, 63, 255, 257, 4095, 4096, 4097, 8193, 32000])
def test_argmax_first_of_the_largest(ops, v):
    x = torch.randint(0, 50, (5, v), device=DEV).float()
    x[1] = -torch.inf
    x[2, v // 2:] = 60.0
    x[3, -1] = 70.0
    x[4, 0] = 70.0
    assert ops.argmax(x).tolist() == [int((r == r.max()).nonzero()[0]) for r in x.cpu()]


def _rms(v, eps):
    return (v.pow(2).mean(1, keepdim=True) + eps).sqrt()


def _ln(v, eps):
    d = v - v.mean(1, keepdim=True)
    return d / (d.pow(2).mean(1, keepdim=True) + eps).sqrt()


def _close(got, want):
    """Within what float32 sums and some ten roundings of a row leave: 2e-6 of its size, and half a unit of a 16-bit type."""
    unit = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[got.dtype]
    err = (got.double() - want).abs()
    assert (err <= 2e-6 * want.abs().amax(1, keepdim=True) + (unit * 1.01) * want.abs()).all(), err.max()


# rows that leave waves without elements, quads a thread of 1, 2, 4 and 8, the last that is kept and the first that is not
WIDTHS = [4, 60, 256, 260, 1024, 1028, 2048, 2052, 4096, 4100, 8188, 8192, 8196]


@pytest.mark.parametrize("width", WIDTHS + [37])
def test_normed_sum_of_few_rows_and_many(ops, width):
    x, y, z = (torch.randn(65, width, device=DEV) for _ in range(3))
    w, b, nw, v = (torch.rand(width, device=DEV) + 0.5 for _ in range(4))
    for bias in (None, b):
        for also in (None, (None, v), (z, v)):
            want = x.double() + (lambda t: t / _rms(t, 1e-5) * w.double())(y.double() + (bias.double() if bias is not None else 0))
            if also:
                want = want + v.double() + (z.double() if also[0] is not None else 0)
            made = {}
            for rows in (1, 64, 65):
                out = x[:rows].clone()
                extra = also and (also[0] if also[0] is None else z[:rows].contiguous(), v)
                ops.rmsnorm_add(out, y[:rows].contiguous(), w, 1e-5, bias, (nw, 1e-6, torch.float16), extra)
                made[rows] = (out, ops.prepared_rmsnorm(out, nw, 1e-6, torch.float16))
                _close(out, want[:rows])
                _close(made[rows][1], (want / _rms(want, 1e-6) * nw.double())[:rows])
            for rows in (1, 64):                              # the two kernels give the same values
                assert all(torch.equal(a, c[:rows]) for a, c in zip(made[rows], made[65]))


@pytest.mark.parametrize("mean", [0.0, 3.0])
@pytest.mark.parametrize("width", WIDTHS + [37])
def test_layer_norms_of_sums(ops, width, mean):
    x, y, y2 = (torch.randn(9, width, device=DEV) + mean for _ in range(3))
    w, b, nw, nb = (torch.rand(width, device=DEV) + 0.5 for _ in range(4))
    xd, yd, y2d = x.double(), y.double(), y2.double()
    out = x.clone()
    ops.layernorm_add(out, y, w, b, 1e-5, (nw, nb, 1e-5, torch.bfloat16))
    want = xd + _ln(yd, 1e-5) * w.double() + b.double()
    _close(out, want)
    _close(ops.prepared_norm(out, nw, 1e-5, torch.bfloat16), _ln(want, 1e-5) * nw.double() + nb.double())
    pair = ops.NormedPair(y, w, y2, b, 1e-5, 0.5)
    out = x.clone()
    ops.layernorm_add(out, pair, nw, nb, 1e-5)
    both = 0.5 * (yd / _rms(yd, 1e-5) * w.double() + y2d / _rms(y2d, 1e-5) * b.double())
    _close(out, xd + _ln(both, 1e-5) * nw.double() + nb.double())
    for adds in ([(y, 0.5)], [(y, 0.5), (y2, 2.0)]):
        out = x.clone()
        copy = ops.add_layernorm(out, 2.0, adds, w, 1e-5, torch.bfloat16)
        want = _ln(2 * xd + sum(s * t.double() for t, s in adds), 1e-5) * w.double()
        _close(out, want)
        assert torch.equal(copy, out.to(torch.bfloat16))


# rows whose pieces come one by one: four and eight a thread, the last workgroup of 512 threads and the first of more, the last row that is
# kept in registers and the first that is not
@pytest.mark.parametrize("width", [8192, 8196, 16384, 16388, 32768, 32772])
def test_layer_norms_of_sums_of_wide_rows(ops, width):
    x, y, y2, w = torch.randn(3, width, device=DEV), torch.randn(3, width, device=DEV) + 2, torch.randn(3, width, device=DEV), torch.rand(width, device=DEV) + 0.5
    for adds in ([(y, 0.5)], [(y, 0.5), (y2, 2.0)]):
        out = x.clone()
        copy = ops.add_layernorm(out, 2.0, adds, w, 1e-5, torch.float16)
        _close(out, _ln(2 * x.double() + sum(s * t.double() for t, s in adds), 1e-5) * w.double())
        assert torch.equal(copy, out.to(torch.float16))


# whole numbers whose mean is 0 and whose squares add up to less than 2^24: every sum is exact in float32 in any order, if the mean is taken
# before the deviations, and then only roots, divisions and products round, once each (numpy's are correctly rounded, as the kernels' are)
@pytest.mark.parametrize("width", WIDTHS + [37])
def test_a_layer_norms_deviations_are_from_the_rows_mean(ops, width):
    v = np.random.default_rng(width).integers(-8, 9, (9, width)).astype(np.float32)
    v[:, -1] -= v.sum(1)
    v += np.sign(v[:, :1] + 0.5) * (np.arange(width) == 0) - np.sign(v[:, :1] + 0.5) * (np.arange(width) == width - 1)
    dev, one = (v * v).sum(1, keepdims=True), torch.ones(width, device=DEV)
    assert v.dtype == np.float32 and (v.sum(1) == 0).all() and dev.max() < 2 ** 24 and dev.min() > 0
    rows = torch.from_numpy(v).to(DEV)
    out = rows.clone()
    ops.add_layernorm(out, 1.0, [(torch.zeros_like(out), 1.0)], one, 0.0)
    assert np.array_equal(out.cpu().numpy(), v / np.sqrt(dev / np.float32(width)))
    out = torch.zeros(9, width, device=DEV)
    ops.layernorm_add(out, rows, one, torch.zeros(width, device=DEV), 0.0)
    assert np.array_equal(out.cpu().numpy(), v * (np.float32(1) / np.sqrt(dev * (np.float32(1) / np.float32(width)))))


@pytest.mark.parametrize("n", WIDTHS + [37, 14336, 16384, 16388])
def test_gated_norm_and_polynorm_of_a_row(ops, n):
    o, w = torch.randn(3, n, device=DEV), torch.rand(n, device=DEV) + 0.5
    want = o.double() / _rms(o.double(), 1e-5) * w.double()
    for stride, col in ((n, 0), (n + 8, 4), (n + 3, 3)):           # gates that are 16-byte aligned and not
        gate = torch.randn(3, stride, device=DEV)
        _close(ops.gated_rmsnorm(o, w, gate, col, 1e-5, torch.float16), want * torch.sigmoid(gate[:, col:col + n].double()))
    coef = torch.tensor([0.5, -0.3, 0.2, 0.1], device=DEV)
    d = o.double()
    _close(ops.polynorm(o, coef, 1e-5, torch.bfloat16), sum(c * d ** k / _rms(d ** k, 1e-5) for k, c in ((1, 0.5), (2, -0.3), (3, 0.2))) + 0.1)


# a row's sum over every number of waves that a workgroup may have (whole numbers: exact in any order, and a wave left out or taken twice shows)
@pytest.mark.parametrize("waves", range(1, 17))
def test_sums_over_any_number_of_waves(ops, waves):
    n = 256 * waves
    v = np.random.default_rng(waves).integers(-8, 9, (3, n)).astype(np.float32)
    v[:, :64] = 16.0 + waves
    squares = (v * v).sum(1, keepdims=True)
    assert squares.max() < 2 ** 24
    out = ops.gated_rmsnorm(torch.from_numpy(v).to(DEV), torch.ones(n, device=DEV), torch.full((3, n), 100.0, device=DEV), 0, 0.0, torch.float32)
    assert np.array_equal(out.cpu().numpy(), v / np.sqrt(squares / np.float32(n)))     # (the sigmoid of 100 is 1)


# many rows, a workgroup of 256 threads: the last and first of 16, 24 and 32 elements a thread, and of batches of 8
@pytest.mark.parametrize("n", [4096, 4097, 6144, 6145, 8192, 8193, 10240, 10241])
def test_gated_norm_of_many_wide_rows(ops, n):
    o, w, gate = torch.randn(256, n, device=DEV), torch.rand(n, device=DEV) + 0.5, torch.randn(256, n, device=DEV)
    want = o.double() / _rms(o.double(), 1e-5) * w.double() * torch.sigmoid(gate.double())
    for dt in (torch.float16, torch.float32):
        _close(ops.gated_rmsnorm(o, w, gate, 0, 1e-5, dt), want)


@pytest.mark.parametrize("terms", [1, 3, 4, 5, 9])
@pytest.mark.parametrize("width", WIDTHS[:-1])
def test_average_over_depth_with_its_norms(ops, width, terms):
    hist, weights = torch.randn(terms + 1, 3, width, device=DEV), torch.rand(terms, device=DEV)
    hist[terms] = torch.nan                                        # behind the last term: nothing of it may be seen
    nw = torch.rand(width, device=DEV) + 0.5
    norms = [(nw, 1e-5, torch.float16), (nw, 1e-6, torch.float32)]
    out = torch.empty(3, width, device=DEV)
    ops.average_norms(hist, terms, weights, out, norms)
    plain = ops.depth_average(hist, terms, weights, torch.empty_like(out))
    assert torch.equal(out, plain)
    for w, eps, dt in norms:
        assert torch.equal(ops.prepared_norm(out, w, eps, dt), ops.rmsnorm(plain, w, eps, dt))
    each = hist[:terms].double() * weights.double()[:, None, None]
    # a rounding of 2^-24 for every product and sum
    assert ((out - each.sum(0)).abs() <= 2 * terms * 2.0 ** -24 * each.abs().sum(0)).all()
    weights[0] = 0.0                                               # a term of weight 0 that is not finite shows, there and nowhere else
    hist[0, 1, width - 1], hist[0, 2, 0] = torch.inf, torch.nan
    got = ops.average_norms(hist, terms, weights, torch.empty_like(out), norms)
    bad = torch.zeros(3, width, dtype=torch.bool, device=DEV)
    bad[1, width - 1] = bad[2, 0] = True
    assert torch.equal(got.isnan(), bad) and torch.equal(ops.depth_average(hist, terms, weights, torch.empty_like(out)).isnan(), bad)


# a row shorter than a wave's first loads, ragged against them, whole, of the wider form and beyond it; few tokens against many
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("t,width,n", [(1, 4, 1), (3, 260, 8), (5, 2048, 16), (2, 2052, 9), (255, 1028, 17), (4, 4096, 9), (2, 66, 4), (2, 4100, 4)])
def test_router_logits_of_few_tokens(ops, dtype, t, width, n):
    h, w, bias = torch.randn(t, width, device=DEV).to(dtype), torch.randn(n, width, device=DEV) * width ** -0.5, torch.randn(n, device=DEV)
    z = ops.small_logits(h, w, bias)
    want = h.double() @ w.double().T + bias.double()
    # 16 sums of a lane, 4 of lanes, 2 of quads, 4 of waves: some 30 roundings at the most, 2^-19 of the products' absolute sum
    assert ((z - want).abs() <= 2.0 ** -19 * (1 + h.double().abs() @ w.double().abs().T + bias.double().abs())).all()
    assert torch.equal(ops.small_logits(h.repeat(256 // t + 1, 1), w, bias)[:t], z)


# rows of a state that divide among a thread's and not, columns that split over workgroups and not; a sequence alone (its heads'
# columns over several workgroups where they can) and among 256 (a workgroup a head), step by step, bit for bit, and against 64 bits
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d,dv", [(4, 80, 96), (16, 128, 128), (3, 33, 64), (2, 256, 64), (5, 20, 48), (1, 7, 1), (2, 128, 256)])
def test_decay_recurrence_of_one_sequence_and_many(ops, dtype, H, d, dv):
    n, steps = 256, 3
    decay = torch.linspace(0.5, 0.99, H, device=DEV)
    many, alone = torch.randn(n, H, d, dv, device=DEV), None
    alone = many[7:8].clone()
    S = alone.double()[0].cpu()
    rounded = dtype if dtype != torch.float32 else None
    for _ in range(steps):
        proj = torch.randn(n, H * (2 * d + dv), device=DEV)
        o = ops.decay_attention(proj, 0, H * d, 2 * H * d, many, decay, torch.arange(n, device=DEV, dtype=torch.int32), None, None, n, H, d, dv,
                                round_to=rounded)
        one = ops.decay_attention(proj[7:8].contiguous(), 0, H * d, 2 * H * d, alone, decay, torch.zeros(1, device=DEV, dtype=torch.int32), None, None, 1,
                                  H, d, dv, round_to=rounded)
        assert torch.equal(one[0], o[7]) and torch.equal(alone[0], many[7])
        if rounded is None:
            q, k, v = (torch.nn.functional.silu(p.double()) for p in proj[7].cpu().split([H * d, H * d, H * dv]))
            S = decay.double().cpu()[:, None, None] * S + k.view(H, d, 1) * v.view(H, 1, dv)
            want = (S * q.view(H, d, 1)).sum(1)
            # some 100 roundings of 2^-24 in a sum of up to 256 products of the order of 1
            assert ((one[0].view(H, dv).double().cpu() - want).abs() <= 2.0 ** -17 * (S * q.view(H, d, 1)).abs().sum(1) + 1e-6).all()


# tokens one by one and all at once, for one workgroup a CU and for more, of 32 and 64 rows a thread, whole and not, columns that split and
# that do not: the same arithmetic in the same order
@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (100, 128), (128, 256), (256, 256), (200, 256), (256, 255), (200, 255)])
@pytest.mark.parametrize("n", [1, 70])
def test_decayed_attention_steps_and_prompts(ops, d, dv, n):
    H, T = 4, 5
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    proj, decay = torch.randn(n * T, H * (2 * d + dv), device=DEV), torch.rand(H, device=DEV) * 0.5 + 0.5
    at_once = torch.randn(n, H, d, dv, device=DEV)
    by_one, S = at_once.clone(), at_once[0].double().cpu()
    args = (0, H * d, 2 * H * d)
    o = ops.decay_attention(proj, *args, at_once, decay, i32(list(range(n))), i32([i * T for i in range(n)]), i32([T] * n), n, H, d, dv)
    for t in range(T):
        one = ops.decay_attention(proj[t::T].contiguous(), *args, by_one, decay, i32(list(range(n))), None, None, n, H, d, dv)
        assert torch.equal(one, o[t::T])
        q, k, v = (torch.nn.functional.silu(p.double()) for p in proj[t].cpu().split([H * d, H * d, H * dv]))
        S = decay.double().cpu()[:, None, None] * S + k.view(H, d, 1) * v.view(H, 1, dv)
        size = (S * q.view(H, d, 1)).abs().sum(1)
        # some 100 roundings of 2^-24 in a sum of up to 256 products of the order of 1
        assert ((one[0].view(H, dv).double().cpu() - (S * q.view(H, d, 1)).sum(1)).abs() <= 2.0 ** -17 * size + 1e-6).all()
    assert torch.equal(at_once, by_one)


# tokens one by one and all at once, by the kernel that knows of one token and by the one that walks a prompt: the same bits
@pytest.mark.parametrize("rows,cols", [(16, 64), (20, 30), (64, 64), (128, 64), (100, 100), (256, 70)])
@pytest.mark.parametrize("n", [1, 40])
def test_state_space_steps_and_prompts(ops, rows, cols, n):
    from types import SimpleNamespace
    H, T = 4, 5
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    step = SimpleNamespace(seq_slot=i32(list(range(n))), n_seqs=n, n_tokens=n)
    prompt = SimpleNamespace(seq_slot=step.seq_slot, n_seqs=n, n_tokens=n * T, seq_qstart=i32([i * T for i in range(n)]), seq_qlen=i32([T] * n))
    xbc, proj = torch.randn(n * T, H * cols + 2 * rows, device=DEV), torch.randn(n * T, H, device=DEV)
    bias, alog, skip = torch.randn(H, device=DEV), torch.randn(H, device=DEV) * 0.3, torch.randn(H, device=DEV)
    at_once = torch.randn(n, H, rows, cols, device=DEV)
    by_one = at_once.clone()
    y = ops.ssm_scan(xbc, proj, 0, bias, alog, skip, at_once, prompt, H, 1, rows, cols, None)
    for t in range(T):
        one = ops.ssm_scan(xbc[t::T].contiguous(), proj[t::T].contiguous(), 0, bias, alog, skip, by_one, step, H, 1, rows, cols, None)
        assert torch.equal(one, y[t::T])
    assert torch.equal(at_once, by_one)


# one token a sequence with a state whose rows and columns are all there (fetched under no condition), and with rows or columns that a
# wave has not; three steps in a row against 64 bits
@pytest.mark.parametrize("rows,cols", [(64, 64), (128, 128), (64, 40), (100, 64), (7, 130), (16, 64), (256, 64)])
def test_recurrences_with_whole_and_ragged_states(ops, rows, cols):
    from types import SimpleNamespace
    n, H = 3, 2
    ctx = SimpleNamespace(seq_slot=torch.tensor([2, 0, 1], dtype=torch.int32, device=DEV), n_seqs=n, n_tokens=n)
    slot = ctx.seq_slot.long()
    r = lambda *s: torch.randn(*s, device=DEV)
    # a sum of up to 256 products takes up to 8 + rows / 4 roundings of 2^-24 in a row; three steps, factors of the order of 1
    near = lambda got, want, size: bool(((got.double() - want).abs() <= 2.0 ** -16 * (1 + size)).all())
    delta, ssm, wkv = r(n, H, rows, cols), r(n, H, rows, cols), r(n, H, rows, rows)
    D, M, W = (s.double()[slot].clone() for s in (delta, ssm, wkv))
    for _ in range(3):
        x, g, kq = r(n, 2 * H * rows + H * cols) * rows ** -0.5, torch.stack([-torch.rand(n, H, device=DEV), torch.rand(n, H, device=DEV)], -1), r(n, H)
        q, k, v = (p.double() for p in x.split([H * rows, H * rows, H * cols], 1))
        q, k, v = q.view(n, H, rows, 1), k.view(n, H, rows, 1), v.view(n, H, 1, cols)
        kq = (q * k).sum((2, 3)).float().contiguous()
        o = ops.delta_scan(x, g.contiguous(), kq, delta, ctx, H, H, rows, cols).view(n, H, cols)
        D = D * g[..., 0].double().exp()[..., None, None]
        D = D + k * (g[..., 1].double()[..., None, None] * (v - (D * k).sum(2, keepdim=True)))
        assert near(o, (D * q).sum(2), (D * q).abs().sum(2)) and near(delta[slot], D, D.abs())

        xbc, proj, bias, alog, skip = r(n, H * cols + 2 * rows), r(n, H), r(H), r(H) * 0.3, r(H)
        y = ops.ssm_scan(xbc, proj, 0, bias, alog, skip, ssm, ctx, H, 1, rows, cols, None).view(n, H, cols)
        xs, B, C = (p.double() for p in xbc.split([H * cols, rows, rows], 1))
        dt = torch.nn.functional.softplus(proj.double() + bias.double())[..., None, None]
        M = M * (-alog.double().exp()[:, None, None] * dt).exp() + dt * B.view(n, 1, rows, 1) * xs.view(n, H, 1, cols)
        want = (M * C.view(n, 1, rows, 1)).sum(2) + skip.double()[:, None] * xs.view(n, H, cols)
        assert near(y, want, (M * C.view(n, 1, rows, 1)).abs().sum(2)) and near(ssm[slot], M, M.abs())

        a, kk, vv, raw, bonus = r(n, H * rows), r(n, H * rows), r(n, H * rows), r(n, H * rows), r(H, rows)
        o = ops.wkv_scan(a, kk, vv, raw, bonus, wkv, ctx, H, rows).view(n, H, rows)
        ad, kd, vd = a.double().view(n, H, rows, 1), kk.double().view(n, H, rows, 1), vv.double().view(n, H, 1, rows)
        seen = W + bonus.double()[..., None] * kd * vd
        assert near(o, (seen * ad).sum(2), (seen * ad).abs().sum(2))
        W = W * (-raw.double().view(n, H, rows, 1).exp()).exp() + kd * vd
        assert near(wkv[slot], W, W.abs())


# the first addition of a wave's sum takes its product unrounded: (1 + 2^-12)^2 in lane 0 and its rounding, with the other sign, half a wave
# on leave 2^-24
@pytest.mark.parametrize("d", [64, 128])
def test_a_bonus_enters_its_sum_unrounded(ops, d):
    from types import SimpleNamespace
    ctx = SimpleNamespace(seq_slot=torch.zeros(1, dtype=torch.int32, device=DEV), n_seqs=1, n_tokens=1)
    r, k, bonus, v = torch.zeros(1, d, device=DEV), torch.zeros(1, d, device=DEV), torch.ones(1, d, device=DEV), torch.ones(1, d, device=DEV)
    r[0, 0] = k[0, 0] = 1 + 2.0 ** -12
    r[0, 32], k[0, 32] = -(1 + 2.0 ** -11), 1.0
    o = ops.wkv_scan(r, k, v, torch.zeros_like(r), bonus, torch.zeros(1, 1, d, d, device=DEV), ctx, 1, d)
    assert torch.equal(o, torch.full_like(o, 2.0 ** -24))


# value sizes in whole fours (four dimensions a store) and not, one split and several, against the kernel that takes a key after
# the other
@pytest.mark.parametrize("dk,dv,vdim", [(16, 32, 32), (16, 30, 32), (64, 64, 64), (64, 49, 64), (64, 60, 64)])
@pytest.mark.parametrize("H", [6, 66])                 # query heads of a KV head for one workgroup and for two
def test_sigmoid_attention_value_sizes(ops, dk, dv, vdim, H):
    G, n, B = 2, 150, 3
    pages = 3
    k = (torch.randn(B * pages, G, 64 * dk, device=DEV) * 0.5).bfloat16()
    v = torch.randn(B * pages, G, 64 * ((vdim + 31) // 32 * 32), device=DEV).bfloat16()
    table = torch.arange(B * pages, device=DEV, dtype=torch.int32).view(B, pages).contiguous()
    slot = torch.arange(B, device=DEV, dtype=torch.int32)
    wide = max(k.stride(0), v.stride(0))                           # pages of keys and of values have one stride
    k, v = (torch.nn.functional.pad(p.view(B * pages, -1), (0, wide - p.stride(0))).contiguous() for p in (k, v))
    kv = (k, v, k.stride(0), table)
    q = torch.randn(B, H, dk, device=DEV).bfloat16()
    ctx = torch.tensor([n, 64, 1], device=DEV, dtype=torch.int32)
    want = ops.sigmoid_attention(q, kv, ctx - 1, slot, None, H, G, dk, dv, vdim, dk ** -0.5).float()
    for splits in (1, 3):
        got = ops.sigmoid_attention_decode(q, kv, slot, ctx, B, None, H, G, dk, dv, vdim, dk ** -0.5, None, splits).float()
        # weights as two 16-bit numbers and in float32: 2^-16 of the up to 150 addends' absolute sum, some 120; then both round to 8
        # bits, where sums that differ by a hair may become neighbours, up to 2^-7 of their size apart
        assert got.shape == want.shape and ((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -9).all(), splits


# outputs of a head in whole fours and not, rows and heads that begin at fours and not, with and without a gate
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n_in,n_out,col,pad", [(64, 64, 0, 0), (64, 64, 2, 0), (128, 36, 0, 4), (40, 100, 4, 3), (96, 33, 0, 0), (8, 6, 0, 2)])
def test_products_per_head_of_few_tokens(ops, dtype, n_in, n_out, col, pad):
    H, t = 3, 5
    w, x = (torch.randn(H, n_out, n_in, device=DEV) * n_in ** -0.5).to(dtype), torch.randn(t, H * n_in, device=DEV).to(dtype)
    want = torch.einsum("hji,thi->thj", w.double().cpu(), x.double().cpu().view(t, H, n_in))
    for gate_col in (None, 0, 1):
        out = torch.full((t, col + H * (n_out + pad) + 1), 7.0, device=DEV, dtype=dtype)
        gate = torch.randn(t, H * n_out + 5, device=DEV)
        kw = {} if gate_col is None else {"gate": gate, "gate_col": gate_col}
        ops.head_linear(x, 0, n_in, w, out, col, n_out + pad, **kw)
        ref = want if gate_col is None else want * torch.sigmoid(gate.double().cpu())[:, gate_col:gate_col + H * n_out].view(t, H, n_out)
        got = out[:, col:col + H * (n_out + pad)].reshape(t, H, n_out + pad).double().cpu()
        eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
        assert ((got[:, :, :n_out] - ref).abs() <= eps * ref.abs() + 2.0 ** -16).all()       # one rounding, and float32 sums
        assert (got[:, :, n_out:] == 7.0).all() and (out[:, :col] == 7.0).all() and (out[:, -1] == 7.0).all()
