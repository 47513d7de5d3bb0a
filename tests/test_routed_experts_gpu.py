"""Routed experts of long prompts (``RoutedExperts``): tokens sorted by expert, products by pairs of token and chosen expert,
against a plain implementation in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

GATED, CLAMPED, PLAIN_IN, PLAIN_OUT = "gated", "clamped", "without a gate, weight on the input", "without a gate, weight on the output"
FORMS = (GATED, CLAMPED, PLAIN_IN, PLAIN_OUT)
LIMIT, ALPHA, SHIFT = 1.2, 1.702, 1.0


def build(form, d, n, ff, top, identity=0, shared=0, seed=0):
    """The part and its tensors: matrices of bfloat16 numbers, a router that reads one column an output."""
    from llm_infer_amd.parts.feed_forward import RoutedExperts
    from llm_infer_amd.weights.loader import place_tensor
    kinds = {GATED: {}, CLAMPED: dict(activation="clamped_swish", limit=LIMIT, alpha=ALPHA, up_shift=SHIFT),
             PLAIN_IN: dict(gated=False, activation="relu2", weight_on="input"), PLAIN_OUT: dict(gated=False, activation="silu")}
    part = RoutedExperts(hidden_size=d, n_experts=n, expert_ff=ff, top=top, n_identity=identity, correction=True, route_scale=1.3,
                         shared_ff=shared, shared_gate=False, prefix="", dtype=torch.bfloat16, device=DEV, **kinds[form])
    g = torch.Generator().manual_seed(seed)
    wanted = part.params()
    W = {k: (torch.randn(*v.shape, generator=g) * v.shape[-1] ** -0.5 * 1.5).bfloat16() for k, v in wanted.items()}
    W["router.weight"] = torch.zeros(n + identity, d, dtype=torch.bfloat16)
    W["router.weight"][torch.arange(n + identity), torch.arange(n + identity)] = 2.0
    W["router.correction"] = torch.zeros(n + identity, dtype=torch.bfloat16)
    part.bind({k: place_tensor(W[k], wanted[k].kind, torch.bfloat16, DEV) for k in wanted})
    return part, W


def inputs(T, d, outputs, seed=1):
    """Rows whose router logits are far apart, every token its own order of the outputs."""
    g = torch.Generator().manual_seed(seed)
    h = 0.3 * torch.randn(T, d, generator=g)
    h[:, :outputs] = torch.rand(T, outputs, generator=g).argsort(-1).float() * (3.0 / outputs)
    return h.bfloat16()


def test_a_long_prompt_takes_bounded_memory():
    """Portions of the tokens: the same numbers, bit for bit, and a working memory that does not grow with the prompt."""
    for form in FORMS:
        part, W = build(form, 64, 4, 96, 2)
        T = 3001
        h = inputs(T, 64, 4).to(DEV)
        outs, peaks = [], []
        for numbers in (part.PAIR_NUMBERS, 2 * 96 * 500, 2 * 96 * 21):     # one portion; seven; the first 63 tokens in three, of the tiles of few rows
            part.PAIR_NUMBERS = numbers
            rows = h if numbers != 2 * 96 * 21 else h[:63].contiguous()
            res = torch.zeros(rows.shape[0], 64, device=DEV)
            weights = part._weights(rows, res, None)
            part._by_pairs(rows, res, weights)                             # (kernels loaded, scratch kept)
            res.zero_()
            torch.cuda.synchronize()
            before = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            part._by_pairs(rows, res, weights)
            peaks.append(torch.cuda.max_memory_allocated() - before)
            outs.append(res)
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0][:63], outs[2]), form
        # rows, the up product's sums and the hidden rows of 500 tokens' pairs, the pairs' lists, and the allocator's rounding
        assert peaks[1] < 500 * 2 * (4 * 64 + 4 * 96 + 2 * 96 + 40) + (1 << 16) < peaks[0], (form, peaks)


def hidden(form, z):
    """(value, weight goes inside) of an expert's up products in float64."""
    if form == GATED:
        return torch.nn.functional.silu(z[..., 0::2]) * z[..., 1::2]
    if form == CLAMPED:
        g, u = z[..., 0::2].clamp(max=LIMIT), z[..., 1::2].clamp(-LIMIT, LIMIT)
        return g * torch.sigmoid(ALPHA * g) * (u + SHIFT)
    return torch.relu(z) ** 2 if form == PLAIN_IN else torch.nn.functional.silu(z)


def plain(form, h, W, n, outputs, top, shared):
    """What the layer adds to a token's row, and per element the sum of the absolute products (what rounding errors scale with)."""
    h, W = h.double(), {k: v.double() for k, v in W.items()}
    s = torch.softmax(h @ W["router.weight"].T, -1)
    chosen = torch.topk(s, top, dim=-1).indices
    w = torch.zeros(h.shape[0], outputs, dtype=torch.float64).scatter_(1, chosen, torch.gather(s, 1, chosen))
    w = w / (w.sum(-1, keepdim=True) + 1e-20) * 1.3
    out = w[:, n:].sum(-1, keepdim=True) * h
    size = out.abs()
    for p, we in [(f"e{e}.", w[:, e:e + 1]) for e in range(n)] + ([("shared.", torch.ones(h.shape[0], 1, dtype=torch.float64))] if shared else []):
        up = W[p + "up"]
        if form in (GATED, CLAMPED):
            up = torch.stack([W[p + "gate"], up], 1).reshape(2 * up.shape[0], -1)
        z = h @ up.T
        t = hidden(form, we * z) if form == PLAIN_IN else we * hidden(form, z)
        t = torch.where(we == 0, torch.zeros_like(t), t)
        out, size = out + t @ W[p + "down"].T, size + t.abs() @ W[p + "down"].abs().T
    return out, size, w


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("ff", [48, 64])       # 64: by pairs, 48 (no multiple of 32): one expert after another
def test_sorted_by_expert_and_every_token_through_every_expert(form, ff):
    d, n, identity, top, shared, T = 64, 4, 2, 3, 32, 700
    part, W = build(form, d, n, ff, top, identity, shared)
    assert (part.pair_weights is not None) == (ff % 32 == 0) and part.per_expert is not None
    h = inputs(T, d, n + identity)
    ref, size, w = plain(form, h, W, n, n + identity, top, shared)
    used = (w[:, :n] != 0).sum(-1)
    assert used.min() == 1 and used.max() == top         # tokens with fewer pairs than `top`: the others of theirs pass them on
    for limit in (1, 10 ** 9):
        part.GROUPED_FROM = limit
        res = torch.ones(T, d, device=DEV)
        part.forward(h.to(DEV), res)
        # a hidden value is rounded to bfloat16 (8 bits) at most twice (before and after its weight), each time by 2^-8 of itself at
        # most; what float32 adds is far below
        assert bool(((res.cpu().double() - 1.0 - ref).abs() <= 2.0 ** -7 * size + 1e-5).all()), limit
        into = torch.full((T, d), 7.0, device=DEV)
        part.forward_into(h.to(DEV), into)
        assert bool(((into.cpu().double() - ref).abs() <= 2.0 ** -7 * size + 1e-5).all()), limit


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,K,F,counts", [(4, 2080, 48, [0, 17, 1, 33]), (3, 128, 160, [129, 0, 400]), (9, 64, 64, [64, 65, 0, 128, 1, 127, 0, 63, 300]),
                                          (70, 96, 16, [0] * 30 + [2] + [0] * 30 + [40, 1] + [0] * 7)])
def test_clamped_activation_by_pairs_in_every_kernel(dtype, E, K, F, counts):
    """Every tile, at experts without pairs, with one, and at a tile's edges."""
    from llm_infer_amd.kernels import ops
    g = torch.Generator().manual_seed(E + K)
    T = sum(counts)
    expert = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)]
    dense = torch.zeros(T, E)
    dense[torch.arange(T), expert] = 1.0
    p = ops.pairs_of_weights(dense.to(DEV), E, 1)
    x = torch.randn(T, K, generator=g).to(dtype)
    w = (torch.randn(E, 2 * F, K, generator=g) * K ** -0.5 * 2).to(dtype)
    wt = ops.prepare_weight(w.view(E * 2 * F, K).to(DEV))
    row_of = p.row_of.cpu().long()
    for gather in (True, False):
        rows = x[row_of].double() if gather else x.double()
        own = w[expert[row_of]].double()
        z = torch.bmm(own, rows[:, :, None])[:, :, 0]
        ref = hidden(CLAMPED, z)
        # the result's rounding to its type (2^-8 of itself at most in bfloat16, 2^-11 in float16), and a product's own error, K roundings of float32 of the sum of
        # its absolute terms, times what the activation makes of it: gate and up within the limit of 1.2, a slope below 4
        bound = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * 1.01 * ref.abs() + 4 * K * 2.0 ** -24 * torch.bmm(own.abs(), rows.abs()[:, :, None])[:, 0::2, 0] + 1e-6
        bound = bound + 4 * K * 2.0 ** -24 * torch.bmm(own.abs(), rows.abs()[:, :, None])[:, 1::2, 0]
        params = ops.glu_params(None, LIMIT, None, ALPHA, SHIFT)
        for force in (None, "wreg:0:0", "wreg:1:0", "wreg:2:0", "wreg:2:1"):
            got = ops.linear_pairs(x.to(DEV), wt, p, ops.EPI_CLAMPGLU, gather, force=force, params=params).cpu()
            assert got.dtype == dtype and bool(((got.double() - ref).abs() <= bound).all()), (gather, force)


@pytest.mark.parametrize("rows", [1, 5, 255, 256, 263])
@pytest.mark.parametrize("width,n", [(4, 1), (260, 4), (2048, 9), (4092, 17), (4096, 3), (4100, 2)])
def test_router_logits_are_the_same_bits_whatever_the_kernel(rows, width, n):
    """Rows in whole quads run on a wave each; the same rows one element off their alignment on a workgroup an output: the order of
    every sum is one and the same (a choice of experts near a tie does not depend on the kernel)."""
    from llm_infer_amd.kernels import ops
    g = torch.Generator().manual_seed(rows + width)
    w, bias = torch.randn(n, width, generator=g).cuda(), torch.randn(n, generator=g).cuda()
    for dt in (torch.float32, torch.float16, torch.bfloat16):
        h = torch.randn(rows, width, generator=g).to(dt).cuda()
        flat = torch.empty(rows * width + 1, dtype=dt, device="cuda")
        off = flat[1:].view(rows, width)
        off.copy_(h)
        for b in (None, bias):
            got = ops.small_logits(h, w, b)
            assert torch.equal(got, ops.small_logits(off, w, b))
            ref = h.double() @ w.double().t() + (0 if b is None else b.double())
            # float32 sums of `width` products (a pairwise tree of 256 sums of 16): 24 roundings of the terms' magnitudes at most
            assert ((got.double() - ref).abs() <= 24 * 2.0 ** -24 * (h.double().abs() @ w.double().abs().t() + 1)).all()
