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
