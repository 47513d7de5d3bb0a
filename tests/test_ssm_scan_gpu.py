"""The state-space recurrence of a prompt by chunks, as products of matrices, against the recurrence in 64 bits, and the gated norm
behind it."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _step(lens, slots):
    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device=DEV)
    starts = [sum(lens[:i]) for i in range(len(lens))]
    made = {}
    return types.SimpleNamespace(host_qlens=lens, device=DEV, n_seqs=len(lens), n_tokens=sum(lens), seq_slot=i32(slots),
                                 seq_qstart=i32(starts), seq_qlen=i32(lens),
                                 shared=lambda key, make: made[key] if key in made else made.setdefault(key, make()))


def _recurrence(xbc, raw, bias, a_log, d, state, lens, slots, P, G, N, dv):
    xbc, raw, bias, a_log, state = (v.double() for v in (xbc, raw, bias, a_log, state))
    out, q = [], 0
    for n, slot in zip(lens, slots):
        for t in range(q, q + n):
            x, b, c = xbc[t].split([P * dv, G * N, G * N])
            x, b, c = x.view(P, dv), b.view(G, N).repeat_interleave(P // G, 0), c.view(G, N).repeat_interleave(P // G, 0)
            dt = torch.nn.functional.softplus(raw[t] + bias)
            state[slot] = torch.exp(-torch.exp(a_log) * dt)[:, None, None] * state[slot] + (dt[:, None] * b)[:, :, None] * x[:, None]
            y = (state[slot] * c[:, :, None]).sum(1)
            out.append((y if d is None else y + d.double()[:, None] * x).reshape(-1))
        q += n
    return torch.stack(out), state


# segments that are whole, of one token, of an edge; states below, at and between the registers' sizes; values of less than a wave, of one
# and beyond; heads that share B and C, and heads with their own
@pytest.mark.parametrize("lens,P,G,N,dv", [([1], 1, 1, 16, 16), ([64, 1, 65], 4, 2, 48, 32), ([16, 17, 15], 6, 3, 64, 80),
                                           ([128, 200, 63], 4, 1, 128, 64), ([300], 2, 2, 144, 48), ([33, 130], 3, 1, 256, 160)])
@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("length", [16, 64])
def test_segments_against_the_recurrence(lens, P, G, N, dv, fast, length):
    """Results and states, from states that are not zero, in slots of any order; ``fast``: decays down to exp(-200) a token.  No
    further off than four times the token-by-token kernel (both round every product to 32 bits, in other orders)."""
    from llm_infer_amd.kernels import ops
    g = torch.Generator().manual_seed(sum(lens) + N + dv)
    T, slots = sum(lens), [2 * i + 1 for i in reversed(range(len(lens)))]

    def r(*s):
        return torch.randn(*s, generator=g)
    proj = r(T, 8 + P)
    xbc, bias, a_log, d = r(T, P * dv + 2 * G * N), r(P) - (0 if fast else 2), torch.log(1 + (40 if fast else 15) * torch.rand(P, generator=g)), r(P)
    state = r(2 * len(lens) + 1, P, N, dv)
    dev = [v.to(DEV) for v in (xbc, proj, bias, a_log, d)]
    for skip in (d, None):
        want, want_state = _recurrence(xbc, proj[:, 8:], bias, a_log, skip, state, lens, slots, P, G, N, dv)
        errors = []
        for segments in (False, True):
            ctx, s = _step(lens, slots), state.to(DEV)
            y = ops.ssm_scan(dev[0], dev[1], 8, dev[2], dev[3], None if skip is None else dev[4], s, ctx, P, G, N, dv,
                             ops.ssm_segments(ctx, length) if segments else None)
            errors.append([((a.double().cpu() - b).norm() / b.norm()).item() for a, b in ((y, want), (s, want_state))])
            idle = [i for i in range(len(state)) if i not in slots]
            assert torch.equal(s.cpu()[idle], state[idle])
        for token, cut in zip(*errors):
            assert cut < 4 * token + 1e-8, errors
            assert cut < 1e-6


def _mixer(P, G, N, dv, width=96):
    """A state-space mixer of a 16-bit model with random weights."""
    from llm_infer_amd.parts.state_space import SelectiveStateSpace
    from llm_infer_amd.weights.loader import place_tensor
    part = SelectiveStateSpace(hidden_size=width, n_heads=P, head_dim=dv, n_state=N, n_groups=G, conv_taps=4, norm_groups=1, norm_eps=1e-5,
                               prefix="", dtype=torch.bfloat16, device=DEV)
    g = torch.Generator().manual_seed(P + N + dv)
    part.bind({n: place_tensor(torch.randn(p.shape, generator=g) * (0.1 if len(p.shape) == 2 else 0.5), p.kind, torch.bfloat16, DEV)
               for n, p in part.params().items()})
    return part


def _run(part, h, lens, monkeypatch):
    """What the mixer adds to the residual rows, and the operands and the result of its recurrence."""
    from llm_infer_amd.cache import Cache
    from llm_infer_amd.engine.step import StepContext
    from llm_infer_amd.kernels import ops
    specs, seen, scan = part.cache_specs(), {}, ops.ssm_scan

    def watched(*args):
        args = list(args)
        seen["args"], seen["state"] = args, args[6].clone()
        seen["y"] = scan(*args)
        return seen["y"]
    monkeypatch.setattr(ops, "ssm_scan", watched)
    cache = Cache(specs, 4096, 4096, torch.bfloat16, DEV)
    slots = [cache.alloc_slot() for _ in lens]
    cache.grow(slots, lens, filled=True)
    ctx = StepContext(DEV, slots, [[0] * n for n in lens], [0] * len(lens), [[] for _ in lens])
    residual = torch.zeros(h.shape, dtype=torch.float32, device=DEV)
    part.forward(h, ctx, [cache.view(i) for i in range(len(specs))], residual)
    monkeypatch.setattr(ops, "ssm_scan", scan)
    return residual, ctx, seen


# few tokens, some of several lengths, many tokens (segments of 16, 16 and 64 tokens)
@pytest.mark.parametrize("lens,P,G,N,dv", [([20], 8, 1, 128, 64), ([300, 1, 70], 4, 2, 48, 32), ([1100, 900], 128, 1, 16, 64)])
def test_a_prompt_is_rounded_as_in_its_segments(lens, P, G, N, dv, monkeypatch):
    """The order in which the recurrence rounds is part of a 16-bit model's result: behind it a token whose experts' scores nearly tie may
    choose otherwise, and a whole model's logits then differ by more than rounding.  So the values are these, bit for bit: segments
    short enough for 3,072 waves, 16 to 128 tokens."""
    from llm_infer_amd.kernels import ops
    part = _mixer(P, G, N, dv)
    h = torch.randn(sum(lens), 96, generator=torch.Generator().manual_seed(7)).to(DEV, torch.bfloat16)
    _, ctx, seen = _run(part, h, lens, monkeypatch)
    length = 16
    while length < 128 and 2 * length <= sum(lens) * P * -(-dv // 64) // 3072:
        length *= 2
    args = seen["args"][:12]
    args[6] = seen["state"]
    assert max(lens) > length
    assert torch.equal(seen["y"], ops.ssm_scan(*args, ops.ssm_segments(ctx, length)))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_token_that_is_not_finite_leaves_the_ones_before_it_alone(bad, monkeypatch):
    part, lens, at = _mixer(4, 1, 128, 64), [200, 40], 133
    h = torch.randn(sum(lens), 96, generator=torch.Generator().manual_seed(9)).to(DEV, torch.bfloat16)
    clean, _, _ = _run(part, h, lens, monkeypatch)
    h[at] = bad
    got, _, _ = _run(part, h, lens, monkeypatch)
    assert torch.isfinite(clean).all() and not torch.isfinite(got[at]).any()
    for rows in (slice(0, at), slice(lens[0], sum(lens))):                     # its own sequence's earlier tokens, another sequence
        assert torch.equal(got[rows], clean[rows])


# elements of a group around what a thread keeps (2, 4 and 8 of them for 256, 512 and 1,024 threads), and beyond that
@pytest.mark.parametrize("part", [1, 255, 512, 513, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 8192, 8193])
@pytest.mark.parametrize("groups", [1, 3])
def test_gated_norm_of_every_width(part, groups):
    from llm_infer_amd.kernels import ops
    g = torch.Generator().manual_seed(part + groups)
    n = part * groups
    y, rows, w = torch.randn(3, n, generator=g), torch.randn(3, n + 5, generator=g), torch.randn(n, generator=g)
    got = ops.gated_group_norm(y.to(DEV), rows.to(DEV), 5, w.to(DEV), groups, 1e-4, torch.float32).cpu().double()
    v = (y.double() * torch.nn.functional.silu(rows[:, 5:].double())).view(3, groups, part)
    want = (v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-4)).view(3, n) * w.double()
    # an exponential, a division, a root and four products of 32 bits, and the sum of squares' own rounding: under 16 roundings
    assert ((got - want).abs() <= 16 * 2.0 ** -24 * want.abs() + 1e-7).all()


@pytest.mark.parametrize("part", [4096, 5000, 8191, 8192])
def test_gated_norm_is_the_same_kept_in_registers_or_not(part):
    """A row followed by three times as many zeros, with a quarter of eps, has twice the norm's factor, exactly: beyond 8,192 elements
    by the kernel that fetches them twice, up to there, with as many threads, by the one that keeps them."""
    from llm_infer_amd.kernels import ops
    g = torch.Generator().manual_seed(part)
    y, z, w = torch.randn(3, part, generator=g), torch.randn(3, part, generator=g), torch.randn(part, generator=g)

    def run(times):
        def pad(t):
            return torch.nn.functional.pad(t, (0, (times - 1) * part)).contiguous().to(DEV)
        return ops.gated_group_norm(pad(y), pad(z), 0, pad(w), 1, 2.0 ** -10 / times, torch.float32)[:, :part]
    assert torch.equal(2 * run(1), run(4))
