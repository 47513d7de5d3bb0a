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


# chunks that are whole, of one token, of a tile's edge; every number of tiles of the state a wave takes; values of one tile, of a
# workgroup's four and beyond; heads that share B and C, and heads with their own
@pytest.mark.parametrize("lens,P,G,N,dv", [([1], 1, 1, 16, 16), ([64, 1, 65], 4, 2, 48, 32), ([16, 17, 15], 6, 3, 64, 80),
                                           ([128, 200, 63], 4, 1, 128, 64), ([300], 2, 2, 144, 48), ([33, 130], 3, 1, 256, 160)])
@pytest.mark.parametrize("fast", [False, True])
def test_chunks_against_the_recurrence(lens, P, G, N, dv, fast):
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
        for chunks in (False, True):
            ctx, s = _step(lens, slots), state.to(DEV)
            y = ops.ssm_scan(dev[0], dev[1], 8, dev[2], dev[3], None if skip is None else dev[4], s, ctx, P, G, N, dv,
                             ops.ssm_segments(ctx, ops.SSM_CHUNK) if chunks else None, chunks)
            errors.append([((a.double().cpu() - b).norm() / b.norm()).item() for a, b in ((y, want), (s, want_state))])
            idle = [i for i in range(len(state)) if i not in slots]
            assert torch.equal(s.cpu()[idle], state[idle])
        for token, chunk in zip(*errors):
            assert chunk < 4 * token + 1e-8, errors
            assert chunk < 1e-6


def test_sizes_that_chunks_do_not_take_are_refused():
    from llm_infer_amd.kernels import ops
    ctx = _step([3], [0])
    seg = ops.ssm_segments(ctx, ops.SSM_CHUNK)
    for N, dv in ((24, 16), (16, 24), (272, 16)):
        assert not ops.ssm_chunks_fit(N, dv)
        with pytest.raises(ops.KernelError):
            ops.ssm_scan(torch.zeros(3, dv + 2 * N, device=DEV), torch.zeros(3, 1, device=DEV), 0, torch.zeros(1, device=DEV),
                         torch.zeros(1, device=DEV), None, torch.zeros(1, 1, N, dv, device=DEV), ctx, 1, 1, N, dv, seg, True)


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
