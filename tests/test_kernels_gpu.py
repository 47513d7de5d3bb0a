"""Each HIP kernel alone against a plain float64/float32 PyTorch reference of the same
operation, at sizes other than the engine's test models."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
F16S = [torch.bfloat16, torch.float16]


@pytest.fixture(scope="module")
def ops():
    import llm_infer_amd  # noqa: F401
    from llm_infer_amd.kernels import ops as o
    return o


def _tol(dtype):
    return {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype]


def test_embed(ops):
    g = torch.Generator().manual_seed(0)
    for dt in [torch.float32] + F16S:
        table = torch.randn(331, 80, generator=g).to(dt).to(DEV)
        toks = torch.tensor([0, 330, 17, 17, 5], dtype=torch.int32, device=DEV)
        out = ops.embed(table, toks)
        assert out.dtype == torch.float32
        assert torch.equal(out, table[toks.long()].float())


@pytest.mark.parametrize("d", [30, 64, 96, 100, 1000, 1022, 4096, 8192, 10000])
def test_rmsnorm(ops, d):
    g = torch.Generator().manual_seed(d)
    x = (torch.randn(7, d, generator=g) * 3).to(DEV)
    w = (1 + 0.1 * torch.randn(d, generator=g)).to(DEV)
    for eps in (1e-5, 1e-2):
        ref = (x.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + eps) * w.double())
        for dt in [torch.float32] + F16S:
            out = ops.rmsnorm(x, w, eps, dt)
            assert out.dtype == dt
            assert torch.allclose(out.double(), ref, rtol=_tol(dt), atol=_tol(dt))
    rows = torch.tensor([5, 0, 5], dtype=torch.int32, device=DEV)
    out = ops.rmsnorm(x, w, 1e-5, torch.float32, rows)
    assert torch.equal(out, ops.rmsnorm(x, w, 1e-5, torch.float32)[rows.long()])
    # eps inside the root: tiny inputs are scaled by 1/sqrt(eps), not blown up
    tiny = torch.full((1, d), 1e-4, device=DEV)
    out = ops.rmsnorm(tiny, torch.ones(d, device=DEV), 1e-2, torch.float32)
    assert torch.allclose(out, torch.full_like(out, 1e-4 / math.sqrt(1e-8 + 1e-2)), rtol=1e-5)


def _linear_ref(x, w, mode, res=None):
    y = x.double() @ w.double().t()
    if mode == 1:
        return res.double() + y
    if mode == 2:
        g, u = y[:, 0::2], y[:, 1::2]
        return g / (1 + torch.exp(-g)) * u
    if mode == 4:                                   # the gate's other activation: gelu in its tanh form
        g, u = y[:, 0::2], y[:, 1::2]
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    return y


LIN_CASES = [  # M, N, K
    (1, 64, 64), (2, 16400, 4096), (16, 1000, 2056), (9, 40, 4104), (3, 172, 96), (8, 100, 256), (5, 6, 8), (13, 344, 64), (33, 130, 136),
    (64, 256, 512), (70, 200, 1024), (129, 384, 320), (200, 136, 72), (256, 512, 2048), (384, 256, 192),
    (927, 96, 16), (140, 40, 24),                   # K shorter than any tile's depth: the chunks past K are masked, not read
]


@pytest.mark.parametrize("M,N,K", LIN_CASES)
@pytest.mark.parametrize("dt", [torch.float32] + F16S)
def test_linear_all_kernels_and_epilogues(ops, M, N, K, dt):
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
    res = torch.randn(M, N, generator=g).to(DEV)
    kinds = ["fma"]
    if dt != torch.float32:
        if M <= 16:
            kinds.append("gemv_mfma")
        kinds += ["mfma:0:1", "mfma:1:1", "mfma:2:1", "mfma:2:3", "mfma:0:2", "big:0", "big:1", "big:0:3", None]
    for kind in kinds:
        for mode in (0, 1, 2, 4):
            if mode in (2, 4) and N % 2:
                continue
            ref = _linear_ref(x, w, mode, res)
            if mode == 1:
                out = res.clone()
                ops.linear(x, w, mode, out=out, force=kind)
                tol = 1e-5 if dt == torch.float32 else 2e-4
            elif mode in (2, 4):
                out = ops.linear(x, w, mode, out_dtype=torch.float32, force=kind)
                tol = 1e-5 if dt == torch.float32 else 2e-4
            else:
                out = ops.linear(x, w, mode, out_dtype=torch.float32, force=kind)
                tol = 1e-5 if dt == torch.float32 else 2e-4
            err = (out.double() - ref).abs().max().item()
            assert err < tol * (1 + ref.abs().max().item()), (kind, mode, err)
            if dt != torch.float32 and mode != 1:
                out16 = ops.linear(x, w, mode, out_dtype=dt, force=kind)
                assert out16.dtype == dt
                assert torch.allclose(out16.double(), ref, rtol=_tol(dt), atol=_tol(dt))


# the edges of the tiles of 16 and 64 rows, of the chains of 256 k, of the steps of 16 and 32, and of the rules by rows and sizes
F32_CASES = [(1, 1, 16), (3, 33, 48), (8, 16400, 256), (9, 16400, 272), (16, 130, 4352), (17, 257, 528), (33, 64, 1040), (40, 16400, 288),
             (64, 100, 4096), (65, 64, 32), (100, 200, 2064), (128, 4112, 512), (129, 130, 304), (300, 514, 8208)]
# half blocks: chains that are single, short, missing beside the last; one to sixteen pairs and more than one round of them
F32_CASES += [(1, 8, 256), (2, 7, 272), (8, 2048, 768), (7, 2050, 2320), (5, 100, 4112), (8, 40, 8448), (4, 64, 16400)]
# whole chains and pairs of them in the order that is written: one round of waves and several, a last round that some waves sit out, half blocks of
# few rows beyond 256 blocks and the sizes on either side of their rule
F32_CASES += [(3, 2050, 512), (8, 24, 9216), (2, 4112, 4096), (3, 6130, 4608), (4, 6144, 4352), (5, 4112, 4096), (3, 6160, 4096), (9, 36, 256), (16, 4096, 4352),
              (12, 2100, 2048), (8, 2064, 1024)]


@pytest.mark.parametrize("M,N,K", F32_CASES)
def test_float32_products_on_the_matrix_cores_are_bit_equal(ops, M, N, K):
    """gemm_f32's kernels against gemm_fma, whose order of sums they keep: bit for bit, with rows of every magnitude."""
    g = torch.Generator().manual_seed(M + N + K)
    scale = torch.exp2(torch.randint(-40, 40, (N, 1), generator=g).float())
    x, w = torch.randn(M, K, generator=g).to(DEV), (torch.randn(N, K, generator=g) * scale).to(DEV)
    res = torch.randn(M, N, generator=g).to(DEV)
    for kind in [None, "f32:2"] + (["f32:1"] if M <= 128 else []):
        for mode in (0, 1, 2):
            if mode == 2 and N % 2:
                continue
            outs = []
            for k in ("fma", kind):
                out = res.clone() if mode == 1 else None
                outs.append(ops.linear(x, w, mode, out=out, force=k))
            assert torch.equal(*outs), (kind, mode)
    # an address that is not 16-byte aligned goes to gemm_fma
    if N * K > 4:
        flat = torch.empty(N * K + 1, device=DEV)
        off = flat[1:].view(N, K)
        off.copy_(w)
        assert torch.equal(ops.linear(x, off), ops.linear(x, w))


@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (33, 30, 512), (32, 33, 768), (64, 130, 1024), (65, 64, 1280), (31, 2050, 2304), (200, 520, 8192),
                                   (21, 4096, 2048), (20, 6144, 2048), (9, 6160, 2048), (256, 3072, 2048), (300, 4112, 512)])
def test_float32_products_that_share_their_chains_among_waves_are_bit_equal(ops, M, N, K):
    """gemm_f32_chains against gemm_fma: one chain (three waves without), rounds of four that are full and not, ragged tiles, rows of
    every magnitude and subnormal products; and the kernel that the sizes choose, on either side of its rules."""
    g = torch.Generator().manual_seed(M + N + K)
    scale = torch.exp2(torch.randint(-40, 40, (N, 1), generator=g).float())
    x, w = torch.randn(M, K, generator=g).to(DEV), (torch.randn(N, K, generator=g) * scale).to(DEV)
    res = torch.randn(M, N, generator=g).to(DEV)
    for kind in (None, "f32:3"):
        for mode in (0, 1, 2):
            if mode == 2 and N % 2:
                continue
            outs = [ops.linear(x, w, mode, out=res.clone() if mode == 1 else None, force=k) for k in ("fma", kind)]
            assert torch.equal(*outs), (kind, mode)
    tiny = (x * 2.0 ** -100).contiguous()
    assert torch.equal(ops.linear(tiny, w, force="f32:3"), ops.linear(tiny, w, force="fma"))
    if M * K > 4096:
        x[0, 5], x[-1, 7] = float("inf"), float("nan")
        assert torch.equal(ops.linear(x, w, force="f32:3").isnan(), ops.linear(x, w, force="fma").isnan())
    with pytest.raises(ops.KernelError):
        ops.linear(x[:, :240].contiguous(), w[:, :240].contiguous(), force="f32:3")


@pytest.mark.parametrize("M,N,K", [(3, 33, 48), (17, 257, 528), (100, 200, 2064), (129, 130, 304)])
def test_float32_products_of_subnormal_numbers_are_bit_equal(ops, M, N, K):
    """Operands, products and sums below 2^-126: no kernel takes them for zeros."""
    g = torch.Generator().manual_seed(M + K)
    tiny = 2.0 ** -126
    for sx, sw in ((2.0 ** -70, 2.0 ** -70), (tiny / 64, 1.0), (1.0, tiny / 1024), (2.0 ** -60, 2.0 ** -66)):
        x, w = (torch.randn(M, K, generator=g) * sx).to(DEV), (torch.randn(N, K, generator=g) * sw).to(DEV)
        ref = ops.linear(x, w, force="fma")
        assert bool((ref != 0).any()) and ref.abs().min().item() < tiny
        for kind in [None, "f32:2"] + (["f32:1"] if M <= 128 else []):
            assert torch.equal(ops.linear(x, w, force=kind), ref), (sx, sw, kind)
        # what flushing products below 2^-126 would give is something else
        assert not torch.equal(torch.where(ref.abs() < tiny, torch.zeros_like(ref), ref), ref)
    one = (torch.randn(M, K, generator=g) * tiny / 8).to(DEV)
    assert bool((one.abs() < tiny).any()) and bool((ops.linear(one, torch.ones(N, K, device=DEV)) != 0).any())


# rows, experts, hidden columns of one and of a shared expert: widths that no tile or batch of steps divides, one expert, many
EXPERT_CASES = [(1, 8, 40, 24), (8, 8, 3584, 3584), (3, 3, 272, 0), (2, 40, 48, 16), (5, 1, 96, 32)]


@pytest.mark.parametrize("M,n,ff,tail", EXPERT_CASES)
@pytest.mark.parametrize("dt", F16S)
def test_products_of_chosen_experts(ops, M, n, ff, tail, dt):
    """Experts side by side with those that no token chose left out, against the same products of all of them: the same sums
    in the hidden rows; the down product takes its own in another order."""
    d, g = 256, torch.Generator().manual_seed(M + n + ff)
    x = torch.randn(M, d, generator=g).to(dt).to(DEV)
    weights = torch.rand(M, n + int(tail > 0), generator=g) + 0.1
    weights[:, torch.randperm(n, generator=g)[:n // 2 + 1]] = 0.0        # (one expert: chosen by nobody)
    weights = weights.to(DEV)
    cols = n * ff + tail
    gu = ops.tile_weight((torch.randn(2 * cols, d, generator=g) / 16).to(dt).to(DEV))
    up = ops.tile_weight((torch.randn(cols, d, generator=g) / 16).to(dt).to(DEV))
    assert ops.experts_fit(x[:1], gu, 8, 2, ff, True) and not ops.experts_fit(x, gu, n, n, ff, True)
    glu = ops.glu_params(None, 0.9, 0.7, 1.702, 1.0, n * ff)
    for mode, params in ((2, None), (ops.EPI_CLAMPGLU, glu)):
        all_ = ops.scale_blocks(ops.linear(x, gu, mode, out_dtype=dt, params=params), weights, n, ff, tail)
        few = ops.linear(x, gu, mode, out_dtype=dt, params=params, experts=(weights, n, ff, ops.EXPERTS_GATED))
        # one product times one weight, rounded to float32 on the way or at once to the type: at most a step of the type apart
        step = 2.0 ** -10 if dt == torch.float16 else 2.0 ** -7
        assert bool(((all_.float() - few.float()).abs() <= step * all_.float().abs()).all()), mode
        assert (all_ != few).float().mean().item() < 1e-3, mode
    z = [ops.linear(x, up, out_dtype=torch.float32, experts=e) for e in (None, (weights, n, ff, ops.EXPERTS_IN_N))]
    hidden = [ops.expert_act(v, weights, n, ff, tail, "relu2", True, dt) for v in z]
    assert torch.equal(*hidden)
    if cols % 32 == 0:
        wd = (torch.randn(d, cols, generator=g) / 16).to(dt).to(DEV)
        down = ops.tile_weight(wd)
        for mode in (0, 1):
            res = torch.randn(M, d, generator=g).to(DEV)
            ref = few.double() @ wd.double().t() + (res.double() if mode else 0.0)
            out = ops.linear(few, down, mode, out=res, experts=(weights, n, ff, ops.EXPERTS_IN_K))
            # sums of `cols` products in float32: half a rounding step for each addition at most
            bound = 2.0 ** -24 * cols * (few.double().abs() @ wd.double().abs().t()).max().item() + 1e-6
            assert (out.double() - ref).abs().max().item() < bound, mode


def test_experts_are_refused_where_no_kernel_takes_them(ops):
    """Not run as if every expert were chosen (which would leave the weights out)."""
    w = torch.zeros(64, 32, dtype=torch.bfloat16, device=DEV)
    x = torch.zeros(40, 32, dtype=torch.bfloat16, device=DEV)
    for rows, wt, mode, over in ((40, ops.tile_weight(w), 0, ops.EXPERTS_IN_N), (40, ops.tile_weight(w), 2, ops.EXPERTS_GATED), (2, w, 0, ops.EXPERTS_IN_N)):
        with pytest.raises(ops.KernelError):
            ops.linear(x[:rows], wt, mode, experts=(torch.ones(rows, 2, device=DEV), 2, 16 if over == ops.EXPERTS_GATED else 32, over))


def test_when_unchosen_experts_are_left_out(ops):
    """By the share of experts that is likely to go unread: of all the router's outputs, those that pass a token on among them."""
    w = ops.tile_weight(torch.zeros(64, 32, dtype=torch.bfloat16, device=DEV))
    x = torch.zeros(9, 32, dtype=torch.bfloat16, device=DEV)
    fit = lambda rows, n, top, outputs=None: ops.experts_fit(x[:rows], w, n, top, 16, True, outputs)
    assert fit(4, 8, 2) and not fit(5, 8, 2) and fit(8, 60, 6) and not fit(9, 60, 6) and not fit(1, 64, 2)
    assert not fit(2, 4, 4) and not fit(1, 1, 1)
    assert fit(2, 2, 2, 4) and not fit(3, 2, 2, 4) and not fit(2, 2, 4, 4)      # two experts and two outputs that pass a token on
    assert not fit(2, 2, 5, 6) and not fit(4, 1, 3, 4)                          # (more are chosen than there are experts)


@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (3, 8, 2), (1023, 5, 3), (1024, 8, 2), (1025, 3, 3), (2500, 70, 4)])
def test_pairs_of_dense_routing_weights(ops, T, E, top):
    g = torch.Generator().manual_seed(T + E)
    w = torch.zeros(T, E + 1)
    for t in range(T):
        n = int(torch.randint(0, min(top, E) + 1, (1,), generator=g))          # a token may have fewer than `top`, or none
        w[t, torch.randperm(E, generator=g)[:n]] = torch.rand(n, generator=g) + 0.1
    p = ops.pairs_of_weights(w.to(DEV), E, top)
    rows = [t for e in range(E) for t in range(T) if w[t, e] != 0]
    counts = [(w[:, e] != 0).sum().item() for e in range(E)]
    assert p.counts.tolist() == counts and p.offsets.tolist() == [sum(counts[:e]) for e in range(E)]
    assert p.row_of[:len(rows)].tolist() == rows
    place, slots, own = {}, torch.full((T, top), -1), torch.zeros(T, top)
    for i, (e, t) in enumerate((e, t) for e in range(E) for t in range(T) if w[t, e] != 0):
        j = place.get(t, 0)
        slots[t, j], own[t, j], place[t] = i, w[t, e], j + 1
    assert torch.equal(p.slot_of.cpu().long(), slots) and torch.equal(p.weights.cpu(), own)
    assert p.weight_of[:len(rows), 0].tolist() == [w[t, e].item() for e in range(E) for t in range(T) if w[t, e] != 0]


@pytest.mark.parametrize("T,E,top", [(40, 9, 2), (1024, 8, 2), (1500, 70, 4), (77, 20, 3), (33, 32, 1), (300, 64, 5), (130, 65, 2), (7, 5, 1)])
def test_pairs_of_rows_with_more_weights_than_are_chosen(ops, T, E, top):
    """A row with more than `top` weights has the pairs of the first `top`: what is counted is what is dealt out, so no place
    beyond T * top is named (nothing checks on the host how many weights of a row are not 0)."""
    g = torch.Generator().manual_seed(T)
    w = torch.rand(T, E + 1, generator=g) + 0.1
    w[torch.rand(T, E + 1, generator=g) < 0.5] = 0.0
    w[::7, -2] = 0.25                                                          # an expert that many rows name last
    assert int((w[:, :E] != 0).sum(1).max()) > top
    p = ops.pairs_of_weights(w.to(DEV), E, top)
    kept = [(w[t, :E] != 0).nonzero().flatten()[:top].tolist() for t in range(T)]
    pairs = [(e, t) for e in range(E) for t in range(T) if e in kept[t]]
    counts = [sum(e in k for k in kept) for e in range(E)]
    assert p.counts.tolist() == counts and p.offsets.tolist() == [sum(counts[:e]) for e in range(E)]
    assert p.row_of[:len(pairs)].tolist() == [t for _, t in pairs]
    assert p.weight_of[:len(pairs), 0].tolist() == [w[t, e].item() for e, t in pairs]
    slot = {pair: i for i, pair in enumerate(pairs)}
    assert p.slot_of.tolist() == [[slot[e, t] for e in kept[t]] + [-1] * (top - len(kept[t])) for t in range(T)]
    assert p.weights.tolist() == [[w[t, e].item() for e in kept[t]] + [0.0] * (top - len(kept[t])) for t in range(T)]


TILED_CASES = [(1, 64, 64), (3, 172, 96), (16, 40, 4096), (9, 16400, 256), (17, 100, 64), (64, 256, 512),
               (33, 4100, 2048), (48, 72, 8192), (50, 6144, 4096), (65, 48, 32), (97, 200, 14336), (30, 520, 96), (128, 16, 160),
               (70, 200, 1024), (96, 1000, 416), (128, 136, 2048), (129, 384, 320), (256, 520, 2048), (384, 512, 192), (300, 1000, 96)]


@pytest.mark.parametrize("M,N,K", TILED_CASES)
@pytest.mark.parametrize("dt", F16S)
def test_linear_tiled_weights(ops, M, N, K, dt):
    """The same products with W kept in matrix-core order: every kernel that reads it, every epilogue."""
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
    res = torch.randn(M, N, generator=g).to(DEV)
    wt = ops.tile_weight(w)
    assert ops.is_tiled(wt) and wt.logical == (N, K) and wt.numel() == (N + 15) // 16 * 16 * K and wt.owner == "device"
    assert torch.equal(ops.untile(wt), w.to(DEV))
    kinds = [None, "mfma:0:1", "mfma:1:2", "mfma:2:1", "big:0", "big:1", "big:0:2", "big:1:5"] + (["gemv_mfma"] if M <= 16 else [])
    # W into registers (tiles of 256, 192, 128 rows of W): the planner's choice and every tile, K whole and split
    kinds += ["wreg", "wreg:0", "wreg:1", "wreg:2", "wreg:0:2", "wreg:1:5", "wreg:2:3"]
    # the narrowest tile with W four steps ahead, with 64 rows of X (:1) and with 128 (:2), K whole and split
    kinds += ["wreg:2:1:1", "wreg:2:3:1", "wreg:2:1:2", "wreg:2:4:2", "wreg:2:1:3", "wreg:2:4:3"]        # (:3: three steps ahead)
    # workgroups that take fewer blocks of 16 rows of W than their tile has (the last field), for every tile
    kinds += ["wreg:2:1:1:7", "wreg:2:3:1:5", "wreg:2:1:2:6", "wreg:0:2:0:13", "wreg:1:1:0:9", "wreg:2:1:0:1"]
    # all of K in one workgroup, the rows of X through LDS of each wave's own (up to 128 rows): one and two tiles of W
    kinds += ["rows", "rows:1", "rows:2"] if M <= 128 else []
    for kind in kinds:
        for mode in (0, 1, 2, 4):
            if mode in (2, 4) and N % 2:
                continue
            ref = _linear_ref(x, w, mode, res)
            if mode == 1:
                out = res.clone()
                ops.linear(x, wt, mode, out=out, force=kind)
            else:
                out = ops.linear(x, wt, mode, out_dtype=torch.float32, force=kind)
            err = (out.double() - ref).abs().max().item()
            assert err < 2e-4 * (1 + ref.abs().max().item()), (kind, mode, err)
    if M <= 64:
        for nt, kw in ((1, 4), (1, 8), (2, 4), (2, 8)):
            if M > 32 and nt == 1:            # three or four tiles of rows of X go with two tiles of W
                continue
            out = ops.gemv_tiled(x, wt, out_dtype=torch.float32, nt=nt, kw=kw)
            assert (out.double() - _linear_ref(x, w, 0)).abs().max().item() < 2e-4 * 4
    if N % 32 == 0:
        head = ops.linear(x, wt.prefix(N // 2), out_dtype=torch.float32)
        assert (head.double() - _linear_ref(x, w[:N // 2], 0)).abs().max().item() < 2e-4 * 4
    with pytest.raises(ops.KernelError):
        ops.linear(x, wt, force="fma")
    with pytest.raises(ops.KernelError):
        ops.tile_weight(w[:, :K - 8].contiguous())


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M,N,K", [(17, 16, 32), (32, 40, 96), (33, 100, 544), (48, 520, 1056), (49, 72, 64), (64, 48, 4128),       # blocks of rows of X
                                   (12, 2064, 8192), (16, 2048, 4096), (9, 32, 4128), (11, 2064, 8192), (12, 16, 4064),             # few rows and a long K
                                   (17, 12288, 1024), (32, 12304, 96), (32, 12272, 1024), (24, 12288, 1056)])                        # wide and shallow
def test_more_rows_than_one_block_and_the_rules_beside_them(ops, M, N, K, dt):
    """gemm_rows with one to four blocks of 16 rows of X, shares of K with and without whole stages, and the planner's choice on
    either side of its rules, as tall products with the residual sum and without (K sums in float32: 2e-4 as above)."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
    res = torch.randn(M, N, generator=g).to(DEV)
    wt = ops.tile_weight(w)
    for kind in (None, "rows:1:4", "rows:1:8", "rows:2:4", "rows:2:8"):
        ref = _linear_ref(x, w, 0)
        out = ops.linear(x, wt, out_dtype=torch.float32, force=kind)
        assert (out.double() - ref).abs().max().item() < 2e-4 * (1 + ref.abs().max().item()), kind
        out = res.clone()
        ops.linear(x, wt, 1, out=out, force=kind)
        ref = _linear_ref(x, w, 1, res)
        assert (out.double() - ref).abs().max().item() < 2e-4 * (1 + ref.abs().max().item()), kind


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M,N,K,rows", [(17, 512, 512, (1, 8)), (24, 4096, 4096, (1, 8)), (32, 2048, 8192, (1, 8)), (19, 320, 1408, (1, 8)),
                                        (24, 3072, 2048, (1, 8)), (32, 48, 320, (1, 8)), (17, 6144, 2048, (2, 8)), (24, 4112, 1024, (2, 8)),
                                        (32, 8192, 4096, (2, 8)), (17, 10240, 512, (2, 4)), (24, 14336, 1024, (2, 4)), (18, 14352, 1280, (2, 4)),
                                        (32, 16384, 2048, (2, 4)), (9, 1024, 8192, (1, 8)), (16, 2032, 8192, (1, 8)), (12, 256, 14336, (1, 8)),
                                        (9, 5120, 13824, (1, 8)), (11, 2064, 12288, (1, 8)),
                                        (31, 100, 864, None), (24, 1024, 1056, None), (20, 8192, 512, None), (32, 14352, 1024, None),
                                        (20, 10240, 288, None), (12, 1024, 8224, None), (16, 2048, 4096, "short"), (12, 512, 8128, "short")])
def test_a_products_sums_do_not_depend_on_the_kernel_of_few_rows(ops, M, N, K, rows, dt):
    """Products of 9 to 32 rows that gemm_rows takes in gemv_tiled's place (tiles, waves; None: it does not): K in the same parts, added up
    in the same order, so the same bits with every epilogue that either side of the rules meets (fewer parts would be a larger error
    against 64 bits)."""
    assert rows == "short" or ops._rows_like_tiled(M, N, K) == rows
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
    wt = ops.tile_weight((torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV))
    res, nw = torch.randn(M, N, generator=g).to(DEV), torch.randn(N, generator=g).to(DEV)
    assert torch.equal(ops.linear(x, wt, out_dtype=torch.float32), ops.linear(x, wt, out_dtype=torch.float32, force="gemv_mfma"))
    assert torch.equal(ops.linear(x, wt, 2), ops.linear(x, wt, 2, force="gemv_mfma"))
    bias = ops.glu_params(nw, act="tanh")
    assert torch.equal(ops.linear(x, wt, ops.EPI_BIAS, params=bias), ops.linear(x, wt, ops.EPI_BIAS, params=bias, force="gemv_mfma"))
    outs = [res.clone(), res.clone()]
    for out, kind in zip(outs, (None, "gemv_mfma")):
        ops.expect_norm(out, nw, 1e-5)
        ops.linear(x, wt, 1, out=out, force=kind)
    assert torch.equal(*outs)
    recs = [getattr(out, "_li_rows", None) for out in outs]
    assert (recs[0] is None) == (recs[1] is None)
    if recs[0] is not None:                              # (what the product left for the norm behind it)
        assert torch.equal(recs[0][0], recs[1][0]) and torch.equal(recs[0][1], recs[1][1])


@pytest.mark.parametrize("M,N,K,kind", [(33, 10240, 1536, "rows:2"), (64, 12288, 1536, "rows:2"), (48, 28672, 512, "rows:2"), (128, 32000, 512, "rows:2"),
                                        (48, 4096, 8192, "wreg"), (32, 4096, 11008, "wreg"), (24, 16384, 5120, "wreg"), (40, 4096, 4096, "rows:1")])
def test_the_parts_in_which_some_dozen_rows_sum_their_products(ops, M, N, K, kind):
    """On either side of the estimate between gemm_rows (K in four parts) and gemm_wreg (in its splits): the kernel that the sums
    belong to, bit for bit."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    wt = ops.tile_weight((torch.randn(N, K, generator=g) / math.sqrt(K)).to(torch.bfloat16).to(DEV))
    assert torch.equal(ops.linear(x, wt, out_dtype=torch.float32), ops.linear(x, wt, out_dtype=torch.float32, force=kind))


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M", [1, 2, 7, 8])
@pytest.mark.parametrize("N,K", [(8, 32), (16, 64), (24, 96), (100, 544), (2048, 1056), (2050, 160), (4096, 8192)])
def test_half_tiles(ops, M, N, K, dt):
    """gemv_tiled with half a tile of W's rows a workgroup: odd numbers of steps, a last tile of less than half its rows, every
    epilogue; the same sums of W's rows as with whole tiles but for the order of K (K sums in float32: 2e-4 as above)."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
    res = torch.randn(M, N, generator=g).to(DEV)
    wt = ops.tile_weight(w)
    for kw in (4, 8):
        for mode in (0, 2, 4):
            ref = _linear_ref(x, w, mode)
            out = ops.gemv_tiled(x, wt, mode, torch.float32, -1, kw)
            assert (out.double() - ref).abs().max().item() < 2e-4 * (1 + ref.abs().max().item()), (kw, mode)
    out = ops.linear(x, wt, 1, out=res.clone())              # (whichever the rule takes)
    assert (out.double() - _linear_ref(x, w, 1, res)).abs().max().item() < 2e-4 * 6
    with pytest.raises(ops.KernelError):
        ops.gemv_tiled(torch.zeros(9, K, dtype=dt, device=DEV), wt, nt=-1)


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 15, 16, 17, 24, 31])
def test_few_rows_with_shares_of_every_length(ops, steps, dt):
    """gemv_tiled's waves with so many steps of K each, and with a last wave that has fewer: every depth of its ring, what the ring
    leaves, whole tiles, two of them and halves (sums of up to 8,000 products of numbers of about 1 / sqrt(K): 2e-4 as above)."""
    g = torch.Generator().manual_seed(steps)
    for kw in (4, 8):
        for K in (32 * kw * steps, 32 * (kw * steps - 1)):
            for N in (48, 30):
                w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
                wt = ops.tile_weight(w)
                for M, nt in ((1, -1), (8, -1), (1, 1), (16, 1), (5, 2), (17, 1), (32, 2)):
                    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
                    ref = _linear_ref(x, w, 0)
                    out = ops.gemv_tiled(x, wt, out_dtype=torch.float32, nt=nt, kw=kw)
                    assert (out.double() - ref).abs().max().item() < 2e-4 * (1 + ref.abs().max().item()), (kw, K, N, M, nt)


@pytest.mark.parametrize("parts", [1, 15, 16, 64, 255, 256, 257, 512, 700])
@pytest.mark.parametrize("M,N,K", [(1, 48, 64), (8, 4096, 256), (9, 100, 2048), (16, 6144, 4096)])
def test_a_norm_of_many_partial_sums_finished_by_the_product(ops, parts, M, N, K):
    """The rows' sums of squares come in any number of parts: those that the product asks for ahead of W and those behind them."""
    g = torch.Generator().manual_seed(parts + K)
    dt = torch.bfloat16
    xw, w = torch.randn(M, K, generator=g).to(dt).to(DEV), (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
    ss = torch.rand(parts, 16, generator=g).to(DEV) + 0.1
    lazy = ops.LazyNorm(torch.zeros(M, K, device=DEV), None, 1e-5, dt, xw, ss, 1.0)
    out = ops.linear(lazy, ops.tile_weight(w), out_dtype=torch.float32)
    ref = _linear_ref(xw, w, 0) / (ss.double().sum(0)[:M, None] / K + 1e-5).sqrt()
    assert ((out.double() - ref) / (1 + ref.abs().max())).abs().max().item() < 2e-4


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M,N,K", [(129, 72, 32), (130, 256, 64), (257, 200, 160), (300, 1000, 96), (511, 528, 96), (384, 1024, 256)])
def test_tiled_products_write_whole_rows(ops, M, N, K, dt):
    """The epilogues that store whole rows of a tile, 16 bytes a lane, beside the ones that go through it quad by quad (taken
    where a wave's columns are not all there or the rows are not aligned to 16 bytes): the same numbers bit for bit, for every
    tile, kind of result and type, and nothing written beside them."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dt).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dt).to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    wt = ops.tile_weight(w)
    s = x.double() @ w.double().t()
    b = s + bias.double()
    glu = lambda v: torch.clamp(v[:, 0::2], max=1.0) * torch.sigmoid(1.702 * torch.clamp(v[:, 0::2], max=1.0)) * (v[:, 1::2].clamp(-1.0, 1.0) + 1)  # noqa: E731
    refs = {(0, None): s, (2, None): torch.nn.functional.silu(s[:, 0::2]) * s[:, 1::2],
            (4, None): torch.nn.functional.gelu(s[:, 0::2], approximate="tanh") * s[:, 1::2],
            (5, "plain"): b, (5, "relu2"): torch.relu(b) ** 2, (5, "tanh"): torch.tanh(b), (6, None): glu(b)}
    for (mode, act), ref in refs.items():
        params = ops.glu_params(bias=bias, act=None if act == "plain" else act) if mode >= 5 else None
        for out_dt in (dt, torch.float32):
            for kind in ("wreg:0", "wreg:1", "wreg:2"):
                rows = ref.shape[1]
                got = []
                for offset in (0, 8 // (2 if out_dt == dt else 4)):              # rows that begin 16 and 8 bytes aligned
                    flat = torch.full((M * rows + 64,), 7.0, dtype=out_dt, device=DEV)
                    out = flat[offset:offset + M * rows].view(M, rows)
                    ops.linear(x, wt, mode, out=out, force=kind, params=params)
                    assert (flat[:offset] == 7.0).all() and (flat[offset + M * rows:] == 7.0).all()
                    got.append(out)
                assert torch.equal(*got), (mode, act, out_dt, kind)
                # 2e-4 for K sums in float32 as above, and half a unit in the last place of what is stored
                ulp = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[out_dt]
                err = (got[0].double() - ref).abs() - ulp * ref.abs()
                assert err.max().item() < 2e-4 * (1 + ref.abs().max().item()), (mode, act, out_dt, kind)


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M,d,K2,N2", [(1, 4096, 4096, 6144), (8, 4096, 14336, 28672), (16, 96, 160, 200), (5, 2048, 64, 128256),
                                       (12, 4096, 14336, 28672), (16, 4096, 4096, 22016), (14, 4096, 4096, 6144)])
def test_norm_split_over_two_products(ops, M, d, K2, N2, dt):
    """A decode step's product that adds into the residual stream prepares the norm that reads the rows
    next (x * weight in 16 bits, sums of squares), and the product behind the norm finishes it: the same
    result as norm kernel + product, without the kernel.  The preparation is void as soon as anything
    else writes to the rows, and for any other norm.  (From 9 rows on, gate and up against a wide matrix finish
    the norm in the tiled GEMM's epilogue instead of gemv_tiled's: the last two cases.)"""
    g = torch.Generator().manual_seed(M + d)
    x0 = torch.randn(M, d, generator=g) * 3
    a = (torch.randn(M, K2, generator=g) * 0.5).to(dt)
    wo = (torch.randn(d, K2, generator=g) * 0.05).to(dt)
    wn = (1 + 0.1 * torch.randn(d, generator=g)).to(DEV)
    w2 = (torch.randn(N2, d, generator=g) * 0.05).to(dt)
    eps = 1e-5
    wot = ops.tile_weight(wo.to(DEV))
    x = x0.to(DEV)
    ops.linear(a.to(DEV), wot, ops.EPI_ADD, out=x)
    assert ops.lazy_rmsnorm(x, wn, eps, dt) is None                         # nobody said which norm comes next
    x = x0.to(DEV)
    ops.expect_norm(x, wn)
    ops.linear(a.to(DEV), wot, ops.EPI_ADD, out=x)
    x_ref = x0.double() + a.double() @ wo.double().t()
    assert (x.double().cpu() - x_ref).abs().max().item() < 1e-3 * (1 + x_ref.abs().max().item())
    ln = ops.lazy_rmsnorm(x, wn, eps, dt)
    assert isinstance(ln, ops.LazyNorm) and ln.dtype == dt and tuple(ln.shape) == (M, d)
    assert torch.allclose(ln.ss.double().sum(0).cpu()[:M], (x.double().cpu() ** 2).sum(1), rtol=1e-5)
    assert torch.allclose(ln.xw.double().cpu(), x.double().cpu() * wn.double().cpu() * ln.scale, rtol=2.0 ** -8)
    w2t = ops.tile_weight(w2.to(DEV))
    fused = ops.linear(ln, w2t, out_dtype=torch.float32)
    h = ops.rmsnorm(x, wn, eps, dt)
    assert torch.equal(ln.tensor(), h)
    plain = ops.linear(h, w2t, out_dtype=torch.float32)
    xd = x.double().cpu()
    ref = (xd / torch.sqrt((xd ** 2).mean(1, keepdim=True) + eps) * wn.double().cpu()) @ w2.double().t()
    own = (plain.double().cpu() - ref).abs().max().item()                   # what rounding the normed rows to 16 bits costs
    assert (fused.double().cpu() - ref).abs().max().item() < 1.5 * own + 1e-6
    # the gated epilogue, and a weight that is not tiled (the norm is then taken by its kernel)
    if N2 % 2 == 0:
        gated = ops.linear(ln, w2t, ops.EPI_SWIGLU, out_dtype=torch.float32)
        g_ref = torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]
        g_own = (ops.linear(h, w2t, ops.EPI_SWIGLU, out_dtype=torch.float32).double().cpu() - g_ref).abs().max().item()
        assert (gated.double().cpu() - g_ref).abs().max().item() < 1.5 * g_own + 1e-6
    assert torch.equal(ops.linear(ln, w2.to(DEV)[:64].contiguous(), out_dtype=torch.float32),
                       ops.linear(h, w2.to(DEV)[:64].contiguous(), out_dtype=torch.float32))
    # anything else that writes to the rows voids the preparation; so does another norm's weight
    assert ops.lazy_rmsnorm(x, wn.clone(), eps, dt) is None
    assert ops.lazy_rmsnorm(x, wn, eps, torch.float32) is None              # a 32-bit norm is never deferred
    x += 1.0
    assert ops.lazy_rmsnorm(x, wn, eps, dt) is None
    ops.linear(a.to(DEV), wot, ops.EPI_ADD, out=x)
    assert ops.lazy_rmsnorm(x, wn, eps, dt) is not None
    ops.linear(a.to(DEV), wo.to(DEV), ops.EPI_ADD, out=x)                   # a kernel that prepares nothing
    assert ops.lazy_rmsnorm(x, wn, eps, dt) is None
    ops.linear(a.to(DEV), wot, ops.EPI_ADD, out=x)
    assert ops.lazy_rmsnorm(x.view(M, d), wn, eps, dt) is None              # another tensor object, no record
    if M < 16:
        big = torch.zeros(17, d, device=DEV)
        ops.expect_norm(big, wn)
        ops.linear(torch.zeros(17, K2, device=DEV, dtype=dt), wot, ops.EPI_ADD, out=big)
        assert ops.lazy_rmsnorm(big, wn, eps, dt) is None                   # more than 16 rows: the norm kernel


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M,N2", [(7, 768), (12, 65536)])
@pytest.mark.parametrize("rms,wscale", [(1e-2, 0.02), (1e3, 0.02), (1e3, 4.0), (3.0, 1.0)])
def test_norm_split_over_two_products_at_a_models_own_scale(ops, rms, wscale, M, N2, dt):
    """The rows that travel in 16 bits between the two products are x * weight; a checkpoint's residual stream
    may be of the order of 0.01 or of 1000 and its norm weights of 0.02.  In float16 each row is scaled by a
    power of two taken from the norm before (left by the norm kernel, then by each product that finishes a
    norm), so the split norm is as exact as norm kernel + product at every scale, down a chain of layers in
    which the rows grow; a view of the rows that a kernel writes through voids the preparation too.  The second
    shape is gate and up of 12 rows against a wide matrix, where the tiled GEMM finishes the norm and leaves the
    scales."""
    d, K2 = 1024, 512
    gated = N2 > 768
    assert not gated or ops._wreg_plan(M, N2, d) == (2, 1)
    mode = ops.EPI_SWIGLU if gated else ops.EPI_STORE
    g = torch.Generator().manual_seed(3)
    x0 = torch.randn(M, d, generator=g) * rms
    x0[2, 5] = 40 * rms                                            # a row with one large element
    wn = (wscale * (1 + 0.3 * torch.randn(d, generator=g))).to(DEV)
    # (the product's own operands stay of moderate size in 16 bits: what it adds is of the order of rms 3^layer)
    wo = (torch.randn(d, K2, generator=g) * 0.05 * rms / 34).to(dt)
    w2 = (torch.randn(N2, d, generator=g) * 0.05).to(dt)
    wot, w2t = ops.tile_weight(wo.to(DEV)), ops.tile_weight(w2.to(DEV))
    eps = 1e-6
    x = x0.to(DEV)
    ops.rmsnorm(x, wn, eps, dt)                                    # the norm before: in float16 it leaves the rows' scales
    assert (getattr(x, "_li_row_scale", None) is not None) == (dt == torch.float16)
    for layer in range(3):                                         # the rows grow by a factor of about 3 a layer
        a = (torch.randn(M, K2, generator=g) * 30 * 3 ** layer).to(dt)
        ops.expect_norm(x, wn)
        ops.linear(a.to(DEV), wot, ops.EPI_ADD, out=x)
        ln = ops.lazy_rmsnorm(x, wn, eps, dt)
        assert ln is not None and (ln.row_scales is not None) == (dt == torch.float16)
        assert torch.isfinite(ln.xw.float()).all()
        fused = ops.linear(ln, w2t, mode, out_dtype=torch.float32)
        assert (getattr(x, "_li_row_scale", None) is not None) == (dt == torch.float16)
        xd = x.double().cpu()
        ref = (xd / torch.sqrt((xd ** 2).mean(1, keepdim=True) + eps) * wn.double().cpu()) @ w2.double().t()
        if gated:
            ref = torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]
        plain = ops.linear(ops.rmsnorm(x.clone(), wn, eps, dt), w2t, mode, out_dtype=torch.float32)
        # (a gated product's largest errors sit at its few largest outputs, and the largest of them differs by a
        # factor of two between two roundings of the same quality: there the root mean square is compared)
        size = (lambda e: e.pow(2).mean().sqrt().item()) if gated else (lambda e: e.abs().max().item())
        own = size(plain.double().cpu() - ref)
        err = size(fused.double().cpu() - ref)
        assert err < 1.5 * own + 1e-6 * size(ref), (layer, err, own)
    # a kernel that writes through a view of the rows voids what was prepared for the rows themselves
    ops.expect_norm(x, wn)
    ops.linear(a.to(DEV), wot, ops.EPI_ADD, out=x)
    assert ops.lazy_rmsnorm(x, wn, eps, dt) is not None
    ops.linear(a.to(DEV)[:4].contiguous(), wot, ops.EPI_ADD, out=x[:4])
    assert ops.lazy_rmsnorm(x, wn, eps, dt) is None


def test_gate_activation_alone(ops):
    """act(gate) * up on interleaved columns, for a product that was stored unactivated."""
    g = torch.Generator().manual_seed(3)
    gu = (torch.randn(5, 2 * 173, generator=g) * 3).to(DEV)
    gate, up = gu[:, 0::2].double(), gu[:, 1::2].double()
    for gelu, ref in ((False, gate / (1 + torch.exp(-gate)) * up),
                      (True, torch.nn.functional.gelu(gate, approximate="tanh") * up)):
        out = ops.swiglu(gu, torch.float32, gelu=gelu)
        assert out.shape == (5, 173) and (out.double() - ref).abs().max() < 1e-5 * (1 + ref.abs().max())
        assert ops.swiglu(gu, torch.bfloat16, gelu=gelu).dtype == torch.bfloat16


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("M,d,K2", [(17, 256, 2048), (64, 4096, 4096), (200, 1000, 8192), (300, 96, 2080)])
def test_norm_taken_by_the_sum_of_split_products(ops, M, d, K2, dt):
    """With K split, the kernel that adds the partial sums into the residual rows also takes the norm that
    reads them next: bit for bit what the reduction and the norm kernel give, one kernel less.  Void as soon
    as anything else writes to the rows, for another weight or eps, and never made when K is not split."""
    g = torch.Generator().manual_seed(M + d)
    x0 = torch.randn(M, d, generator=g) * 3
    a = (torch.randn(M, K2, generator=g) * 0.5).to(dt).to(DEV)
    wot = ops.tile_weight((torch.randn(d, K2, generator=g) * 0.05).to(dt).to(DEV))
    wn = (1 + 0.1 * torch.randn(d, generator=g)).to(DEV)
    eps = 1e-5
    plain = x0.to(DEV)
    ops.linear(a, wot, ops.EPI_ADD, out=plain, force="wreg:2:2")
    assert ops.prepared_rmsnorm(plain, wn, eps, dt) is None                 # nobody said which norm comes next
    x = x0.to(DEV)
    ops.expect_norm(x, wn, eps)
    ops.linear(a, wot, ops.EPI_ADD, out=x, force="wreg:2:2")
    assert torch.equal(x, plain)
    ready = ops.prepared_rmsnorm(x, wn, eps, dt)
    assert ready is not None and ready.dtype == dt and torch.equal(ready, ops.rmsnorm(x, wn, eps, dt))
    assert ops.prepared_rmsnorm(x, wn.clone(), eps, dt) is None and ops.prepared_rmsnorm(x, wn, 2 * eps, dt) is None
    assert ops.prepared_rmsnorm(x, wn, eps, torch.float32) is None
    x += 1.0
    assert ops.prepared_rmsnorm(x, wn, eps, dt) is None                     # torch wrote to the rows
    y = x0.to(DEV)
    ops.expect_norm(y, wn, eps)
    ops.linear(a, wot, ops.EPI_ADD, out=y, force="wreg:2:2")
    ops.linear(a, wot, ops.EPI_ADD, out=y, force="wreg:2:1")                # a product without a split wrote to them
    assert ops.prepared_rmsnorm(y, wn, eps, dt) is None
    # the planner's own choice at these sizes
    z = x0.to(DEV)
    ops.expect_norm(z, wn, eps)
    ops.linear(a, wot, ops.EPI_ADD, out=z)
    ready = ops.prepared_rmsnorm(z, wn, eps, dt)
    assert ready is None or torch.equal(ready, ops.rmsnorm(z, wn, eps, dt))
    # (where the product runs as gemm_rows, all of K in a workgroup, there is no second kernel to take the norm)
    assert M < 64 or ops._wreg_plan(M, d, K2)[1] == 1 or ops._rows_plan(M, d, K2, True) or ready is not None


@pytest.mark.parametrize("M,N,K", [(2048, 8560, 736), (5000, 4048, 736), (1300, 12288, 4096)])
def test_large_products(ops, M, N, K):
    """Products of many tiles as the planner runs them: a K that is 32 more than a multiple of 64, widths and
    heights that end inside a tile."""
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(torch.float16).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(torch.float16).to(DEV)
    out = ops.linear(x, ops.tile_weight(w), out_dtype=torch.float32)
    for r0 in range(0, M, 4096):                       # the reference in slices: it is float64
        ref = x[r0:r0 + 4096].double() @ w.double().t()
        assert (out[r0:r0 + 4096].double() - ref).abs().max().item() < 2e-4 * (1 + ref.abs().max().item())


def test_linear_rows_do_not_depend_on_the_batch_in_float32(ops):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(70, 136, generator=g).to(DEV)
    w = torch.randn(100, 136, generator=g).to(DEV)
    whole = ops.linear(x, w, out_dtype=torch.float32)
    for r in (0, 63, 64, 69):
        assert torch.equal(ops.linear(x[r:r + 1].contiguous(), w, out_dtype=torch.float32)[0], whole[r])


def test_linear_mixed_precision_weights_stay_32_bit(ops):
    g = torch.Generator().manual_seed(2)
    x = torch.randn(5, 64, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(32, 64, generator=g).to(DEV)                     # float32 weight, bfloat16 activations
    out = ops.linear(x, w, out_dtype=torch.float32)
    assert torch.allclose(out.double(), x.double() @ w.double().t(), atol=1e-4)


def test_linear_refuses_what_it_cannot_do(ops):
    x = torch.randn(4, 12).to(torch.bfloat16).to(DEV)
    w = torch.randn(6, 12).to(torch.bfloat16).to(DEV)
    with pytest.raises(ops.KernelError):
        ops.linear(x, w, force="gemv_mfma")                           # K = 12 is no multiple of 8
    with pytest.raises(ops.KernelError):
        ops.linear(x, w, force="mfma:0:1")
    out = ops.linear(x, w, out_dtype=torch.float32)                  # the general kernel takes it
    assert torch.allclose(out.double(), x.double() @ w.double().t(), atol=1e-4)
    with pytest.raises(ops.KernelError):
        ops.linear(x, w[:5].contiguous(), 2)                          # SwiGLU needs gate/up pairs


# ---------------------------------------------------------------------------
# the cache's bookkeeping
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("n0,n1,n_pages", [(0, 0, 0), (1, 0, 0), (0, 3, 1), (448, 0, 0), (448, 1, 0), (300, 200, 7), (0, 0, 900), (1000, 449, 897)])
def test_cache_edit(ops, n0, n1, n_pages):
    """Words and pages around what one launch's arguments hold (896 numbers); pages of one workgroup and of several."""
    import numpy as np
    rng = np.random.default_rng(n0 * 7 + n1 + n_pages)
    a = torch.arange(4096, dtype=torch.int32, device=DEV).view(64, 64)
    b = torch.arange(1000, dtype=torch.int64, device=DEV)
    for elems in (64, 32768 // 2 + 64):
        pool = torch.randint(1, 99, (1000 if elems == 64 else 40, elems), device=DEV).half()
        want_a, want_b, want_pool = a.clone(), b.clone(), pool.clone()
        wa, wb = rng.permutation(4096)[:n0], rng.permutation(2000)[:n1]
        va, vb = rng.integers(-9, 9, len(wa)), rng.integers(0, 9, len(wb))
        pages = rng.permutation(len(pool))[:n_pages]
        want_a.view(-1)[torch.from_numpy(wa).to(DEV)] = torch.from_numpy(va).int().to(DEV)
        want_b.view(torch.int32)[torch.from_numpy(wb).to(DEV)] = torch.from_numpy(vb).int().to(DEV)
        want_pool[torch.from_numpy(pages).to(DEV)] = 0
        got_a, got_b = a.clone(), b.clone()
        ops.cache_edit([(got_a, wa, va), (got_b, wb, vb)], pool, pages)
        assert torch.equal(got_a, want_a) and torch.equal(got_b, want_b) and torch.equal(pool, want_pool)
    with pytest.raises(ops.KernelError, match="outside"):
        ops.cache_edit([(got_a, np.array([4096]), np.array([0]))])
    with pytest.raises(ops.KernelError, match="outside"):
        ops.cache_edit((), pool, [len(pool)])


def test_clear_rows(ops):
    """Rows of 16-byte, 4-byte and odd lengths, longer than a workgroup's share, and more tables than one launch takes."""
    shapes = [((3, 5, 7), torch.float32), ((2, 5, 3), torch.float16), ((1, 5), torch.int32), ((4, 5, 64, 300), torch.float32),
              ((1, 5, 2), torch.int64)] * 7
    tables = [torch.randint(1, 99, s, device=DEV).to(dt) for s, dt in shapes]
    want = [t.clone() for t in tables]
    for t in want:
        t[:, 3] = 0
    ops.clear_rows(tables, 3)
    assert all(torch.equal(t, w) for t, w in zip(tables, want))
    with pytest.raises(ops.KernelError, match="no such row"):
        ops.clear_rows(tables, 5)


# ---------------------------------------------------------------------------
# attention over the paged cache
# ---------------------------------------------------------------------------
def _fill_cache(ops, dtype, K, hd, seqs, n_slots=8, window=None):
    """Writes k, v (no rotation) for sequences given as (slot, k [n, K, hd], v) into a fresh cache."""
    from llm_infer_amd.cache import Cache, KVSpec
    total = sum(k.shape[0] for _, k, _ in seqs)
    cache = Cache([KVSpec(K, hd, window)], max_tokens=total + 64 * len(seqs) + 64, max_positions=4096,
                  dtype=dtype, device=DEV, n_slots=n_slots)
    view = None
    for slot_hint, k, v in seqs:
        slot = cache.alloc_slot()
        assert slot == slot_hint
        n = k.shape[0]
        cache.grow([slot], [n])
        view = cache.view(0)
        qkv = torch.cat([torch.zeros(n, 1 * hd), k.reshape(n, K * hd).float(), v.reshape(n, K * hd).float()], 1).to(DEV)
        pos = torch.arange(n, dtype=torch.int32, device=DEV)
        ts = torch.full((n,), slot, dtype=torch.int32, device=DEV)
        ops.rope_store(qkv.contiguous(), None, 0, False, pos, ts, view.page_table, view.page_stride, view.k, view.v,
                       1, K, hd, dtype)
    return cache, view


def _attn_ref(q, k, v, window=None):
    import plain_llama as P
    return P.attention(q.double(), k.double(), v.double(), window)


ATTN_CASES = [  # H, K, hd, lengths
    (4, 2, 16, [7, 1, 13]), (3, 1, 32, [1, 4, 9, 16, 31]), (5, 5, 48, [70, 64, 65]),
    (8, 2, 64, [200, 3]), (8, 1, 128, [130, 257]), (2, 2, 80, [66]), (40, 1, 16, [5, 90]),
]


@pytest.mark.parametrize("H,K,hd,lens", ATTN_CASES)
@pytest.mark.parametrize("dt", [torch.float32] + F16S)
def test_attention_whole_prompts_and_decode(ops, H, K, hd, lens, dt):
    g = torch.Generator().manual_seed(H * 100 + hd)
    seqs, qs = [], []
    for i, n in enumerate(lens):
        k = torch.randn(n, K, hd, generator=g).to(dt)
        v = torch.randn(n, K, hd, generator=g).to(dt)
        q = (torch.randn(n, H, hd, generator=g) * 1.5).to(dt)
        seqs.append((i, k, v))
        qs.append(q)
    cache, view = _fill_cache(ops, dt, K, hd, seqs)
    scale = hd ** -0.5
    refs = [_attn_ref(q.float(), k.float(), v.float()) for q, (_, k, v) in zip(qs, seqs)]
    tol = {torch.float32: 2e-5, torch.float16: 3e-3, torch.bfloat16: 2.5e-2}[dt]
    # all sequences whole, in one step
    from llm_infer_amd.engine.step import StepContext
    ctx = StepContext(DEV, list(range(len(lens))), [[0] * n for n in lens], [0] * len(lens), [[] for _ in lens])
    q_all = torch.cat(qs).to(DEV).contiguous()
    if dt == torch.float32:
        out = ops.attention_f32(q_all, view.as_tuple(), ctx.pos, ctx.tok_slot, H, K, hd, scale, None)
    else:
        out = ops.attention_prefill(q_all, view.as_tuple(), ops.prefill_meta(ctx), H, K, hd, scale, None)
    ref_all = torch.cat(refs)
    err = (out.double().cpu() - ref_all).abs().max().item()
    assert err < tol, err
    # the last token of every sequence as a decode step, with every split count
    q_last = torch.stack([q[-1] for q in qs]).to(DEV).contiguous()
    ref_last = torch.stack([r[-1] for r in refs])
    seq_slot = torch.arange(len(lens), dtype=torch.int32, device=DEV)
    seq_ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    if dt == torch.float32:
        pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
        out = ops.attention_f32(q_last, view.as_tuple(), pos, seq_slot, H, K, hd, scale, None)
        assert (out.double().cpu() - ref_last).abs().max().item() < tol
    else:
        for splits in (1, 2, 3, 4, 8, 16, 24):               # merged inside a workgroup, by the merge kernel, or both
            out = ops.attention_decode(q_last, view.as_tuple(), seq_slot, seq_ctx, len(lens), H, K, hd, scale,
                                       None, splits)
            err = (out.double().cpu() - ref_last).abs().max().item()
            assert err < tol, (splits, err)


# query heads of a KV head around the 16 rows of the narrow tile (beyond them the tile of 32 rows, and chunks of it), for head sizes
# of one 32 up to the largest, and sizes of 16 that are none of 32; contexts of one key, at the edges of a score tile's eights and of a
# page; the form for steady splits too (heads of up to 128 have it, the others take no notice)
@pytest.mark.parametrize("G,K,hd", [(1, 2, 32), (15, 1, 64), (16, 2, 128), (17, 1, 128), (4, 3, 96), (33, 1, 32), (7, 1, 256), (16, 1, 160),
                                    (3, 2, 80), (18, 1, 112), (33, 2, 64)])
@pytest.mark.parametrize("dt", F16S)
def test_decode_attention_in_tiles_of_16_and_32_rows(ops, G, K, hd, dt):
    g = torch.Generator().manual_seed(G * 100 + hd)
    H, lens, scale = G * K, [1, 8, 25, 63, 64, 65, 130, 300], hd ** -0.5
    seqs = [(i, torch.randn(n, K, hd, generator=g).to(dt), torch.randn(n, K, hd, generator=g).to(dt)) for i, n in enumerate(lens)]
    q = (torch.randn(len(lens), H, hd, generator=g) * 1.5).to(dt)
    sink, slopes = torch.randn(H, generator=g), torch.rand(H, generator=g) * 0.1
    cache, view = _fill_cache(ops, dt, K, hd, seqs)
    slot, ctx = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in (list(range(len(lens))), lens))
    # as test_attention_whole_prompts_and_decode: half a unit in the last place of probabilities and results of the order of 1, four times
    tol = {torch.float16: 3e-3, torch.bfloat16: 2.5e-2}[dt]
    for extra in ({}, {"window": 70, "keep_first": 5}, {"sink": sink, "slopes": slopes, "softcap": 20.0}):
        refs = []
        for i, (_, k, v) in enumerate(seqs):
            n = lens[i]
            s = torch.einsum("hd,nhd->hn", q[i].double(), k.double().repeat_interleave(G, 1)) * scale
            j = torch.arange(n)
            if "softcap" in extra:
                s = 20.0 * torch.tanh(s / 20.0) - slopes.double()[:, None] * (n - 1 - j)
            if "window" in extra:
                s = s.masked_fill((j <= n - 1 - 70) & (j >= 5), -math.inf)
            if "sink" in extra:
                p = torch.softmax(torch.cat([s, sink.double()[:, None]], 1), 1)[:, :n]
            else:
                p = torch.softmax(s, 1)
            refs.append(torch.einsum("hn,nhd->hd", p, v.double().repeat_interleave(G, 1)))
        kw = {name: t.to(DEV) if torch.is_tensor(t) else t for name, t in extra.items() if name != "window"}
        for splits, steady in ((1, False), (2, False), (4, False), (8, False), (1, True), (2, True), (4, True), (8, True)):
            out = ops.attention_decode(q.to(DEV), view.as_tuple(), slot, ctx, len(lens), H, K, hd, scale, extra.get("window"), splits,
                                       steady=steady, **kw)
            assert (out.double().cpu() - torch.stack(refs)).abs().max().item() < tol, (splits, steady, list(extra))


# many tokens, so that heads of a KV head share a workgroup (as many as 256 / hd holds and H / K has divisors for); lengths at
# the edges of the sixteens and of the 256 keys that are taken at a time; with and without a window that cuts into both
@pytest.mark.parametrize("H,K,hd,n", [(4, 1, 64, 273), (12, 2, 16, 256), (6, 2, 48, 259), (32, 8, 128, 40)])
def test_float32_attention_with_heads_in_one_workgroup(ops, H, K, hd, n):
    from llm_infer_amd.engine.step import StepContext
    g = torch.Generator().manual_seed(hd + n)
    k, v, q = (torch.randn(n, m, hd, generator=g) for m in (K, K, H))
    cache, view = _fill_cache(ops, torch.float32, K, hd, [(0, k, v)])
    ctx = StepContext(DEV, [0], [[0] * n], [0], [[]])
    qd = q.to(DEV)
    for window in (None, 37):
        out = ops.attention_f32(qd, view.as_tuple(), ctx.pos, ctx.tok_slot, H, K, hd, hd ** -0.5, window)
        assert (out.double().cpu() - _attn_ref(q, k, v, window)).abs().max().item() < 2e-5      # (as for whole prompts above)
        # a token by itself, its heads in workgroups of their own: the same sums in the same order
        for t in (0, 15, 16, n - 1):
            one = ops.attention_f32(qd[t:t + 1].contiguous(), view.as_tuple(), ctx.pos[t:t + 1], ctx.tok_slot[t:t + 1], H, K, hd,
                                    hd ** -0.5, window)
            assert torch.equal(one[0], out[t]), (window, t)


# a token by itself (the kernel for few tokens) against all of a prompt together, bit for bit: contexts that end at the edges of
# pages and of the 256 keys taken at a time, windows that begin within a page, at its edge and beyond 256 keys; what lies behind a
# token in its page is no number and must not reach it
@pytest.mark.parametrize("H,K,hd", [(4, 1, 16), (6, 2, 64), (5, 1, 112), (3, 1, 256)])
def test_float32_attention_of_few_tokens(ops, H, K, hd):
    from llm_infer_amd.engine.step import StepContext
    g = torch.Generator().manual_seed(hd)
    n, held = 450, 400
    k, v, q = (torch.randn(n, m, hd, generator=g) for m in (K, K, H))
    v[held:] = float("nan")
    cache, view = _fill_cache(ops, torch.float32, K, hd, [(0, k, v)])
    ctx = StepContext(DEV, [0], [[0] * n], [0], [[]])
    qd = q.to(DEV)
    for window in (None, 37, 64, 100, 300):
        every = ops.attention_f32(qd, view.as_tuple(), ctx.pos, ctx.tok_slot, H, K, hd, hd ** -0.5, window)[:held]
        assert torch.isfinite(every).all()
        for some in ([0, 62, 63], [64, 127, 128, 191], [254, 255, 256], [319, 320, held - 1]):
            t = torch.tensor(some, device=DEV)
            few = ops.attention_f32(qd[t].contiguous(), view.as_tuple(), t.to(torch.int32), ctx.tok_slot[t].contiguous(), H, K, hd,
                                    hd ** -0.5, window)
            assert torch.equal(few, every[t]), (window, some)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_attention_window_and_far_key(ops, dt):
    """One far key among hundreds stands out by its score; the window cuts it off exactly at its edge."""
    H, K, hd, n = 2, 1, 32, 300
    g = torch.Generator().manual_seed(5)
    k = (torch.randn(n, K, hd, generator=g) * 0.1)
    v = torch.randn(n, K, hd, generator=g)
    q = torch.randn(n, H, hd, generator=g) * 0.1
    far = 37
    k[far, 0, :] = 0
    k[far, 0, 3] = 12.0
    q[:, :, 3] = 6.0                      # every query looks hard at key `far`
    k, v, q = k.to(dt), v.to(dt), q.to(dt)
    cache, view = _fill_cache(ops, dt, K, hd, [(0, k, v)])
    from llm_infer_amd.engine.step import StepContext
    ctx = StepContext(DEV, [0], [[0] * n], [0], [[]])
    scale = hd ** -0.5
    tol = 2e-5 if dt == torch.float32 else 2.5e-2
    for window in (None, 100, 64, 1):
        ref = _attn_ref(q.float(), k.float(), v.float(), window)
        qd = q.to(DEV).contiguous()
        if dt == torch.float32:
            out = ops.attention_f32(qd, view.as_tuple(), ctx.pos, ctx.tok_slot, H, K, hd, scale, window)
        else:
            out = ops.attention_prefill(qd, view.as_tuple(), ops.prefill_meta(ctx), H, K, hd, scale, window)
        assert (out.double().cpu() - ref).abs().max().item() < tol, window
        if window == 100:
            # position far+99 still sees the far key, far+100 does not
            o = out.float().cpu()
            assert (o[far + 99, 0] - v[far, 0].float()).abs().max() < 0.05
            assert (o[far + 100, 0] - v[far, 0].float()).abs().max() > 0.2
        if dt != torch.float32:
            last = qd[-1:].contiguous()
            out1 = ops.attention_decode(last, view.as_tuple(), torch.zeros(1, dtype=torch.int32, device=DEV),
                                        torch.tensor([n], dtype=torch.int32, device=DEV), 1, H, K, hd, scale,
                                        window, 2)
            assert (out1.double().cpu()[0] - ref[-1]).abs().max().item() < tol


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("window", [100, 64])
def test_decode_attention_at_the_window_edge(ops, dt, window):
    """The 16-bit decode kernel cuts the window exactly: a far key that outweighs all others is seen by
    the last position that may see it and not by the next, with every count of splits; and with the
    pages below the window given back and everything free filled with NaN."""
    H, K, hd, n = 2, 1, 32, 300
    scale = hd ** -0.5
    tol = 3e-3 if dt == torch.float16 else 2.5e-2

    def make(far):
        g = torch.Generator().manual_seed(far)
        k = torch.randn(n, K, hd, generator=g) * 0.1
        v = torch.randn(n, K, hd, generator=g)
        q = torch.randn(n, H, hd, generator=g) * 0.1
        k[far, 0, :] = 0
        k[far, 0, 3] = 12.0
        q[:, :, 3] = 6.0
        return k.to(dt), v.to(dt), q.to(dt)

    def decode(view, q_row, ctx_len, splits):
        return ops.attention_decode(q_row.to(DEV).contiguous(), view.as_tuple(), torch.zeros(1, dtype=torch.int32, device=DEV),
                                    torch.tensor([ctx_len], dtype=torch.int32, device=DEV), 1, H, K, hd, scale,
                                    window, splits).float().cpu()[0]

    # a cache that keeps everything; the context length moves over the edge
    far = 37
    k, v, q = make(far)
    cache, view = _fill_cache(ops, dt, K, hd, [(0, k, v)])
    ref = _attn_ref(q.float(), k.float(), v.float(), window)
    for splits in (1, 2, 8):
        for ctx_len, sees in ((far + window, True), (far + window + 1, False)):
            out = decode(view, q[ctx_len - 1:ctx_len], ctx_len, splits)
            assert (out.double() - ref[ctx_len - 1]).abs().max().item() < tol, (splits, ctx_len)
            assert ((out[0] - v[far, 0].float()).abs().max() < 0.05) == sees, (splits, ctx_len)
    # a cache of a window group: pages that lie wholly below the window are given back, and whatever is
    # free (the page that free table entries point at included) holds NaN
    for far, sees in ((n - window, True), (n - window - 1, False)):
        k, v, q = make(far)
        cache, view = _fill_cache(ops, dt, K, hd, [(0, k, v)], window=window)
        cache.trim_windows([0])
        group = cache.groups[0]
        first = group.first_needed_page(n)
        assert first >= 3 and sorted(group.pages_of[0]) == list(range(first, (n + 63) // 64))
        free = [p for p in range(group.n_pages) if p not in group.pool.held()]
        group.storage[torch.tensor(free, device=DEV)] = float("nan")
        ref = _attn_ref(q.float(), k.float(), v.float(), window)[-1]
        for splits in (1, 2, 8):
            out = decode(view, q[-1:], n, splits)
            assert torch.isfinite(out).all(), (far, splits)
            assert (out.double() - ref).abs().max().item() < tol, (far, splits)
            assert ((out[0] - v[far, 0].float()).abs().max() < 0.05) == sees, (far, splits)


def test_rope_store_rotation_and_cache_layout(ops):
    """Rotation against the plain formula, both pairings, partial rotary dim; keys read back
    through attention with a one-hot query."""
    import plain_llama as P
    H, K, hd, rot, n = 2, 2, 32, 16, 70
    g = torch.Generator().manual_seed(3)
    qkv = torch.randn(n, (H + 2 * K) * hd, generator=g)
    from llm_infer_amd.cache import Cache, KVSpec
    cache = Cache([KVSpec(K, hd)], 256, 1024, torch.float32, DEV, 2)
    slot = cache.alloc_slot()
    cache.grow([slot], [n])
    view = cache.view(0)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)
    ts = torch.zeros(n, dtype=torch.int32, device=DEV)
    i = torch.arange(0, rot, 2, dtype=torch.float32)
    inv = (1.0 / torch.pow(torch.tensor(10000.0), i / rot)).to(DEV)
    q = ops.rope_store(qkv.to(DEV), inv, rot, False, pos, ts, view.page_table, view.page_stride, view.k, view.v,
                       H, K, hd, torch.float32)
    ref_q = P.rope(qkv[:, :H * hd].view(n, H, hd).double(), torch.arange(n), 10000.0, rot)
    assert torch.allclose(q.double().cpu(), ref_q, atol=2e-5)
    ref_k = P.rope(qkv[:, H * hd:(H + K) * hd].view(n, K, hd).double(), torch.arange(n), 10000.0, rot)
    ref_v = qkv[:, (H + K) * hd:].view(n, K, hd).double()
    # read keys back: a one-hot query at dim j gives scores k[t, j]; check through decode attention
    # on the values instead: attention with all-equal scores averages v
    zero_q = torch.zeros(1, H, hd, device=DEV)
    out = ops.attention_f32(zero_q, view.as_tuple(), torch.tensor([n - 1], dtype=torch.int32, device=DEV),
                            torch.zeros(1, dtype=torch.int32, device=DEV), H, K, hd, 1.0, None)
    assert torch.allclose(out[0].double().cpu(), ref_v.mean(0), atol=1e-5)
    # keys: q = e_j * big picks the token with the largest k[:, j]
    for j in (0, 5, 17, 31):
        qq = torch.zeros(1, H, hd, device=DEV)
        qq[0, :, j] = 200.0
        out = ops.attention_f32(qq, view.as_tuple(), torch.tensor([n - 1], dtype=torch.int32, device=DEV),
                                torch.zeros(1, dtype=torch.int32, device=DEV), H, K, hd, 1.0, None)
        for h in range(H):
            best = ref_k[:, h, j].argmax().item()
            assert torch.allclose(out[0, h].double().cpu(), ref_v[best, h], atol=1e-3), (j, h)
    # half pairing equals the plain rotation applied to de-interleaved heads
    q2 = ops.rope_store(qkv.to(DEV), inv, rot, True, pos, ts, None, None, None, None, H, 0, hd, torch.float32)
    x = qkv[:, :H * hd].view(n, H, hd).double()
    perm = torch.cat([torch.stack([torch.arange(rot // 2), torch.arange(rot // 2) + rot // 2], 1).reshape(-1),
                      torch.arange(rot, hd)])
    ref_half = torch.empty_like(x)
    ref_half[..., perm] = P.rope(x[..., perm], torch.arange(n), 10000.0, rot)
    assert torch.allclose(q2.double().cpu(), ref_half, atol=2e-5)


@pytest.mark.parametrize("dt", F16S)
@pytest.mark.parametrize("T,H,K,hd,rot,d", [(1, 4, 2, 16, 16, 64), (9, 3, 1, 32, 16, 96), (70, 5, 5, 48, 24, 160),
                                           (200, 8, 2, 64, 64, 256), (3, 2, 0, 32, 32, 64)])
def test_rotation_fused_into_the_projection(ops, dt, T, H, K, hd, rot, d):
    """The product whose epilogue rotates and stores equals the product followed by rope_store:
    q and the cache pages within one rounding of the stored dtype when both use the same sums."""
    from llm_infer_amd.cache import Cache, KVSpec
    g = torch.Generator().manual_seed(T + hd)
    x = torch.randn(T, d, generator=g).to(dt).to(DEV)
    w = (torch.randn((H + 2 * K) * hd, d, generator=g) / math.sqrt(d)).to(dt).to(DEV)
    inv = (1.0 / torch.pow(torch.tensor(500.0), torch.arange(0, rot, 2, dtype=torch.float32) / rot)).to(DEV)
    pos = (torch.arange(T, dtype=torch.int32) + 60).to(DEV)
    ts = torch.zeros(T, dtype=torch.int32, device=DEV)

    def fresh():
        c = Cache([KVSpec(max(K, 1), hd)], 512, 1024, dt, DEV, 2)
        s_ = c.alloc_slot()
        c.grow([s_], [60 + T])
        return c, c.view(0)

    c0, v0 = fresh()
    qkv = ops.linear(x, w, out_dtype=torch.float32, force="fma")
    args0 = (v0.page_table, v0.page_stride, v0.k, v0.v) if K else (None, None, None, None)
    q0 = ops.rope_store(qkv, inv, rot, False, pos, ts, *args0, H, K, hd, dt)
    kinds = ["fma", None] + (["gemv_mfma"] if T <= 16 else []) + ["mfma:0:1", "mfma:2:2"]
    for tiled in (False, True):
        if tiled and d % 32:
            continue
        ww = ops.tile_weight(w) if tiled else w
        for kind in kinds + (["wreg:0", "wreg:1:2", "wreg:2"] if tiled else []):
            if tiled and kind == "fma":
                continue
            c1, v1 = fresh()
            args1 = (v1.page_table, v1.page_stride, v1.k, v1.v) if K else (None, None, None, None)
            table = ops.rope_table(inv, pos, T) if kind != "fma" else None     # with and without the table
            q1 = ops.linear_rope_store(x, ww, inv, rot, pos, ts, *args1, H, K, hd, dt, force=kind, cos_sin=table)
            # the same float32 sums on the "fma" path: at most one rounding of the stored dtype apart
            tol = (2.0 ** -9 if dt == torch.float16 else 2.0 ** -7) if kind == "fma" else 2e-2
            assert (q1.float() - q0.float()).abs().max().item() <= tol * (1 + q0.float().abs().max().item()), kind
            if K:
                a, b = c0.groups[0].storage.float(), c1.groups[0].storage.float()
                assert (a - b).abs().max().item() <= tol * (1 + a.abs().max().item()), kind
                assert (b != 0).sum().item() >= 0.9 * T * 2 * K * hd


def test_token_probability(ops):
    import plain_llama as P
    g = torch.Generator().manual_seed(5)
    for V in (7, 65, 331, 5000, 128256, 300007):
        logits = torch.randn(5, V, generator=g) * 4
        logits[0, V // 2] = 40.0                                   # nearly all the mass on one token
        tokens = [V // 2, 0, V - 1, V, -1]                         # the last two lie outside the vocabulary
        got = ops.token_prob(logits.to(DEV), torch.tensor(tokens, dtype=torch.int32, device=DEV)).cpu()
        want = torch.tensor([P.token_prob(logits[i].double(), t) for i, t in enumerate(tokens)])
        assert got[3] == 0 and got[4] == 0
        torch.testing.assert_close(got, want.float(), rtol=2e-5, atol=1e-12)
        assert got[0] > 0.999
        # all tokens of a row add up to one
        row = logits[1:2].expand(V, V).contiguous().to(DEV) if V <= 331 else None
        if row is not None:
            every = ops.token_prob(row, torch.arange(V, dtype=torch.int32, device=DEV))
            assert abs(every.double().sum().item() - 1.0) < 1e-5


def test_sampling_kernels(ops):
    import plain_llama as P
    g = torch.Generator().manual_seed(0)
    for V in (7, 64, 65, 256, 331, 5000, 128256, 300007):      # one chunk, 32 chunks, chunks longer than 4,096
        logits = torch.randn(6, V, generator=g) * 3
        logits[1, 3] = logits[1, V - 2] = 50.0                    # a tie: the first wins
        logits[2, V - 1] = 60.0
        d = logits.to(DEV)
        got = ops.argmax(d).tolist()
        assert got == [P.sample_greedy(r) for r in logits]
        assert got[1] == 3 and got[2] == V - 1
        for T in (0.01, 0.8, 2.0, 1e6):             # from nearly only the maximum to nearly equal chances
            rs = [0.0, 0.25, 0.5, 0.75, 0.999, 0.9999999]
            r = torch.tensor(rs, dtype=torch.float32, device=DEV)
            got = ops.sample(d, T, forced_r=r).tolist()
            for b in range(6):
                p = P.probabilities(logits[b].double(), T)
                c = torch.cumsum(p, 0)
                lo = c[got[b] - 1].item() if got[b] > 0 else 0.0
                hi = c[got[b]].item()
                assert lo - 1e-5 <= rs[b] < hi + 1e-5, (V, T, b, got[b])
        assert ops.sample(d, 0.0).tolist() == ops.argmax(d).tolist()
    # the generator: host twin equals the device, streams differ by key, counter advances
    state = torch.tensor([[11, 0], [12, 0]], dtype=torch.int64, device=DEV)
    slots = torch.tensor([1, 0], dtype=torch.int32, device=DEV)
    logits = torch.zeros(2, 64, device=DEV)                     # uniform distribution: token = floor(r * 64)
    t1 = ops.sample(logits, 1.0, slots, state).tolist()
    t2 = ops.sample(logits, 1.0, slots, state).tolist()
    assert state[:, 1].tolist() == [2, 2]
    assert t1 == [int(ops.uniform01(12, 0) * 64), int(ops.uniform01(11, 0) * 64)]
    assert t2 == [int(ops.uniform01(12, 1) * 64), int(ops.uniform01(11, 1) * 64)]
    us = [ops.uniform01(5, i) for i in range(2000)]
    assert 0.45 < sum(us) / len(us) < 0.55 and min(us) >= 0.0 and max(us) < 1.0
    # drawn tokens follow the probabilities: 8192 sequences with generators of their own, one draw each
    n, V = 8192, 7
    row = torch.tensor([2.0, 0.5, -1.0, 1.5, 0.0, -3.0, 1.0])
    p = P.probabilities(row.double(), 0.7)
    state = torch.stack([torch.arange(n, dtype=torch.int64) + 1000, torch.zeros(n, dtype=torch.int64)], 1).to(DEV)
    drawn = ops.sample(row.repeat(n, 1).to(DEV), 0.7, torch.arange(n, dtype=torch.int32, device=DEV), state)
    freq = torch.bincount(drawn.cpu().long(), minlength=V).double() / n
    sigma = torch.sqrt(p * (1 - p) / n)
    assert ((freq - p).abs() < 5 * sigma + 1e-9).all(), (freq.tolist(), p.tolist())


@pytest.mark.parametrize("M,N,K", [(1, 2050, 256), (8, 3000, 512), (17, 130, 96), (40, 72, 160), (130, 520, 2048), (3, 33, 40)])
def test_a_soft_cap_in_the_products_epilogue(ops, M, N, K):
    """Bit for bit the product and the pass over its values behind it, for every kernel that the sizes and types choose."""
    g = torch.Generator().manual_seed(M + N + K)
    for dt in (torch.float32, torch.float16, torch.bfloat16):
        x, w = torch.randn(M, K, generator=g).to(DEV, dt), torch.randn(N, K, generator=g).to(DEV, dt)
        for weight in (w, ops.prepare_weight(w)):
            got = ops.linear(x, weight, ops.EPI_BIAS, out_dtype=torch.float32, params=ops.glu_params(act="softcap", limit=3.5))
            assert torch.equal(got, ops.softcap(ops.linear(x, weight, out_dtype=torch.float32), 3.5))
    with pytest.raises(ops.KernelError):
        ops.linear(x, w, ops.EPI_BIAS, out_dtype=torch.float32, params=ops.glu_params(act="softcap", limit=0.0))


@pytest.mark.parametrize("N", [592, 583])
@pytest.mark.parametrize("M,force", [(300, "wreg:0"), (300, "wreg:1"), (300, "wreg:2"), (50, "wreg:2:1:1"), (100, "wreg:2:1:3"), (129, "wreg:2:2")])
def test_activations_in_the_epilogue_of_prompts_products(ops, M, force, N):
    """Bit for bit the activation of the stored float32 sums, with a bias and without: whole rows and the last columns, every tile, K whole and
    split.  tanh is the soft cap of 1."""
    g = torch.Generator().manual_seed(M + N)
    for dt in (torch.float16, torch.bfloat16):
        x, w = torch.randn(M, 256, generator=g).to(DEV, dt), ops.prepare_weight((torch.randn(N, 256, generator=g) / 8).to(DEV, dt))
        bias = torch.randn(N, generator=g).to(DEV)
        run = lambda out=torch.float32, **p: ops.linear(x, w, ops.EPI_BIAS, out_dtype=out, force=force, params=ops.glu_params(**p))
        plain = ops.linear(x, w, out_dtype=torch.float32, force=force)
        for b, sums in ((None, plain), (bias, plain + bias)):
            for out in (torch.float32, dt):
                assert torch.equal(run(out, bias=b, act="relu2"), sums.clamp(min=0).square().to(out))
                assert torch.equal(run(out, bias=b, act="tanh"), ops.softcap(sums.clone(), 1.0).to(out))
                assert torch.equal(run(out, bias=b, act="softcap", limit=3.5), ops.softcap(sums.clone(), 3.5).to(out))
        assert torch.equal(run(bias=bias), plain + bias)


@pytest.mark.parametrize("rows,n", [(1, 1), (5, 3), (130, 130), (130, 66)])
def test_a_steps_first_kernel_sends_the_tokens_before_it_to_the_host(ops, rows, n):
    """decode_prepare's ring of tokens, recorded and replayed: every step's own tokens, rows that a smaller step leaves out keep
    count, a number that no step had is an error and not a wait for ever."""
    from llm_infer_amd.tensor import Tensor
    i32 = lambda v: torch.full((rows,), v, dtype=torch.int32, device=DEV)
    slots = torch.arange(rows, dtype=torch.int32, device=DEV)
    lens, pos, ctx, tokens, steps = i32(7), i32(0), i32(0), i32(0), i32(0)
    ring = Tensor.pinned((ops.TOKEN_RING, rows), torch.int64)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())                  # (the kernel indexes by what the lines above fill in)
    torch.cuda.synchronize()
    assert slots.tolist() == list(range(rows)) and lens.tolist() == [7] * rows
    graphs = {}
    with torch.cuda.stream(side):
        ops.decode_prepare(slots, lens, pos, ctx, rows, -1, None, (tokens, steps, ring))
        assert ops.wait_tokens(ring, rows, 1) == [0] * rows
        for k in (rows, n):
            graphs[k] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graphs[k], stream=side):
                ops.decode_prepare(slots, lens, pos, ctx, k, -1, None, (tokens, steps, ring))
        for step in range(2, 12):
            k = rows if step % 3 else n
            tokens.copy_(torch.arange(rows, dtype=torch.int32) * 1000 + step - (1 << 20))
            graphs[k].replay()
            assert ops.wait_tokens(ring, k, step) == [r * 1000 + step - (1 << 20) for r in range(k)]
        with pytest.raises(ops.KernelError):
            ops.wait_tokens(ring, n, 12)
    assert steps.tolist() == [11] * rows
    with pytest.raises(ops.KernelError):
        ops.decode_prepare(slots, lens, pos, ctx, rows, -1, None, (tokens, steps, ring[:2]))
    with pytest.raises(ops.KernelError):
        ops.wait_tokens(ring, rows + 1, 1)
