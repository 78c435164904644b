"""Each HIP kernel alone against a plain float32 reference of the same op, at sizes other than
the engine's (odd widths, head sizes in steps of 16, page sizes 8..64)."""
import math

import pytest
import torch
import torch.nn.functional as F

import plain_qwen2 as P
from gpu_util import DEV, DTYPES, flat_batch, paged_cache, tol
from test_plain import REFERENCE_CASES

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from pico_vllm_amd.ops import kernels
    return kernels


def close(a, b, dtype, scale=1.0):
    rtol, atol = tol(dtype)
    a, b = a.float().cpu(), b.float().cpu()
    assert a.shape == b.shape
    err = (a - b).abs()
    bound = atol * scale + rtol * b.abs()
    assert bool((err <= bound).all()), f"max err {float(err.max()):.3e} (bound {float(bound.min()):.3e}..)"


@pytest.mark.parametrize("dtype", DTYPES)
def test_embedding(K, dtype):
    table = torch.randn(301, 136).to(dtype)
    ids = torch.tensor([0, 300, 5, 5, 17], dtype=torch.int32)
    out = K.embedding(table.to(DEV), ids.to(DEV))
    assert out.dtype == torch.float32
    assert torch.equal(out.cpu(), table.float()[ids.long()])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H", [64, 136, 1536, 5000])
def test_add_rmsnorm(K, dtype, H):
    T, eps = 7, 1e-5
    resid = torch.randn(T, H) * 3
    delta = (torch.randn(T, H)).to(dtype)
    w = 1 + 0.1 * torch.randn(H)
    want_sum = resid + delta.float()
    r = resid.clone().to(DEV)
    out = K.add_rmsnorm(r, delta.to(DEV), w.to(DEV), eps, dtype)
    close(r, want_sum, torch.float32)                                   # the residual stream is float32
    close(out, P.rms_norm(want_sum, w, eps), dtype)
    # no delta: the stream is untouched
    r2 = resid.clone().to(DEV)
    out = K.add_rmsnorm(r2, None, w.to(DEV), eps, dtype)
    assert torch.equal(r2.cpu(), resid)
    close(out, P.rms_norm(resid, w, eps), dtype)
    # wanted rows only: the stream is untouched, rows are gathered
    rows = torch.tensor([6, 0, 3], dtype=torch.int32)
    r3 = resid.clone().to(DEV)
    out = K.add_rmsnorm(r3, delta.to(DEV), w.to(DEV), eps, dtype, rows=rows.to(DEV))
    assert torch.equal(r3.cpu(), resid)
    close(out, P.rms_norm(want_sum[rows.long()], w, eps), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_residual_add(K, dtype):
    # the add without a norm, for an arrangement of parts that ends on an add
    resid, delta = torch.randn(7, 136) * 3, torch.randn(7, 136).to(dtype)
    r = resid.clone().to(DEV)
    assert K.residual_add(r, delta.to(DEV)) is r
    assert torch.equal(r.cpu(), resid + delta.float())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1027])
def test_residual_add_in_fours_and_what_is_left(K, dtype, n):
    # whole fours, what they leave, and rows that start on no sixteen bytes: one float32 sum an entry, so exact
    resid, delta = torch.randn(n + 3) * 3, torch.randn(n + 3).to(dtype)
    for at in (0, 1):
        r, d = resid.clone().to(DEV), delta.to(DEV)
        K.residual_add(r[at:at + n], d[at:at + n])
        want = resid.clone()
        want[at:at + n] += delta[at:at + n].float()
        assert torch.equal(r.cpu(), want)


def test_rmsnorm_eps_is_inside_the_root(K):
    x = torch.full((1, 64), 1e-4)
    out = K.add_rmsnorm(x.to(DEV), None, torch.ones(64, device=DEV), 1e-2, torch.float32)
    close(out, x / math.sqrt(1e-8 + 1e-2), torch.float32)


@pytest.mark.parametrize("dtype", DTYPES)
def test_swiglu(K, dtype):
    gu = (torch.randn(5, 2 * 172) * 2).to(dtype)
    close(K.swiglu(gu.to(DEV)), P.swiglu(gu), dtype)
    g = gu[:, :172].float()
    close(K.swiglu(torch.cat([gu[:, :172], torch.ones(5, 172).to(dtype)], -1).to(DEV)), F.silu(g), dtype)
    # halves that are multiples of 8 take the kernel with 16-byte loads in bfloat16
    for T, I in ((3, 8), (70, 320), (33, 8960)):
        gu = (torch.randn(T, 2 * I) * 2).to(dtype)
        close(K.swiglu(gu.to(DEV)), P.swiglu(gu), dtype)


@pytest.mark.parametrize("T,I", [(1, 4), (3, 1020), (7, 1028), (300, 8960), (65536, 4)])
def test_swiglu_of_float32_rows(K, T, I):
    # four elements a thread at the edges of a workgroup and of the grid; the same bits as rows that start elsewhere, one element a thread
    gu = torch.randn(T, 2 * I, device=DEV)
    odd = torch.empty(2 * I * T + 1, device=DEV)[1:].view(T, 2 * I)
    odd.copy_(gu)
    out = K.swiglu(gu)
    assert torch.equal(out, K.swiglu(odd))
    want = F.silu(gu[:, :I].double()) * gu[:, I:].double()
    assert bool(((out.double() - want).abs() <= 2.0 ** -21 * want.abs() + 1e-30).all())     # exponential, sum, quotient, product: under 8 roundings of 2^-24


@pytest.mark.parametrize("counts,D,F_", [([0, 1, 63, 64, 65], 72, 40), ([129, 0, 48, 2], 64, 264), ([1, 127, 128, 129, 700], 136, 1000),
                                         ([0, 1100], 328, 200), ([0, 0, 5], 1536, 8),
                                         ([200, 1, 129], 8328, 72), ([128, 300], 5440, 328), ([129] * 16, 1152, 456), ([129] * 16, 1728, 72)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_moe_grouped(K, counts, D, F_, mode):
    # experts with rows up to, at and behind the edges of tiles of 64 and 128 rows and of strips of tiles, columns and k that
    # end inside a tile and a stage; a row with a stride; a number that has no matrices; a second product of one round of tiles of 128
    # columns, of 192, and of more; choices so uneven that what was taken for one round is 288 tiles for 256 workgroups
    g = torch.Generator().manual_seed(D + F_)
    E, which = len(counts), [e for e, n in enumerate(counts) for _ in range(n)] + [len(counts)]
    R = len(which)
    which = torch.tensor(which)[torch.randperm(R, generator=g)]
    h = torch.randn(R, D + 8, generator=g).bfloat16().to(DEV)[:, 8:]
    gate_up = (torch.randn(E, 2 * F_, D, generator=g) * D ** -0.5).bfloat16().to(DEV)
    down = (torch.randn(E, D, F_, generator=g) * F_ ** -0.5).bfloat16().to(DEV)
    wt = torch.rand(R, 1, generator=g).to(DEV)
    got = K.moe_experts(h, gate_up, down, which.int().view(R, 1).to(DEV), wt, 0.7, 1.702, grouped=True, mode=mode).double()
    for e in range(E + 1):
        at = (which == e).nonzero().view(-1).to(DEV)
        if e == E:
            assert not got[at].any()                 # one slot a token: rows of no expert are left zero
            continue
        w = wt[at].double()
        z = (h[at].double() * (w if mode == 0 else 1.0)) @ gate_up[e].double().T
        gate, up = z[:, :F_], z[:, F_:]
        if mode != 1:
            gate, up = gate.clamp(max=0.7), up.clamp(-0.7, 0.7) + 1
        y = gate * torch.sigmoid((1.0 if mode == 1 else 1.702) * gate) * up * (w if mode else 1.0)
        want = y @ down[e].double().T
        # y is rounded once to bfloat16 (eight bits: at most 2^-8 of its size), the sums are float32 (1e-5 of a row's size each)
        slack = (y.abs() * 2.0 ** -8 + 1e-5 * (1 + 2 * z.abs().max() if at.numel() else 1.0)) @ down[e].double().abs().T + 1e-5
        assert bool(((got[at] - want).abs() <= slack).all())


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_experts_activation_has_the_same_bits_by_every_kernel(K, mode):
    # a gate that is one number of the row and an up that is another: every finite bfloat16 number through the activation by the grouped products,
    # the kernel that streams matrices and the plain one.  All other sums are exact, so the bits are the activation's: a last bit here sends
    # later tokens to other experts
    x = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = x[torch.isfinite(x.float())]
    T = x.numel()
    h = torch.zeros(T, 16, dtype=torch.bfloat16)
    h[:, 0], h[:, 1] = x, (torch.arange(T) % 13 - 6) / 8
    gate_up, down = torch.zeros(1, 16, 16, dtype=torch.bfloat16), torch.zeros(1, 16, 8, dtype=torch.bfloat16)
    gate_up[0, :8, 0], gate_up[0, 8:, 1], down[0, :8] = 1, 1, torch.eye(8)
    which, wt = torch.zeros(T, 1, dtype=torch.int32), torch.full((T, 1), 1.0 if mode == 0 else 0.3)
    args = [t.to(DEV) for t in (h, gate_up, down, which, wt)]
    plain = K.moe_experts_plain(*args, 7.0, 1.702, mode=mode)
    for grouped in (True, False):
        assert torch.equal(K.moe_experts(*args, 7.0, 1.702, grouped=grouped, mode=mode), plain)


@pytest.mark.parametrize("T,top,E,F,D", [(4, 2, 16, 2240, 1536), (5, 4, 7, 24, 40), (8, 2, 2, 200, 72), (16, 1, 3, 136, 520), (16, 4, 40, 64, 64), (17, 4, 6, 48, 56), (64, 1, 64, 32, 8)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_rows_that_share_an_expert_have_the_bits_of_rows_alone(K, T, top, E, F, D, mode):
    # a wave's 64 rows and more, experts that all rows and that none chose, a slot without an expert (from E on: left as it is), padding tokens
    g = torch.Generator(device=DEV).manual_seed(T * top + E)
    h = torch.randn(T, D, device=DEV, generator=g).bfloat16()
    gate_up = torch.randn(E, 2 * F, D, device=DEV, generator=g).mul(D ** -0.5).bfloat16()
    down = torch.randn(E, D, F, device=DEV, generator=g).mul(F ** -0.5).bfloat16()
    which = torch.stack([torch.randperm(E + 1, device=DEV, generator=g)[:top] for _ in range(T)]).int()
    wt = torch.rand(T, top, device=DEV, generator=g)
    live = torch.randint(0, 3, (T,), device=DEV, generator=g).int()
    live[-1] = 5
    slabs = lambda t: t.reshape(top, -1, D)
    alone = torch.cat([slabs(K.moe_experts(h[t:t + 1], gate_up, down, which[t:t + 1], wt[t:t + 1], 0.7, 1.702, grouped=False, mode=mode)) for t in range(T)], 1)
    got = slabs(K.moe_experts(h, gate_up, down, which, wt, 0.7, 1.702, grouped=False, mode=mode))
    padded = slabs(K.moe_experts(h, gate_up, down, which, wt, 0.7, 1.702, grouped=False, mode=mode, live=live))
    there = (which < E).t()                       # a slot without an expert is not written
    assert torch.equal(got[there], alone[there])
    keep = there & (live > 0)
    assert torch.equal(padded[keep], alone[keep])
    if 3 < T and T * top <= 64:
        assert float(padded[:, live == 0].abs().sum()) == 0
    # sorted by expert: what padding tokens would read and write is left out, the others' rows keep their bits
    sort = [slabs(K.moe_experts(h, gate_up, down, which, wt, 0.7, 1.702, grouped=True, mode=mode, live=x)) for x in (None, live)]
    assert torch.equal(sort[1][keep], sort[0][keep]) and (T * top > min(64, 2 * E) or float(sort[1][:, live == 0].abs().sum()) == 0)


@pytest.mark.parametrize("F", [524280, 524288, 1048560])
def test_experts_of_few_rows_and_very_many_columns(K, F):
    # 65,535 tiles of sixteen columns a row alone, of eight where rows share an expert, and beyond
    g = torch.Generator(device=DEV).manual_seed(F)
    h, gate_up = torch.randn(4, 8, device=DEV, generator=g).bfloat16(), torch.randn(1, 2 * F, 8, device=DEV, generator=g).bfloat16()
    down, wt = torch.randn(1, 8, F, device=DEV, generator=g).mul(F ** -0.5).bfloat16(), torch.rand(4, 1, device=DEV, generator=g)
    which = torch.zeros(4, 1, dtype=torch.int32, device=DEV)
    alone = torch.cat([K.moe_experts(h[t:t + 1], gate_up, down, which[t:t + 1], wt[t:t + 1], 0.7, 1.702, grouped=False) for t in range(4)])
    for share in (None, True):
        assert torch.equal(K.moe_experts(h, gate_up, down, which, wt, 0.7, 1.702, grouped=False, share=share), alone)


@pytest.mark.parametrize("T,top,E,F,D", [(1, 1, 1, 8, 8), (3, 4, 4, 40, 24), (4, 2, 16, 2240, 1536), (5, 4, 7, 24, 40), (8, 2, 2, 200, 72), (16, 1, 3, 136, 520),
                                         (16, 4, 40, 64, 64), (64, 1, 64, 32, 8), (8, 2, 16, 2240, 1536)])
@pytest.mark.parametrize("share", [True, False])
def test_rows_that_share_a_stream_and_rows_that_do_not(K, T, top, E, F, D, share):
    # either way the bits of rows one by one, a slot without an expert left as it is, padding tokens zero; as the rule has it in the last
    g = torch.Generator(device=DEV).manual_seed(T * top + F)
    h = torch.randn(T, D, device=DEV, generator=g).bfloat16()
    gate_up = torch.randn(E, 2 * F, D, device=DEV, generator=g).mul(D ** -0.5).bfloat16()
    down = torch.randn(E, D, F, device=DEV, generator=g).mul(F ** -0.5).bfloat16()
    which = torch.stack([torch.randperm(E + 1, device=DEV, generator=g)[:top] for _ in range(T)]).int()
    wt = torch.rand(T, top, device=DEV, generator=g)
    live = torch.randint(0, 2, (T,), device=DEV, generator=g).int()
    run = lambda rows, **more: K.moe_experts(h[rows], gate_up, down, which[rows], wt[rows], 7.0, 1.702, grouped=False, **more).reshape(top, -1, D)
    alone = torch.cat([run(slice(t, t + 1), share=False) for t in range(T)], 1)
    there = (which < E).t()
    every = slice(None)
    assert torch.equal(run(every, share=share)[there], alone[there])
    padded = run(every, share=share, live=live)
    assert torch.equal(padded[there & (live > 0)], alone[there & (live > 0)]) and float(padded[:, live == 0].abs().sum()) == 0
    assert torch.equal(run(every)[there], alone[there])


def test_moe_experts_of_operands_beyond_the_grouped_products_reach(K):
    # activations that span 2^31 bytes and more, and an expert of as many
    g = torch.Generator(device=DEV).manual_seed(1)
    which = torch.arange(40, device=DEV).int().view(40, 1) % 3
    wt = torch.rand(40, 1, generator=g, device=DEV)
    for D, F_, stride in ((64, 48, 2 ** 25), (16384, 32768, 16384)):
        wide = torch.empty(39 * stride + D, device=DEV, dtype=torch.bfloat16)
        h = wide.as_strided((40, D), (stride, 1))
        h.normal_(generator=g)
        gate_up = torch.empty(3, 2 * F_, D, device=DEV, dtype=torch.bfloat16).normal_(0, D ** -0.5, generator=g)
        down = torch.empty(3, D, F_, device=DEV, dtype=torch.bfloat16).normal_(0, F_ ** -0.5, generator=g)
        assert K.moe_fast_ok(h, gate_up, down) and not K.moe_grouped_ok(h, down)
        got = K.moe_experts(h, gate_up, down, which, wt, 0.7, 1.702)
        assert torch.equal(got, K.moe_experts(h.contiguous(), gate_up, down, which, wt, 0.7, 1.702, grouped=False))
        want = K.moe_experts_plain(h.contiguous(), gate_up, down, which, wt, 0.7, 1.702)
        assert torch.allclose(got, want, rtol=2e-2, atol=2e-2)
        del wide, h, gate_up, down, got, want


@pytest.mark.parametrize("M,N,K_", [(1, 301, 136), (5, 64, 172), (70, 130, 64), (130, 17, 33)])
def test_gemm_f32(K, M, N, K_):
    a, w, b = torch.randn(M, K_), torch.randn(N, K_), torch.randn(N)
    out = K.gemm_f32(a.to(DEV), w.to(DEV), b.to(DEV))
    want = a.double() @ w.double().T + b.double()
    assert torch.allclose(out.cpu().double(), want, rtol=1e-5, atol=1e-4)
    # a row's result does not depend on the other rows of the call: bitwise
    one = K.gemm_f32(a[M // 2:M // 2 + 1].to(DEV), w.to(DEV), b.to(DEV))
    assert torch.equal(one.cpu()[0], out.cpu()[M // 2])
    # strided rows (a view into a wider buffer), bfloat16 activations
    wide = torch.randn(M, K_ + 24).to(DEV)
    out2 = K.gemm_f32(wide[:, 8:8 + K_], w.to(DEV))
    assert torch.allclose(out2.cpu().double(), wide[:, 8:8 + K_].cpu().double() @ w.double().T, rtol=1e-5, atol=1e-4)
    ab = a.to(torch.bfloat16)
    out3 = K.gemm_f32(ab.to(DEV), w.to(DEV))
    assert torch.allclose(out3.cpu().double(), ab.double() @ w.double().T, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("M", [1, 31, 33, 64, 65])
@pytest.mark.parametrize("N,K_", [(63, 3), (65, 33), (129, 255), (64, 256), (200, 260), (70, 1028), (33000, 516)])
def test_gemm_f32_at_the_edges_of_tiles_and_ranges(K, M, N, K_):
    # a row has the same bits in any call: alone or in tiles of 32 or 64 rows, its ranges of K in one workgroup (33,000
    # columns) or in one each (fewer)
    g = torch.Generator().manual_seed(M * K_)
    a, w, b = (torch.randn(*s, generator=g).to(DEV) for s in ((M, K_), (N, K_), (N,)))
    out = K.gemm_f32(a, w, b)
    rows = slice(0, None) if N < 1000 else slice(N - 300, None)
    want = a.cpu().double() @ w[rows].cpu().double().T
    err = out[:, rows].cpu().double() - b[rows].cpu().double() - want
    # the tree's bound (below) at four levels, and the bias's own rounding; five sigma for the largest
    bound = (1.69 * 2 + 1) * 2.0 ** -24 * float((K_ + 1) ** 0.5)
    assert float(err.abs().max()) <= 5 * bound
    assert torch.equal(K.gemm_f32(a[M // 2:M // 2 + 1].contiguous(), w, b)[0], out[M // 2])
    assert torch.equal(K.gemm_f32(a, w[rows].contiguous(), b[rows].contiguous()), out[:, rows])


@pytest.mark.parametrize("K_", [64, 1000, 1536, 3584, 5120, 8960, 18944, 27648])
def test_gemm_f32_rounding_does_not_grow_with_the_inner_size(K, K_):
    # The sums are trees of radix 16 with L = ceil(log16 K) levels (at most 4).  An addition rounds its partial sum
    # by up to eps = 2^-24 of it, 0.58 eps rms; the partial sums of a group of 16 have on average 8.5 / 16 of the
    # group's mean square, and the groups' mean squares add up to the result's (random signs): every level adds
    # (0.58 eps)^2 * 8.5 to the relative mean square error, so rms error <= 0.58 sqrt(8.5 L) eps = 1.69 sqrt(L) eps
    # of the result's rms at ANY inner size.  One running sum over K terms would give 0.2 sqrt(K) eps: 19 eps at 8,960.
    g = torch.Generator().manual_seed(K_)
    a, w = torch.randn(8, K_, generator=g), torch.randn(96, K_, generator=g)
    want = a.double() @ w.double().T
    err = K.gemm_f32(a.to(DEV), w.to(DEV)).cpu().double() - want
    eps, levels = 2.0 ** -24, min(4, math.ceil(math.log(K_, 16)))
    rms = float(err.pow(2).mean().sqrt() / want.pow(2).mean().sqrt())
    print(f"[gemm_f32] K={K_}: rms error {rms / eps:.2f} eps, bound {1.69 * math.sqrt(levels):.2f} eps")
    assert rms <= 1.69 * math.sqrt(levels) * eps
    assert float(err.abs().max() / want.pow(2).mean().sqrt()) <= 5 * 1.69 * math.sqrt(levels) * eps     # 768 outputs: five sigma


@pytest.mark.parametrize("M,N,K_", [(1, 16, 8), (65, 48, 64), (128, 400, 72), (129, 208, 1000), (200, 4112, 192), (257, 640, 136),
                                   (450, 2576, 64), (600, 6160, 328)])
@pytest.mark.parametrize("name", ["bf16", "f32", "swiglu", "clipped", "relu2", "gelu"])
def test_gemm_tiles(K, M, N, K_, name):
    # the edges of tiles of 64 to 256 rows and columns, of the stages of 64 k, of one and several rounds of workgroups
    g = torch.Generator().manual_seed(M + N)
    wide = torch.randn(M, K_ + 8, generator=g).bfloat16().to(DEV)
    a, w = wide[:, 8:], (torch.randn(N, K_, generator=g) * K_ ** -0.5).bfloat16().to(DEV)      # rows with a stride
    b = torch.randn(N, generator=g).to(DEV) if name in ("bf16", "f32", "gelu") else None
    epi = {"bf16": K.EPI_BF16, "f32": K.EPI_F32, "swiglu": K.EPI_SWIGLU, "clipped": K.EPI_CLIPPED, "relu2": K.EPI_RELU2, "gelu": K.EPI_GELU}[name]
    clip = (0.7, 1.702) if name == "clipped" else None
    out = K.gemm_tiles(a, w, b, epi, clip)
    z = a.double() @ w.double().T + (b.double() if b is not None else 0.0)
    half = N // 2
    want = {"bf16": lambda: z, "f32": lambda: z, "swiglu": lambda: F.silu(z[:, :half]) * z[:, half:],
            "clipped": lambda: z[:, :half].clamp(max=0.7) * torch.sigmoid(1.702 * z[:, :half].clamp(max=0.7)) * (z[:, half:].clamp(-0.7, 0.7) + 1),
            "relu2": lambda: torch.relu(z) ** 2, "gelu": lambda: F.gelu(z)}[name]()
    # float32 sums of at most 1,000 terms (relative error below 1e-5 of a row's size, which is about 1) through activations
    # with slopes of at most about 2 |z|; then one rounding to bfloat16 (2^-9)
    slack = 1e-5 * (1 + 2 * float(z.abs().max()))
    if name == "f32":
        assert out.dtype == torch.float32 and float((out.double() - want).abs().max()) <= slack
    else:
        assert out.dtype == torch.bfloat16 and bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all())
    # a row's bits do not depend on the rows beside it, nor on the tile that a call of its size takes
    assert torch.equal(K.gemm_tiles(a[M // 2:M // 2 + 1], w, b, epi, clip)[0], out[M // 2])
    assert torch.equal(K.gemm_tiles(a[:(M + 1) // 2], w, b, epi, clip), out[:(M + 1) // 2])


@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 63, 255, 256, 257, 511, 512, 513, 519, 520, 521, 767, 768, 769, 1023, 1025, 1031])
def test_gemm_tiles_deals_every_tile_once(K, tiles):
    # 100 rows and an inner size of one stage: so many tiles of 192 columns, the rows of one each, which the cost of a round gives to workgroups
    # that a compute unit has to itself up to 256 of them and to two a unit beyond.  Grids of every remainder by eight, whole rounds of
    # 512, last rounds of one tile, of an eighth less one, of one tile a compute unit and more, behind one round and two.  A tile
    # is made of exact sums (whole numbers), so one that is left out or written by another shows
    g = torch.Generator(device=DEV).manual_seed(tiles)
    N = 192 * tiles - 32
    a = torch.randint(-4, 5, (100, 64), device=DEV, generator=g).bfloat16()
    w = torch.randint(-4, 5, (N, 64), device=DEV, generator=g).bfloat16()
    want = a.float() @ w.float().T
    for _ in range(2):
        junk = torch.full((100, N), float("nan"), device=DEV)
        del junk                                                  # (what the next tensor of this size finds in its memory)
        assert torch.equal(K.gemm_tiles(a, w, None, K.EPI_F32), want)


@pytest.mark.parametrize("M", [65, 700])
def test_gemm_tiles_gelu_over_its_range(K, M):
    # the epilogue's own error function from end to end, a bias that starts on no 16 bytes beside it
    z = torch.cat([torch.linspace(-9, 9, 4093), torch.tensor([0.0, float("inf"), float("nan")])]).bfloat16()
    w, x = torch.zeros(len(z), 8), torch.zeros(M, 8)
    w[:, 1], x[:, 1] = 1.0, 1.0
    bias = torch.cat([torch.zeros(1), z.float() - 1.0]).to(DEV)[1:]              # exact: z from x . w + bias
    z = (bias.cpu() + 1.0).double()
    out = K.gemm_tiles(x.bfloat16().to(DEV), w.bfloat16().to(DEV), bias, K.EPI_GELU).cpu().double()
    want = z * 0.5 * torch.erfc(-z / math.sqrt(2.0))
    fine = torch.isfinite(z)
    # 4e-6 of a result's size in float32 (the exponent's rounding at |z| = 9), then a rounding to bfloat16 (2^-9)
    assert bool(((out - want).abs() <= want.abs() * 2.0 ** -8)[:, fine].all())
    assert bool((out[:, -2] == float("inf")).all()) and bool(out[:, -1].isnan().all())


@pytest.mark.parametrize("M,N,K_", [(1024, 1168, 8), (700, 1552, 200), (641, 1600, 2560), (1025, 2064, 72), (1920, 2048, 64), (2048, 2048, 328), (1377, 1536, 2736),
                                    (1568, 1680, 2504), (1569, 1680, 2504), (1570, 1664, 3000)])
@pytest.mark.parametrize("bias", [False, True])
def test_products_of_a_single_round(K, M, N, K_, bias):
    # the smallest and largest numbers of tiles, ends inside a tile and a stage, with and without workgroups that read the matrix ahead
    # (the last four), next to no rows in the last tile (1,569 and 1,570: one row more than 32 decides)
    assert K.library.core().pico_gemm_tiles_round(M, N, K_) == (1 if -(-M // 128) * -(-N // 64) <= 256 else 2)
    g = torch.Generator(device=DEV).manual_seed(M)
    a, w = torch.full((M, K_ + 8), float("nan"), device=DEV, dtype=torch.bfloat16), torch.full((N, K_ + 16), float("nan"), device=DEV, dtype=torch.bfloat16)
    a[:, :K_], w[:, :K_] = torch.randn(M, K_, device=DEV, generator=g), torch.randn(N, K_, device=DEV, generator=g)
    b = torch.randn(N, device=DEV, generator=g) if bias else None
    a, w = a[:, :K_], w[:, :K_]
    assert K.tiles_round_ok(a, w)
    out = K.gemm_tiles(a, w, b)
    want = a.double() @ w.double().T + (b.double() if bias else 0.0)
    # float32 sums (a chain of K / 16 additions, 2^-24 of a partial sum each: under 1e-5 of a row's size), rounded to eight bits
    assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-5 * K_ ** 0.5 * 4).all())
    rows = slice(M - 70, M)                              # a row's result does not depend on which tiles it is in
    assert torch.equal(out[rows], K.gemm_tiles(a[rows].contiguous(), w, b))


@pytest.mark.parametrize("M,N,K_,parts,mb,nb,share,want", [
    (65, 13440, 1536, 1, 2, 1, 2, 0), (128, 8960, 1536, 1, 2, 1, 2, 1536), (96, 1536, 13440, 8, 2, 1, 2, 0), (832, 3584, 18944, 2, 4, 2, 1, 0), (352, 18944, 3584, 1, 3, 3, 1, 0),
    (300, 7168, 3584, 1, 2, 2, 1, 3584), (352, 7168, 3584, 1, 2, 2, 1, 3584), (300, 6144, 1536, 1, 2, 1, 2, 1536), (320, 8960, 1536, 1, 2, 2, 1, 0), (768, 4608, 3584, 1, 2, 2, 1, 3008),
    (1700, 1536, 13440, 1, 2, 1, 2, 0), (1024, 1536, 13440, 1, 2, 1, 2, 13440), (2048, 1536, 8960, 1, 2, 2, 1, 8960), (2052, 1536, 8960, 1, 2, 2, 1, 0), (512, 1024, 1536, 1, 2, 1, 2, 0)])
def test_what_is_read_ahead_of_a_product(K, M, N, K_, parts, mb, nb, share, want):
    # both sides of every line of the rule, at points where it was measured: no parts, no large tiles, no matrix that a single row of many tiles
    # reads, no helper with more rows than it gets through
    assert K.library.core().pico_gemm_tiles_ahead(M, N, K_, parts, mb, nb, share) == want


@pytest.mark.parametrize("name", ["swiglu", "clipped"])
def test_activation_of_the_tiled_product_over_all_numbers(K, name):
    # a gate that is one number of the row, an up that is 1 (0, for the clipped form's u + 1): every bfloat16 number through the
    # activation, which is then rounded to bfloat16 (2^-8 of it) from what is within 2^-21 of the quotient in 64 bits (results below 2^-119, of z
    # under -88.7, may be zero)
    x = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    a = torch.zeros(65536, 16, dtype=torch.bfloat16)
    a[:, 0], a[:, 1] = x, 1
    w = torch.zeros(16, 16, dtype=torch.bfloat16)
    w[:8, 0], w[8:, 1] = 1, 1 if name == "swiglu" else 0
    alpha = 1.0 if name == "swiglu" else 1.702
    out = K.gemm_tiles(a.to(DEV), w.to(DEV), None, K.EPI_SWIGLU if name == "swiglu" else K.EPI_CLIPPED, clip=(float("inf"), alpha)).cpu()
    g = x.double()
    want = g / (1 + torch.exp(-(x.float() * alpha).double()))
    bad = ~torch.isfinite(g)                                # (an infinite gate times the up rows' zero is NaN)
    assert bool((out == out[:, :1])[~bad].all())
    got, want = out[:, 0][~bad].double(), want[~bad]
    assert bool(((got - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -21) + 2.0 ** -119).all())      # (eight bits: half of the last is 2^-8 of 1)


@pytest.mark.parametrize("name,gates", [("swiglu", [-86.0, -87.0, -87.5, -88.0, -88.5]), ("clipped", [-51.0, -51.25, -51.5, -51.75, -52.0])])
def test_activation_of_the_tiled_product_keeps_its_smallest_results(K, name, gates):
    # gates at which 1 + exp(-z) is between 2^126 and the largest number: results of about 5e-37 are normal numbers, rounded to eight bits (from
    # within 2^-17 of the quotient: in float32 the exponent alpha g is off by up to 88 2^-24)
    x = torch.tensor(gates).repeat(20).bfloat16()
    a = torch.zeros(x.numel(), 16, dtype=torch.bfloat16)
    a[:, 0], a[:, 1] = x, 1
    w = torch.zeros(16, 16, dtype=torch.bfloat16)
    w[:8, 0], w[8:, 1] = 1, 1 if name == "swiglu" else 0
    alpha = 1.0 if name == "swiglu" else 1.702
    out = K.gemm_tiles(a.to(DEV), w.to(DEV), None, K.EPI_SWIGLU if name == "swiglu" else K.EPI_CLIPPED, clip=(float("inf"), alpha)).cpu().double()
    want = (x.double() / (1 + torch.exp(-alpha * x.double()))).view(-1, 1)
    assert bool(((out - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -17)).all())


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("N,name", [(66000, "f32"), (65536, "f32"), (65600, "swiglu"), (33024, "clipped"), (65536, "swiglu")])
def test_few_rows_of_a_large_matrix(K, M, N, name):
    # both widths of the tiles for few rows, at and behind the sizes where the rule changes over, through ``Linear``
    from pico_vllm_amd.ops.linear import Linear
    g = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, 72, generator=g).bfloat16().to(DEV), (torch.randn(N, 72, generator=g) * 72 ** -0.5).bfloat16().to(DEV)
    z = a.double() @ w.double().T
    gate, up = z[:, :N // 2], z[:, N // 2:]
    slack = 1e-5 * (1 + 2 * float(z.abs().max()))                       # as above
    for out in ([Linear(w)(a, torch.float32), K.gemm_tiles(a, w, None, K.EPI_F32)] if name == "f32" else
                [Linear(w).swiglu(a), K.gemm_tiles(a, w, None, K.EPI_SWIGLU)] if name == "swiglu" else
                [Linear(w).clipped_glu(a, 0.7, 1.702), K.gemm_tiles(a, w, None, K.EPI_CLIPPED, (0.7, 1.702))]):
        if name == "f32":
            assert float((out.double() - z).abs().max()) <= slack
            continue
        want = F.silu(gate) * up if name == "swiglu" else \
            gate.clamp(max=0.7) * torch.sigmoid(1.702 * gate.clamp(max=0.7)) * (up.clamp(-0.7, 0.7) + 1)
        assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + slack).all())


@pytest.mark.parametrize("N,K_,name", [(66000, 72, "f32"), (66064, 1096, "f32"), (65536, 512, "f32"), (65600, 200, "swiglu"), (98320, 832, "swiglu"),
                                       (33024, 264, "clipped")])
def test_a_row_of_a_large_matrix_does_not_depend_on_the_rows_beside_it(K, N, K_, name):
    # up to 64 rows two products share the work, by the number of rows: both make the same sums in the same order
    from pico_vllm_amd.ops.linear import Linear
    g = torch.Generator().manual_seed(N)
    a, w = torch.randn(64, K_, generator=g).bfloat16().to(DEV), (torch.randn(N, K_, generator=g) * K_ ** -0.5).bfloat16().to(DEV)
    lin = Linear(w, torch.randn(N, generator=g).to(DEV) if name == "f32" else None)
    call = {"f32": lambda x: lin(x, torch.float32), "swiglu": lin.swiglu, "clipped": lambda x: lin.clipped_glu(x, 0.7, 1.702)}[name]
    want = call(a)
    for rows in (1, 8, 9, 15, 16, 17, 32, 33, 63):
        assert torch.equal(call(a[:rows]), want[:rows]), rows
    epi, bias, clip = {"f32": (K.EPI_F32, lin.bias_f32, None), "swiglu": (K.EPI_SWIGLU, None, None), "clipped": (K.EPI_CLIPPED, None, (0.7, 1.702))}[name]
    for rows in (1, 16, 17, 64):
        assert torch.equal(K.gemm_tiles(a[:rows], w, bias, epi, clip, few=True), K.gemm_skinny(a[:rows], w, bias, epi, clip=clip)), rows
    with pytest.raises(RuntimeError):
        K.gemm_tiles(a.repeat(2, 1), w, bias, epi, clip, few=True)
    with pytest.raises(RuntimeError):
        K.gemm_tiles(a, w, None, K.EPI_BF16, few=True)


def test_gemm_tiles_refuses(K):
    a, w = torch.zeros(70, 72, device=DEV).bfloat16(), torch.zeros(48, 72, device=DEV).bfloat16()
    for bad in (lambda: K.gemm_tiles(a[:, :68], w[:, :68]), lambda: K.gemm_tiles(a, w[:40]), lambda: K.gemm_tiles(a.float(), w),
                lambda: K.gemm_tiles(a, w, None, K.EPI_CLIPPED), lambda: K.gemm_tiles(a[:, 1:65], w[:, :64]),
                lambda: K.gemm_tiles(a, w, torch.zeros(47, device=DEV)), lambda: K.gemm_tiles(a, w[:, :64])):
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.parametrize("M,N,K_", [(1, 301, 136), (3, 256, 64), (8, 384, 192), (33, 130, 172), (64, 1000, 1536),
                                   (100, 77, 40)])
@pytest.mark.parametrize("out_dtype", DTYPES)
def test_gemm_bf16(K, M, N, K_, out_dtype):
    a, w, b = torch.randn(M, K_).bfloat16(), torch.randn(N, K_).bfloat16(), torch.randn(N)
    out = K.gemm_bf16(a.to(DEV), w.to(DEV), b.to(DEV), out_dtype)
    want = a.double() @ w.double().T + b.double()
    assert out.dtype == out_dtype
    if out_dtype == torch.float32:       # exact products, float32 accumulation
        assert torch.allclose(out.cpu().double(), want, rtol=1e-4, atol=1e-3 * math.sqrt(K_))
    else:
        assert torch.allclose(out.cpu().double(), want, rtol=1e-2, atol=1e-2 * math.sqrt(K_))
    out_nb = K.gemm_bf16(a.to(DEV), w.to(DEV), None, torch.float32)
    assert torch.allclose(out_nb.cpu().double(), a.double() @ w.double().T, rtol=1e-4, atol=1e-3 * math.sqrt(K_))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,rot,Pg", [(4, 1, 16, 16, 16), (6, 3, 32, 32, 8), (5, 5, 48, 48, 16), (2, 2, 64, 32, 32),
                                            (12, 2, 128, 128, 16), (3, 1, 24, 8, 16), (28, 4, 128, 128, 16),
                                            (6, 2, 24, 24, 8), (5, 1, 40, 40, 16), (4, 4, 72, 72, 8), (2, 1, 250, 250, 16)])
def test_rope_and_cache_store(K, dtype, nq, nkv, d, rot, Pg):
    theta = 10000.0
    new_lens, prefix_lens = [5, 1, 9], [14, 33, 0]          # 14..18 crosses a page edge of 16 (store_kvcache.py:107-118)
    pos, seq = flat_batch(new_lens, prefix_lens)
    T = int(pos.numel())
    qkv = torch.randn(T, (nq + 2 * nkv) * d).to(dtype)
    num_pages = 12 * 16 // Pg
    kc = torch.full((num_pages, nkv, Pg, d), 7.0, dtype=dtype, device=DEV)
    vc = torch.full((num_pages, nkv, d, Pg), 7.0, dtype=dtype, device=DEV)
    g = torch.Generator().manual_seed(0)
    perm = torch.randperm(num_pages, generator=g).tolist()
    maxp = max(-(-(n + p) // Pg) for n, p in zip(new_lens, prefix_lens))
    bt = torch.full((3, maxp), -1, dtype=torch.int32)
    for b, (n, p) in enumerate(zip(new_lens, prefix_lens)):
        for j in range(-(-(n + p) // Pg)):
            bt[b, j] = perm.pop()
    inv = (1.0 / (theta ** (torch.arange(0, rot, 2).float() / rot))).to(DEV)
    x = qkv.clone().to(DEV)
    slots = torch.tensor([int(bt[int(b), int(p) // Pg]) * Pg + int(p) % Pg for b, p in zip(seq, pos)],
                         dtype=torch.int32, device=DEV)
    slots[3] = -1                                           # a padding row: rotated, but nothing of it is stored
    table = K.rope_table(pos.to(DEV), inv)
    want_cos, want_sin = P.rope_tables(pos.cpu(), rot, theta)
    assert torch.allclose(table[..., 0].cpu(), want_cos[:, :rot // 2], atol=2e-6)
    assert torch.allclose(table[..., 1].cpu(), want_sin[:, :rot // 2], atol=2e-6)
    K.rope_kv_store(x, table, slots, kc, vc, nq, nkv, d, rot)
    # reference
    q, k, v = P.split_qkv(qkv.float(), nq, nkv, d)
    cos, sin = P.rope_tables(pos.cpu(), rot, theta)

    def rot_part(t):
        return torch.cat([P.apply_rope(t[..., :rot], cos, sin), t[..., rot:]], dim=-1)
    qr, kr = rot_part(q), rot_part(k)
    close(x[:, :nq * d].reshape(T, nq, d), qr, dtype, scale=3)
    assert torch.equal(x[:, nq * d:].cpu(), qkv[:, nq * d:])          # k and v in the activation buffer are untouched
    want_k = torch.full((num_pages, nkv, Pg, d), 7.0)
    want_v = torch.full((num_pages, nkv, d, Pg), 7.0)
    for t in range(T):
        if t == 3:
            continue
        b, p = int(seq[t]), int(pos[t])
        page, off = int(bt[b, p // Pg]), p % Pg
        want_k[page, :, off, :] = kr[t]
        want_v[page, :, :, off] = v[t]
    close(kc, want_k, dtype, scale=3)          # also: every slot that no token owns still holds 7
    close(vc, want_v, dtype, scale=3)


def _attn_case(K, dtype, new_lens, prefix_lens, nq, nkv, d, Pg, window=0, seed=0, boost=None):
    g = torch.Generator().manual_seed(seed)
    totals = [n + p for n, p in zip(new_lens, prefix_lens)]
    ks = [(torch.randn(N, nkv, d, generator=g)).to(dtype).float() for N in totals]
    vs = [(torch.randn(N, nkv, d, generator=g)).to(dtype).float() for N in totals]
    qs = [(torch.randn(n, nq, d, generator=g)).to(dtype).float() for n in new_lens]
    if boost is not None:
        boost(qs, ks, vs)
    num_pages = sum(-(-N // Pg) for N in totals) + 3
    kc, vc, bt = paged_cache(ks, vs, Pg, num_pages, dtype, seed)
    pos, seq = flat_batch(new_lens, prefix_lens)
    q = torch.cat(qs, 0).reshape(-1, nq * d).to(DEV, dtype)
    out = K.paged_attention_ref(q, kc, vc, bt, pos, seq, nq, nkv, d, 1.0 / math.sqrt(d), window)
    want = torch.cat([P.causal_attention(qb, kb, vb, q_positions=torch.arange(p, p + n), window=window)
                      for qb, kb, vb, n, p in zip(qs, ks, vs, new_lens, prefix_lens)], 0)
    return out.reshape(-1, nq, d), want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", range(len(REFERENCE_CASES)))
def test_plain_attention_kernel_on_the_reference_cases(K, dtype, case):
    new_lens, prefix_lens = REFERENCE_CASES[case]
    out, want = _attn_case(K, dtype, new_lens, prefix_lens, 12, 2, 128, 16, seed=case)
    close(out, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,Pg", [(4, 1, 16, 16), (6, 3, 32, 8), (5, 5, 48, 16), (3, 1, 80, 32), (8, 2, 256, 64),
                                        (2, 2, 112, 8)])
def test_plain_attention_kernel_other_sizes(K, dtype, nq, nkv, d, Pg):
    out, want = _attn_case(K, dtype, [7, 1, 30, 2], [0, 70, 45, 129], nq, nkv, d, Pg, seed=3)
    close(out, want, dtype)


@pytest.mark.parametrize("nq,nkv,d,Pg,window", [(12, 2, 128, 16, 0), (7, 1, 60, 4, 0), (5, 5, 132, 12, 100), (8, 2, 256, 64, 33), (40, 2, 8, 16, 0)])
def test_f32_attention_keeps_columns_apart(K, nq, nkv, d, Pg, window):
    # tiles of 16 columns with tokens of several sequences, whose keys end in the middle of a quarter; what a token does not see
    # (its own sequence's later tokens, tokens outside its window, other sequences, the rest of a page) is not finite
    new_lens, prefix_lens = [1, 1, 70, 5, 1], [130, 0, 15, 63, 64]
    clean, want = _attn_case(K, torch.float32, new_lens, prefix_lens, nq, nkv, d, Pg, window, seed=5)
    close(clean, want, torch.float32)
    ends = [sum(new_lens[:b + 1]) for b in range(5)]
    bad_k, bad_v = 15 + 50, 15 + 40                              # of the third sequence, among its new tokens

    def spoil(qs, ks, vs):
        ks[2][bad_k:bad_k + 3], vs[2][bad_v], vs[2][bad_v + 1], vs[4][64] = float("nan"), float("inf"), float("nan"), float("inf")
        ks[0][:20], vs[0][:20] = (float("nan"), float("inf")) if window else (ks[0][:20], vs[0][:20])
    got, _ = _attn_case(K, torch.float32, new_lens, prefix_lens, nq, nkv, d, Pg, window, seed=5, boost=spoil)
    spoiled = set(range(2 + 40, 2 + 70)) | {ends[4] - 1}         # rows that see one of them
    rows = [r for r in range(ends[4]) if r not in spoiled]
    close(got[rows], want[rows], torch.float32)
    assert not torch.isfinite(got[2 + 40]).all()
    # a position's bits do not depend on how its sequence was cut into steps, nor on who shares its tile
    g = torch.Generator().manual_seed(5)
    totals = [n + p for n, p in zip(new_lens, prefix_lens)]
    kv = [[torch.randn(N, nkv, d, generator=g) for N in totals] for _ in range(2)]
    q = [torch.randn(n, nq, d, generator=g) for n in new_lens]

    def last(qs, ks, vs):
        for b in range(5):
            qs[b][:], ks[b][:], vs[b][:] = q[b][-1:], kv[0][b], kv[1][b]
    lone, _ = _attn_case(K, torch.float32, [1] * 5, [n - 1 for n in totals], nq, nkv, d, Pg, window, seed=6, boost=last)
    assert torch.equal(lone, clean[[e - 1 for e in ends]])


@pytest.mark.parametrize("nq,nkv,singles,portion", [(16, 16, 40, 200), (3, 3, 16, 0), (14, 2, 7, 30), (40, 2, 3, 2), (64, 64, 17, 300)])
def test_f32_attention_deals_a_tiles_sequences_out(K, nq, nkv, singles, portion):
    # a workgroup for each of a tile's sequences, for every second, third or fourth of them, or one for all
    new_lens = [1] * singles + ([portion] if portion else [])
    prefix_lens = [(37 * i + 5) % 130 for i in range(singles)] + ([9] if portion else [])
    got, want = _attn_case(K, torch.float32, new_lens, prefix_lens, nq, nkv, 64, 16, seed=8)
    close(got, want, torch.float32)


# Head sizes that are no multiple of 16 (the configuration allows any even one): the matrix-core kernels do not take
# them, so both engine precisions go through this kernel there.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("Pg", [8, 16])
@pytest.mark.parametrize("nq,nkv,d", [(6, 2, 24), (5, 1, 40), (4, 4, 72), (3, 1, 2), (2, 1, 250)])
@pytest.mark.parametrize("case", range(len(REFERENCE_CASES)))
def test_plain_attention_kernel_at_head_sizes_between_the_steps_of_16(K, dtype, Pg, nq, nkv, d, case):
    # the reference's own (new, prefix) cases (tests/test_prefill_paged_attn.py:183-260), with grouped heads
    new_lens, prefix_lens = REFERENCE_CASES[case]
    out, want = _attn_case(K, dtype, new_lens, prefix_lens, nq, nkv, d, Pg, seed=case + d)
    close(out, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d", [24, 40, 72])
def test_attention_finds_one_far_key_at_head_sizes_between_the_steps_of_16(K, dtype, d):
    # as below: a dropped key, page or tail of the head dimension would show
    for far in (0, 7, 8, 63, 64, 301):
        def boost(qs, ks, vs, far=far):
            ks[0][far] = qs[0][-1, 0:1, :] * 8.0          # (a short head: a large factor makes the score stand out)
            vs[0][far] = 100.0
            vs[0][far][..., d - 1] = -100.0          # the last head dimension carries a value of its own
        out, want = _attn_case(K, dtype, [3], [330], 3, 1, d, 8, seed=far, boost=boost)
        assert float(want[-1, 0, :d - 1].mean()) > 50 and float(want[-1, 0, d - 1]) < -50
        close(out, want, dtype, scale=100)


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_finds_one_far_key_among_hundreds(K, dtype):
    # one key far back gets a large score; its value dominates the output.  A kernel that drops a
    # block of keys, a page or a boundary position fails here, whereas with random scores the loss
    # of one key among 600 would hide under the tolerance.
    for far in (0, 15, 16, 63, 64, 200, 511):
        def boost(qs, ks, vs, far=far):
            ks[0][far] = qs[0][-1, 0:1, :] * 2.0          # same direction as the last query of head 0
            vs[0][far] = 100.0
        out, want = _attn_case(K, dtype, [3], [597], 2, 1, 64, 16, seed=far, boost=boost)
        assert float(want[-1, 0].mean()) > 50
        close(out, want, dtype, scale=100)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 5, 16, 17, 64, 100])
def test_attention_window_edge(K, dtype, window):
    # the key just outside the window carries a huge value: reading it would show at once
    def boost(qs, ks, vs):
        n = ks[0].shape[0]
        last = n - 1
        if last - window >= 0:
            vs[0][last - window] = 1000.0
    out, want = _attn_case(K, dtype, [4, 1], [126, 40], 4, 2, 32, 16, window=window, seed=window, boost=boost)
    assert float(want[3].abs().max()) < 50
    close(out, want, dtype)


@pytest.mark.parametrize("nq,nkv,d,rot", [(8, 1, 16, 16), (12, 2, 128, 128), (2, 2, 64, 32)])
def test_rotation_gives_a_token_the_same_bits_whatever_stands_beside_it(K, nq, nkv, d, rot):
    # seven tokens alone take the kernel for few tokens, the same seven among twenty the one with 16-byte accesses: the
    # same rotated queries and the same keys and values in the cache, bit for bit (a step padded for a recorded graph
    # must not differ from the step unpadded)
    g = torch.Generator().manual_seed(d)
    T, n, Pg = 20, 7, 16
    qkv = (torch.randn(T, (nq + 2 * nkv) * d, generator=g) * 2).bfloat16()
    pos = torch.randint(0, 3000, (T,), generator=g, dtype=torch.int32)
    slots = torch.randperm(4 * Pg, generator=g)[:T].to(torch.int32)
    inv = (1.0 / (10000.0 ** (torch.arange(0, rot, 2).float() / rot))).to(DEV)
    got = []
    for rows in (T, n):
        x = qkv[:rows].clone().to(DEV)
        kc = torch.zeros(4, nkv, Pg, d, dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros(4, nkv, d, Pg, dtype=torch.bfloat16, device=DEV)
        K.rope_kv_store(x, K.rope_table(pos[:rows].to(DEV), inv), slots[:rows].to(DEV), kc, vc, nq, nkv, d, rot)
        got.append((x[:n].cpu(), [(kc[int(s) // Pg, :, int(s) % Pg].cpu(), vc[int(s) // Pg, :, :, int(s) % Pg].cpu()) for s in slots[:n]]))
    assert torch.equal(got[0][0], got[1][0])
    for (k1, v1), (k2, v2) in zip(got[0][1], got[1][1]):
        assert torch.equal(k1, k2) and torch.equal(v1, v2)


def test_sampling_greedy_and_ties(K):
    logits = torch.randn(5, 1000)
    logits[1, 7] = logits[1, 900] = 50.0            # tie: the lower index wins
    logits[2, 999] = 60.0
    z = torch.zeros(5)
    out = K.sample(logits.to(DEV), z.to(DEV), torch.ones(5, device=DEV), z.to(DEV))
    want = [P.sample_greedy(l) for l in logits]
    assert out.tolist() == want and want[1] == 7 and want[2] == 999


@pytest.mark.parametrize("R,V", [(1, 17), (5, 1000), (8, 151936), (64, 4099)])
def test_argmax_in_two_launches_is_the_greedy_sample(K, R, V):
    g = torch.Generator().manual_seed(V)
    logits = torch.randn(R, V, generator=g)
    logits[0, V // 3] = logits[0, V - 1] = 40.0                  # a tie across chunks: the lower index wins
    if R > 1:
        logits[1, V - 1] = 50.0                                  # the last element of the last chunk
        logits[R - 1, 0] = 50.0
    dev = logits.to(DEV)
    out = torch.full((R,), -1, dtype=torch.int32, device=DEV)
    K.argmax(dev, out, K.argmax_workspace(R, DEV))
    z = torch.zeros(R, device=DEV)
    assert out.tolist() == [P.sample_greedy(l) for l in logits] == K.sample(dev, z, z + 1, z).tolist()
    assert out[0] == V // 3
    wide = torch.randn(R, V + 5, generator=g).to(DEV)            # rows with a stride of their own
    K.argmax(wide[:, :V], out, K.argmax_workspace(R + 3, DEV))
    assert out.tolist() == wide[:, :V].argmax(1).tolist()
    with pytest.raises(K.KernelError):
        K.argmax(dev, out, K.argmax_workspace(max(R - 1, 0), DEV))


@pytest.mark.parametrize("V", [301, 5000, 151936, 300007])      # (the last: a thread's piece of a chunk is beyond what it holds in registers)
def test_sampling_temperature_follows_the_inverse_cdf(K, V):
    g = torch.Generator().manual_seed(V)
    R = 64
    logits = torch.randn(R, V, generator=g) * 3
    temps = torch.rand(R, generator=g) * 1.5 + 0.2
    us = torch.rand(R, generator=g)
    out = K.sample(logits.to(DEV), temps.to(DEV), torch.ones(R, device=DEV), us.to(DEV)).tolist()
    agree = 0
    for r in range(R):
        p = P.temperature_probs(logits[r], float(temps[r]))
        want = P.inverse_cdf(p, float(us[r]))
        cum = torch.cumsum(p, 0)
        # equal, or u falls within float32 rounding of a boundary of the CDF
        if out[r] == want:
            agree += 1
        else:
            lo, hi = sorted((out[r], want))
            assert hi - lo <= 2 and abs(float(cum[lo]) - float(us[r])) < 1e-5, (r, out[r], want)
    assert agree >= R - 3


def test_sampling_top_p_keeps_a_prefix_of_tied_tokens(K):
    # tokens of equal probability at the threshold: the sorted rule keeps as many of them as it takes to reach
    # top_p, not all (pico_vllm/sampler.py:25-32); which ones is the sort's choice, here the lowest indices
    cases = [(torch.tensor([0.2, 0.4, 0.2, 0.2]), 0.5, {1, 0}), (torch.tensor([0.2, 0.4, 0.2, 0.2]), 0.7, {1, 0, 2}),
             (torch.tensor([0.2, 0.4, 0.2, 0.2]), 0.95, {0, 1, 2, 3}), (torch.full((100,), 0.01), 0.305, set(range(31))),
             (torch.tensor([0.25, 0.25, 0.25, 0.25]), 0.1, {0})]
    for probs, top_p, kept in cases:
        logits = probs.log()[None, :].contiguous()
        assert set(torch.nonzero(P.top_p_probs(logits[0], 1.0, top_p)).flatten().tolist()) == kept
        seen = set()
        for u in torch.linspace(0.001, 0.999, 97):
            tok = K.sample(logits.to(DEV), torch.ones(1, device=DEV), torch.tensor([top_p], device=DEV), u.reshape(1).to(DEV))
            seen.add(int(tok[0]))
        assert seen == kept, (probs.tolist()[:5], top_p, sorted(seen))


def test_sampling_at_the_real_vocabulary_row_by_row(K):
    # 151,936 logits a row, rows of every kind side by side: greedy, plain temperature, wide and narrow nuclei, flat and
    # peaked distributions.  Every row against the plain rule, and the same token when the row is sampled alone.
    g = torch.Generator().manual_seed(21)
    R, V = 14, 151936
    logits = torch.randn(R, V, generator=g) * torch.tensor([1, 1, 3, 3, 3, 8, 8, 0.1, 0.1, 20, 20, 3, 3, 3.0])[:, None]
    temps = torch.tensor([0.0, 1.0, 0.7, 0.7, 1.3, 1.0, 0.5, 1.0, 1.0, 1.0, 2.0, 0.0, 0.9, 1.1])
    top_ps = torch.tensor([1.0, 1.0, 0.9, 0.5, 0.05, 0.95, 0.3, 0.9, 0.999, 0.8, 0.6, 0.5, 1.0, 0.99])
    us = torch.rand(R, generator=g)
    dev = logits.to(DEV)
    work = K.sample_workspace(R, DEV)
    out = K.sample(dev, temps.to(DEV), top_ps.to(DEV), us.to(DEV), work=work).tolist()
    assert out == K.sample(dev, temps.to(DEV), top_ps.to(DEV), us.to(DEV), work=work).tolist()      # and again: the same
    exact = 0
    for r in range(R):
        alone = K.sample(dev[r:r + 1], temps[r:r + 1].to(DEV), top_ps[r:r + 1].to(DEV), us[r:r + 1].to(DEV))
        assert int(alone[0]) == out[r], (r, int(alone[0]), out[r])
        if temps[r] == 0:
            assert out[r] == P.sample_greedy(logits[r])
            continue
        p = P.top_p_probs(logits[r].double(), float(temps[r]), float(top_ps[r]))
        assert float(p[out[r]]) > 0, (r, "a token outside the kept set")
        want = P.inverse_cdf(p, float(us[r]))
        cum = torch.cumsum(p, 0)
        exact += out[r] == want
        # equal, or u falls within rounding of a boundary of the CDF (float32 exponentials against float64 ones)
        assert out[r] == want or abs(float(cum[min(out[r], want)]) - float(us[r])) < 1e-4, (r, out[r], want)
    assert exact >= R - 3
    # rows that are known to have no nucleus skip the search for it
    plain_rows = torch.ones(R, device=DEV)
    assert K.sample(dev, temps.to(DEV), plain_rows, us.to(DEV), top_p_rows=False).tolist() \
        == K.sample(dev, temps.to(DEV), plain_rows, us.to(DEV)).tolist()
    with pytest.raises(K.KernelError, match="workspace"):
        K.sample(dev, temps.to(DEV), top_ps.to(DEV), us.to(DEV), work=K.sample_workspace(R - 1, DEV))


@pytest.mark.parametrize("M,N,K_", [(3, 100, 516), (40, 200, 516), (400, 6500, 260), (300, 15403, 516)])
@pytest.mark.parametrize("ea,ew", [(0, 0), (-120, 110), (-140, 120), (30, -80), (31, -120), (100, -140), (-40, -20), (60, 60), (126, -20), (0, -140), (30, -140),
                                   (30, -136), (-140, 30), (70, -70), (-80, 70), (-80, 84), (-70, -70)])
def test_gemm_f32_at_the_limits_of_its_numbers(K, M, N, K_, ea, ew):
    # numbers are taken apart into bfloat16 pieces: operands and results of any size keep float32's precision (bound: the tree of four
    # levels above; each of its sums is a multiple of 2^-149, two ranges and their sum here), through copies, registers and bfloat16 rows;
    # what is not finite stays in its row and column.  The last shape has tiles of 64 x 128
    g = torch.Generator().manual_seed(5)
    a, w = (torch.ldexp(torch.randn(*s, generator=g).clamp(-3, 3), torch.tensor(e)).to(DEV) for s, e in (((M, K_), ea), ((N, K_), ew)))
    odd = torch.zeros(M, K_ + 1, device=DEV)[:, :K_]
    odd.copy_(a)
    want = a.double() @ w.double().T
    out = K.gemm_f32(a, w)
    for got, ref in ((out, want), (K.gemm_f32(odd, w), want), (K.gemm_f32(a.to(torch.bfloat16), w), a.to(torch.bfloat16).double() @ w.double().T)):
        assert (got.double() - ref).pow(2).mean().sqrt() <= 3.4 * 2.0 ** -24 * ref.pow(2).mean().sqrt() + 3 * 2.0 ** -150
    a[1, 7], a[2, 9], w[5, 3] = float("inf"), float("nan"), float("-inf")
    hit = K.gemm_f32(a, w)
    rows, cols = [r for r in range(M) if r not in (1, 2)], [c for c in range(N) if c != 5]
    assert torch.equal(hit[rows][:, cols], out[rows][:, cols])
    assert torch.isnan(hit[2]).all()
    assert torch.allclose(hit[1, cols], a[1, 7] * w[cols, 7], equal_nan=True)      # infinities, and NaN where a tiny number has become 0
    assert torch.allclose(hit[rows, 5], a[rows, 3] * w[5, 3], equal_nan=True)
    assert torch.equal(K.gemm_f32(torch.zeros_like(a), w[cols]), torch.zeros(M, N - 1, device=DEV))


@pytest.mark.parametrize("M,N,K_", [(33, 65, 1), (64, 63, 255), (65, 2050, 517), (200, 200, 2051), (300, 33000, 66), (300, 15403, 515), (31, 64, 37)])
def test_gemm_f32_of_rows_that_end_anywhere(K, M, N, K_):
    # no multiple of four: the bits are those of the same rows with zeros up to whole fours, whatever stands behind a row
    g = torch.Generator(device=DEV).manual_seed(M + N)
    even = (K_ + 3) // 4 * 4
    out = []
    for width, cols, fill in ((even, even, 0.0), (K_ + 2, K_, float("nan"))):
        g.manual_seed(M + N)
        a, w = (torch.full((r, width), fill, device=DEV) for r in (M, N))
        for t in (a, w):
            t[:, :K_] = torch.randn(t.shape[0], K_, device=DEV, generator=g)
        out.append(K.gemm_f32(a[:, :cols], w[:, :cols]))
    assert torch.equal(*out)
    a[1, 0] = float("inf")                                  # and those that are made again
    assert torch.equal(K.gemm_f32(a[:, :K_], w[:, :K_])[2:], out[0][2:])


@pytest.mark.parametrize("M,N,K_", [(1, 70, 4), (1, 5000, 1540), (31, 64, 36), (32, 130, 256), (33, 65, 288), (64, 63, 260), (65, 2050, 512),
                                    (200, 200, 2052), (300, 33000, 68)])
def test_gemm_f32_has_the_same_bits_by_copies_and_through_registers(K, M, N, K_):
    # rows of whole aligned fours are copied straight to LDS; the same numbers in rows that start elsewhere go through registers.  Edges of
    # tiles, of stages of 32 k and of ranges, with and without slabs; not-a-numbers behind every row
    g = torch.Generator(device=DEV).manual_seed(M + N)
    wide_a, wide_w = (torch.full((r, K_ + 8), float("nan"), device=DEV) for r in (M, N))
    wide_a[:, :K_], wide_w[:, :K_] = torch.randn(M, K_, device=DEV, generator=g), torch.randn(N, K_, device=DEV, generator=g)
    b = torch.randn(N, device=DEV, generator=g)
    odd = torch.full((M, K_ + 1), float("nan"), device=DEV)
    odd[:, :K_] = wide_a[:, :K_]
    out = K.gemm_f32(wide_a[:, :K_], wide_w[:, :K_], b)
    want = wide_a[:, :K_].double() @ wide_w[:, :K_].double().T + b.double()
    # a tree of L = 4 levels of 16 rounds a sum with an rms error of at most 1.69 sqrt(L) 2^-24 of the result's rms, 3.4; the bias
    # and the rounding of the result itself come under it (measured 1.9 to 2.4 at inner sizes of thousands)
    assert (out.double() - want).pow(2).mean().sqrt() <= 3.4 * 2.0 ** -24 * want.pow(2).mean().sqrt()
    if M > 1:                                       # (the stride of a single row is its length)
        assert torch.equal(out, K.gemm_f32(odd[:, :K_], wide_w[:, :K_], b))


@pytest.mark.parametrize("V", [40, 3000, 151936, 300001])
def test_sampling_searches_classes_of_any_size(K, V):
    # classes that hold a few elements, more than a chunk lists (nearly flat rows), the whole row (equal logits), and chunks of more
    # elements than a thread holds: every draw against the plain rule, as far from a boundary of the CDF as sums of 32-bit
    # exponentials are off (the exponentials by 3e-7 each, at 17,000 kept tokens a row and more)
    g = torch.Generator().manual_seed(V)
    R = 12
    logits = torch.randn(R, V, generator=g) * torch.tensor([3, 3, 1, 1, 0.2, 0.2, 0.01, 0.01, 0, 0, 6, 6.0])[:, None]
    top_ps = torch.tensor([0.9, 0.3, 0.9, 0.999, 0.5, 0.95, 0.9, 0.02, 0.25, 0.9, 0.99, 1e-5])
    temps, us = torch.full((R,), 0.8), torch.rand(R, generator=g)
    out = K.sample(logits.to(DEV), temps.to(DEV), top_ps.to(DEV), us.to(DEV)).tolist()
    assert out == K.sample(logits.to(DEV), temps.to(DEV), top_ps.to(DEV), us.to(DEV)).tolist()
    for r in range(R):
        p = P.top_p_probs(logits[r].double(), 0.8, float(top_ps[r]))
        want, cum = P.inverse_cdf(p, float(us[r])), torch.cumsum(p, 0)
        assert 0 <= out[r] < V and (out[r] == want or abs(float(cum[min(out[r], want)]) - float(us[r])) < 2e-6), (r, out[r], want)
        assert float(p[out[r]]) > 0 or abs(float(us[r]) - 1) < 2e-6, (r, "a token outside the kept set")


@pytest.mark.parametrize("V", [9000, 151936, 300001])
def test_sampling_among_many_equal_logits(K, V):
    # classes whose elements are one value (listed once), one value in some chunks and several in others, and one value but for a
    # single element; every draw against the plain rule, in which tied tokens stay in vocabulary order
    g = torch.Generator().manual_seed(V)
    R = 10
    logits = (torch.randn(R, V, generator=g) * 2).round() / 2
    logits[3:6] = logits[3:6].clamp(min=1.0)                      # most of the row one value
    logits[6:8] = 0.0
    logits[8:] = 0.0
    logits[8, V // 3], logits[9, V - 2] = -0.01, 0.02
    top_ps = torch.tensor([0.3, 0.9, 0.999, 0.4, 0.8, 0.97, 0.51307, 0.98703, 0.70291, 0.01003])     # (no whole number of equal tokens)
    us = torch.rand(R, generator=g)
    out = K.sample(logits.to(DEV), torch.full((R,), 0.9).to(DEV), top_ps.to(DEV), us.to(DEV)).tolist()
    for r in range(R):
        p = P.top_p_probs(logits[r].double(), 0.9, float(top_ps[r]))
        want, cum = P.inverse_cdf(p, float(us[r])), torch.cumsum(p, 0)
        # as far from a boundary as sums of 32-bit exponentials are off
        assert out[r] == want or abs(float(cum[min(out[r], want)]) - float(us[r])) < 2e-6, (r, out[r], want)
        assert float(p[out[r]]) > 0 or abs(float(us[r]) - 1) < 2e-6, (r, "a token outside the kept set")


def test_sampling_of_more_rows_than_a_search_takes_at_a_time(K):
    # 256 rows share the room for lists and classes, the next ones write it again; greedy, plain and top_p rows in turn
    R, V = 515, 333
    g = torch.Generator().manual_seed(5)
    logits, us = (torch.randn(R, V, generator=g) * 2).to(DEV), torch.rand(R, generator=g).to(DEV)
    temps, top_ps = torch.tensor([0.0, 0.8, 0.8, 1.3])[torch.arange(R) % 4].to(DEV), torch.tensor([1.0, 0.9, 1.0, 0.4])[torch.arange(R) % 4].to(DEV)
    out = K.sample(logits, temps, top_ps, us)
    alone = [K.sample(logits[r:r + 1], temps[r:r + 1], top_ps[r:r + 1], us[r:r + 1]) for r in (0, 1, 2, 3, 255, 256, 257, 258, 511, 512, 513, 514)]
    assert out[[0, 1, 2, 3, 255, 256, 257, 258, 511, 512, 513, 514]].tolist() == [int(t[0]) for t in alone]
    assert torch.equal(out, torch.cat([K.sample(logits[r:r + 103], temps[r:r + 103], top_ps[r:r + 103], us[r:r + 103]) for r in range(0, R, 103)]))


def test_the_room_that_sampling_holds(K):
    # bytes a row: 640, and what a search takes: classes, a row's length (rounded up a chunk) and at most 623 KB, for 256 rows at most
    from pico_vllm_amd.sampling.sampler import Sampler
    size = lambda *a, **k: 4 * K.sample_workspace(*a, **k).numel()
    assert size(64, DEV, top_p_rows=False) == size(64, DEV, 151936, top_p_rows=False) == 640 * 64
    assert size(1, DEV, 5000) == 640 + 16400 + 4 * 32 * 160
    assert size(8, DEV, 151936) == 8 * (640 + 16400 + 4 * 151936 + 0) and size(8, DEV) == 8 * (640 + 16400 + 4 * 32 * 4864)
    assert size(4096, DEV, 151936) == 4096 * 640 + 256 * (16400 + 4 * 151936)
    sampler, logits = Sampler(torch.device(DEV), 64), torch.randn(2, 700, device=DEV)
    for temps, top_ps in (([0.0, 0.0], [1.0, 1.0]), ([0.0, 0.7], [0.5, 1.0])):
        sampler.sample(logits, temps, top_ps, [1, 2], [0, 0])
    assert sampler._top_p_work is None
    first = [sampler.sample(torch.cat([logits] * n, 1), [0.7, 0.0], [0.5, 1.0], [1, 2], [0, 0]) for n in (1, 3, 1)]
    assert first[0] == first[2] and 4 * sampler._top_p_work[1].numel() == size(64, DEV, 2100)
    with pytest.raises(K.KernelError, match="workspace"):
        K.sample(logits, *(torch.full((2,), 0.5, device=DEV) for _ in range(3)), work=K.sample_workspace(2, DEV, top_p_rows=False))


@pytest.mark.parametrize("R", [1, 63, 64, 65, 256, 257, 300])
def test_options_that_travel_with_the_launch(K, R):
    # the sampler's rows against the launches that read them from the GPU, at the edges of how many travel with one launch; two launches
    # unread at a time
    from pico_vllm_amd.sampling.sampler import Sampler, uniform
    g = torch.Generator().manual_seed(R)
    seeds = torch.randint(-2 ** 62, 2 ** 62, (R,), generator=g).tolist()
    seeds[0] = 2 ** 70 + 5
    at = torch.randint(0, 5000, (R,), generator=g).tolist()
    assert K.sample_uniforms(seeds, at).tolist() == [uniform(s, i) for s, i in zip(seeds, at)]
    temps, top_ps = [[0.0, 0.7, 1.0, 0.8][i % 4] for i in range(R)], [[1.0, 0.9, 1.0, 0.95][i % 4] for i in range(R)]
    sampler = Sampler(torch.device(DEV), R + 3)
    tickets, want = [], []
    for step, (t, p) in enumerate([(temps, top_ps), ([0.0] * R, top_ps), (temps, [1.0] * R), (temps[::-1], top_ps)]):
        logits = torch.randn(R, 3000, generator=g).to(DEV) * 2.5
        us = [uniform(s, i + step) if x > 0 else 0.0 for s, i, x in zip(seeds, at, t)]
        want.append(K.sample(logits, *(torch.tensor(x, device=DEV) for x in (t, p, us))).tolist())
        tickets.append(sampler.launch(logits, t, p, [s if x > 0 else None for s, x in zip(seeds, t)], [i + step for i in at]))
        assert sampler.device_tokens[:R].tolist() == want[-1]
        if step % 2:
            assert [sampler.read(x) for x in tickets[-2:]] == want[-2:]


@pytest.mark.parametrize("V", [40, 2049, 65535, 65537, 131073, 196608, 196641, 262145])
def test_sampling_finds_every_element_of_a_chunk(K, V):
    # likely tokens at the edges of a row's 32 chunks and of what a thread reads of one at a time, all others next to impossible: each is drawn
    # where its share of the row lies
    step = -(-V // 32)
    at = sorted({c * step + o for c in (0, 13, 31) for o in (0, 255, 256, 2047, 2048, 4095, 4096, 6143, 6144, 8191, step - 1) if o < step and c * step + o < V})
    n = len(at)
    logits = torch.full((n, V), -40.0)
    logits[:, at] = 3.0
    u = (torch.arange(n) + 0.5) / n
    got = K.sample(logits.to(DEV), torch.ones(n, device=DEV), torch.full((n,), 0.999, device=DEV), u.to(DEV))
    assert got.tolist() == at


def test_sampling_at_the_edges_of_its_options(K):
    # a nucleus so small that only the likeliest token fits, a temperature so low that it holds all the mass, one so high
    # that the distribution is flat, and a vocabulary smaller than the number of chunks a row is read in
    g = torch.Generator().manual_seed(3)
    for V in (5, 31, 33, 1000, 151936):
        logits = torch.randn(6, V, generator=g) * 2
        best = logits.argmax(1).tolist()
        temps = torch.tensor([1.0, 1e-4, 1.0, 50.0, 50.0, 0.3])
        top_ps = torch.tensor([1e-6, 1.0, 1e-6, 1.0, 0.999999, 1e-3])
        for u in (0.0, 0.37, 0.999999):
            us = torch.full((6,), u)
            out = K.sample(logits.to(DEV), temps.to(DEV), top_ps.to(DEV), us.to(DEV)).tolist()
            assert [out[0], out[1], out[2], out[5]] == [best[0], best[1], best[2], best[5]], (V, u, out, best)
            for r in (3, 4):                                   # nearly flat: the token at which the CDF passes u
                p = P.top_p_probs(logits[r].double(), 50.0, float(top_ps[r]))
                want = P.inverse_cdf(p, u)
                assert 0 <= out[r] < V and (out[r] == want or abs(float(torch.cumsum(p, 0)[min(out[r], want)]) - u) < 1e-4), (V, u, r, out[r], want)


def test_sampling_never_returns_a_token_whose_probability_underflowed(K):
    # a low temperature leaves a handful of tokens with a probability above zero; with u just below 1 the running sum
    # of a thread may stop short of the target by rounding, and the fallback must then be the last token that has
    # any probability, never one of the thousands behind it whose exp() is 0
    g = torch.Generator().manual_seed(5)
    for V in (1000, 151936):
        logits = torch.randn(4, V, generator=g)
        alive = [sorted(torch.randperm(V, generator=g)[:3].tolist()) for _ in range(4)]
        for r, idx in enumerate(alive):
            logits[r, idx] = torch.tensor([30.0, 30.5, 29.5])
        temps = torch.full((4,), 0.05)                       # exp((x - 30.5) / 0.05) is 0 for every other token
        for u in (0.0, 0.5, 0.9999999, 1.0 - 2.0 ** -24):
            out = K.sample(logits.to(DEV), temps.to(DEV), torch.ones(4, device=DEV), torch.full((4,), u).to(DEV),
                           top_p_rows=False).tolist()
            assert all(out[r] in alive[r] for r in range(4)), (V, u, out, alive)
            out = K.sample(logits.to(DEV), temps.to(DEV), torch.tensor([1.0, 0.9, 0.5, 1.0]).to(DEV),
                           torch.full((4,), u).to(DEV)).tolist()
            assert all(out[r] in alive[r] for r in range(4)), (V, u, out, alive)


def test_sampling_refuses_a_workspace_that_is_not_16_byte_aligned(K):
    logits = torch.randn(2, 100).to(DEV)
    ones = torch.ones(2, device=DEV)
    work = K.sample_workspace(3, DEV)
    with pytest.raises(K.KernelError, match="workspace"):
        K.sample(logits, ones, ones, ones * 0.5, work=work[2:])          # 8 bytes off


def test_sampling_top_p(K):
    probs = torch.tensor([[0.05, 0.5, 0.15, 0.3]])
    logits = torch.log(probs)
    for top_p, kept in ((0.81, {1, 3, 2}), (0.79, {1, 3}), (0.2, {1})):
        seen = set()
        for i in range(200):
            u = torch.tensor([(i + 0.5) / 200])
            tok = K.sample(logits.to(DEV), torch.ones(1, device=DEV), torch.tensor([top_p], device=DEV), u.to(DEV))
            seen.add(int(tok[0]))
            want = P.inverse_cdf(P.top_p_probs(logits[0], 1.0, top_p), float(u))
            p_kept = P.top_p_probs(logits[0], 1.0, top_p)
            cum = torch.cumsum(p_kept, 0)
            assert int(tok[0]) == want or min(abs(float(c) - float(u)) for c in cum) < 1e-5
        assert seen == kept
    # a large vocabulary with random logits: every draw lies in the kept set of the plain rule
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(16, 5000, generator=g) * 4
    us = torch.rand(16, generator=g)
    out = K.sample(logits.to(DEV), torch.full((16,), 0.7, device=DEV), torch.full((16,), 0.9, device=DEV), us.to(DEV))
    for r in range(16):
        p = P.top_p_probs(logits[r], 0.7, 0.9)
        assert float(p[int(out[r])]) > 0
        want = P.inverse_cdf(p, float(us[r]))
        assert abs(int(out[r]) - want) <= 0 or abs(float(torch.cumsum(p, 0)[min(int(out[r]), want)]) - float(us[r])) < 1e-4


# ---- matrix-core attention (bfloat16) ----------------------------------------------------------
def _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=0, boost=None, decode=False, nsplit=1, teams=0, as_step=False,
               window=0, chunk_len=0, max_chunks=0, order=None, cut=None, whole=False):
    from pico_vllm_amd.ops.attention_fast import FastAttention
    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(seed)
    totals = [n + p for n, p in zip(new_lens, prefix_lens)]
    ks = [torch.randn(N, nkv, d, generator=g).to(dtype).float() for N in totals]
    vs = [torch.randn(N, nkv, d, generator=g).to(dtype).float() for N in totals]
    qs = [torch.randn(n, nq, d, generator=g).to(dtype).float() for n in new_lens]
    if boost is not None:
        boost(qs, ks, vs)
    num_pages = sum(-(-N // Pg) for N in totals) + 3
    kc, vc, bt = paged_cache(ks, vs, Pg, num_pages, dtype, seed)
    B = len(new_lens)
    cu = torch.tensor([0] + list(torch.tensor(new_lens).cumsum(0)), dtype=torch.int32, device=DEV)
    ctxl = torch.tensor(totals, dtype=torch.int32, device=DEV)
    # queries live inside a wider buffer, as q does inside the qkv activations
    T = sum(new_lens)
    wide = torch.zeros(T, (nq + 2 * nkv) * d, dtype=dtype, device=DEV)
    wide[:, :nq * d] = torch.cat(qs, 0).reshape(T, nq * d).to(DEV, dtype)
    fa = FastAttention(nq, nkv, d, window)
    scale = 1.0 / math.sqrt(d)
    if as_step:          # the way the attention part calls it: the kernels are chosen from the shape of the batch
        from types import SimpleNamespace
        step = SimpleNamespace(num_seqs=B, all_decode=max(new_lens) == 1, max_context=max(totals), cu_seqlens=cu,
                               context_lens=ctxl, host={"cu_seqlens": cu.cpu().numpy(), "context_lens": ctxl.cpu().numpy()}, shared={})
        out = fa(wide, SimpleNamespace(k=kc, v=vc), bt, step, scale)
    elif decode:
        if cut is not None:             # a cut to fill: the contexts of all sequences in pieces of one length
            cut.append(fa.decode_cut(B, nsplit, DEV))
        out = fa.decode(wide, kc, vc, bt, ctxl, B, scale, nsplit, cut=cut[0] if cut is not None else None, whole=whole)
    else:
        if order is not None:           # a list to fill: the query tiles of all sequences longest first
            order.append(fa.order_list(T, B, DEV))
        out = fa.prefill(wide, kc, vc, bt, cu, ctxl, B, scale, teams=teams, chunk_len=chunk_len,
                         max_chunks=max_chunks or (-(-max(totals) // chunk_len) if chunk_len else 0),
                         order=order[0] if order is not None else None)
    want = torch.cat([P.causal_attention(qb, kb, vb, q_positions=torch.arange(p, p + n), window=window)
                      for qb, kb, vb, n, p in zip(qs, ks, vs, new_lens, prefix_lens)], 0)
    return out.reshape(-1, nq, d), want


@pytest.mark.parametrize("window", [1, 20, 64, 100, 129, 1000])
@pytest.mark.parametrize("nq,nkv,d,Pg", [(12, 2, 128, 16), (6, 3, 32, 8), (4, 1, 64, 16), (5, 5, 48, 16), (4, 1, 16, 16), (4, 2, 256, 32),
                                        (4, 1, 96, 16)])
def test_fast_attention_with_a_window(K, nq, nkv, d, Pg, window):
    # only the last `window` keys count: prompt portions (the window's edge inside a key tile, at a tile's end, beyond the
    # prefix), decode tokens with every split, a mixed step; keys before the window are made large so that one that is
    # let in shows (their pages are what a cache manager gives back)
    def boost(qs, ks, vs):
        for q in qs:
            q *= 2.0
    new_lens, prefix_lens = [70, 1, 200, 2, 1, 130], [0, 300, 131, 63, 17, 500]
    for teams in (1, 2, 3, 4, 6):
        out, want = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=window, boost=boost, teams=teams, window=window)
        close(out, want, torch.bfloat16)
    for nsplit in (1, 3, 8):
        out, want = _fast_case([1, 1, 1, 1], [300, 17, 0, 1000], nq, nkv, d, Pg, seed=window + 1, boost=boost, decode=True,
                               nsplit=nsplit, window=window)
        close(out, want, torch.bfloat16)
    out, want = _fast_case([1, 1, 40, 9], [300, 64, 100, 0], nq, nkv, d, Pg, seed=window + 2, boost=boost, as_step=True, window=window)
    close(out, want, torch.bfloat16)


def test_a_window_reads_nothing_before_it(K):
    # pages before the window hold not-a-number: a kernel that let one of their keys or values into a sum would show it
    from pico_vllm_amd.ops.attention_fast import FastAttention
    nq, nkv, d, Pg, window = 4, 2, 64, 16, 40
    g = torch.Generator().manual_seed(3)
    N = 400
    k = torch.randn(N, nkv, d, generator=g).bfloat16().float()
    v = torch.randn(N, nkv, d, generator=g).bfloat16().float()
    dead = N - window                                     # the one query, at position N - 1, sees keys dead .. N - 1
    k[:dead], v[:dead] = float("nan"), float("nan")
    kc, vc, bt = paged_cache([k], [v], Pg, N // Pg + 2, torch.bfloat16, 1, garbage=False)
    q = torch.randn(1, nq, d, generator=g).bfloat16()
    fa = FastAttention(nq, nkv, d, window)
    ctxl = torch.tensor([N], dtype=torch.int32, device=DEV)
    want = P.causal_attention(q.float(), k[dead:], v[dead:], window=window)
    for nsplit in (1, 4):
        out = fa.decode(q.reshape(1, -1).to(DEV), kc, vc, bt, ctxl, 1, d ** -0.5, nsplit)
        close(out.reshape(1, nq, d), want, torch.bfloat16)
    cu = torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    out = fa.prefill(q.reshape(1, -1).to(DEV), kc, vc, bt, cu, ctxl, 1, d ** -0.5)
    close(out.reshape(1, nq, d), want, torch.bfloat16)


@pytest.mark.parametrize("case", range(len(REFERENCE_CASES)))
def test_fast_prefill_on_the_reference_cases(K, case):
    new_lens, prefix_lens = REFERENCE_CASES[case]
    out, want = _fast_case(new_lens, prefix_lens, 12, 2, 128, 16, seed=case)
    close(out, want, torch.bfloat16)


@pytest.mark.parametrize("nq,nkv,d,Pg", [(4, 1, 16, 16), (6, 3, 32, 8), (5, 5, 48, 16), (3, 1, 80, 32), (8, 2, 256, 64),
                                        (2, 2, 64, 8), (12, 2, 128, 16)])
def test_fast_prefill_other_sizes_and_long_portions(K, nq, nkv, d, Pg):
    # portions longer than one 128-query tile, a decode token, a 2-token portion, long prefixes
    out, want = _fast_case([7, 1, 300, 2, 129], [0, 70, 45, 129, 500], nq, nkv, d, Pg, seed=3)
    close(out, want, torch.bfloat16)


@pytest.mark.parametrize("teams", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("nq,nkv,d,Pg", [(6, 3, 32, 8), (2, 2, 64, 8), (12, 2, 128, 16), (8, 2, 256, 64), (4, 1, 96, 32),
                                        (4, 1, 96, 16), (4, 1, 96, 8), (8, 2, 256, 16), (2, 1, 160, 8)])
def test_fast_prefill_with_every_shape_of_workgroup(K, nq, nkv, d, Pg, teams):
    # the shape of the workgroups (1 to 3 teams on a 64-query tile, 4: two query blocks a wave, 128-query tiles, 6: two teams of those)
    # is a hint: every value gives the same attention; lengths around the 64- and 128-query tiles and the
    # 64-, 128- and 192-key tiles of one to three teams; pages of 8 and 16 keys take the short way in whole tiles
    out, want = _fast_case([63, 1, 65, 130, 2, 200, 193, 127, 257], [0, 127, 1, 62, 191, 129, 383, 1, 64], nq, nkv, d, Pg, seed=5,
                           teams=teams)
    close(out, want, torch.bfloat16)


@pytest.mark.parametrize("teams,chunk_len", [(1, 0), (2, 0), (3, 0), (4, 0), (6, 0), (1, 256), (4, 128)])
@pytest.mark.parametrize("nq,nkv,d,Pg", [(12, 2, 128, 16), (6, 3, 32, 8), (4, 1, 96, 32), (2, 1, 160, 8)])
def test_fast_prefill_takes_the_tiles_of_several_sequences_longest_first(K, nq, nkv, d, Pg, teams, chunk_len):
    # with a list to fill, the workgroups take the query tiles of all sequences by the keys they read, most first: the
    # list is a permutation of the tiles in that order, and the attention is the same bits as sequence by sequence
    new_lens, prefix_lens = [63, 1, 65, 130, 2, 200, 193, 127, 257], [0, 127, 1, 62, 191, 129, 383, 1, 64]
    plain, want = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=5, teams=teams, chunk_len=chunk_len)
    order = []
    out, _ = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=5, teams=teams, chunk_len=chunk_len, order=order)
    close(out, want, torch.bfloat16)
    assert torch.equal(out, plain)
    bmq = 128 if teams in (4, 6) and d <= 128 else 64
    tiles = [(b, t) for b, n in enumerate(new_lens) for t in range(-(-n // bmq))]
    grid = sum(new_lens) // bmq + len(new_lens)                 # tiles the launch has room for; the list may be longer
    got = order[0].cpu().tolist()[:grid]
    assert got[len(tiles):] == [-1] * (grid - len(tiles)) and order[0].numel() >= grid
    listed = [(e >> 16, e & 0xffff) for e in got[:len(tiles)]]
    assert sorted(listed) == tiles
    keys = [min(prefix_lens[b] + new_lens[b], prefix_lens[b] + (t + 1) * bmq) for b, t in listed]
    assert keys == sorted(keys, reverse=True)
    if nq == 12 and teams == 1 and not chunk_len:
        # a list that was never written names no tile the kernel accepts: nothing is read through it, nothing is written
        from pico_vllm_amd.ops.attention_fast import FastAttention
        fa, B, T = FastAttention(nq, nkv, d), len(new_lens), sum(new_lens)
        g = torch.Generator().manual_seed(1)
        ks = [torch.randn(n + p, nkv, d, generator=g).bfloat16().float() for n, p in zip(new_lens, prefix_lens)]
        kc, vc, bt = paged_cache(ks, ks, Pg, sum(-(-k.shape[0] // Pg) for k in ks) + 3, torch.bfloat16, 1)
        cu = torch.tensor([0] + list(torch.tensor(new_lens).cumsum(0)), dtype=torch.int32, device=DEV)
        ctxl = torch.tensor([n + p for n, p in zip(new_lens, prefix_lens)], dtype=torch.int32, device=DEV)
        q = torch.randn(T, (nq + 2 * nkv) * d, generator=g).bfloat16().to(DEV)
        for junk in (1 << 30, (3 << 16) | 40, 0x7fff0000):
            lst = fa.order_list(T, B, DEV).fill_(junk)
            res = fa.prefill(q, kc, vc, bt, cu, ctxl, B, d ** -0.5, out=torch.zeros(T, nq * d, dtype=torch.bfloat16, device=DEV),
                             teams=teams, order=lst, order_build=False)
            assert not res.float().abs().sum().item()


@pytest.mark.parametrize("Pg", [8, 16, 32])
@pytest.mark.parametrize("d", list(range(16, 257, 16)))
def test_fast_prefill_whole_key_tiles_at_every_head_size_and_page_size(K, d, Pg):
    # contexts of three and more whole key tiles: where a thread's chunks of K are a whole number of pages
    # apart the kernel prepares its addresses once per tile, elsewhere it must not; queries are scaled up so
    # that a few keys carry each row's weight and a wrong key or row part shows
    def boost(qs, ks, vs):
        for q in qs:
            q *= 4.0            # a power of two: the scaled queries are bfloat16 numbers still
    out, want = _fast_case([200, 70, 3], [0, 330, 400], 2, 1, d, Pg, seed=17 + d + Pg, boost=boost)
    assert float(want.abs().mean()) > 0.3
    close(out, want, torch.bfloat16)
    # and the decode kernels of that head size, whole and split
    for nsplit in (1, 5):
        out, want = _fast_case([1, 1], [330, 65], 2, 1, d, Pg, seed=d + Pg, boost=boost, decode=True, nsplit=nsplit)
        close(out, want, torch.bfloat16)


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("nq,nkv,d,Pg,nsplit", [(12, 2, 128, 16, 8), (6, 3, 32, 8, 2), (5, 5, 48, 16, 3), (4, 1, 256, 32, 4), (8, 2, 96, 16, 16)])
def test_fast_decode_with_the_contexts_cut_into_pieces_of_one_length(K, nq, nkv, d, Pg, nsplit, window):
    # from 17 sequences on (32, counted as a recorded step is padded) the contexts of a decode step are cut into pieces of one length over all sequences (the pieces of
    # a long context are as long as a short context's): the cut covers every sequence's keys once, in order, in whole units
    # of 32 keys (of an LDS tile where the kernel stages tiles), in no more pieces than nsplit splits of 32 sequences
    # would be and with the smallest length that allows that; the attention is the plain one; and sequences without a context
    # behind the others (the padding of a recorded step) change no bit of the others
    from pico_vllm_amd.ops.attention_fast import FastAttention
    def boost(qs, ks, vs):
        for q in qs:
            q *= 2.0
    prefix_lens = [3000, 17, 0, 1000, 64, 129, 2047, 5, 700, 31, 32, 33, 1500, 95, 96, 2, 260, 511, 4100, 1]
    new_lens = [1] * len(prefix_lens)
    cut = []
    out, want = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=nsplit + window, boost=boost, decode=True, nsplit=nsplit,
                           window=window, cut=cut)
    close(out, want, torch.bfloat16)
    plan, slots = cut[0]
    B = len(prefix_lens)
    assert slots == 32 * nsplit
    pieces = plan[:4 * slots].reshape(slots, 4).cpu().tolist()
    rows = plan[4 * slots:4 * slots + 2 * B].reshape(B, 2).cpu().tolist()
    unit = 32 if (d % 32 == 0 and d <= 128 and nq // nkv <= 16) else (64 if d <= 128 else 32)
    used = sum(n for _, n in rows)
    assert used <= slots and all(p[0] == -1 for p in pieces[used:])
    lengths = set()
    for b, (first, n) in enumerate(rows):
        ctx = prefix_lens[b] + 1
        low = max(0, ctx - window) // unit * unit if window else 0
        mine = pieces[first:first + n]
        assert [p[0] for p in mine] == [b] * n and all(p[3] == ctx for p in mine) and 1 <= n <= 256
        assert mine[0][1] == low and mine[-1][2] == ctx and all(x[2] == y[1] for x, y in zip(mine, mine[1:]))
        lengths |= {p[2] - p[1] for p in mine[:-1]}
        T = mine[0][2] - mine[0][1] if n > 1 else None
        assert all(p[2] - p[1] == T for p in mine[:-1])
    assert len(lengths) <= 1 and all(t % unit == 0 for t in lengths)
    if lengths:                                            # a unit shorter, the pieces would not fit the launch
        T = lengths.pop()
        spans = [prefix_lens[b] + 1 - (max(0, prefix_lens[b] + 1 - window) // unit * unit if window else 0) for b in range(B)]
        assert all(-(-x // T) == n for x, (_, n) in zip(spans, rows))
        assert T == unit or sum(-(-x // (T - unit)) for x in spans) > slots or -(-max(spans) // (T - unit)) > 256
    # the same sequences with three rows without a context behind them: the same bits
    fa = FastAttention(nq, nkv, d, window)
    g = torch.Generator().manual_seed(7)
    totals = [p + 1 for p in prefix_lens]
    ks = [torch.randn(N, nkv, d, generator=g).bfloat16().float() for N in totals]
    vs = [torch.randn(N, nkv, d, generator=g).bfloat16().float() for N in totals]
    kc, vc, bt = paged_cache(ks, vs, Pg, sum(-(-N // Pg) for N in totals) + 3, torch.bfloat16, 1)
    q = torch.randn(B + 3, (nq + 2 * nkv) * d, generator=g).bfloat16().to(DEV)
    ctxl = torch.tensor(totals + [0, 0, 0], dtype=torch.int32, device=DEV)
    bt16 = torch.full((B + 3, bt.shape[1]), -1, dtype=torch.int32, device=DEV)
    bt16[:B] = bt
    real = fa.decode(q[:B], kc, vc, bt, ctxl[:B], B, d ** -0.5, nsplit, cut=fa.decode_cut(B, nsplit, DEV))
    padded = fa.decode(q, kc, vc, bt16, ctxl, B + 3, d ** -0.5, nsplit, cut=fa.decode_cut(B + 3, nsplit, DEV))
    assert torch.equal(real, padded[:B]) and not padded[B:].float().abs().sum().item()
    # a cut that was never written names no piece of this step: nothing is read through it, every row comes out empty
    plan, slots = fa.decode_cut(B, nsplit, DEV)
    for junk in (1 << 30, -7):
        plan.fill_(junk)
        out = fa.decode(q[:B], kc, vc, bt, ctxl[:B], B, d ** -0.5, nsplit, cut=(plan, slots), cut_build=False)
        assert not out.float().abs().sum().item()


@pytest.mark.parametrize("nq,nkv,d,Pg", [(12, 2, 128, 16), (6, 3, 32, 8), (5, 5, 48, 16), (4, 1, 16, 16)])
@pytest.mark.parametrize("new_lens,prefix_lens", [([1, 1, 1, 70, 2, 1], [300, 17, 64, 33, 129, 5]),     # decode rows first, as the scheduler orders them
                                                  ([1, 1, 1, 1], [300, 17, 64, 0]),                      # decode only
                                                  ([1, 40], [1000, 0]), ([9, 1, 1], [0, 20, 30])])      # no decode row in front
def test_fast_attention_of_a_mixed_step(K, nq, nkv, d, Pg, new_lens, prefix_lens):
    # leading single-token sequences go through the decode kernel, the rest through the prefill kernel
    out, want = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=9, as_step=True)
    close(out, want, torch.bfloat16)


def test_fast_attention_of_a_step_with_much_work(K):
    # eight portions of 256 tokens after 2,048 with 16 heads: the step is served by the workgroups of 128 queries
    from pico_vllm_amd.ops.attention_fast import FastAttention
    fa = FastAttention.__new__(FastAttention)
    fa.nq = 16
    assert fa.prefill_teams([256] * 8, [2304] * 8) == 4
    out, want = _fast_case([256] * 8, [2048] * 8, 16, 4, 32, 16, seed=13, as_step=True)
    close(out, want, torch.bfloat16)


@pytest.mark.parametrize("teams", [0, 1, 2, 4, 6])
@pytest.mark.parametrize("nq,nkv,d,Pg,chunk_len", [(12, 2, 128, 16, 256), (6, 3, 32, 8, 128), (2, 2, 64, 8, 384), (4, 1, 96, 32, 128),
                                                  (4, 2, 256, 16, 512), (2, 1, 160, 8, 256)])
def test_fast_prefill_with_the_keys_cut_into_chunks(K, nq, nkv, d, Pg, chunk_len, teams):
    # every chunk of a tile's keys is a workgroup of its own and a second launch joins them: tiles of one chunk and of
    # many in one batch, a chunk's edge inside a tile's own positions (its first queries see no key of the last
    # chunk), portions of one and two tokens, a context that ends one key into a chunk, more room for chunks than needed;
    # queries are scaled up so that few keys carry a row's weight and a chunk that is lost or joined wrongly shows
    def boost(qs, ks, vs):
        for q in qs:
            q *= 2.0
    new_lens, prefix_lens = [300, 77, 1, 130, 2, 64], [1000, 0, 555, 2 * chunk_len - 129, chunk_len - 1, 3 * chunk_len]
    out, want = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=chunk_len + d, boost=boost, teams=teams, chunk_len=chunk_len)
    close(out, want, torch.bfloat16)
    more, _ = _fast_case(new_lens, prefix_lens, nq, nkv, d, Pg, seed=chunk_len + d, boost=boost, teams=teams, chunk_len=chunk_len,
                         max_chunks=-(-max(n + p for n, p in zip(new_lens, prefix_lens)) // chunk_len) + 3)
    assert torch.equal(out, more)


def test_fast_prefill_refuses_chunks_it_cannot_cut(K):
    from pico_vllm_amd.ops.kernels import KernelError
    for kw in (dict(teams=3, chunk_len=256), dict(teams=1, chunk_len=200), dict(teams=1, chunk_len=256, window=50),
               dict(teams=1, chunk_len=256, max_chunks=65)):
        with pytest.raises(KernelError):
            _fast_case([70], [300], 4, 2, 64, 16, **kw)
    with pytest.raises(KernelError):            # a head size that the 16-query kernel does not serve
        _fast_case([70], [300], 4, 2, 48, 16, teams=1, chunk_len=256)


def test_a_step_behind_a_long_prefix_cuts_its_keys_into_chunks(K):
    # the host's choice (FastAttention.prefill_chunks) and the step that it serves
    from pico_vllm_amd.ops.attention_fast import FastAttention
    fa = FastAttention.__new__(FastAttention)
    fa.nq, fa.nkv, fa.d, fa.window, fa.cus = 12, 2, 128, 0, 256
    assert fa.prefill_chunks([2048], [2048]) is None                    # no prefix: short tiles
    assert fa.prefill_chunks([2048] * 8, [4096] * 8) is None            # work for every compute unit
    assert fa.prefill_chunks([2048], [16384]) == (4, 8192, 2)           # 192 workgroups of 256 key tiles each on 512 places
    assert fa.prefill_chunks([2048], [32768]) == (4, 4096, 8)
    assert fa.prefill_chunks([64], [8064]) == (1, 2048, 4)              # one tile per head
    fa.nq = 28
    assert fa.prefill_chunks([2048], [16384]) is None                   # 448 workgroups on 512 places
    fa.window = 100
    assert fa.prefill_chunks([64], [8064]) is None
    fa.nq, fa.nkv, fa.d, fa.window = 4, 2, 64, 0
    assert fa.prefill_chunks([64, 70], [8064, 7070]) == (1, 2048, 4)
    out, want = _fast_case([1, 64, 70], [300, 8000, 7000], 4, 2, 64, 16, seed=21, as_step=True)      # behind a decode row
    close(out, want, torch.bfloat16)


def test_fast_prefill_chooses_teams_by_the_shape_of_the_batch():
    from pico_vllm_amd.ops.attention_fast import FastAttention
    fa = FastAttention.__new__(FastAttention)
    fa.nq = 12
    assert fa.prefill_teams([2048], [2048]) == 3            # a causal triangle: the longest tile decides
    assert fa.prefill_teams([512], [4096]) == 3             # few tiles
    assert fa.prefill_teams([1] * 8, [4000] * 8) == 3       # decode tokens inside a mixed step
    assert fa.prefill_teams([2048], [16384]) == 4           # many long, equal tiles that fill 128 queries
    assert fa.prefill_teams([32] * 64, [2032] * 64) == 1    # much work in short portions
    assert fa.prefill_teams([2048] * 2, [2048] * 2) == 6    # more than the longest tile's worth for every unit, not much more
    assert fa.prefill_teams([512] * 4, [1024] * 4) == 6
    assert fa.prefill_teams([2048] * 4, [2048] * 4) == 4    # much work


def test_fast_prefill_with_a_cache_of_4_gib(K):
    # offsets into such a cache do not fit 32 bits: the kernel with 64-bit addresses serves it;
    # the pages used lie at both ends of the cache
    from pico_vllm_amd.ops.attention_fast import FastAttention
    nq, nkv, d, Pg = 2, 1, 64, 16
    pages = (1 << 32) // (nkv * Pg * d * 2) + 7
    g = torch.Generator().manual_seed(11)
    n, prefix = 70, 90
    N = n + prefix
    k = torch.randn(N, nkv, d, generator=g).bfloat16().float()
    v = torch.randn(N, nkv, d, generator=g).bfloat16().float()
    q = torch.randn(n, nq, d, generator=g).bfloat16().float()
    kc = torch.zeros(pages, nkv, Pg, d, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros(pages, nkv, d, Pg, dtype=torch.bfloat16, device=DEV)
    need = -(-N // Pg)
    ids = [pages - 1 - 3 * j if j % 2 else 5 * j for j in range(need)]
    for j, page in enumerate(ids):
        m = min(Pg, N - j * Pg)
        kc[page, :, :m, :] = k[j * Pg:j * Pg + m].transpose(0, 1).to(DEV, torch.bfloat16)
        vc[page, :, :, :m] = v[j * Pg:j * Pg + m].permute(1, 2, 0).to(DEV, torch.bfloat16)
    bt = torch.tensor([ids], dtype=torch.int32, device=DEV)
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    ctxl = torch.tensor([N], dtype=torch.int32, device=DEV)
    fa = FastAttention(nq, nkv, d)
    out = fa.prefill(q.reshape(n, nq * d).to(DEV, torch.bfloat16), kc, vc, bt, cu, ctxl, 1, 1.0 / math.sqrt(d))
    want = P.causal_attention(q, k, v, q_positions=torch.arange(prefix, N))
    close(out.reshape(n, nq, d), want, torch.bfloat16)
    del kc, vc
    torch.cuda.empty_cache()


@pytest.mark.parametrize("nq,nkv,d,Pg", [(4, 1, 16, 16), (6, 3, 32, 8), (5, 5, 48, 16), (3, 1, 80, 32), (8, 2, 256, 64),
                                        (12, 2, 128, 16), (32, 1, 64, 16)])
@pytest.mark.parametrize("nsplit", [1, 3, 8, 65, 256])
def test_fast_decode(K, nq, nkv, d, Pg, nsplit):
    out, want = _fast_case([1, 1, 1, 1, 1], [0, 70, 45, 129, 1000], nq, nkv, d, Pg, seed=4, decode=True, nsplit=nsplit)
    close(out, want, torch.bfloat16)


@pytest.mark.parametrize("nq,nkv,d", [(1, 1, 32), (12, 2, 128), (16, 1, 96), (32, 2, 64), (30, 2, 128)])
@pytest.mark.parametrize("window", [0, 40])
def test_fast_decode_of_whole_sequences(K, nq, nkv, d, window):
    # one split: no merging launch.  Contexts at the edges of blocks of 32 keys and of the turns of the workgroup's eight waves, groups of
    # one to sixteen heads; a sequence without a context (the padding of a recorded step) is left zero and no other is touched
    from pico_vllm_amd.ops.attention_fast import FastAttention
    out, want = _fast_case([1] * 8, [0, 30, 31, 32, 255, 256, 511, 700], nq, nkv, d, 16, seed=nq + d, decode=True, nsplit=1, window=window, whole=True)
    close(out, want, torch.bfloat16)
    fa = FastAttention(nq, nkv, d, window)
    kc, vc = torch.randn(4, nkv, 16, d, device=DEV).bfloat16(), torch.randn(4, nkv, d, 16, device=DEV).bfloat16()
    q, bt = torch.randn(3, nq * d, device=DEV).bfloat16(), torch.arange(4, dtype=torch.int32, device=DEV).view(1, 4).repeat(3, 1)
    some = fa.decode(q, kc, vc, bt, torch.tensor([50, 0, 64], dtype=torch.int32, device=DEV), 3, d ** -0.5, 1, whole=True)
    alone = fa.decode(q[2:], kc, vc, bt[2:], torch.tensor([64], dtype=torch.int32, device=DEV), 1, d ** -0.5, 1, whole=True)
    assert not some[1].any() and torch.equal(some[2:], alone)
    with pytest.raises(K.KernelError, match="not read whole"):
        fa.decode(q, kc, vc, bt, torch.tensor([50, 0, 64], dtype=torch.int32, device=DEV), 3, d ** -0.5, 2, whole=True)


def test_fast_kernels_find_one_far_key_among_hundreds(K):
    for far in (0, 15, 16, 31, 32, 63, 64, 127, 128, 200, 511, 596):
        def boost(qs, ks, vs, far=far):
            ks[0][far] = qs[0][-1, 0:1, :] * 2.0
            vs[0][far] = 100.0
        out, want = _fast_case([3], [597], 2, 1, 64, 16, seed=far, boost=boost)
        assert float(want[-1, 0].mean()) > 50
        close(out, want, torch.bfloat16, scale=100)
        for nsplit in (1, 4):
            out, want = _fast_case([1], [599], 2, 1, 64, 16, seed=far, boost=boost, decode=True, nsplit=nsplit)
            assert float(want[-1, 0].mean()) > 50
            close(out, want, torch.bfloat16, scale=100)


@pytest.mark.parametrize("far", [2, 9000, 20470])
def test_fast_attention_finds_a_far_key_among_twenty_thousand(K, far):
    # 20,480 cached keys (1,280 pages) and one key that matters: every split of decode, and a portion of a
    # prompt after that prefix, reach it through the block table
    def boost(qs, ks, vs, far=far):
        for q in qs:
            ks[0][far] = q[-1, 0:1, :] * 3.0
        vs[0][far] = 100.0
    for nsplit in (1, 7, 32, 100, 256):
        out, want = _fast_case([1], [20480], 4, 2, 64, 16, seed=far, boost=boost, decode=True, nsplit=nsplit)
        assert float(want[-1, 0].mean()) > 50
        close(out, want, torch.bfloat16, scale=100)
    out, want = _fast_case([1], [20480], 4, 2, 64, 16, seed=far, boost=boost, as_step=True)
    close(out, want, torch.bfloat16, scale=100)
    for teams in (0, 1, 3):
        out, want = _fast_case([70], [20411], 4, 2, 64, 16, seed=far, boost=boost, teams=teams)
        assert float(want[-1, 0].mean()) > 50
        close(out, want, torch.bfloat16, scale=100)


def test_fast_kernels_refuse_what_they_cannot_do(K):
    from pico_vllm_amd.ops.attention_fast import choose, supported
    assert choose(4, 2, 24, 0) is None and choose(4, 2, 512, 0) is None and choose(4, 2, 64, -1) is None
    assert supported(12, 2, 128, 0) and supported(12, 2, 128, 4096)


# ---- weight-streaming GEMM --------------------------------------------------------------------
@pytest.mark.parametrize("M,N,K_", [(1, 2048, 1536), (8, 1536, 1536), (64, 1536, 8960), (33, 301, 136), (5, 384, 192),
                                   (2, 64, 320), (17, 1000, 264), (12, 1536, 1536), (16, 90, 64), (24, 512, 1024),
                                   (32, 301, 256), (9, 1000, 8960),
                                   # more than 32 tokens and many tiles: two tiles a workgroup (an odd number of tiles,
                                   # an odd number of slices, a single slice)
                                   (50, 10270, 192), (40, 10400, 64), (64, 10240, 320),
                                   # more than 64 tokens of a small matrix: blocks of 64 tokens, the last one partial
                                   # (with 1 to 32 and with more than 32 tokens)
                                   (65, 301, 136), (100, 1536, 1536), (130, 2048, 1536), (256, 1000, 264), (200, 90, 8960),
                                   # the four projections at the 7B sizes (hidden 3584, 28 + 2 * 4 heads of 128, 18944) ...
                                   (1, 4608, 3584), (64, 3584, 3584), (40, 37888, 3584), (8, 3584, 18944),
                                   # ... and at the 32B sizes (hidden 5120, 40 + 2 * 8 heads of 128, 27648)
                                   (3, 7168, 5120), (1, 5120, 5120), (64, 55296, 5120), (17, 5120, 27648)])
def test_gemm_skinny_epilogues(K, M, N, K_):
    g = torch.Generator().manual_seed(M * N)
    a = torch.randn(M, K_, generator=g).bfloat16()
    w = (torch.randn(N, K_, generator=g) / math.sqrt(K_)).bfloat16()
    b = torch.randn(N, generator=g)
    want = a.double() @ w.double().T
    out = K.gemm_skinny(a.to(DEV), w.to(DEV), b.to(DEV), K.EPI_F32)
    assert torch.allclose(out.cpu().double(), want + b.double(), rtol=1e-4, atol=1e-4)
    out = K.gemm_skinny(a.to(DEV), w.to(DEV), b.to(DEV), K.EPI_BF16)
    assert out.dtype == torch.bfloat16 and torch.allclose(out.cpu().double(), want + b.double(), rtol=1e-2, atol=1e-2)
    # partial sums over ranges of k add up to the product; the bias is in the first slab only
    for splits in range(2, 9):
        per = -(-(-(-K_ // splits)) // 256) * 256
        if -(-K_ // per) != splits:
            continue
        slabs = K.gemm_skinny(a.to(DEV), w.to(DEV), b.to(DEV), K.EPI_F32, splits)
        assert slabs.shape == (splits, M, N)
        assert torch.allclose(slabs.cpu().double().sum(0), want + b.double(), rtol=1e-4, atol=1e-4)
        assert torch.allclose(slabs[1:].cpu().double().sum(0) + slabs[0].cpu().double(), want + b.double(), rtol=1e-4, atol=1e-4)
    # the stack goes into the norm kernel as delta
    if N >= 64:
        splits = K.skinny_k_splits(N, K_)
        delta = K.gemm_skinny(a.to(DEV), w.to(DEV), None, K.EPI_F32, splits)
        resid = torch.randn(M, N, generator=g)
        r = resid.clone().to(DEV)
        out = K.add_rmsnorm(r, delta, torch.ones(N, device=DEV), 1e-6, torch.float32)
        assert torch.allclose(r.cpu().double(), resid.double() + want, rtol=1e-4, atol=1e-4)
        close(out, P.rms_norm((resid.double() + want).float(), torch.ones(N), 1e-6), torch.float32, scale=10)
    # SwiGLU epilogue: w = [gate rows; up rows]
    if N % 2 == 0:
        out = K.gemm_skinny(a.to(DEV), w.to(DEV), None, K.EPI_SWIGLU)
        close(out, P.swiglu(want.float()), torch.bfloat16, scale=2)
    # a row's result does not depend on the other rows of the call
    one = K.gemm_skinny(a[M // 2:M // 2 + 1].to(DEV), w.to(DEV), b.to(DEV), K.EPI_F32)
    full = K.gemm_skinny(a.to(DEV), w.to(DEV), b.to(DEV), K.EPI_F32)
    assert torch.equal(one.cpu()[0], full.cpu()[M // 2])


@pytest.mark.parametrize("M,nq,nkv,d,H,Pg,bias", [(1, 12, 2, 128, 1536, 16, True), (8, 12, 2, 128, 1536, 16, True),
                                                  (64, 6, 3, 32, 192, 8, True), (37, 3, 1, 64, 136, 32, False),
                                                  (5, 2, 2, 96, 264, 16, True), (13, 4, 2, 64, 320, 16, True),
                                                  (29, 2, 1, 128, 128, 8, False),
                                                  # several blocks of 64 tokens
                                                  (70, 12, 2, 128, 1536, 16, True), (256, 6, 3, 32, 192, 8, True),
                                                  (150, 3, 1, 64, 136, 32, False)])
def test_gemm_skinny_with_rotation_and_cache_store(K, M, nq, nkv, d, H, Pg, bias):
    # projection + bias + rotate-half + store in one kernel against the plain steps one after the other
    theta = 1e6
    g = torch.Generator().manual_seed(M + d)
    x = torch.randn(M, H, generator=g).bfloat16()
    N = (nq + 2 * nkv) * d
    w = (torch.randn(N, H, generator=g) / math.sqrt(H)).bfloat16()
    b = torch.randn(N, generator=g) if bias else None
    pos = torch.randint(0, 5000, (M,), generator=g, dtype=torch.int32)
    num_pages = M + 4
    pages = torch.randperm(num_pages, generator=g)[:M]
    offs = torch.randint(0, Pg, (M,), generator=g)
    slots = (pages * Pg + offs).to(torch.int32)
    if M > 2:
        slots[M // 2] = -1                                  # a padding row stores nothing
    kc = torch.full((num_pages, nkv, Pg, d), 7.0, dtype=torch.bfloat16, device=DEV)
    vc = torch.full((num_pages, nkv, d, Pg), 7.0, dtype=torch.bfloat16, device=DEV)
    inv = (1.0 / (theta ** (torch.arange(0, d, 2).float() / d))).to(DEV)
    q_out = K.gemm_skinny_rope(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), K.rope_table(pos.to(DEV), inv),
                               slots.to(DEV), kc, vc, nq, nkv, d)
    qkv = (x.double() @ w.double().T + (0 if b is None else b.double())).float()
    q, k, v = P.split_qkv(qkv, nq, nkv, d)
    cos, sin = P.rope_tables(pos, d, theta)
    qr, kr = P.apply_rope(q, cos, sin), P.apply_rope(k, cos, sin)
    close(q_out.reshape(M, nq, d), qr, torch.bfloat16, scale=4)
    want_k = torch.full((num_pages, nkv, Pg, d), 7.0)
    want_v = torch.full((num_pages, nkv, d, Pg), 7.0)
    for t in range(M):
        if int(slots[t]) < 0:
            continue
        want_k[int(pages[t]), :, int(offs[t]), :] = kr[t]
        want_v[int(pages[t]), :, :, int(offs[t])] = v[t]
    close(kc, want_k, torch.bfloat16, scale=4)             # also: every slot that no token owns still holds 7
    close(vc, want_v, torch.bfloat16, scale=4)


@pytest.mark.parametrize("N,K_,slabs", [(2048, 1536, 5), (17920, 1536, 3), (1000, 320, 1), (90, 64, 0), (640, 2048, 8),
                                        (2 * 323, 512, -1), (1000, 3584, 6), (512, 4096, 8), (384, 2112, 0),
                                        (4608, 3584, 7), (37888, 3584, 5)])
def test_gemm_skinny_with_the_norm_in_front(K, N, K_, slabs):
    # norm(resid + partial sums) W^T of one row in one kernel against the norm kernel followed by the product;
    # slabs: 0 = nothing to add, -1 = one sum [1, K], else a stack [slabs, 1, K]
    g = torch.Generator().manual_seed(N + K_)
    resid = torch.randn(1, K_, generator=g)
    delta = None if slabs == 0 else torch.randn((1, K_) if slabs < 0 else (slabs, 1, K_), generator=g)
    nw = 1 + 0.1 * torch.randn(K_, generator=g)
    w = (torch.randn(N, K_, generator=g) / math.sqrt(K_)).bfloat16().to(DEV)
    eps = 1e-5
    d_dev = None if delta is None else delta.to(DEV)
    assert K.skinny_norm_ok(resid.to(DEV), d_dev, w)
    assert not K.skinny_norm_ok(torch.randn(2, K_).to(DEV), None, w)
    r2 = resid.clone().to(DEV)
    h = K.add_rmsnorm(r2, d_dev, nw.to(DEV), eps, torch.bfloat16)              # the two kernels: r2 is summed in place
    total = resid.double() + (0 if delta is None else delta.double().reshape(-1, 1, K_).sum(0))
    for epi in (K.EPI_F32, K.EPI_BF16, K.EPI_SWIGLU):
        out, r_out = K.gemm_skinny_norm(resid.to(DEV), d_dev, nw.to(DEV), eps, w, epi)
        assert torch.equal(r_out, r2)                                            # the same sums in the same order
        want = K.gemm_skinny(h, w, None, epi)
        scale = float(want.float().abs().max())
        # the sum of squares is formed by other threads: the normed row may differ in a last bfloat16 bit
        assert float((out.float() - want.float()).abs().max()) <= 2e-2 * scale, epi
        assert float((out.float() - want.float()).abs().mean()) <= 1e-3 * scale, epi
        if epi == K.EPI_F32:
            close(out, (P.rms_norm(total.float(), nw, eps).bfloat16().double() @ w.cpu().double().T).float(), torch.bfloat16, scale=4)
    assert torch.allclose(r_out.cpu().double(), total, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("nq,nkv,d,H,Pg,bias,slabs", [(12, 2, 128, 1536, 16, True, 5), (6, 3, 32, 192, 8, True, 0),
                                                      (3, 1, 64, 128, 32, False, 1), (4, 2, 64, 320, 16, True, 3),
                                                      (28, 4, 128, 3584, 16, True, 5)])
def test_gemm_skinny_with_the_norm_in_front_and_rotation_and_cache_store(K, nq, nkv, d, H, Pg, bias, slabs):
    theta = 1e6
    g = torch.Generator().manual_seed(d + H)
    resid = torch.randn(1, H, generator=g)
    delta = None if slabs == 0 else torch.randn(slabs, 1, H, generator=g)
    nw = 1 + 0.1 * torch.randn(H, generator=g)
    N = (nq + 2 * nkv) * d
    w = (torch.randn(N, H, generator=g) / math.sqrt(H)).bfloat16().to(DEV)
    b = torch.randn(N, generator=g).to(DEV) if bias else None
    pos = torch.randint(0, 5000, (1,), generator=g, dtype=torch.int32)
    slots = torch.tensor([3 * Pg + 5], dtype=torch.int32, device=DEV)
    inv = (1.0 / (theta ** (torch.arange(0, d, 2).float() / d))).to(DEV)
    table = K.rope_table(pos.to(DEV), inv)
    d_dev = None if delta is None else delta.to(DEV)
    caches = []
    for fused in (False, True):
        kc = torch.full((6, nkv, Pg, d), 7.0, dtype=torch.bfloat16, device=DEV)
        vc = torch.full((6, nkv, d, Pg), 7.0, dtype=torch.bfloat16, device=DEV)
        if fused:
            q, r_out = K.gemm_skinny_rope_norm(resid.to(DEV), d_dev, nw.to(DEV), 1e-6, w, b, table, slots, kc, vc, nq, nkv, d)
        else:
            r_out = resid.clone().to(DEV)
            h = K.add_rmsnorm(r_out, d_dev, nw.to(DEV), 1e-6, torch.bfloat16)
            q = K.gemm_skinny_rope(h, w, b, table, slots, kc, vc, nq, nkv, d)
        caches.append((q.float(), r_out, kc.float(), vc.float()))
    (q0, r0, k0, v0), (q1, r1, k1, v1) = caches
    assert torch.equal(r0, r1)
    for a, c in ((q0, q1), (k0, k1), (v0, v1)):
        scale = float(a.abs().max())
        assert float((a - c).abs().max()) <= 2e-2 * scale and float((a - c).abs().mean()) <= 1e-3 * scale
    assert float((k0 == 7.0).float().mean()) > 0.5 and torch.equal(k0 == 7.0, k1 == 7.0)     # only the token's slot was written


def test_the_norm_in_front_is_refused_beyond_its_widest_row(K):
    # a width of 5,120 (the 32B size) does not fit the kernel's row buffer: the caller is told so and runs the norm itself
    w = torch.zeros(256, 5120, dtype=torch.bfloat16, device=DEV)
    resid = torch.zeros(1, 5120, device=DEV)
    assert not K.skinny_norm_ok(resid, None, w)
    with pytest.raises(K.KernelError):
        K.gemm_skinny_norm(resid, None, torch.ones(5120, device=DEV), 1e-6, w)


def test_gemm_skinny_refuses_misaligned_operands(K):
    a = torch.randn(4, 172).bfloat16().to(DEV)          # K = 172 is no multiple of 8
    w = torch.randn(64, 172).bfloat16().to(DEV)
    assert not K.skinny_ok(a, w)
    with pytest.raises(K.KernelError):
        K.gemm_skinny(a, w)
    # more than 64 rows: small matrices only, and never more than 256
    small, large = torch.randn(64, 64).bfloat16().to(DEV), torch.zeros(4104, 1024, dtype=torch.bfloat16, device=DEV)
    assert K.skinny_ok(torch.randn(65, 64).bfloat16().to(DEV), small)
    assert K.skinny_ok(torch.randn(64, 1024).bfloat16().to(DEV), large)
    assert not K.skinny_ok(torch.randn(65, 1024).bfloat16().to(DEV), large)
    assert not K.skinny_ok(torch.randn(257, 64).bfloat16().to(DEV), small)
    with pytest.raises(K.KernelError):
        K.gemm_skinny(torch.randn(257, 64).bfloat16().to(DEV), small)


def test_the_wrappers_refuse_operands_that_do_not_fit_before_anything_is_launched(K):
    # a kernel trusts the sizes it is given; what does not fit them is refused on the host, by name
    from pico_vllm_amd.ops.attention_fast import FastAttention
    bf, f32, i32 = torch.bfloat16, torch.float32, torch.int32

    def dev(*shape, dtype=f32):
        return torch.zeros(*shape, dtype=dtype, device=DEV)

    def refused(message, fn, *args, **kw):
        with pytest.raises(K.KernelError, match=message):
            fn(*args, **kw)

    T, H, V = 5, 64, 30
    ids, table = dev(T, dtype=i32), dev(V, H)
    refused("GPU only", K.embedding, table.cpu(), ids)
    refused("not supported", K.embedding, table.half(), ids)
    refused("contiguous int32", K.embedding, table, ids.long())
    refused("table must be contiguous", K.embedding, dev(V, 2 * H)[:, ::2], ids)
    refused("out must be", K.embedding, table, ids, out=dev(T, H, dtype=bf))
    refused("softcap", K.softcap, dev(4, 4, dtype=bf), 2.0)
    refused("softcap", K.softcap, dev(4, 4), 0.0)
    resid, w = dev(T, H), dev(H)
    refused("residual stream", K.add_rmsnorm, resid.to(bf), None, w, 1e-6, bf)
    refused("norm weight", K.add_rmsnorm, resid, None, dev(H + 1), 1e-6, bf)
    refused("partial sums must be float32", K.add_rmsnorm, resid, dev(2, T, H, dtype=bf), w, 1e-6, bf)
    refused("shaped like the residual", K.add_rmsnorm, resid, dev(T, H + 8), w, 1e-6, bf)
    refused("rows must be a contiguous int32", K.add_rmsnorm, resid, None, w, 1e-6, bf, rows=dev(2, dtype=torch.int64))
    refused("out has the wrong shape", K.add_rmsnorm, resid, None, w, 1e-6, bf, out=dev(T, H))
    refused("residual_add", K.residual_add, resid, dev(T, H + 8))
    refused("swiglu: input", K.swiglu, dev(T, 7))
    refused("swiglu: out", K.swiglu, dev(T, 8), out=dev(T, 8))
    a, wf = dev(T, H), dev(9, H)
    refused("inner sizes differ", K.gemm_f32, a, dev(9, H + 1))
    refused("w must be float32", K.gemm_f32, a, wf.to(bf))
    refused("bias must be", K.gemm_f32, a, wf, dev(8))
    refused("out has the wrong", K.gemm_f32, a, wf, None, dev(T, 9, dtype=bf))
    ab, wb = dev(T, H, dtype=bf), dev(16, H, dtype=bf)
    refused("inner sizes differ", K.gemm_bf16, ab, dev(16, H + 8, dtype=bf))
    refused("must be bfloat16", K.gemm_bf16, a, wb)
    refused("bias must be", K.gemm_bf16, ab, wb, dev(16, dtype=bf))
    refused("out has the wrong", K.gemm_bf16, ab, wb, None, bf, dev(T, 16))
    refused("inner sizes differ", K.gemm_skinny, ab, dev(16, H + 8, dtype=bf))
    refused("skinny_ok", K.gemm_skinny, dev(65, H, dtype=bf), dev((1 << 16) + 8, H, dtype=bf))   # many rows, a large matrix
    refused("skinny_ok", K.gemm_skinny, dev(T, 60, dtype=bf), dev(16, 60, dtype=bf))       # K no multiple of 8
    refused("bias must be", K.gemm_skinny, ab, wb, dev(15))
    refused("partial sums", K.gemm_skinny, ab, wb, None, K.EPI_BF16, 2)
    refused("even number", K.gemm_skinny, ab, dev(15, H, dtype=bf), None, K.EPI_SWIGLU)
    assert not K.skinny_norm_ok(dev(2, H), None, wb) and not K.skinny_norm_ok(dev(1, H), dev(9, 1, H), wb)
    assert K.skinny_norm_ok(dev(1, H), dev(3, 1, H), wb)
    refused("skinny_norm_ok", K.gemm_skinny_norm, dev(2, H), None, w, 1e-6, wb)
    refused("norm weight", K.gemm_skinny_norm, dev(1, H), None, dev(H + 1), 1e-6, wb)
    refused("even number", K.gemm_skinny_norm, dev(1, H), None, w, 1e-6, dev(15, H, dtype=bf), K.EPI_SWIGLU)
    # rotation and the cache: 2 query heads, 1 kv head of size 32, pages of 8
    nq, nkv, d, Pg = 2, 1, 32, 8
    kc, vc = dev(4, nkv, Pg, d, dtype=bf), dev(4, nkv, d, Pg, dtype=bf)
    qkv, slots, cs = dev(T, (nq + 2 * nkv) * d, dtype=bf), dev(T, dtype=i32), dev(T, d // 2, 2)
    K.rope_kv_store(qkv, cs, slots, kc, vc, nq, nkv, d, d)
    refused("qkv must be contiguous", K.rope_kv_store, dev(T, 100, dtype=bf), cs, slots, kc, vc, nq, nkv, d, d)
    refused("4-dimensional", K.rope_kv_store, qkv, cs, slots, kc[0], vc, nq, nkv, d, d)
    refused("do not fit", K.rope_kv_store, qkv, cs, slots, kc, dev(4, nkv, Pg, d, dtype=bf), nq, nkv, d, d)
    refused("differ in dtype", K.rope_kv_store, qkv, cs, slots, kc.float(), vc.float(), nq, nkv, d, d)
    refused("slots has 5 entries, 6 are needed", K.rope_kv_store, dev(6, (nq + 2 * nkv) * d, dtype=bf), cs, slots, kc, vc, nq, nkv, d, d)
    refused("table of cosines", K.rope_kv_store, qkv, dev(T, d // 2), slots, kc, vc, nq, nkv, d, d)
    refused("table of cosines", K.rope_kv_store, qkv, None, slots, kc, vc, nq, nkv, d, d)
    refused("inv_freq", K.rope_table, slots, dev(4, dtype=bf))
    wq, bq = dev((nq + 2 * nkv) * d, H, dtype=bf), dev((nq + 2 * nkv) * d)
    K.gemm_skinny_rope(ab, wq, bq, cs, slots, kc, vc, nq, nkv, d)
    refused("weight .* is not", K.gemm_skinny_rope, ab, wb, None, cs, slots, kc, vc, nq, nkv, d)
    refused("skinny_ok", K.gemm_skinny_rope, a, wq.float(), bq, cs, slots, kc, vc, nq, nkv, d)
    refused("bias must be", K.gemm_skinny_rope, ab, wq, bq[:-1], cs, slots, kc, vc, nq, nkv, d)
    refused("cache must be bfloat16", K.gemm_skinny_rope, ab, wq, bq, cs, slots, kc.float(), vc.float(), nq, nkv, d)
    refused("multiple of 32", K.gemm_skinny_rope, ab, dev(4 * 16, H, dtype=bf), None, dev(T, 8, 2), slots,
            dev(4, 1, Pg, 16, dtype=bf), dev(4, 1, 16, Pg, dtype=bf), 2, 1, 16)
    r1, cs1 = dev(1, H), dev(1, d // 2, 2)
    K.gemm_skinny_rope_norm(r1, None, w, 1e-6, wq, bq, cs1, slots, kc, vc, nq, nkv, d)
    refused("skinny_norm_ok", K.gemm_skinny_rope_norm, dev(2, H), None, w, 1e-6, wq, bq, cs1, slots, kc, vc, nq, nkv, d)
    refused("weight .* is not", K.gemm_skinny_rope_norm, r1, None, w, 1e-6, wb, None, cs1, slots, kc, vc, nq, nkv, d)
    refused("bias must be", K.gemm_skinny_rope_norm, r1, None, w, 1e-6, wq, bq[:-1], cs1, slots, kc, vc, nq, nkv, d)
    refused("cache must be bfloat16", K.gemm_skinny_rope_norm, r1, None, w, 1e-6, wq, bq, cs1, slots, kc.float(), vc.float(), nq, nkv, d)
    refused("multiple of 32", K.gemm_skinny_rope_norm, r1, None, w, 1e-6, dev(4 * 16, H, dtype=bf), None, dev(1, 8, 2), slots,
            dev(4, 1, Pg, 16, dtype=bf), dev(4, 1, 16, Pg, dtype=bf), 2, 1, 16)
    # attention
    q, bt, pos, seq = dev(T, nq * d, dtype=bf), dev(1, 4, dtype=i32), dev(T, dtype=i32), dev(T, dtype=i32)
    K.paged_attention_ref(q, kc, vc, bt, pos, seq, nq, nkv, d, 0.1)
    refused("unit stride", K.paged_attention_ref, q[:, :d], kc, vc, bt, pos, seq, nq, nkv, d, 0.1)
    refused("differ in dtype", K.paged_attention_ref, q.float(), kc, vc, bt, pos, seq, nq, nkv, d, 0.1)
    refused("block_table", K.paged_attention_ref, q, kc, vc, bt.long(), pos, seq, nq, nkv, d, 0.1)
    refused("out has the wrong", K.paged_attention_ref, q, kc, vc, bt, pos, seq, nq, nkv, d, 0.1, out=dev(T, nq * d))
    fa = FastAttention(nq, nkv, d)
    ctxl, cu = torch.ones(T, dtype=i32, device=DEV), torch.arange(T + 1, dtype=i32, device=DEV)
    bt5 = dev(T, 4, dtype=i32)
    fa.decode(q, kc, vc, bt5, ctxl, T, 0.1, 1)
    refused("one query token per sequence", fa.decode, q, kc, vc, bt5, ctxl, T - 1, 0.1, 1)
    refused("at most 32 query heads", FastAttention(33, 1, d).decode, dev(T, 33 * d, dtype=bf), kc, vc, bt5, ctxl, T, 0.1, 1)
    refused("bfloat16 tensors", fa.decode, q.float(), kc, vc, bt5, ctxl, T, 0.1, 1)
    refused("unit stride", fa.prefill, q[:, :d], kc, vc, bt5, cu, ctxl, T, 0.1)
    refused("block_table", fa.prefill, q, kc, vc, bt, cu, ctxl, T, 0.1)              # a table for one sequence, five given
    refused("sequence metadata", fa.prefill, q, kc, vc, bt5, cu.long(), ctxl, T, 0.1)
    refused("sequence metadata", fa.decode, q, kc, vc, bt5, ctxl[:2], T, 0.1, 1)
    # sampling
    logits, t1 = dev(3, V), dev(3)
    K.sample(logits, t1, t1 + 1, t1)
    refused("logits must be float32", K.sample, logits.to(bf), t1, t1, t1)
    refused("top_p must be", K.sample, logits, t1, dev(2), t1)
    refused("out must be", K.sample, logits, t1, t1, t1, dev(3))
    work = K.argmax_workspace(3, DEV)
    K.argmax(logits, dev(3, dtype=i32), work)
    refused("logits must be float32", K.argmax, logits.to(bf), dev(3, dtype=i32), work)
    refused("out must be", K.argmax, logits, dev(2, dtype=i32), work)
    refused("workspace", K.argmax, logits, dev(3, dtype=i32), K.argmax_workspace(2, DEV))
    torch.cuda.synchronize()


def test_the_library_product_with_its_tuner_on_gives_the_same_and_hands_the_mode_back():
    # rows in multiples of 512 are timed by the library's tuner when asked; other counts take its default; off again
    # torch's own mode is as it was
    from pico_vllm_amd.ops import linear as L
    g = torch.Generator().manual_seed(0)
    x, w, b = torch.randn(1024, 320, generator=g).bfloat16(), torch.randn(200, 320, generator=g).bfloat16(), torch.randn(200, generator=g)
    lin = L.Linear(w.to(DEV), b.to(DEV))
    want = x.double() @ w.double().T + b.bfloat16().double()
    before = lin(x.to(DEV))
    assert not torch.cuda.tunable.is_enabled()
    L.set_library_tuning(True)
    try:
        tuned = lin(x.to(DEV))                    # 1,024 rows: tuned
        assert torch.cuda.tunable.is_enabled() and torch.cuda.tunable.tuning_is_enabled()
        other = lin(x[:300].to(DEV))              # 300 rows: the library's default choice, nothing is timed
        assert not torch.cuda.tunable.tuning_is_enabled()
        no_bias = L.Linear(w.to(DEV))(x[:512].to(DEV))
    finally:
        L.set_library_tuning(False)
    assert not torch.cuda.tunable.is_enabled() and not torch.cuda.tunable.tuning_is_enabled()
    for got, ref in ((before, want), (tuned, want), (other, want[:300]), (no_bias, want[:512] - b.bfloat16().double())):
        assert got.dtype == torch.bfloat16
        assert torch.allclose(got.cpu().double(), ref, rtol=1e-2, atol=1e-2 * math.sqrt(320))


@pytest.mark.parametrize("nq,nkv,dk,dv,more", [(12, 1, 320, 256, {}), (6, 2, 64, 128, {"window": 50, "keep_first": 5, "softcap": 20.0}),
                                               (5, 5, 128, 16, {"chunk": 64, "sink": True}), (40, 2, 32, 96, {"slope_span": 8.0})])
@pytest.mark.parametrize("lens,prefix", [([1], 0), ([11, 10], 0), ([65, 1, 130], 37), ([3, 300], 500)])
@pytest.mark.parametrize("Pg", [8, 64])
def test_bias_attention_shared_keys(nq, nkv, dk, dv, more, lens, prefix, Pg):
    # 128 columns that share staged keys (columns run over tokens whatever the heads a group), against blocks whose keys four
    # waves share: edges of workgroups, of stages of 32 and 64 keys, of windows, kept keys and chunks, several sequences
    from pico_vllm_amd.ops.attention_bias_fast import FastBiasAttention
    fast = FastBiasAttention(nq, nkv, dk, dv, dk ** -0.5, **more)
    g = torch.Generator(device=DEV).manual_seed(dk + len(lens))
    B, T, per = len(lens), sum(lens), -(-(max(lens) + prefix) // Pg)
    kc, vc = (torch.randn(B * per + 3, nkv, *s, device=DEV, generator=g).bfloat16() for s in ((Pg, dk), (dv, Pg)))
    bt = torch.randperm(B * per + 3, device=DEV, generator=g)[:B * per].int().reshape(B, per).contiguous()
    q = torch.randn(T, nq * dk, device=DEV, generator=g).bfloat16()
    cu = torch.tensor([0] + [sum(lens[:i + 1]) for i in range(B)], dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(prefix, prefix + n) for n in lens]).int().to(DEV)
    got, want = (fast.run(q, kc, vc, bt, cu, pos, B, split=s, chunks=1).double() for s in (False, True))
    # both round probabilities (2^-9 each, against maxima that may differ) and the output to bfloat16
    assert float((got - want).abs().max()) <= 2.0 ** -7 * float(vc.float().abs().max())


@pytest.mark.parametrize("nq,nkv,dk,dv,more", [(12, 1, 320, 256, {}), (28, 1, 64, 64, {"window": 100}), (5, 5, 128, 128, {"chunk": 64, "sink": True}),
                                               (12, 2, 64, 32, {"window": 40, "keep_first": 6, "softcap": 20.0}),
                                               (8, 4, 64, 128, {"v_div": 2, "temp_coef": 0.1, "temp_every": 32, "slope_span": 8.0})])
@pytest.mark.parametrize("new_lens,prefix_lens", [([200], [0]), ([3, 90, 64, 1], [130, 37, 64, 70])])
def test_shared_keys_keep_columns_apart(K, nq, nkv, dk, dv, more, new_lens, prefix_lens):
    # against the equations in 64 bits; and what a token does not see (later tokens of its sequence, tokens that its window has
    # passed, another chunk's, the rest of a page) does not reach it: a row that sees no value of Inf or NaN keeps its bits
    from pico_vllm_amd.ops.attention_bias_fast import FastBiasAttention
    fast = FastBiasAttention(nq, nkv, dk, dv, dk ** -0.5, **more)
    g = torch.Generator().manual_seed(dk + nq)
    R, nv, Pg, T = nq // nkv, nkv // more.get("v_div", 1), 16, sum(new_lens)
    totals = [n + p for n, p in zip(new_lens, prefix_lens)]
    ks, vs = ([torch.randn(N, *s, generator=g).bfloat16() for N in totals] for s in ((nkv, dk), (nv, dv)))
    q = torch.randn(T, nq, dk, generator=g).bfloat16()
    bt = torch.randperm(sum(-(-N // Pg) for N in totals) + 3, generator=g).int()
    cu = torch.tensor([0] + [sum(new_lens[:b + 1]) for b in range(len(new_lens))], dtype=torch.int32)
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(new_lens, prefix_lens)]).int()
    per = -(-max(totals) // Pg)

    def run(ks, vs):
        kc, vc = torch.full((len(bt), nkv, Pg, dk), float("nan")).bfloat16(), torch.full((len(bt), nv, dv, Pg), float("nan")).bfloat16()
        table, at = torch.zeros(len(new_lens), per, dtype=torch.int32), 0
        for b, N in enumerate(totals):
            pages = bt[at:at + -(-N // Pg)]
            at += len(pages)
            table[b, :len(pages)] = pages
            for j in range(N):
                kc[pages[j // Pg], :, j % Pg], vc[pages[j // Pg], :, :, j % Pg] = ks[b][j], vs[b][j]
        return fast.run(q.reshape(T, -1).to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), cu.to(DEV), pos.to(DEV), len(new_lens), split=False).cpu()

    def seen(b, i):                                     # the keys that the token at position i sees
        j = torch.arange(totals[b])
        lo = i // more["chunk"] * more["chunk"] if "chunk" in more else max(0, i - more["window"] + 1) if "window" in more else 0
        return (j <= i) & ((j >= lo) | (j < more.get("keep_first", 0)))
    clean = run(ks, vs)
    for b in range(len(new_lens)):
        for t in range(int(cu[b]), int(cu[b + 1])):
            i, see = int(pos[t]), seen(b, int(pos[t]))
            s = torch.einsum("ghd,jgd->ghj", q[t].double().view(nkv, R, dk), ks[b].double()) * dk ** -0.5
            s = s * (1 + more.get("temp_coef", 0.0) * math.log((i + 1) // more["temp_every"] + 1) if "temp_every" in more else 1.0)
            if "slope_span" in more:
                slope = 2.0 ** (-more["slope_span"] * torch.arange(1, nq + 1).double() / nq)
                s = s - slope.view(nkv, R, 1) * (i - torch.arange(totals[b])).double()
            s = 20.0 * torch.tanh(s / 20.0) if "softcap" in more else s
            p = s.masked_fill(~see, float("-inf")).exp()
            p = p / (p.sum(-1, keepdim=True) + (1.0 if more.get("sink") else 0.0))
            want = torch.einsum("ghj,jgd->ghd", p, vs[b].double().repeat_interleave(nkv // nv, 1)).reshape(-1)
            # the weights and the output are rounded to bfloat16, whose unit is 2^-7: each by at most 2^-8 of its size, the
            # weights' share of the output being at most that of sum p |v|; the scores' float32 sums are the rest
            bound = 2.0 ** -7 * torch.einsum("ghj,jgd->ghd", p, vs[b].double().abs().repeat_interleave(nkv // nv, 1)).reshape(-1) + 1e-5
            assert bool(((clean[t].double() - want).abs() <= bound).all()), (b, i)
    bad = {0: [totals[0] - 2], 1: [1, 60, 62, 126], 2: [127]} if len(totals) > 1 else {0: [0, 7, 63, 64, 150, 190]}
    odd_k, odd_v = [k.clone() for k in ks], [v.clone() for v in vs]
    for b, keys in bad.items():
        for n, j in enumerate(keys):
            odd_v[b][j, :, ::3] = (float("inf"), float("nan"), float("-inf"))[n % 3]
    last = max(bad)
    odd_k[last][bad[last][-1]] = float("nan")
    got = run(odd_k, odd_v)
    for b in range(len(new_lens)):
        for t in range(int(cu[b]), int(cu[b + 1])):
            hit = bool(seen(b, int(pos[t]))[bad.get(b, [])].any())
            assert torch.isfinite(got[t]).all() != hit, (b, int(pos[t]))
            if not hit:
                assert torch.equal(got[t], clean[t]), (b, int(pos[t]))


@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 64), (6, 1, 40, 72), (3, 3, 96, 128)])
@pytest.mark.parametrize("lens", [[1], [64, 63], [65, 1, 200], [130]])
@pytest.mark.parametrize("steps", [(0.01, 0.2), (0.5, 60.0)])
def test_ssd_chunks(K, H, G, dk, dv, lens, steps):
    # a decay a token and head, from slow ones to ones that a float cannot hold, over the edges of chunks of 64 and several
    # sequences, against the walk token by token in 64 bits
    g = torch.Generator().manual_seed(dk + sum(lens))
    T, B = sum(lens), len(lens)
    x = torch.randn(T, H * dv + 2 * G * dk, generator=g).bfloat16()
    dt = torch.empty(T, H).uniform_(*steps, generator=g)
    a = torch.empty(H).uniform_(0.5, 4.5, generator=g)
    decay = torch.exp(-a * dt)
    state = torch.randn(B + 1, H, dk, dv, generator=g)
    cu = torch.tensor([0] + [sum(lens[:i + 1]) for i in range(B)], dtype=torch.int32)
    slots = torch.arange(B, 0, -1, dtype=torch.int32)
    st = state.to(DEV)
    out = K.ssd_chunks(x.to(DEV), H * dv + G * dk, H * dv, 0, decay.to(DEV), dt.to(DEV), cu.to(DEV), slots.to(DEV), st, B, H, G, dk, dv).cpu().double()
    v, k, q = x[:, :H * dv].double().view(T, H, dv), x[:, H * dv:H * dv + G * dk].double().view(T, G, dk), x[:, H * dv + G * dk:].double().view(T, G, dk)
    k, q = k.repeat_interleave(H // G, 1), q.repeat_interleave(H // G, 1)
    for b in range(B):
        S = state[slots[b]].double()
        size = S.abs()                              # the same sums of absolute values: what rounding is relative to
        for t in range(cu[b], cu[b + 1]):
            w = decay[t].double().view(H, 1, 1)
            add = k[t].unsqueeze(-1) * (dt[t].double().view(H, 1) * v[t]).unsqueeze(1)
            S, size = w * S + add, w * size + add.abs()
            bound = (size * q[t].abs().unsqueeze(-1)).sum(1)
            # sums of up to dk + 64 float32 products of float32 products: 2^-24 of the absolute sums a rounding, at most
            # some twenty in a row (chains of 64 at random, decays and factors)
            err = (out[t].view(H, dv) - (S * q[t].unsqueeze(-1)).sum(1)).abs()
            assert bool((err <= 20 * 2.0 ** -24 * bound + 1e-30).all())
        assert bool(((st[slots[b]].cpu().double() - S).abs() <= 20 * 2.0 ** -24 * size + 1e-30).all())
    assert torch.equal(st[0].cpu(), state[0])       # a slot that no sequence holds


@pytest.mark.parametrize("dk,dv", [(32, 64), (40, 72), (96, 128), (128, 200)])
@pytest.mark.parametrize("n", [1, 31, 64, 150])
def test_decay_chunks_scale_and_odd_states(K, dk, dv, n):
    # a constant decay with a scale on the queries against the walk in 64 bits; an infinite element of the state and an Inf among the
    # values stay in their columns (and, of the value, in its own and later tokens)
    g = torch.Generator().manual_seed(dk + n)
    H = 3
    x, fixed, state = torch.randn(n, 2 * H * dk + H * dv, generator=g).bfloat16(), torch.tensor([0.6, 0.97, 1.0]), torch.randn(1, H, dk, dv, generator=g)
    cu, slots = torch.tensor([0, n], dtype=torch.int32).to(DEV), torch.zeros(1, dtype=torch.int32, device=DEV)

    def run(rows, start):
        st = start.to(DEV)
        return K.gla_scan(rows.to(DEV), 0, H * dk, 2 * H * dk, None, cu, slots, st, 1, H, dk, dv, 0.3, 64, head_decay=fixed.to(DEV)).view(n, H, dv).cpu(), st.cpu()
    out, st = run(x, state)
    q, k, v = x[:, :H * dk].double().view(n, H, dk), x[:, H * dk:2 * H * dk].double().view(n, H, dk), x[:, 2 * H * dk:].double().view(n, H, dv)
    S = state[0].double()
    size = S.abs()
    for t in range(n):
        add, w = k[t].unsqueeze(-1) * v[t].unsqueeze(1), fixed.double().view(H, 1, 1)
        S, size = w * S + add, w * size + add.abs()
        # (test_ssd_chunks' bound, and powers of the decay that are made from its float32 logarithm: 2^-24 of an exponent of up to 64 a chunk)
        assert bool(((out[t].double() - 0.3 * (S * q[t].unsqueeze(-1)).sum(1)).abs() <= (20 + 64) * 2.0 ** -24 * 0.3 * (size * q[t].abs().unsqueeze(-1)).sum(1)).all())
    odd_state, odd_x = state.clone(), x.clone()
    odd_state[0, 1, 5, 3], odd_x[n // 2, 2 * H * dk + 7] = float("inf"), float("-inf")
    got, st2 = run(odd_x, odd_state)
    hit = torch.zeros(n, H, dv, dtype=torch.bool)
    hit[:, 1, 3], hit[n // 2:, 0, 7] = True, True
    assert torch.equal(got[~hit], out[~hit]) and not torch.isfinite(got[hit]).any()
    assert torch.equal(st2[0, 2], st[0, 2]) and st2[0, 1, 5, 3] == float("inf") and torch.isinf(st2[0, 0, :, 7]).all()


@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 64), (6, 1, 40, 72), (3, 3, 8, 8)])
@pytest.mark.parametrize("lens", [[1] * 70 + [130, 17, 64], [33, 0, 1, 32, 8, 200], [9] * 5])
def test_decay_chunks_of_many_sequences(K, H, G, dk, dv, lens):
    # many sequences walk four state elements a thread, few one; a sequence has the bits that it has alone
    g = torch.Generator().manual_seed(len(lens))
    T, B = sum(lens), len(lens)
    x = torch.randn(T, H * dv + 2 * H * dk, generator=g).bfloat16().to(DEV)
    dt, decay = (torch.rand(T, H, generator=g) + 0.1).to(DEV), (torch.rand(T, H, generator=g) * 0.3 + 0.7).to(DEV)
    state, fixed = torch.randn(B, H, dk, dv, generator=g).to(DEV), torch.linspace(0.7, 1.0, H).to(DEV)

    def run(rows, cu, slots, st, varies):
        cu, slots = torch.tensor(cu, dtype=torch.int32, device=DEV), torch.tensor(slots, dtype=torch.int32, device=DEV)
        if varies:
            return K.ssd_chunks(x[rows], H * dv + G * dk, H * dv, 0, decay[rows], dt[rows], cu, slots, st, len(slots), H, G, dk, dv)
        return K.gla_scan(x[rows], H * dv + H * dk, H * dv, 0, None, cu, slots, st, len(slots), H, dk, dv, 1.0, chunk=64, head_decay=fixed)
    cu = [sum(lens[:i]) for i in range(B + 1)]
    for varies in (True, False):
        st = state.clone()
        out = run(slice(None), cu, list(range(B)), st, varies)
        for b in range(B):
            if lens[b]:
                alone = state.clone()
                assert torch.equal(run(slice(cu[b], cu[b + 1]), [0, lens[b]], [b], alone, varies), out[cu[b]:cu[b + 1]]), b
                assert torch.equal(alone[b], st[b]), b
            else:
                assert torch.equal(state[b], st[b]), b


@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 64), (6, 1, 40, 72), (3, 3, 96, 128)])
@pytest.mark.parametrize("varies", [True, False])
def test_decay_chunks_keep_tokens_apart(K, H, G, dk, dv, varies):
    # a token's rows keep their bits whatever a later token of its chunk brings, another column of values, another head, another
    # sequence; from the token on the column (a value), or the head (a key, a decay) is not finite, and so is what is left of it
    if not varies and H != G:
        G = H                                            # one decay a head: every head has its own queries and keys
    g = torch.Generator().manual_seed(dk)
    lens = [65, 1, 200]
    T, B = sum(lens), len(lens)
    x = torch.randn(T, H * dv + 2 * G * dk, generator=g).bfloat16()
    dt, decay = torch.rand(T, H, generator=g) + 0.1, torch.rand(T, H, generator=g) * 0.3 + 0.7
    state = torch.randn(B, H, dk, dv, generator=g)
    cu = torch.tensor([0, 65, 66, 266], dtype=torch.int32).to(DEV)
    slots = torch.arange(B, dtype=torch.int32).to(DEV)
    q_col, k_col = H * dv + G * dk, H * dv

    def run(x, decay):
        st = state.to(DEV)
        if varies:
            out = K.ssd_chunks(x.to(DEV), q_col, k_col, 0, decay.to(DEV), dt.to(DEV), cu, slots, st, B, H, G, dk, dv)
        else:
            out = K.gla_scan(x.to(DEV), q_col, k_col, 0, None, cu, slots, st, B, H, dk, dv, 1.0, chunk=64,
                             head_decay=torch.linspace(0.7, 1.0, H).to(DEV), silu=True)
        return out.cpu().view(T, H, dv), st.cpu()
    clean, left = run(x, decay)
    for what, value in (("value", float("inf")), ("value", float("nan")), ("key", float("nan")), ("decay", float("nan"))):
        if what == "decay" and not varies:
            continue
        for at in (40, 66 + 31, 66 + 70, 66 + 199):
            b, h = (0, 2) if at < 65 else (2, 1)
            bad_x, bad_g = x.clone(), decay.clone()
            heads, cols = slice(h, h + 1), slice(None)
            if what == "value":
                cols = slice(5, 6)
                bad_x[at, h * dv + 5] = value
            elif what == "key":
                share = H // G
                heads = slice(h // share * share, (h // share + 1) * share)
                bad_x[at, k_col + h // share * dk + 3] = value
            else:
                bad_g[at, h] = value
            got, st = run(bad_x, bad_g)
            hit, hit_state = torch.zeros_like(got, dtype=torch.bool), torch.zeros_like(st, dtype=torch.bool)
            hit[at:int(cu[b + 1]), heads, cols] = True
            hit_state[b, heads, 3 if what == "key" else slice(None), cols] = True
            assert not torch.isfinite(got[hit]).any() and not torch.isfinite(st[hit_state]).any(), (what, at)
            assert torch.equal(got[~hit], clean[~hit]) and torch.equal(st[~hit_state], left[~hit_state]), (what, at)


@pytest.mark.parametrize("dk", [16, 17, 32, 64, 96, 128, 192, 256])
@pytest.mark.parametrize("lens,dv", [([1], 16), ([64, 65], 40), ([3, 700, 128], 72), ([130, 1, 80], 104), ([70, 16], 96), ([100], 97), ([17, 64], 128)])
def test_delta_chunks(K, dk, lens, dv):
    # the walk over the chunks' states on the matrix cores (key sizes of whole 64s) and without (96), value sizes that end inside
    # a tile of 16 columns, one and many chunks, a slot that no sequence holds, against the rule token by token in 64 bits
    g = torch.Generator().manual_seed(dk + sum(lens))
    T, B, H, G = sum(lens), len(lens), 4, 2
    q, k = (F.normalize(torch.randn(T, G, dk, generator=g), dim=-1) for _ in range(2))
    v, decay, beta = torch.randn(T, H * dv, generator=g).bfloat16(), torch.rand(T, H, generator=g) * 0.2 + 0.8, torch.rand(T, H, generator=g)
    state = torch.randn(B + 1, H, dk, dv, generator=g)
    cu = torch.tensor([0] + [sum(lens[:i + 1]) for i in range(B)], dtype=torch.int32)
    slots = torch.arange(B, 0, -1, dtype=torch.int32)
    st = state.to(DEV)
    out = K.delta_scan(q.reshape(T, -1).to(DEV), k.reshape(T, -1).to(DEV), v.to(DEV), decay.to(DEV), beta.to(DEV), cu.to(DEV), slots.to(DEV),
                       st, B, H, G, dk, dv, delta=True, chunk=64).cpu().double().view(T, H, dv)
    q, k, v = q.double().repeat_interleave(H // G, 1), k.double().repeat_interleave(H // G, 1), v.double().view(T, H, dv)
    # a chunk's sums are chains of at most 128 and its walk of 64 steps of three roundings, each chain at random about 0.2 of
    # the root of its length in units of 2^-24: 3.6; what a decay of 0.8 to 1 and the rule leave of earlier chunks' adds a
    # fifth; three times that for the spread
    tol = 13 * 2.0 ** -24

    def rms(x):
        return float(x.pow(2).mean().sqrt())
    for b in range(B):
        S, want = state[slots[b]].double(), []
        for t in range(cu[b], cu[b + 1]):
            S = S * decay[t].double().view(H, 1, 1)
            S = S + k[t].unsqueeze(-1) * (beta[t].double().view(H, 1) * (v[t] - (S * k[t].unsqueeze(-1)).sum(1))).unsqueeze(1)
            want.append((S * q[t].unsqueeze(-1)).sum(1))
        want = torch.stack(want)
        assert rms(out[cu[b]:cu[b + 1]] - want) <= tol * rms(want)
        assert rms(st[slots[b]].cpu().double() - S) <= tol * rms(S)
    assert torch.equal(st[0].cpu(), state[0])


@pytest.mark.parametrize("E,top", [(1, 1), (5, 5), (63, 4), (64, 2), (65, 16), (130, 3)])
def test_moe_route_among_equal_and_odd_logits(K, E, top):
    # the lowest of equal logits first; a NaN only where it is the first that is left; all of a row minus infinity
    g = torch.Generator().manual_seed(E)
    z = torch.randint(-3, 4, (41, E), generator=g).float()
    z[3], z[4, E // 2], z[5, 0], z[6, E - 1] = float("-inf"), float("nan"), float("nan"), float("inf")
    z[7, ::2] = float("nan")
    experts, weights = K.moe_route(z.to(DEV), top)
    for t in range(41):
        row, left = z[t].tolist(), list(range(E))
        for k in range(top):
            best = left[0]
            for e in left:
                best = e if row[e] > row[best] else best
            left.remove(best)
            assert int(experts[t, k]) == best, (t, k)
    want = torch.sigmoid(torch.gather(z, 1, experts.cpu().long()))
    assert torch.allclose(weights.cpu(), want, rtol=1e-6, atol=0, equal_nan=True)      # one exponential and a quotient


@pytest.mark.parametrize("T,H", [(1, 4), (7, 44), (3, 45), (130, 1536)])
@pytest.mark.parametrize("slabs,gated,scaled,b_dtype", [(1, False, False, None), (3, True, True, torch.bfloat16), (2, False, True, torch.float32),
                                                        (0, True, False, torch.float32)])
def test_scaled_add(K, T, H, slabs, gated, scaled, b_dtype):
    # four entries a thread (rows of whole fours on aligned addresses) and one
    g = torch.Generator().manual_seed(T + H)
    x, a = torch.randn(T, H, generator=g), torch.randn(slabs, T, H, generator=g) if slabs else None
    b = torch.randn(T, H, generator=g).to(b_dtype) if b_dtype else None
    gate, scale = (torch.randn(T, 1, generator=g) if gated and b_dtype else None), (torch.randn(H, generator=g) if scaled else None)
    want = (a.double().sum(0) if slabs else 0) + (0 if b is None else b.double() * (torch.sigmoid(gate.double()) if gate is not None else 1))
    want = x.double() + (want * scale.double() if scaled else want)
    size = x.abs().double() + ((a.abs().double().sum(0) if slabs else 0) + (0 if b is None else b.abs().double())) * (scale.abs().double() if scaled else 1)
    for off in (0, 1):                                                   # the stream on 16 bytes, and 4 behind
        buf = torch.zeros(T * H + 1)
        buf[off:off + T * H] = x.view(-1)
        resid = buf.to(DEV)[off:off + T * H].view(T, H)
        K.scaled_add(resid, None if a is None else a.to(DEV) if slabs > 1 else a[0].to(DEV), None if b is None else b.to(DEV),
                     None if gate is None else gate.to(DEV), None if scale is None else scale.to(DEV))
        # eight float32 roundings at most, of parts of `size`
        assert bool(((resid.cpu().double() - want).abs() <= 8 * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("M,N,K_,parts", [(65, 16, 200, 2), (1, 16, 520, 5), (64, 80, 128, 2), (129, 208, 1000, 4), (300, 1552, 8960, 8), (257, 3584, 18944, 3)])
def test_products_in_parts_of_the_inner_size(K, M, N, K_, parts):
    """Parts of whole 64, the last one shorter and in remainders of 8; rows in a wider matrix; with a bias and without."""
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K_ + 8, generator=g).bfloat16().to(DEV)[:, :K_]
    w = torch.randn(N, K_, generator=g).bfloat16().to(DEV)
    b = torch.randn(N, generator=g).to(DEV)
    xd, wd = x.double().cpu(), w.double().cpu()
    size = xd.abs() @ wd.abs().T
    for bias in (b, None):
        got = K.gemm_tiles_split(x, w, bias, parts).double().cpu()
        want = xd @ wd.T + (0 if bias is None else bias.double().cpu())
        # one rounding to bfloat16, and float32 sums of K terms
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + K_ * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("M,N,K_", [(65, 1536, 8960), (1000, 3584, 18944), (1536, 64, 6656)])
def test_the_layer_takes_a_long_inner_size_in_parts(K, M, N, K_):
    from pico_vllm_amd.ops.linear import Linear
    g = torch.Generator().manual_seed(N)
    x, w = torch.randn(M, K_, generator=g).bfloat16().to(DEV), torch.randn(N, K_, generator=g).bfloat16().to(DEV)
    b = torch.randn(N, generator=g).bfloat16().to(DEV)
    parts = K.tiles_parts(x, w)
    assert parts > 1
    assert torch.equal(Linear(w, b)(x), K.gemm_tiles_split(x, w, b.float(), parts))
    assert K.tiles_parts(x[:, :K_ - 4], w[:, :K_ - 4]) == 1 and K.tiles_parts(x[:, :6144], w[:, :6144]) == 1


def test_the_layer_takes_a_bias_that_starts_anywhere(K):
    # a float32 bias is kept where it lies: one that starts on no 16 bytes is the library's product's, as it was before there were parts
    from pico_vllm_amd.ops.linear import Linear
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(300, 8960, generator=g).bfloat16().to(DEV), torch.randn(1536, 8960, generator=g).bfloat16().to(DEV)
    b = torch.randn(1537, generator=g).to(DEV)[1:]
    assert K.tiles_parts(x, w, b) == 1 < K.tiles_parts(x, w, b.clone())
    got, want = Linear(w, b)(x).double().cpu(), x.double().cpu() @ w.double().cpu().T + b.double().cpu()
    # the bias and the result are rounded to bfloat16, and float32 sums of 8,960 terms
    assert bool(((got - want).abs() <= 2.0 ** -8 * (want.abs() + b.double().cpu().abs()) + 8960 * 2.0 ** -24 * (x.double().cpu().abs() @ w.double().cpu().abs().T)).all())


@pytest.mark.parametrize("nq,nkv,dk,dv,more", [(12, 2, 128, 128, {"window": 300, "slope_span": 8.0}), (6, 2, 64, 128, {"window": 50, "keep_first": 5, "softcap": 20.0}),
                                               (5, 5, 128, 16, {"chunk": 64, "sink": True}), (12, 1, 320, 256, {})])
@pytest.mark.parametrize("most", [128, 129, 384, 600])
def test_bias_attention_of_single_tokens_in_as_many_pieces_as_keys(nq, nkv, dk, dv, more, most):
    # the pieces that contexts up to `most` keys have, against the most there are (the rest of them empty): the same keys a piece, so the same bits
    # but for a single piece, which is rounded once without a merge
    from pico_vllm_amd.ops.attention_bias_fast import MAX_CHUNKS, FastBiasAttention
    fast = FastBiasAttention(nq, nkv, dk, dv, dk ** -0.5, **more)
    g = torch.Generator(device=DEV).manual_seed(most)
    contexts = [n for n in (1, 31, 127, 128, 129, 256, 257, 383, 600) if n <= most]
    B, per = len(contexts), -(-most // 16)
    kc, vc = (torch.randn(B * per, nkv, *s, device=DEV, generator=g).bfloat16() for s in ((16, dk), (dv, 16)))
    bt = torch.randperm(B * per, device=DEV, generator=g).int().reshape(B, per).contiguous()
    q = torch.randn(B, nq * dk, device=DEV, generator=g).bfloat16()
    cu, pos = torch.arange(B + 1, dtype=torch.int32, device=DEV), torch.tensor(contexts, dtype=torch.int32, device=DEV) - 1
    keys = min(most, fast.window + 31) if fast.window else most
    pieces = fast.chunks(B, B, keys)
    assert pieces == min(-(-keys // 128), fast.chunks(B, B))
    got, want = (fast.run(q, kc, vc, bt, cu, pos, B, split=True, chunks=n) for n in (pieces, MAX_CHUNKS))
    if pieces > 1:
        assert torch.equal(got, want)
    else:
        assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -9)        # an ulp of bfloat16 where the last bit of the sum differs


@pytest.mark.parametrize("nq,nkv,dk,dv,more", [(12, 2, 64, 64, {}), (20, 1, 32, 16, {"window": 30}), (5, 5, 32, 32, {"chunk": 16, "sink": True})])
@pytest.mark.parametrize("B", [1, 7, 8, 63, 64, 65, 130])
def test_a_block_of_columns_finds_its_sequence(nq, nkv, dk, dv, more, B):
    # one by one and 64 at a time: sequences without tokens, of one, of a block and of several; each has the bits it has alone
    from pico_vllm_amd.ops.attention_bias_fast import FastBiasAttention
    fast = FastBiasAttention(nq, nkv, dk, dv, dk ** -0.5, **more)
    g = torch.Generator().manual_seed(B + nq)
    lens = [int(n) for n in torch.tensor([0, 1, 1, 1, 2, 16, 40])[torch.randint(0, 7, (B,), generator=g)]]
    lens[-1] = 3
    ends = [n + int(p) for n, p in zip(lens, torch.randint(0, 200, (B,), generator=g))]
    per = -(-max(ends) // 16)
    dev = torch.Generator(device=DEV).manual_seed(B)
    kc, vc = (torch.randn(B * per, nkv, *s, device=DEV, generator=dev).bfloat16() for s in ((16, dk), (dv, 16)))
    bt = torch.randperm(B * per, generator=g).int().reshape(B, per).to(DEV)
    q = torch.randn(sum(lens), nq * dk, device=DEV, generator=dev).bfloat16()
    at = [sum(lens[:i]) for i in range(B + 1)]
    cu = torch.tensor(at, dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(e - n, e) for n, e in zip(lens, ends)]).int().to(DEV)
    for chunks in (1, 3):
        got = fast.run(q, kc, vc, bt, cu, pos, B, split=True, chunks=chunks)
        for b in range(B):
            if lens[b] and (B < 60 or b % 9 == 0 or b > B - 4):
                own = slice(at[b], at[b + 1])
                alone = fast.run(q[own], kc, vc, bt[b:b + 1], torch.tensor([0, lens[b]], dtype=torch.int32, device=DEV), pos[own].contiguous(), 1,
                                 split=True, chunks=chunks)
                assert torch.equal(got[own], alone), (b, lens[b])


@pytest.mark.parametrize("nq,nkv,d,more", [(12, 2, 64, {"temp_coef": 0.4, "temp_every": 64, "slope_span": 8.0}), (4, 4, 64, {"window": 100}),
                                           (6, 2, 32, {"sink": True, "gated": True, "gate_heads": True, "out_scale": 0.7})])
@pytest.mark.parametrize("B,most", [(33, 4096), (64, 4096), (64, 130), (100, 4096), (257, 600)])
def test_single_tokens_of_many_requests_as_a_step_has_them(nq, nkv, d, more, B, most):
    # by whatever kernel and in as many pieces as the step's plan says, against the equations in 64 bits
    from types import SimpleNamespace
    from pico_vllm_amd.ops.attention_bias_fast import FastBiasAttention
    fast = FastBiasAttention(nq, nkv, d, d, d ** -0.5, **more)
    g = torch.Generator().manual_seed(B + nq)
    contexts = [1 + int(n) for n in torch.randint(0, min(most, 400), (B,), generator=g)]
    per, R = -(-max(contexts) // 16), nq // nkv
    bt = torch.randperm(B * per, generator=g).int().reshape(B, per)
    kc, vc = torch.randn(B * per, nkv, 16, d, generator=g).bfloat16(), torch.randn(B * per, nkv, d, 16, generator=g).bfloat16()
    q, gate, sinks = torch.randn(B, nq * d, generator=g).bfloat16(), torch.randn(B, nq, generator=g).bfloat16(), torch.randn(nq, generator=g)
    extra = fast.sink
    if extra:
        fast.sinks = sinks.to(DEV)
    cu, lens = torch.arange(B + 1, dtype=torch.int32), torch.tensor(contexts, dtype=torch.int32)
    ctx = SimpleNamespace(num_tokens=B, num_seqs=B, all_decode=True, max_context=most, host={"cu_seqlens": cu.numpy(), "context_lens": lens.numpy()}, shared={},
                          cu_seqlens=cu.to(DEV), positions=lens.to(DEV) - 1, context_lens=lens.to(DEV))
    got = fast(q.to(DEV), SimpleNamespace(k=kc.to(DEV), v=vc.to(DEV)), bt.to(DEV), ctx, gate=gate.to(DEV) if extra else None).double().cpu().view(B, nq, d)
    for b, n in enumerate(contexts):
        pages = bt[b, :-(-n // 16)].long()
        k = kc[pages].double().permute(1, 0, 2, 3).reshape(nkv, -1, d)[:, :n].repeat_interleave(R, 0)
        v = vc[pages].double().permute(1, 0, 3, 2).reshape(nkv, -1, d)[:, :n].repeat_interleave(R, 0)
        s = (k @ q[b].double().view(nq, d, 1))[..., 0] * d ** -0.5
        if "temp_every" in more:
            s = s * (1 + 0.4 * math.log(n // 64 + 1))
            s = s - 2.0 ** (-8.0 * torch.arange(1, nq + 1).double() / nq)[:, None] * (n - 1 - torch.arange(n).double())
        if fast.window:
            s[:, :max(0, n - fast.window)] = -math.inf
        p = torch.exp(s - s.amax(1, keepdim=True))
        total = p.sum(1, keepdim=True) + (torch.exp(sinks.double()[:, None] - s.amax(1, keepdim=True)) if extra else 0)
        want = ((p / total)[:, None] @ v)[:, 0]
        if extra:
            want = want * torch.sigmoid(gate[b].double())[:, None] * 0.7
        # probabilities and the output are rounded to bfloat16, and scores are float32 sums of products of bfloat16 numbers
        assert float((got[b] - want).abs().max()) <= 2.0 ** -7 * float(v.abs().max()), (b, n)
