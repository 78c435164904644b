"""Prompt portions of attention through a latent with the heads' own keys and values, against the equations in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# q (turned), k, v, the probabilities and the output are rounded to bfloat16: each 2^-9 / sqrt 3 of its size in the mean, the scores'
# two (of scores about 1) in the exponent: 2.5e-3 together, and twice that
TOL = 5e-3


def inputs(H, d, r, dv, C, seqs, P=16, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)

    def rn(*s):
        return torch.randn(*s, device=DEV, generator=g)
    pages = [-(-(c + n) // P) for c, n in seqs]
    bt = torch.full((len(seqs), max(pages)), -1, dtype=torch.int32, device=DEV)
    order, at = torch.randperm(sum(pages) + 2, device=DEV, generator=g).int(), 0
    for b, k in enumerate(pages):
        bt[b, :k] = order[at:at + k]
        at += k
    T = sum(n for _, n in seqs)
    k_cache = rn(sum(pages) + 2, 1, P, C + r).bfloat16()
    angles = torch.rand(T, r // 2, device=DEV, generator=g) * 6.28
    starts = torch.tensor([0] + [n for _, n in seqs]).cumsum(0)
    return dict(q=rn(T, H * (d + r) + 4).bfloat16(), table=torch.stack([angles.cos(), angles.sin()], -1).contiguous(), k_cache=k_cache,
                v_cache=k_cache[..., :C].transpose(2, 3).contiguous(), uk=(rn(H * d, C) * C ** -0.5).bfloat16(),
                uv=(rn(H * dv, C) * C ** -0.5).bfloat16(), gate=rn(T, H).bfloat16(), bt=bt, cu=starts.int().to(DEV),
                ctx=torch.tensor([c + n for c, n in seqs], dtype=torch.int32, device=DEV))


def exact(x, H, d, r, dv, C, seqs, P=16):
    q = x["q"][:, :H * (d + r)].double().view(-1, H, d + r)
    u, v, c, s = q[..., d::2], q[..., d + 1::2], x["table"][:, None, :, 0].double(), x["table"][:, None, :, 1].double()
    q = torch.cat([q[..., :d], torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)], -1)
    out, t = [], 0
    for b, (cached, n) in enumerate(seqs):
        L = cached + n
        rows = x["k_cache"][x["bt"][b, :-(-L // P)].long(), 0].reshape(-1, C + r)[:L].double()
        seen = torch.arange(L, device=DEV)[None] <= torch.arange(cached, L, device=DEV)[:, None]
        for h in range(H):
            k = torch.cat([rows[:, :C] @ x["uk"][h * d:(h + 1) * d].double().T, rows[:, C:]], 1)
            val = rows[:, :C] @ x["uv"][h * dv:(h + 1) * dv].double().T
            w = torch.softmax((q[t:t + n, h] @ k.T * (d + r) ** -0.5).masked_fill(~seen, float("-inf")), -1)
            out.append(torch.sigmoid(x["gate"][t:t + n, h:h + 1].double()) * (w @ val))
        t += n
    at, rows = 0, []
    for _, n in seqs:
        rows.append(torch.cat(out[at:at + H], 1))
        at += H
    return torch.cat(rows)


def served(x, H, d, r, dv, C, seqs, lead=0, slots=None):
    from pico_vllm_amd.ops import latent_prompt
    p = latent_prompt.LatentPrompt(H, d, r, dv, C, (d + r) ** -0.5, x["uk"], x["uv"])
    p.slots = slots or p.slots
    room = sum(-(-(c + n) // 64) for c, n in seqs[lead:])
    T = x["q"].shape[0]
    out = torch.full((T, H * dv), 7.0, dtype=torch.bfloat16, device=DEV)
    p.run(x["q"], x["table"], x["k_cache"], x["v_cache"], x["bt"][lead:], x["cu"][lead:], x["ctx"][lead:], len(seqs) - lead,
          sum(n for _, n in seqs[:lead]), room, out, x["gate"])
    return out


SIZES = [(12, 128, 64, 128, 256), (3, 64, 32, 64, 128), (5, 32, 64, 32, 96), (2, 64, 128, 128, 32)]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("seqs", [
    [(0, 2)], [(0, 64)], [(0, 129)], [(100, 128)], [(63, 127), (1, 1), (0, 65), (700, 30)], [(2000, 300)],
    [(5, 3)] * 70, [(0, 700), (0, 40), (1200, 33)]])
def test_against_the_equations(sizes, seqs):
    # tiles of queries and keys that are full, one more and one less; a piece of keys that ends inside a tile, covers several tiles and
    # several sequences; more sequences than lanes
    x = inputs(*sizes, seqs)
    want, got = exact(x, *sizes, seqs), served(x, *sizes, seqs)
    assert (got.double() - want).norm() <= TOL * want.norm()
    assert torch.equal(got, served(x, *sizes, seqs))


@pytest.mark.parametrize("slots", [1, 2, 7])
def test_pieces_of_any_length(slots):
    sizes, seqs = SIZES[1], [(300, 200), (0, 500), (1000, 2)]
    x = inputs(*sizes, seqs)
    want, got = exact(x, *sizes, seqs), served(x, *sizes, seqs, slots=slots)
    assert (got.double() - want).norm() <= TOL * want.norm()


@pytest.mark.parametrize("P", [8, 64])
def test_rows_in_front_and_pages(P):
    sizes, seqs = SIZES[1], [(40, 1), (90, 1), (0, 1), (17, 150), (0, 70)]
    x = inputs(*sizes, seqs, P=P)
    want, got = exact(x, *sizes, seqs, P=P), served(x, *sizes, seqs, lead=3)
    assert (got[:3] == 7.0).all()                     # single tokens are served elsewhere
    assert (got[3:].double() - want[3:]).norm() <= TOL * want[3:].norm()


@pytest.mark.parametrize("odd", [float("nan"), float("inf")])
def test_a_value_that_is_not_finite_reaches_its_readers_alone(odd):
    sizes, seqs, P = SIZES[0], [(70, 200), (0, 90)], 16
    H, d, r, dv, C = sizes
    x = inputs(*sizes, seqs)
    plain = served(x, *sizes, seqs)
    at = 70 + 133                                     # a token in the middle of a tile: those in front of it do not see it
    x["k_cache"][x["bt"][0, at // P].long(), 0, at % P, 3] = odd
    got = served(x, *sizes, seqs)
    assert torch.equal(got[:133], plain[:133]) and torch.equal(got[200:], plain[200:])
    assert not torch.isfinite(got[133:200]).any()


def test_single_tokens_beside_portions_through_the_layer():
    # the layer's two ways in one step, against the step whose portions are served in the latent's space like the single tokens
    from types import SimpleNamespace
    from pico_vllm_amd.parts.latent_attention import LatentAttention
    H, d, r, dv, C = sizes = SIZES[0]
    seqs = [(40, 1), (333, 1), (0, 130), (500, 20)]
    x = inputs(*sizes, seqs)
    T, D = x["q"].shape[0], 256
    g = torch.Generator(device=DEV).manual_seed(5)

    def rn(*s):
        return (torch.randn(*s, device=DEV, generator=g) * s[-1] ** -0.5).bfloat16()
    layer = LatentAttention(D, H, d, r, dv, 0, C, (d + r) ** -0.5, 10000.0, gate_heads=True)
    layer.load({"q": rn(H * (d + r), D), "g": rn(H, D), "dkv": rn(C + r, D), "dkv.norm": torch.ones(C, device=DEV), "uk": x["uk"], "uv": x["uv"],
                "o": rn(D, H * dv)}, torch.device(DEV), torch.bfloat16)
    pos = torch.cat([torch.arange(c, c + n) for c, n in seqs])
    seq = torch.cat([torch.full((n,), b) for b, (_, n) in enumerate(seqs)])
    bt = x["bt"].cpu()
    slots = bt[seq, pos // 16] * 16 + pos % 16
    layer.position.table = lambda ctx: x["table"]
    a = (torch.randn(T, D, device=DEV, generator=g)).bfloat16()

    def run(prompt):
        ctx = SimpleNamespace(num_tokens=T, num_seqs=len(seqs), all_decode=False, shared={}, host={"cu_seqlens": x["cu"].cpu().numpy(), "context_lens": x["ctx"].cpu().numpy()},
                              cu_seqlens=x["cu"], context_lens=x["ctx"], positions=pos.int().to(DEV), token_seq=seq.int().to(DEV), block_tables=[x["bt"]],
                              slot_mapping=[slots.int().to(DEV)], max_context=600)
        cache = SimpleNamespace(group=0, k=x["k_cache"].clone(), v=x["v_cache"].clone())
        layer.prompt, kept = (layer.prompt if prompt else None), layer.prompt
        assert not prompt or layer.prompt.plan(ctx)[0] == 2
        out = layer.attend(a, ctx, cache)
        layer.prompt = kept
        return out
    new, old = run(True), run(False)
    assert (new[:2].float() - old[:2].float()).norm() <= TOL * old[:2].float().norm()
    assert (new.float() - old.float()).norm() <= 2 * TOL * old.float().norm()


def test_matrices_of_the_heads_that_start_anywhere():
    # a checkpoint's tensors may be views on the GPU: those that start on no 16 bytes are copied once
    sizes, seqs = SIZES[1], [(40, 70)]
    x = inputs(*sizes, seqs)
    want = served(x, *sizes, seqs)
    for name in ("uk", "uv"):
        odd = torch.empty(x[name].numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view(x[name].shape)
        x[name] = odd.copy_(x[name])
    assert torch.equal(served(x, *sizes, seqs), want)
