"""GPU tests of the general page's decode precision, against float64 attention
over the pages' dequantized rows.  The RoPE frequencies are 0 (every rotation is
exactly the identity), so that nothing but the arithmetic of scores, weights and
sums is between the two."""

import pytest
import torch

from bmx_amd import k2b, synth

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pages(k, v, rank, group, bits):
    """The committed tokens' decode arguments, and their dense keys and values in float64."""
    h, S, d = k.shape
    c = k2b.CodecConsts.make(head_dim=d)
    consts = k2b.CodecConsts(c.codebook, c.sign_bits, (0.0,) * (d // 2), 1.0)
    pool = synth.PagePool(S // 16, h, rank, DEV, head_dim=d, group=group, k_bits=bits)
    seq = synth.encode_sequence(pool, k.to(DEV), v.float().to(DEV), rank, consts, svd=synth.first_page_svd(k, rank))
    K, V = k2b.dequant(pool.pages, torch.tensor(seq.page_ids, dtype=torch.int32, device=DEV), S, seq.basis16, consts,
                       h_kv=h, rank=rank, group=group, k_bits=bits)

    def decode(q, n=S, **kw):
        return k2b.decode(q[None], pool.pages, synth.page_table([seq], device=DEV),
                          torch.tensor([n], dtype=torch.int32, device=DEV), S, seq.basis16, consts, d ** -0.5,
                          rank=rank, group=group, k_bits=bits, **kw)[0].double()
    return decode, K.double(), V.double()


def test_key_parts_are_not_biased():
    """Packed scores of 500 to 1,000 (base 2) keep their place against window scores of the same size: the share of
    the packed tokens, read back from the output, gives the packed scores' relative error, here of 2,048 rows.
    Key parts rounded to nearest err to either side, as the fp32 sums do (deviation of a row 3e-7, of the mean 7e-9;
    the bound 2^-25 is four of them); parts cut towards zero take up to 2^-21 off every key."""
    h, G, d, n = 16, 16, 64, 128
    errs = []
    for seed in range(8):
        gen = torch.Generator().manual_seed(seed)
        k = torch.randn(h, 1, d, generator=gen).half().expand(h, n, d).contiguous()
        decode, K, V = _pages(k, torch.randn(h, n, d, generator=gen), 16, 32, 3)
        kt, vt = k.to(DEV)[None], torch.randn(1, h, n, d, generator=gen).half().to(DEV)
        size = torch.linspace(500, 1000, G, dtype=torch.float64, device=DEV)[None, :, None]
        q = (K[:, :1] / K[:, :1].square().sum(-1, keepdim=True) * d ** 0.5 / 1.4426950408889634 * size).float()
        out = decode(q, k_tail=kt, v_tail=vt, tail_len=n, tail_cap=n)
        s = torch.matmul(q.double(), torch.cat([K, kt[0].double()], 1).transpose(1, 2).contiguous()) * d ** -0.5

        def part(x, val):   # log of the part's weight, its mean value
            return torch.logsumexp(x, -1), torch.matmul(torch.softmax(x, -1), val)
        (lp, P), (lw, W) = part(s[..., :n], V), part(s[..., n:], vt[0].double())
        share = ((out - W) * (P - W)).sum(-1) / (P - W).square().sum(-1)
        assert share.min() > 0.02 and share.max() < 0.98
        errs.append((torch.logit(share) - (lp - lw)) / s[..., :n].mean(-1))
    err = torch.stack(errs)
    print(f"mean {err.mean().item():.2e}, deviation {err.std().item():.2e}", flush=True)
    assert abs(err.mean().item()) <= 2 ** -25


@pytest.mark.parametrize("S,split", [(2048, 0), (4096, 4096)])     # few pages a wave; all of them on one workgroup
@pytest.mark.parametrize("d,rank,G", [(64, 16, 4), (128, 64, 1), (32, 32, 16)])
@pytest.mark.parametrize("norm,sink_norm,gap", [
    (8.0, 8.0, 0), (0.1, 0.1, 0), (1e-2, 1e-2, 0), (1e-4, 1e-4, 0),      # norms of all tokens, no sink
    (0.16, 0.16, 11), (1e-2, 1e-2, 13), (1e-4, 1e-4, 11),                # all tokens gap nats below the first
    (8.0, 1e-2, 11), (8.0, 0.0, 13), (1e-2, 100.0, 11), (1e-2, 100.0, -11),
])
def test_value_product(norm, sink_norm, gap, d, rank, G, S, split):
    """The output against float64 where values are small, or where the first token's score stands gap nats above (or
    below) the others, with a norm of its own.  An operand keeps 2^-22 of itself, a score of up to 30 (base 2) the
    roundings of its fp32 sum, 4 of 2^-20, and with it the weight (times ln 2): 2.7e-6; the fp32 sums of 4,096 terms,
    largest first or last, 2^-24 times 64 at most in the mean: 3.8e-6.  Together below 8e-6."""
    h = 3
    gen = torch.Generator().manual_seed(S + d)
    v = torch.randn(h, S, d, generator=gen) * norm / d ** 0.5
    v[:, 0] *= sink_norm / norm
    decode, K, V = _pages(synth.k2b_keys(h, S, rank, gen, head_dim=d), v, rank, 32, 3)
    q = torch.randn(h, G, d, generator=gen).to(DEV)
    q = (q + K[:, :1] / K[:, :1].square().sum(-1, keepdim=True) * gap * d ** 0.5).float().contiguous()
    out = decode(q, split_tokens=split)
    s = torch.matmul(q.double(), K.transpose(1, 2).contiguous()) * d ** -0.5
    ref = torch.matmul(torch.softmax(s, -1), V)
    err = ((out - ref).norm() / ref.norm()).item()
    print(f"error {err:.2e}", flush=True)
    assert err <= 8e-6


@pytest.mark.parametrize("size", [1.0, 2.0 ** -12, 2.0 ** 9])     # of the window's keys; the query is 1 / size
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,rank,G", [(64, 16, 4), (128, 64, 1), (32, 32, 16)])
def test_window_scores(d, rank, G, dtype, size):
    """Window scores carry the fp32 query: a window alone against float64, scores of up to 30 (base 2), the query far
    below and above 1 and its elements over 2^10 (the bound is test_value_product's, for the same kind of sums)."""
    h, T = 3, 100
    gen = torch.Generator().manual_seed(d)
    decode, _, _ = _pages(synth.k2b_keys(h, 128, rank, gen, head_dim=d), torch.randn(h, 128, d, generator=gen), rank,
                          32, 3)
    ramp = torch.logspace(-5, 5, d, base=2.0)
    kt = (torch.randn(1, h, T, d, generator=gen) / ramp * size).to(dtype).to(DEV)
    vt = torch.randn(1, h, T, d, generator=gen).to(dtype).to(DEV)
    q = (torch.randn(h, G, d, generator=gen) * ramp / size * 5).to(DEV)
    out = decode(q, n=0, k_tail=kt, v_tail=vt, tail_len=T, tail_cap=T)
    s = torch.matmul(q.double(), kt[0].double().transpose(1, 2).contiguous()) * d ** -0.5
    ref = torch.matmul(torch.softmax(s, -1), vt[0].double())
    err = ((out - ref).norm() / ref.norm()).item()
    print(f"error {err:.2e}, scores to {s.abs().max().item() * 1.4427:.0f}", flush=True)
    assert err <= 8e-6


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_window_key_of_minus_infinite_score(dtype):
    """A window row whose key is infinite, at a score of minus infinity for every query, has no weight."""
    h, d, rank, G, T = 2, 64, 16, 4, 20
    gen = torch.Generator().manual_seed(2)
    decode, _, _ = _pages(synth.k2b_keys(h, 128, rank, gen, head_dim=d), torch.randn(h, 128, d, generator=gen), rank,
                          32, 3)
    kt, vt = (torch.randn(1, h, T, d, generator=gen).to(dtype).to(DEV) for _ in range(2))
    q = torch.randn(h, G, d, generator=gen).to(DEV)
    q[..., 5] = -1 - q[..., 5].abs()
    kt[:, :, 7, 5] = float("inf")
    out = decode(q, k_tail=kt, v_tail=vt, tail_len=T, tail_cap=T)
    keep = [t for t in range(T) if t != 7]
    want = decode(q, k_tail=kt[:, :, keep].contiguous(), v_tail=vt[:, :, keep].contiguous(), tail_len=T - 1,
                  tail_cap=T - 1)
    assert torch.isfinite(want).all() and (out - want).abs().max().item() <= 2e-6
