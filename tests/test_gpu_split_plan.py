"""GPU tests of the decode grid (k2b and RTN): heads spread over several
workgroups and the window on workgroups of its own give what the plain grid
gives, bit for bit (the same 64-token splits and the same merge), and a bound
call holds at any window length."""

import pytest
import torch

from bmx_amd import k2b, rtn, synth

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _window(gen, h, T, dtype):
    return tuple(torch.randn(1, h, T, 128, generator=gen).to(dtype).to(DEV) for _ in range(2))


# (h_kv, G, tokens, window, dtype): blocks of 1, 2 and 4 heads; room for the window's workgroups or not
GRID = [(8, 4, 256, 60, torch.float16), (8, 4, 2048, 128, torch.bfloat16), (3, 16, 640, 17, torch.float32),
        (8, 1, 4096, 1, torch.float16), (5, 8, 8192, 255, torch.bfloat16), (8, 4, 16256, 128, torch.float32),
        (1, 2, 384, 31, torch.float16)]


@pytest.mark.parametrize("h,G,S,T,dtype", GRID)
def test_k2b_grid_equals_plain_splits(h, G, S, T, dtype):
    gen = torch.Generator().manual_seed(h * 100 + G)
    wdt = torch.bfloat16 if dtype == torch.bfloat16 else torch.float16
    consts = k2b.CodecConsts.make()
    k_pre, v = synth.k2b_keys(h, S, 16, gen), synth.values(h, S, gen)
    pool = synth.PagePool(S // 16, h, 16, DEV, gen=gen)
    seq = synth.encode_sequence(pool, k_pre.to(DEV), v.to(DEV), 16, consts)
    kt, vt = _window(gen, h, T, wdt)
    q = torch.randn(1, h, G, 128, generator=gen).to(dtype).to(DEV)
    ln = torch.tensor([S], dtype=torch.int32, device=DEV)
    outs = [k2b.decode(q, pool.pages, synth.page_table([seq], device=DEV), ln, S, seq.basis16, consts, 128 ** -0.5,
                       rank=16, k_tail=kt, v_tail=vt, tail_len=T, tail_cap=T, split_tokens=st) for st in (0, 64)]
    if S // 64 >= (T + 15) // 16:   # else the plain grid has more (empty) splits
        assert torch.equal(*outs)
    else:
        assert (outs[0].float() - outs[1].float()).abs().max().item() <= 2 ** -8 * outs[1].float().abs().max().item()


@pytest.mark.parametrize("h,G,S,T,dtype", GRID)
def test_rtn_grid_equals_plain_splits(h, G, S, T, dtype):
    gen = torch.Generator().manual_seed(h * 100 + G)
    wdt = torch.bfloat16 if dtype == torch.bfloat16 else torch.float16
    codec = dict(k_bits=4, v_bits=4, k_group=32, v_group=64)
    k, v = (torch.randn(h, S, 128, generator=gen).half().to(DEV) for _ in range(2))
    pages = torch.zeros(S // 16, rtn.page_bytes(h, **codec), dtype=torch.uint8, device=DEV)
    ids = torch.arange(S // 16, dtype=torch.int32, device=DEV)
    rtn.append(k, v, pages, ids, **codec)
    kt, vt = _window(gen, h, T, wdt)
    q = torch.randn(1, h, G, 128, generator=gen).to(dtype).to(DEV)
    ln = torch.tensor([S], dtype=torch.int32, device=DEV)
    outs = [rtn.decode(q, pages, ids[None], ln, S, 128 ** -0.5, k_tail=kt, v_tail=vt, tail_len=T, tail_cap=T,
                       split_tokens=st, **codec) for st in (0, 64)]
    if S // 64 >= (T + 15) // 16:
        assert torch.equal(*outs)
    else:
        assert (outs[0].float() - outs[1].float()).abs().max().item() <= 2 ** -8 * outs[1].float().abs().max().item()


@pytest.mark.parametrize("S", [0, 128, 2048, 16256])
def test_bound_call_at_any_window_length(S):
    """A plan bound with a short window runs with every length up to its buffers' rows."""
    h, G, cap = 8, 4, 288
    gen = torch.Generator().manual_seed(S)
    consts = k2b.CodecConsts.make()
    n = max(S, 128)
    pool = synth.PagePool(n // 16, h, 16, DEV)
    seq = synth.encode_sequence(pool, synth.k2b_keys(h, n, 16, gen).to(DEV), synth.values(h, n, gen).to(DEV), 16,
                                consts)
    kt, vt = _window(gen, h, cap, torch.float16)
    q = torch.randn(1, h, G, 128, generator=gen).half().to(DEV)
    ln = torch.tensor([S], dtype=torch.int32, device=DEV)
    kw = dict(rank=16, k_tail=kt, v_tail=vt, tail_cap=cap)
    plan = k2b.DecodePlan(q, pool.pages, None, ln, S, seq.basis16, consts, 128 ** -0.5, tail_len=1, **kw)
    for T in (1, 15, 16, 17, 128, 255, 288):
        new = (kt[:, :, T - 1:T].clone(), vt[:, :, T - 1:T].clone())
        got = plan.run(tail_len=T, new_kv=new).clone()
        want = k2b.decode(q, pool.pages, None, ln, S, seq.basis16, consts, 128 ** -0.5, tail_len=T, **kw)
        assert torch.equal(got, want)


@pytest.mark.parametrize("B,h,S,T,on_device", [(3, 8, 640, 16, False), (3, 2, 2688, 16, True), (5, 8, 384, 5, True),
                                               (7, 4, 512, 17, True)])
def test_rtn_batch_of_spread_heads(B, h, S, T, on_device):
    """Batches that do not divide the CUs, whose heads the plan may spread: the plain grid's outputs, bit for bit, with
    lengths and windows shorter than their bounds."""
    gen = torch.Generator().manual_seed(B)
    codec = dict(k_bits=4, v_bits=4, k_group=32, v_group=64)
    k, v = (torch.randn(h, S, 128, generator=gen).half().to(DEV) for _ in range(2))
    pages = torch.zeros(S // 16, rtn.page_bytes(h, **codec), dtype=torch.uint8, device=DEV)
    ids = torch.arange(S // 16, dtype=torch.int32, device=DEV)
    rtn.append(k, v, pages, ids, **codec)
    kt, vt = (torch.randn(B, h, T, 128, generator=gen).half().to(DEV) for _ in range(2))
    q = torch.randn(B, h, 4, 128, generator=gen).to(DEV)
    ln = torch.tensor([S - 128 * (b % 3) for b in range(B)], dtype=torch.int32, device=DEV)
    n = torch.tensor([T - b % 3 for b in range(B)], dtype=torch.int32, device=DEV) if on_device else T - 1
    outs = [rtn.decode(q, pages, ids.repeat(B, 1), ln, S, 128 ** -0.5, k_tail=kt, v_tail=vt, tail_len=n, tail_cap=T,
                       split_tokens=st, **codec) for st in (0, 64)]
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)


@pytest.mark.parametrize("T", [48, 49, 300])    # 8 heads x 3, 4 or 19 tiles over 3 splits: 24 pairs is the line
@pytest.mark.parametrize("page", ["k2b", "rtn"])
def test_windows_of_more_pairs_than_the_first_waves_take(page, T):
    """72 sequences (3 splits each) score their windows behind the groups, on 4 waves or on all 8: each sequence's
    output is that of the sequence alone (other splits; fp16 partial records)."""
    B, h, G, S = 72, 8, 2, 256
    gen = torch.Generator().manual_seed(T)
    kt, vt = (torch.randn(B, h, T, 128, generator=gen).half().to(DEV) for _ in range(2))
    q = torch.randn(B, h, G, 128, generator=gen).to(DEV)
    ln = torch.full((B,), S, dtype=torch.int32, device=DEV)
    if page == "k2b":
        consts = k2b.CodecConsts.make()
        pool = synth.PagePool(S // 16, h, 16, DEV)
        seq = synth.encode_sequence(pool, synth.k2b_keys(h, S, 16, gen).to(DEV), synth.values(h, S, gen).to(DEV), 16,
                                    consts)

        def decode(s):
            return k2b.decode(q[s], pool.pages, synth.page_table([seq] * len(q[s]), device=DEV), ln[s], S, seq.basis16,
                              consts, 128 ** -0.5, rank=16, k_tail=kt[s], v_tail=vt[s], tail_len=T, tail_cap=T)
    else:
        codec = dict(k_bits=4, v_bits=4, k_group=32, v_group=64)
        k, v = (torch.randn(h, S, 128, generator=gen).half().to(DEV) for _ in range(2))
        pages = torch.zeros(S // 16, rtn.page_bytes(h, **codec), dtype=torch.uint8, device=DEV)
        ids = torch.arange(S // 16, dtype=torch.int32, device=DEV)
        rtn.append(k, v, pages, ids, **codec)

        def decode(s):
            return rtn.decode(q[s], pages, ids.repeat(len(q[s]), 1), ln[s], S, 128 ** -0.5, k_tail=kt[s], v_tail=vt[s],
                              tail_len=T, tail_cap=T, **codec)
    out = decode(slice(0, B))
    for b in (0, 35, 71):
        alone = decode(slice(b, b + 1))[0]
        assert (out[b] - alone).abs().max().item() <= 2 ** -10 * alone.abs().max().item()
