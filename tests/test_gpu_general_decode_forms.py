"""GPU tests of the general page's decode at the forms that take their own
branch: head counts that give a head several waves or a call several head
blocks, every compaction width, residual groups inside and across a wave's 4
pages, ranges longer than the RoPE tables and than the page-id window, a basis
that is not 16-byte aligned, a codebook with no affine fp16 image, and a batch
whose workspace is served in parts.

Bar: 2-norm error 1e-3.  The rotation tables are fp16 as the oracle's; an entry
next to a rounding boundary may round the other way (2^-11 of it, in about one
of 200), the other differences are below 1e-5."""

import pytest
import torch

from bmx_amd import k2b, synth
from test_gpu_k2b_geom import _attention_ref, _case_pages, _oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rel(out, ref):
    return ((out - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("h,d,rank,group,bits,G,S,T,split", [
    (1, 64, 16, 16, 3, 16, 2048, 33, 0),       # 8 waves of one head, 16 columns
    (3, 32, 32, 128, 4, 5, 1152, 7, 0),        # two waves a head, a group of two quads
    (12, 64, 16, 32, 3, 2, 640, 20, 0),        # two head blocks
    (5, 128, 16, 16, 2, 8, 512, 0, 0),         # 4-wave workgroups, two head blocks
    (2, 64, 32, 64, 3, 4, 4096, 16, 4096),     # one workgroup: 64 quads, 16 table sets, 4 id windows
    (1, 128, 128, 128, 3, 1, 2048, 130, 1024),
    (8, 32, 64, 64, 4, 7, 256, 4, 64),
])
def test_decode_forms(h, d, rank, group, bits, G, S, T, split):
    gen = torch.Generator().manual_seed(h + d + rank + group)
    k_pre, v, svd, consts, pool, seq = _case_pages(gen, h, d, rank, group, bits, S)
    kt = vt = None
    if T:
        kt = synth.rope_keys(synth.k2b_keys(h, T, rank, gen, head_dim=d), S, consts).unsqueeze(0).to(DEV)
        vt = synth.values(h, T, gen, head_dim=d).unsqueeze(0).to(DEV)
    q = torch.randn(1, h, G, d, generator=gen).to(DEV)
    cache = _oracle(k_pre, v, svd, consts, h, d, rank, group, bits, 0, S)
    ref = _attention_ref(q[0].cpu().reshape(h * G, 1, d), cache, consts, kt[0].cpu() if T else None,
                         vt[0].cpu() if T else None, G, d).reshape(1, h, G, d)
    odd = torch.zeros(seq.basis16.numel() + 1, dtype=torch.float16, device=DEV)
    odd[1:] = seq.basis16.reshape(-1)
    for basis in (seq.basis16, odd[1:].view_as(seq.basis16)):
        out = k2b.decode(q, pool.pages, synth.page_table([seq], device=DEV),
                         torch.tensor([S], dtype=torch.int32, device=DEV), S, basis, consts, d ** -0.5, rank=rank,
                         k_tail=kt, v_tail=vt, tail_len=T, tail_cap=T, group=group, k_bits=bits, split_tokens=split)
        assert _rel(out.cpu(), ref) <= 1e-3


def test_decode_of_a_shorter_sequence_than_the_bound():
    """packed_len below max_packed_len, down to none: the rest of the table is not attended to."""
    h, d, rank, group, bits, G = 2, 64, 16, 32, 3, 4
    gen = torch.Generator().manual_seed(5)
    k_pre, v, svd, consts, pool, seq = _case_pages(gen, h, d, rank, group, bits, 1024)
    q = torch.randn(1, h, G, d, generator=gen).to(DEV)
    table = synth.page_table([seq], device=DEV)
    for S in (1024, 896, 128, 0):
        out = k2b.decode(q, pool.pages, table, torch.tensor([S], dtype=torch.int32, device=DEV), 1024, seq.basis16,
                         consts, d ** -0.5, rank=rank, group=group, k_bits=bits)
        if S == 0:
            assert not out.any()
            continue
        cache = _oracle(k_pre, v, svd, consts, h, d, rank, group, bits, 0, S)
        ref = _attention_ref(q[0].cpu().reshape(h * G, 1, d), cache, consts, None, None, G, d).reshape(1, h, G, d)
        assert _rel(out.cpu(), ref) <= 1e-3


def test_decode_any_codebook():
    """Levels that are no affine image of fp16 numbers, in any order."""
    h, d, rank, group, bits, G, S = 2, 64, 16, 32, 3, 4, 512
    gen = torch.Generator().manual_seed(6)
    k_pre, v, svd, consts, pool, seq = _case_pages(gen, h, d, rank, group, bits, S)
    levels = (0.8137, -1.6180339, 0.1234567, 2.7182818)
    other = k2b.CodecConsts(levels, consts.sign_bits, consts.inv_freq, consts.rope_scaling)
    cache = _oracle(k_pre, v, svd, consts, h, d, rank, group, bits, 0, S)
    V = cache.dense_v()
    # values of the same codes with the other levels, through the dequant kernel's fp32 output
    _, V2 = k2b.dequant(pool.pages, torch.tensor(seq.page_ids, dtype=torch.int32, device=DEV), S, seq.basis16, other,
                        h_kv=h, rank=rank, dtype=torch.float32, group=group, k_bits=bits)
    q = torch.randn(1, h, G, d, generator=gen).to(DEV)
    out = k2b.decode(q, pool.pages, synth.page_table([seq], device=DEV),
                     torch.tensor([S], dtype=torch.int32, device=DEV), S, seq.basis16, other, d ** -0.5, rank=rank,
                     group=group, k_bits=bits)
    cache.dense_v = lambda: V2.cpu().reshape(V.shape)
    ref = _attention_ref(q[0].cpu().reshape(h * G, 1, d), cache, consts, None, None, G, d).reshape(1, h, G, d)
    assert _rel(out.cpu(), ref) <= 1e-3


def test_decode_batch_served_in_parts():
    """64 sequences with 4096-row window buffers: the workspace of the call stays below 24 MiB and every sequence
    equals the same sequence alone (to fp32 summation: the splits differ)."""
    h, d, rank, group, bits, G, B, S, T = 8, 32, 16, 32, 3, 4, 64, 128, 5
    gen = torch.Generator().manual_seed(7)
    _, _, _, consts, pool, seq = _case_pages(gen, h, d, rank, group, bits, S * 4)
    pages = torch.tensor(seq.page_ids, dtype=torch.int32)
    table = torch.stack([pages.roll(-8 * (b % 4))[:8] for b in range(B)]).contiguous().to(DEV)
    kt = torch.zeros(B, h, 4096, d, dtype=torch.float16, device=DEV)
    vt = torch.zeros_like(kt)
    kt[:, :, :T] = torch.randn(B, h, T, d, generator=gen).half().to(DEV)
    vt[:, :, :T] = torch.randn(B, h, T, d, generator=gen).half().to(DEV)
    q = torch.randn(B, h, G, d, generator=gen).to(DEV)
    lens = torch.full((B,), S, dtype=torch.int32, device=DEV)
    lens[3::7] = 0
    ws = k2b.DecodeWorkspace()
    kw = dict(rank=rank, tail_cap=4096, group=group, k_bits=bits, workspace=ws)
    new = (torch.randn(B, h, 1, d, generator=gen).half().to(DEV), torch.randn(B, h, 1, d, generator=gen).half().to(DEV))
    one_k, one_v = kt.clone(), vt.clone()
    out = k2b.decode(q, pool.pages, table, lens, S, seq.basis16, consts, d ** -0.5, k_tail=kt, v_tail=vt, tail_len=T,
                     new_kv=new, **kw)
    assert ws.buf.numel() <= 24 << 20
    assert torch.equal(kt[:, :, T - 1:T], new[0]) and torch.equal(vt[:, :, T - 1:T], new[1])
    for b in (0, 3, 31, 32, 33, 63):
        s = slice(b, b + 1)
        alone = k2b.decode(q[s], pool.pages, table[s], lens[s], S, seq.basis16, consts, d ** -0.5, k_tail=one_k[s],
                           v_tail=one_v[s], tail_len=T, new_kv=(new[0][s], new[1][s]), **kw)
        assert (out[s] - alone).abs().max().item() <= 2e-6


def test_decode_with_more_splits_than_the_workspace_holds():
    """256 splits of 16 heads x 16 queries with room for 157: the call without split_tokens, to fp32 summation."""
    h, d, rank, group, bits, G, S, cap = 16, 128, 16, 16, 2, 16, 16384, 4096
    gen = torch.Generator().manual_seed(9)
    consts = k2b.CodecConsts.make(head_dim=d)
    pages = torch.randint(0, 256, (S // 16, k2b.page_bytes(h, rank, head_dim=d, group=group, k_bits=bits)),
                          generator=gen, dtype=torch.uint8).to(DEV)
    k = torch.randn(h, S, d, generator=gen).half().to(DEV)
    basis = torch.linalg.qr(torch.randn(h * d, rank, generator=gen))[0].contiguous().to(DEV)
    ids = torch.arange(S // 16, dtype=torch.int32, device=DEV)
    k2b.append(k, k.flip(1), basis, basis.half(), pages, ids, consts, rank=rank, group=group, k_bits=bits)
    kt, vt = (torch.randn(1, h, cap, d, generator=gen).half().to(DEV) for _ in range(2))
    q = torch.randn(1, h, G, d, generator=gen).to(DEV)
    ws = k2b.DecodeWorkspace()
    outs = [k2b.decode(q, pages, ids[None], torch.tensor([S], dtype=torch.int32, device=DEV), S, basis.half(), consts,
                       d ** -0.5, rank=rank, k_tail=kt, v_tail=vt, tail_len=77, tail_cap=cap, group=group, k_bits=bits,
                       split_tokens=st, workspace=ws) for st in (0, 64)]
    assert ws.buf.numel() <= 24 << 20
    assert (outs[0] - outs[1]).abs().max().item() <= 2e-6


@pytest.mark.parametrize("T", [0, 64, 65, 200])      # a window wave's pass is 64 rows
@pytest.mark.parametrize("S,cap", [(256, 200), (4096, 255)])
def test_decode_batch_of_many_rows(S, T, cap):
    """40 sequences of 8 heads and 4 queries (more merge workgroups than the chip holds at a time): every sequence
    equals the same sequence alone, to fp32 summation."""
    h, d, rank, group, bits, G, B = 8, 32, 16, 32, 3, 4, 40
    gen = torch.Generator().manual_seed(8)
    _, _, _, consts, pool, seq = _case_pages(gen, h, d, rank, group, bits, S)
    table = synth.page_table([seq] * B, device=DEV)
    kt, vt = (torch.randn(B, h, cap, d, generator=gen).half().to(DEV) for _ in range(2))
    q = torch.randn(B, h, G, d, generator=gen).to(DEV)
    lens = torch.full((B,), S, dtype=torch.int32, device=DEV)
    lens[1::3] -= 128
    kw = dict(rank=rank, tail_cap=cap, group=group, k_bits=bits, tail_len=T)
    out = k2b.decode(q, pool.pages, table, lens, S, seq.basis16, consts, d ** -0.5, k_tail=kt, v_tail=vt, **kw)
    for b in (0, 1, 20, 39):
        s = slice(b, b + 1)
        alone = k2b.decode(q[s], pool.pages, table[s], lens[s], S, seq.basis16, consts, d ** -0.5, k_tail=kt[s],
                           v_tail=vt[s], **kw)
        assert (out[s] - alone).abs().max().item() <= 2e-6
