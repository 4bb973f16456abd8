"""GPU tests of the decode calls' recent window on all three pages (k2b, RTN,
general): what lies past the window's length in its buffers reaches no output,
and rows given apart are stored whatever the query holds."""

import pytest
import torch

from bmx_amd import k2b, rtn, synth
from test_gpu_k2b_geom import _case_pages

pytestmark = pytest.mark.gpu
DEV = "cuda"
H, G, S = 2, 4, 256


def _page(kind, gen):
    """decode(q, k_tail, v_tail, **window arguments) over S committed tokens, and head_dim."""
    lens = torch.tensor([S], dtype=torch.int32, device=DEV)
    if kind == "rtn":
        codec = dict(k_bits=4, v_bits=4, k_group=32, v_group=64)
        k, v = (torch.randn(H, S, 128, generator=gen).half().to(DEV) for _ in range(2))
        pages = torch.zeros(S // 16, rtn.page_bytes(H, **codec), dtype=torch.uint8, device=DEV)
        ids = torch.arange(S // 16, dtype=torch.int32, device=DEV)
        rtn.append(k, v, pages, ids, **codec)
        return lambda q, kt, vt, **kw: rtn.decode(q, pages, ids[None], lens, S, 128 ** -0.5, k_tail=kt,
                                                  v_tail=vt, **codec, **kw), 128
    if kind == "k2b":
        d, consts = 128, k2b.CodecConsts.make()
        pool = synth.PagePool(S // 16, H, 16, DEV)
        seq = synth.encode_sequence(pool, synth.k2b_keys(H, S, 16, gen).to(DEV), synth.values(H, S, gen).to(DEV), 16,
                                    consts)
        geo = {}
    else:
        d, geo = 64, dict(group=32, k_bits=3)
        _, _, _, consts, pool, seq = _case_pages(gen, H, d, 16, 32, 3, S)
    table = synth.page_table([seq], device=DEV)
    return lambda q, kt, vt, **kw: k2b.decode(q, pool.pages, table, lens, S, seq.basis16, consts, d ** -0.5, rank=16,
                                              k_tail=kt, v_tail=vt, **geo, **kw), d


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("T,cap", [(1, 16), (17, 128), (100, 160)])
@pytest.mark.parametrize("kind", ["k2b", "rtn", "general"])
def test_rows_past_the_window_are_not_attended(kind, T, cap, on_device):
    gen = torch.Generator().manual_seed(T)
    decode, d = _page(kind, gen)
    kt, vt = (torch.randn(1, H, cap, d, generator=gen).half().to(DEV) for _ in range(2))
    q = torch.randn(1, H, G, d, generator=gen).to(DEV)
    n = torch.tensor([T], dtype=torch.int32, device=DEV) if on_device else T
    kt[:, :, T:], vt[:, :, T:] = 0, 0
    want = decode(q, kt, vt, tail_len=n, tail_cap=cap)
    assert torch.isfinite(want).all()
    for bad in (float("nan"), float("inf"), float("-inf")):
        kt[:, :, T:], vt[:, :, T:] = bad, bad
        assert torch.equal(decode(q, kt, vt, tail_len=n, tail_cap=cap), want)


@pytest.mark.parametrize("T,cap", [(1, 16), (17, 128), (150, 160)])
@pytest.mark.parametrize("kind", ["k2b", "rtn", "general"])
def test_rows_given_apart_are_stored_whatever_their_scores(kind, T, cap):
    """A query row that is not a number has no score above minus infinity; the later rows and calls need the window."""
    gen = torch.Generator().manual_seed(T)
    decode, d = _page(kind, gen)
    kt, vt = (torch.randn(1, H, cap, d, generator=gen).half().to(DEV) for _ in range(2))
    q = torch.randn(1, H, G, d, generator=gen).to(DEV)
    q[:, 0, 0] = float("nan")
    new = tuple(torch.randn(1, H, 1, d, generator=gen).half().to(DEV) for _ in range(2))
    out = decode(q, kt, vt, tail_len=T, tail_cap=cap, new_kv=new)
    assert torch.equal(kt[:, :, T - 1:T], new[0]) and torch.equal(vt[:, :, T - 1:T], new[1])
    want = decode(q, kt, vt, tail_len=T, tail_cap=cap)      # the same rows from the buffers
    assert torch.equal(out[0, 0, 1:], want[0, 0, 1:]) and torch.equal(out[0, 1], want[0, 1])
