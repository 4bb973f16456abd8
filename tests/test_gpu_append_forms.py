"""GPU tests of the k2b write kernels at the forms that take their own branch:
every (rank, tokens per thread) instance of the residual kernel on the general
page, key rows that are not 16-byte aligned, value rows outside the range of the
short division, and each value dtype and head_dim.  Codes are compared bit for
bit with the oracle (inputs whose fp32 sums are exact in any order)."""

import numpy as np
import pytest
import torch

from bmx_amd import k2b
from oracle import codecs as OC
from oracle import layout as OL

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _encode(k_pre, v, V, us0, consts, *, h, d, rank, group, bits, via=None):
    """Pages of two codec pages; via(t) re-lays an input out before the call."""
    via = via or (lambda t: t)
    pb = k2b.page_bytes(h, rank, head_dim=d, group=group, k_bits=bits)
    pages = torch.zeros(k_pre.shape[1] // 16, pb, dtype=torch.uint8, device=DEV)
    ids = torch.arange(pages.shape[0], dtype=torch.int32, device=DEV)
    k2b.append(via(k_pre.to(DEV)), via(v.to(DEV)), V.to(DEV), V.to(DEV).half(), pages, ids, consts, rank=rank,
               us_first=us0.to(DEV), group=group, k_bits=bits)
    return pages.cpu().numpy()


def _odd_rows(t):
    """The same values in rows of an odd stride that start 2 (fp16) bytes off 16-byte alignment."""
    buf = torch.zeros(t.shape[0], t.shape[1], t.shape[2] + 3, dtype=t.dtype, device=t.device)
    buf[:, :, 1:1 + t.shape[2]] = t
    return buf[:, :, 1:1 + t.shape[2]]


# (h, d, rank, group, bits): tokens per thread group * d / 512 = 1, 2, 4, 8, 16, 32 with each rank
@pytest.mark.parametrize("h,d,rank,group,bits", [
    (1, 32, 16, 16, 2), (3, 32, 32, 32, 4), (4, 64, 64, 32, 3), (2, 64, 128, 64, 3), (5, 128, 16, 64, 4),
    (1, 128, 128, 128, 3), (2, 128, 64, 16, 2), (1, 128, 32, 64, 3), (7, 128, 16, 64, 3),
    # a wave's share of the channels ends in a chunk of 8, and takes two rounds of chunks
    (5, 32, 16, 16, 2), (16, 128, 32, 64, 3)])
def test_append_forms_bit_exact(h, d, rank, group, bits):
    gen = torch.Generator().manual_seed(h * 1000 + d + rank)
    S, C = 256, h * d
    k_pre = (torch.randint(-24, 25, (h, S, d), generator=gen) / 8.0).half()
    v = (torch.randint(-16, 17, (h, S, d), generator=gen) / 4.0).half()
    V = (torch.randint(-2, 3, (C, rank), generator=gen) / 4.0).float()
    us0 = OC.to_matrix(k_pre[:, :128].float()) @ V
    consts = k2b.CodecConsts.make(v_seed=1, head_dim=d)
    kw = dict(h=h, d=d, rank=rank, group=group, bits=bits)
    pages = _encode(k_pre, v, V, us0, consts, **kw)
    enc = OC.FrozenSubspaceKeyEncoder(rank, bits, group)
    parts = []
    for p in range(2):
        sl = slice(p * 128, (p + 1) * 128)
        kp, _ = enc.encode(OC.to_matrix(k_pre[:, sl].float()), us_override=(us0, V) if p == 0 else None)
        idx, norms, _ = OC.quantize_v_perhead(OC.to_matrix(v[:, sl].float()), bits=2, seed=1, h=h)
        parts.append((kp["Us"].numpy().astype(np.float16), kp["res_Q_int"].numpy(),
                      kp["res_scale"][..., 0].numpy().astype(np.float16), idx.numpy(),
                      norms.numpy().astype(np.float16)))
    us, res, sc, vi, vn = (np.concatenate([x[i] for x in parts], axis=1 if i in (1, 2) else 0) for i in range(5))
    if d == 128 and group == 64 and bits == 3 and rank in (16, 32):
        want = OL.pack_pages(us, res, sc, vi, vn, h, rank)
    else:
        want = OL.pack_general(us, res, sc, vi, vn, h, rank, d, group, bits)
    np.testing.assert_array_equal(pages, want)
    np.testing.assert_array_equal(_encode(k_pre, v, V, us0, consts, via=_odd_rows, **kw), want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_value_rows_of_every_range(d, dtype):
    """Ordinary rows beside rows of tiny values, a norm below fp16's normal range, a norm above fp16's largest
    number and a zero row (norm 0 in fp16: its codes are 0)."""
    h, S, rank = 2, 128, 16
    gen = torch.Generator().manual_seed(d)
    v = torch.randn(h, S, d, generator=gen)
    v[:, 3] *= 1e-7                      # the norm is an fp16 subnormal
    v[:, 9, ::2] = 1e-35                 # far below the row's norm (0 in fp16)
    v[:, 17] *= 4000.0
    v[:, 33] = 60000.0                   # the norm overflows to infinity in fp16
    v[:, 64] = 0.0
    v = v.to(dtype)
    consts = k2b.CodecConsts.make(v_seed=2, head_dim=d)
    group, bits = (64, 3) if d == 128 else (32, 3)
    C = h * d
    pages = _encode(torch.zeros(h, S, d, dtype=torch.float16), v, torch.zeros(C, rank), torch.zeros(128, rank),
                    consts, h=h, d=d, rank=rank, group=group, bits=bits)
    vi, vn = (OL.unpack_pages(pages, h, rank) if d == 128
              else OL.unpack_general(pages, h, rank, d, group, bits))[3:]
    idx, norms, _ = OC.quantize_v_perhead(OC.to_matrix(v.float()), bits=2, seed=2, h=h)
    zero = np.zeros(S, bool)
    zero[64] = True
    np.testing.assert_array_equal(vn.astype(np.float32), norms.numpy())
    np.testing.assert_array_equal(vi[~zero], idx.numpy()[~zero])
    assert not vi[zero].any()
