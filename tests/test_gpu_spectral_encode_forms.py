"""GPU tests of the spectral write kernel at the forms that take their own
branch: key dtypes, rows that are not 16-byte aligned, head counts whose column
blocks are partly empty, and values at the ends of the short division's range.
Pages are compared byte for byte with the oracle's (its products and sums are
rounded one by one, as the format says)."""

import numpy as np
import pytest
import torch

from bmx_amd import k2b, spectral
from oracle import codecs as OC
from oracle import spectral as O

from tests.spectral_util import synthetic_keys, synthetic_pack
from tests.test_gpu_spectral import _lloyd, _values_full_of

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pages(pack, h, k, v, payload, codec):
    dp = spectral.DevicePack(pack, h, DEV, payload, codec)
    n = k.shape[1] // 64
    kp = torch.zeros(n, dp.k_page_bytes, dtype=torch.uint8, device=DEV)
    vp = torch.zeros(4 * n, dp.v_page_bytes, dtype=torch.uint8, device=DEV)
    spectral.append(k, v, dp, kp, torch.arange(n, dtype=torch.int32, device=DEV), vp,
                    torch.arange(4 * n, dtype=torch.int32, device=DEV), k2b.CodecConsts.make(v_seed=0))
    return kp.cpu().numpy(), vp.cpu().numpy()


def _odd_rows(t):
    buf = torch.zeros(t.shape[0], t.shape[1], t.shape[2] + 3, dtype=t.dtype, device=t.device)
    buf[:, :, 1:1 + t.shape[2]] = t
    return buf[:, :, 1:1 + t.shape[2]]


@pytest.mark.parametrize("payload", ["rtn", "lloyd"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("h,budget,edge", [(1, 2.5, False), (2, 2.0, False), (3, 3.0, True)])
def test_key_pages_of_every_form(h, budget, edge, dtype, payload):
    pack = synthetic_pack(h, budget, seed=5)
    M = torch.from_numpy(synthetic_keys(pack, 128, seed=6))
    if edge:   # one group's keys near nothing, the other's large
        M[:64] *= 1e-20 if dtype != torch.float16 else 1e-4
        M[64:] *= 1e25 if dtype != torch.float16 else 3e3
    k = OC.from_matrix(M, h).to(dtype)
    v = torch.randn(h, 128, 128, generator=torch.Generator().manual_seed(1)).to(dtype)
    layout = O.Layout(pack.bits.numpy())
    Y = O.encode(OC.to_matrix(k.float()).numpy(), pack.enc.numpy(), layout)
    codes, scales = O.quantize(Y, layout, _lloyd(payload))
    want = O.pack_pages(codes, scales, layout, lloyd=payload == "lloyd")
    kp, _ = _pages(pack, h, k.to(DEV), v.to(DEV), payload, "perhead")
    np.testing.assert_array_equal(kp, want)
    odd, _ = _pages(pack, h, _odd_rows(k.to(DEV)), _odd_rows(v.to(DEV)), payload, "perhead")
    np.testing.assert_array_equal(odd, want)


@pytest.mark.parametrize("h", [1, 4])
def test_full_values_beside_the_keys(h):
    """The full-C value pages of the launch that encodes the keys: the oracle's codes and norms."""
    pack = synthetic_pack(h, 2.5, seed=5)
    M = torch.from_numpy(synthetic_keys(pack, 192, seed=6))
    v = torch.randn(h, 192, 128, generator=torch.Generator().manual_seed(1)).bfloat16()
    kp, vp = _pages(pack, h, OC.from_matrix(M, h).to(DEV), _odd_rows(v.to(DEV)), "rtn", "full")
    kq, _ = _pages(pack, h, OC.from_matrix(M, h).to(DEV), v.to(DEV), "rtn", "perhead")
    np.testing.assert_array_equal(kp, kq)
    codes, norms = _values_full_of(vp, h)
    idx, want, _ = OC.quantize_v_perhead(OC.to_matrix(v.float()), bits=2, seed=0, h=1)
    np.testing.assert_array_equal(codes, idx.numpy())
    np.testing.assert_array_equal(norms.astype(np.float32), want.numpy()[:, 0])
