"""Infinite values of plain caches in the wide and narrow kernels, whose weights go in
as several pieces: a column with an infinite value in a token that the row keeps is
infinite, with its sign, as weight times value is in f32; the other columns do not
notice.  (The low pieces may be negative or 0, and would make it NaN.)"""
import math

import pytest
import torch

from kaplumba_amd import _lib, ops
from tests import attention_paths as paths

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("dk,dv,masked", [(64, 64, True), (96, 96, False), (128, 128, True), (192, 128, False),
                                          (256, 256, True)])
@pytest.mark.parametrize("Hq,Hkv,L,T,kernel", [(8, 2, 3, 1501, paths.NARROW), (64, 16, 160, 2111, paths.WIDE)])
def test_infinite_values(device, dt, dk, dv, masked, Hq, Hkv, L, T, kernel):
    tdt = torch.float16 if dt == "f16" else torch.bfloat16
    mask = _lib.TQ_MASK_BOOL if masked else _lib.TQ_MASK_NONE
    assert paths.path(1, Hq, Hkv, L, T, dk, dv, plain=dt, q=dt, mask=mask) == kernel
    g = torch.Generator(device=device).manual_seed(dk)
    k = torch.randn(1, Hkv, T, dk, generator=g, device=device).to(tdt)
    v = torch.randn(1, Hkv, T, dv, generator=g, device=device).to(tdt)
    q = torch.randn(1, Hq, L, dk, generator=g, device=device).to(tdt)
    keep = torch.arange(T, device=device)[None] <= torch.arange(T - L, T, device=device)[:, None]
    call = lambda x: ops.attention_plain(q, k, x, 1 / math.sqrt(dk), not masked, mask=keep if masked else None)  # noqa: E731
    clean = call(v)
    bad = v.clone()
    bad[:, :, 5, 0] = math.inf
    bad[:, :, 700, 1] = -math.inf
    bad[:, :, T - 1, 2] = math.inf  # the last query alone sees it, and it ends a split
    bad[:, :, 9, 3] = math.nan
    out = call(bad)
    assert (out[..., 0] == math.inf).all()
    assert (out[..., 1] == -math.inf).all()
    assert (out[..., -1, 2] == math.inf).all()
    assert out[..., 3].isnan().all()
    # (their products are summed apart there, so not bit by bit)
    rest, want = out[..., 4:].float(), clean[..., 4:].float()
    assert ((rest - want).norm() / want.norm()).item() <= (2e-4 if dt == "f16" else 1.5e-3)
