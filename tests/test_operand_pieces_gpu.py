"""The f32-class arithmetic behind 16-bit outputs of the wide and narrow kernels:
operands and weights in several pieces, sums in f32.

Outputs are compared with the float64 result rounded to their type.  With internal
errors below 1e-6 of a row they differ where that result lies within such an error of
a rounding boundary: 0.1-0.5 % of the f16 values and 0.03-0.04 % of the bf16 ones.
Without the weights' second piece (wide) or the keys' (narrow) 34-59 % of the f16
values differ, without a third bf16 piece of the weights 0.24 % of the bf16 ones."""
import math

import pytest
import torch

from kaplumba_amd import _lib, ops
from tests import attention_paths as paths
from tests.test_norm_range_gpu import attention64, random_side

pytestmark = pytest.mark.gpu

SIZES = [(8, 2, 3, 2111, paths.NARROW), (64, 16, 160, 1111, paths.WIDE)]


def masks(kind, L, T, g, device):
    """(keep, the mask to pass): causal as a boolean, or with additive entries."""
    keep = torch.arange(T, device=device)[None] <= torch.arange(T - L, T, device=device)[:, None]
    if kind == "bool":
        return keep, keep, 0.0
    add = torch.randn(L, T, generator=g, device=device).masked_fill(~keep, -math.inf)
    return keep, add, add.double().masked_fill(~keep, 0.0)


def differ(out, want):
    return (out != want.to(out.dtype)).double().mean().item()


@pytest.mark.parametrize("Hq,Hkv,L,T,kernel", SIZES)
@pytest.mark.parametrize("d,rot,mask", [(64, "hadamard", "bool"), (128, "hadamard", "bool"), (128, "hadamard", "add"),
                                        (96, "dense", None), (192, "dense", None), (256, "hadamard", "add")])
def test_packed(device, Hq, Hkv, L, T, kernel, d, rot, mask):
    g = torch.Generator(device=device).manual_seed(d)
    code = {None: _lib.TQ_MASK_NONE, "bool": _lib.TQ_MASK_BOOL, "add": _lib.TQ_MASK_ADD_F32}[mask]
    assert paths.path(1, Hq, Hkv, L, T, d, q="f16", k_rot=rot, mask=code) == kernel
    kc, vc = ops.Codec(d, 4, 0, rotation=rot), ops.Codec(d, 3, 1, rotation=rot)
    norm = lambda s: torch.exp(s * torch.randn(Hkv, T, generator=g, device=device))  # noqa: E731
    k_norms, k_words, k_rows = random_side(g, kc, Hkv, T, math.sqrt(d) * norm(0.2), device)
    v_norms, v_words, v_rows = random_side(g, vc, Hkv, T, norm(1.5), device)  # over a dozen powers of two
    q = torch.randn(1, Hq, L, d, generator=g, device=device).half()
    keep, m, bias = masks(mask or "bool", L, T, g, device)
    want = attention64(q, 1 / math.sqrt(d), kc, vc, k_rows, v_rows, keep, bias)
    out = ops.attention_packed(q, k_norms, k_words, v_norms, v_words, kc, vc, 1 / math.sqrt(d), mask is None,
                               mask=m if mask else None)
    assert differ(out, want) <= 0.01


@pytest.mark.parametrize("Hq,Hkv,L,T,kernel", SIZES)
@pytest.mark.parametrize("d,mask", [(128, "bool"), (96, None), (192, None), (256, "bool")])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
def test_plain(device, Hq, Hkv, L, T, kernel, d, mask, dt):
    if d == 192 and kernel == paths.WIDE:
        T *= 3
    tdt = torch.float16 if dt == "f16" else torch.bfloat16
    assert paths.path(1, Hq, Hkv, L, T, d, plain=dt, q=dt, mask=_lib.TQ_MASK_BOOL if mask else 0) == kernel
    g = torch.Generator(device=device).manual_seed(d)
    k, v = (torch.randn(1, Hkv, T, d, generator=g, device=device).to(tdt) for _ in range(2))
    q = torch.randn(1, Hq, L, d, generator=g, device=device).to(tdt)
    keep, m, _ = masks("bool", L, T, g, device)
    qs = (q * torch.tensor(1 / math.sqrt(d), dtype=tdt)).double().reshape(Hkv, Hq // Hkv * L, d)
    s = qs @ k[0].double().transpose(1, 2).contiguous()
    s = s.reshape(Hkv, Hq // Hkv, L, T).masked_fill(~keep, -math.inf)
    want = (torch.softmax(s, -1).reshape(Hkv, -1, T) @ v[0].double()).reshape(1, Hq, L, d)
    out = ops.attention_plain(q, k, v, 1 / math.sqrt(d), mask is None, mask=m if mask else None)
    assert differ(out, want) <= (0.01 if dt == "f16" else 1e-3)
