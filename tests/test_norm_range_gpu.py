"""Value norms of very unlike size in the matrix-core kernels of the general
attention path (tq_attn_narrow.h, tq_attn_wide.h), whose weights p * n_t go into
f16 pieces: a token that a row masks, or hardly weighs, must not cost the row's
other tokens any bits, whatever its norm.

Against the float64 form on the device.  f16 (bf16) outputs round each value by
at most 2^-11 (2^-8) of it; what lies under that is f32-class (2e-6)."""
import math

import numpy as np
import pytest
import torch

from kaplumba_amd import _lib, ops
from tests import attention_paths as paths

pytestmark = pytest.mark.gpu


def rotation64(codec, device):
    r = torch.from_numpy(np.array(codec.rot_host)).double().to(device)
    if r.dim() == 2:
        return r
    h = torch.ones(1, 1, dtype=torch.float64, device=device)
    while h.shape[0] < r.shape[0]:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h * r[None, :] / math.sqrt(r.shape[0])


def random_side(g, codec, Hkv, T, norms, device):
    """A packed side of random indices: (norms, words, rows (Hkv, T, dim) in the rotated basis)."""
    idx = torch.randint(0, 1 << codec.bits, (Hkv, T, codec.dim), generator=g, device=device)
    at = torch.arange(codec.dim, device=device) * codec.bits
    w = torch.zeros(Hkv, T, codec.packed_width + 1, dtype=torch.int64, device=device)
    w.scatter_add_(2, (at // 32).expand_as(idx), (idx << (at % 32)) & 0xffffffff)
    w.scatter_add_(2, (at // 32 + 1).expand_as(idx), (idx << (at % 32)) >> 32)
    words = w[None, ..., :codec.packed_width].to(torch.uint32)
    cb = torch.from_numpy(codec.codebook.copy()).double().to(device)
    return norms[None], words, norms.double()[..., None] * cb[idx]


def attention64(q, scale, kc, vc, k_rows, v_rows, keep, bias=0.0):
    """(1, Hq, L, Dv) in float64; keep, bias: (L, T)."""
    qs = (q * torch.tensor(scale, dtype=q.dtype)).double()
    Hkv = k_rows.shape[0]
    _, Hq, L, D = q.shape
    qr = (qs @ rotation64(kc, q.device).T).reshape(Hkv, Hq // Hkv * L, D)
    s = (qr @ k_rows.transpose(1, 2).contiguous()).reshape(Hkv, Hq // Hkv, L, -1)
    s = (s + bias).masked_fill(~keep, -math.inf)
    o = torch.softmax(s, -1).reshape(Hkv, Hq // Hkv * L, -1) @ v_rows @ rotation64(vc, q.device)
    return o.reshape(1, Hq, L, -1)


@pytest.mark.parametrize("Hq,Hkv,L,T", [(8, 2, 3, 2111), (64, 16, 160, 1111)])  # narrow; wide
@pytest.mark.parametrize("d,rot", [(64, "hadamard"), (96, "dense"), (128, "hadamard"), (256, "hadamard")])
@pytest.mark.parametrize("kind", ["masked", "faint", "sinking", "tiny"])
def test_unlike_value_norms(device, Hq, Hkv, L, T, d, rot, kind):
    assert paths.path(1, Hq, Hkv, L, T, d, q="f16", k_rot=rot, mask=_lib.TQ_MASK_BOOL) == (paths.NARROW if L == 3 else paths.WIDE)
    g = torch.Generator(device=device).manual_seed(d + L)
    kc, vc = ops.Codec(d, 4, 0, rotation=rot), ops.Codec(d, 4, 1, rotation=rot)
    kn = math.sqrt(d) * torch.exp(0.2 * torch.randn(Hkv, T, generator=g, device=device))
    vn = torch.exp(0.3 * torch.randn(Hkv, T, generator=g, device=device))
    q = torch.randn(1, Hq, L, d, generator=g, device=device)
    i = torch.arange(T - L, T, device=device)[:, None]
    keep = torch.arange(T, device=device)[None] <= i
    if kind == "masked":  # tokens that no row keeps, and one that every row but one keeps not
        vn[:, T // 3] = 1e12
        vn[:, 40] = 1e5
        keep = keep & (torch.arange(T, device=device) != T // 3)
        keep[1:, 40] = False
    elif kind == "tiny":  # every norm far below 1
        vn *= 1e-20
    k_norms, k_words, k_rows = random_side(g, kc, Hkv, T, kn, device)
    if kind in ("faint", "sinking"):
        # queries along one key, whose score stands 40 (in units of e) above the others'
        best = T - L - 70
        along = k_rows[:, best] @ rotation64(kc, device)
        q = (q * 0.1 + 40 * math.sqrt(d) * (along / (along * along).sum(-1, keepdim=True)).float()
             .repeat_interleave(Hq // Hkv, 0)[None, :, None])
        if kind == "faint":
            vn[:, 5] = 3e8  # weighs e^-40 of the best key's 1: 1e-9 of its value
        else:
            vn[:, :600] = 1e4  # large norms first, then the row's maximum rises by 40
    v_norms, v_words, v_rows = random_side(g, vc, Hkv, T, vn, device)
    q = q.to(torch.bfloat16 if kind == "tiny" else torch.float16)  # f16 holds no 1e-20
    want = attention64(q, 1 / math.sqrt(d), kc, vc, k_rows, v_rows, keep)
    out = ops.attention_packed(q, k_norms, k_words, v_norms, v_words, kc, vc, 1 / math.sqrt(d), False, mask=keep)
    err = (out.double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max().item() <= 2.0 ** (-8 if kind == "tiny" else -11) + 2e-6, err.max().item()


@pytest.mark.parametrize("Hq,Hkv,L,T", [(8, 2, 1, 2111), (8, 2, 3, 2111), (64, 16, 160, 1111)])  # narrow or tuned; wide or tile
@pytest.mark.parametrize("d,rot", [(64, "hadamard"), (96, "dense"), (128, "hadamard"), (256, "hadamard")])
@pytest.mark.parametrize("masked", [False, True])
def test_tiny_queries(device, Hq, Hkv, L, T, d, rot, masked):
    """Query rows of 1e-36 and 1e-30 score every key alike: their output is the mean of the values."""
    g = torch.Generator(device=device).manual_seed(d + L)
    kc, vc = ops.Codec(d, 4, 0, rotation=rot), ops.Codec(d, 4, 1, rotation=rot)
    norms = torch.exp(0.3 * torch.randn(Hkv, T, generator=g, device=device))
    k_norms, k_words, k_rows = random_side(g, kc, Hkv, T, norms, device)
    v_norms, v_words, v_rows = random_side(g, vc, Hkv, T, norms, device)
    q = torch.randn(1, Hq, L, d, generator=g, device=device)
    q[0, : Hq // Hkv] *= 1e-36  # a whole kv head's rows: some kernels scale them together
    q[0, Hq // Hkv] *= 1e-36
    q[0, Hq // Hkv + 1] *= 1e-30
    q = q.to(torch.bfloat16)
    keep = torch.arange(T, device=device)[None] <= torch.arange(T - L, T, device=device)[:, None]
    want = attention64(q, 1 / math.sqrt(d), kc, vc, k_rows, v_rows, keep)
    out = ops.attention_packed(q, k_norms, k_words, v_norms, v_words, kc, vc, 1 / math.sqrt(d), not masked,
                               mask=keep if masked else None)
    err = (out.double() - want).norm(dim=-1) / want.norm(dim=-1)
    # bf16 outputs, and the f16 weights of the tuned dims (2^-11 each)
    assert err.max().item() <= 2.0 ** -8 + 2.0 ** -10, err.max().item()
