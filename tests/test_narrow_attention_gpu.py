"""GPU parity of the narrow kernel (tq_attn_narrow.h: few query rows per kv head
at other dims, K / V dims that differ, plain caches and array masks) vs the
float64 oracle: every padded dim, 16-row group edges, sub-chunk and wave
remainders, windows and masks.  Bar as in test_attention_gpu; f32 queries at the
same shapes hold the f32-class error of the kernel that serves them."""
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O
from kaplumba_amd import _lib, ops
from kaplumba_amd.cache import create_causal_mask
from tests import attention_paths as paths
from tests.test_attention_gpu import assert_close, q_tensor
from tests.test_general_attention_gpu import packed_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk,krot,dv,vrot,kb,vb", [
    (64, "hadamard", 64, "dense", 3, 4), (40, "dense", 24, "dense", 1, 1), (80, "dense", 80, "dense", 3, 3),
    (96, "dense", 96, "dense", 4, 2), (128, "hadamard", 64, "hadamard", 2, 4), (100, "dense", 37, "dense", 3, 1),
    (192, "dense", 128, "hadamard", 3, 3), (160, "dense", 160, "dense", 4, 4), (250, "dense", 256, "hadamard", 2, 3)])
@pytest.mark.parametrize("Hq,Hkv,L,T,lengths,starts", [
    (4, 4, 1, 31, None, None),                      # fewer tokens than a sub-chunk; one row
    (8, 2, 4, 257, [257, 33], None),                # 16 rows: a whole group; one token past the 8 waves
    (6, 2, 7, 2100, [2100, 1999], [5, 1900])])      # 21 rows: a group and a remainder; left padding
def test_narrow_packed(device, dk, krot, dv, vrot, kb, vb, Hq, Hkv, L, T, lengths, starts):
    B = 1 if lengths is None else len(lengths)
    qdt = "f16" if L == 7 else "bf16"
    assert paths.path(B, Hq, Hkv, L, T, dk, dv, q=qdt, k_rot=krot, v_rot=vrot) == paths.NARROW
    packed_case(device, 70 + dk + dv + L, B, Hq, Hkv, L, T, dk, dv, kb, vb, krot, vrot, qdt=qdt,
                lengths=lengths, starts=starts, norm="float16" if L == 4 else "float32")


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("L,T,W", [(1, 1500, 200), (5, 700, 33), (3, 90, 512)])
def test_narrow_window_mask(device, d, L, T, W):
    m = create_causal_mask(L, offset=T - L, window_size=W).numpy()
    assert paths.path(2, 8, 2, L, T, d, mask=_lib.TQ_MASK_BOOL) == paths.NARROW
    packed_case(device, 950 + d + L, 2, 8, 2, L, T, d, d, 3, 3, causal=False, mask_np=m)


@pytest.mark.parametrize("d", [96, 128, 256])
def test_narrow_f32_error(device, d):
    """f32 queries and outputs, which take the vector kernel's f32 arithmetic."""
    assert paths.path(1, 8, 2, 3, 1111, d, q="f32", mask=_lib.TQ_MASK_BOOL) == paths.VECTOR
    rng = np.random.default_rng(d)
    B, Hq, Hkv, L, T = 1, 8, 2, 3, 1111
    rot = "dense" if d == 96 else "hadamard"
    kc, vc = ops.Codec(d, 4, 0, rotation=rot), ops.Codec(d, 4, 1, rotation=rot)
    kt, vt = (torch.from_numpy(rng.standard_normal((B, Hkv, T, d)).astype(np.float32)).to(device) for _ in range(2))
    st = []
    for x, c in ((kt, kc), (vt, vc)):
        p = torch.zeros((B, Hkv, T, c.packed_width), dtype=torch.uint32, device=device)
        n = torch.zeros((B, Hkv, T), device=device)
        ops.append_quantize(x, c, p, n, 0)
        st.append((n, p))
    q = rng.standard_normal((B, Hq, L, d)).astype(np.float32)
    m = np.tril(np.ones((L, T), bool), T - L)
    out = ops.attention_packed(torch.from_numpy(q).to(device), st[0][0], st[0][1], st[1][0], st[1][1], kc, vc,
                               1 / math.sqrt(d), False, mask=torch.from_numpy(m).to(device))
    host = lambda t: t.cpu().numpy()  # noqa: E731
    want = O.attention(q, host(st[0][1]).astype(np.uint32), host(st[0][0]), host(st[1][1]).astype(np.uint32),
                       host(st[1][0]), k_bits=4, v_bits=4, k_codebook=O.beta_codebook(d, 4),
                       v_codebook=O.beta_codebook(d, 4), rot_kind=rot, k_rot=kc.rot_host, v_rot=vc.rot_host,
                       scale=1 / math.sqrt(d), q_dtype="f32", causal=False, mask=m)
    rel = np.linalg.norm(host(out) - want) / np.linalg.norm(want)
    assert rel < 2e-6, rel


@pytest.mark.parametrize("kvdt", ["f16", "bf16"])
@pytest.mark.parametrize("dk,dv", [(40, 24), (96, 96), (192, 128), (248, 200)])
@pytest.mark.parametrize("Hq,Hkv,L,T,lengths,window", [(4, 2, 1, 70, None, 0), (6, 2, 7, 777, [777, 300], 0),
                                                       (4, 1, 3, 1400, None, 45)])
def test_narrow_plain(device, kvdt, dk, dv, Hq, Hkv, L, T, lengths, window):
    B = 1 if lengths is None else len(lengths)
    rng = np.random.default_rng(dk + dv + L)
    k = O.round_to_dtype(rng.standard_normal((B, Hkv, T, dk)).astype(np.float32), kvdt)
    v = O.round_to_dtype(rng.standard_normal((B, Hkv, T, dv)).astype(np.float32), kvdt)
    q = O.round_to_dtype(rng.standard_normal((B, Hq, L, dk)).astype(np.float32), kvdt)
    m = create_causal_mask(L, offset=T - L, window_size=window).numpy() if window else None
    assert paths.path(B, Hq, Hkv, L, T, dk, dv, plain=kvdt, q=kvdt, mask=_lib.TQ_MASK_BOOL if window else 0) == paths.NARROW
    want = O.attention_plain(q, k, v, scale=1 / math.sqrt(dk), q_dtype=kvdt, causal=m is None and L > 1,
                             lengths=lengths, mask=m)
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[kvdt]
    buf = [torch.full((B, Hkv, T + 9, x.shape[-1]), float("nan"), dtype=dt, device=device) for x in (k, v)]
    for b, x in zip(buf, (k, v)):
        b[:, :, :T] = torch.from_numpy(x).to(dt).to(device)
    out = ops.attention_plain(q_tensor(q, kvdt, device), buf[0][:, :, :T], buf[1][:, :, :T], 1 / math.sqrt(dk),
                              m is None and L > 1,
                              seq_lens=None if lengths is None else torch.tensor(lengths, dtype=torch.int32),
                              mask=None if m is None else torch.from_numpy(m).to(device))
    assert_close(out, want, kvdt, f"narrow plain {kvdt} k{dk} v{dv} L{L} T{T}")
