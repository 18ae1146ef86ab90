"""GPU parity of the wide kernel (tq_attn_wide.h: many query rows per kv head
outside the packed d = 128 causal case) vs the float64 oracle: every padded
dim it is built for, row and token remainders, windows and masks.  Bar as in
test_attention_gpu."""
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


def kv_heads(least, B, rows, T, dk, dv, tuned=False, plain=False, masked=False):
    """kv heads (``rows`` query rows each) from which the wide kernel takes the
    call: wide_pays in tq_attn_general.hip, in rows of the call and products of 2^28."""
    if tuned and dk in (64, 128):
        all_rows, work = 1536, 16
    elif tuned and dk == 256:
        all_rows, work = 0, 1.25 if plain else 2.5
    elif dv > 128:
        all_rows, work = (1024, 2) if plain else (0, 0.5)
    elif dk > 128:
        all_rows, work = 1024, 1
    else:
        all_rows, work = (8192, 4) if masked else (1024, 8)
    n = max(least, math.ceil(all_rows / (B * rows)), math.ceil(1.02 * work * 2 ** 28 / (B * rows * T * (dk + dv))))
    # the library's own rule, so that a moved line shows here
    got = paths.path(B, n, n, rows, T, dk, dv, plain="f16" if plain else None, q="f16", k_rot="dense",
                     v_rot="dense" if tuned or masked or plain else "hadamard", mask=_lib.TQ_MASK_BOOL if masked else 0)
    assert got == paths.WIDE, (B, n, rows, T, dk, dv, got)
    return n


@pytest.mark.parametrize("dk,krot,dv,vrot,kb,vb", [
    (64, "hadamard", 64, "hadamard", 3, 4),
    (64, "dense", 64, "dense", 1, 2),
    (256, "hadamard", 256, "hadamard", 2, 3),
    (256, "dense", 256, "dense", 4, 2),
    (256, "hadamard", 256, "dense", 4, 4),
    (80, "dense", 80, "dense", 3, 3),
    (96, "dense", 96, "dense", 4, 1),
    (50, "dense", 37, "dense", 3, 3),
    (128, "hadamard", 64, "hadamard", 3, 2),
    (128, "hadamard", 256, "hadamard", 2, 3),
    (192, "dense", 128, "hadamard", 3, 4),
    (130, "dense", 100, "dense", 2, 4),
    (64, "hadamard", 250, "dense", 3, 3)])
@pytest.mark.parametrize("R,Hkv,L,T,lengths,starts", [
    (4, 1, 16, 131, None, None),                  # 64 rows: half the waves idle
    (3, 1, 43, 700, [700, 45], None),             # 129 rows: one past a block of 128
    (4, 2, 70, 1029, [1029, 611], [3, 600])])     # 280 rows; a window shorter than the queries
def test_wide_packed(device, dk, krot, dv, vrot, kb, vb, R, Hkv, L, T, lengths, starts):
    B = 1 if lengths is None else len(lengths)
    Hkv = kv_heads(Hkv, B, R * L, T, dk, dv, tuned=dk == dv and krot == vrot)
    Hq = R * Hkv
    packed_case(device, 40 + dk + dv + L, B, Hq, Hkv, L, T, dk, dv, kb, vb, krot, vrot,
                qdt="f16" if L == 43 else "bf16", lengths=lengths, starts=starts,
                norm="float16" if L == 16 else "float32")


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("W,L,T", [(64, 96, 500), (33, 75, 421)])
def test_wide_window_mask(device, d, W, L, T):
    """A sliding window's rows see a band of keys; rows of one block end at different keys."""
    m = create_causal_mask(L, offset=T - L, window_size=W).numpy()
    Hkv = kv_heads(2, 1, 2 * L, T, d, d, masked=True)
    packed_case(device, 900 + d + W, 1, 2 * Hkv, Hkv, L, T, d, d, 3, 3, causal=False, mask_np=m)


@pytest.mark.parametrize("shape", ["2d", "4d", "5d", "keys"])
def test_wide_bool_mask_shapes_and_empty_rows(device, shape):
    """Rows that keep nothing average every value of their window; a row that
    keeps one key takes it, wherever it lies; a mask broadcast along keys."""
    B, R, L, T = 2, 4, 33, 600
    Hkv = kv_heads(2, B, R * L, T, 128, 128, masked=True)
    Hq = R * Hkv
    rng = np.random.default_rng(77)
    full = {"2d": (L, T), "4d": (B, Hkv, L, T), "5d": (B, Hkv, R, L, T), "keys": (L, 1)}[shape]
    m = rng.random(full) < 0.4
    if shape == "keys":
        m = np.broadcast_to(m, (L, T))
    else:
        m[..., 5, :] = False
        m[..., 6, :] = False
        m[..., 6, T - 1] = True
        m[..., 7, 64:] = False
    mt = torch.from_numpy(np.ascontiguousarray(m[:, :1])).to(device).expand(L, T) if shape == "keys" else None
    packed_case(device, 910, B, Hq, Hkv, L, T, 128, 128, 3, 3, causal=False, lengths=[600, 437],
                starts=[0, 21], mask_np=m, mask_t=mt)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("causal", [False, True])
def test_wide_additive_mask(device, dt, causal):
    """Additive entries, the type's lowest value among them (finite: a row of it is uniform)."""
    B, L, T = 1, 50, 333
    Hkv = kv_heads(2, B, 2 * L, T, 64, 64, masked=True)
    Hq = 2 * Hkv
    rng = np.random.default_rng(78)
    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[dt]
    m = O.round_to_dtype(rng.normal(0, 2.0, size=(L, T)).astype(np.float32), dt)
    m[rng.random((L, T)) < 0.3] = -6e4 if dt != "f16" else float(np.float16(-6e4))
    m = O.round_to_dtype(m, dt)
    if not causal and dt != "f16":
        m[3] = torch.finfo(tdt).min
        m[4, 10:] = torch.finfo(tdt).min
    packed_case(device, 920, B, Hq, Hkv, L, T, 64, 64, 4, 2, causal=causal, mask_np=m,
                mask_t=torch.from_numpy(m).to(tdt).to(device))


def test_wide_minus_infinity_mask(device):
    """-inf entries weigh nothing; the kept keys alone decide."""
    L, T = 40, 300
    rng = np.random.default_rng(79)
    keep = rng.random((L, T)) < 0.2
    keep[:, 11] = True
    add = np.where(keep, 0.0, -np.inf).astype(np.float32)
    Hkv = kv_heads(2, 1, 2 * L, T, 96, 96, masked=True)
    packed_case(device, 930, 1, 2 * Hkv, Hkv, L, T, 96, 96, 3, 3, "dense", "dense", causal=False, mask_np=keep,
                mask_t=torch.from_numpy(add).to(device))


@pytest.mark.parametrize("kvdt", ["f16", "bf16"])
@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (256, 256), (80, 80), (96, 96), (192, 128), (200, 256)])
@pytest.mark.parametrize("R,Hkv,L,T,lengths,window", [(4, 1, 16, 170, None, 0), (3, 2, 91, 777, [777, 300], 0),
                                                      (2, 2, 48, 400, None, 45)])
def test_wide_plain(device, kvdt, dk, dv, R, Hkv, L, T, lengths, window):
    B = 1 if lengths is None else len(lengths)
    Hkv = kv_heads(Hkv, B, R * L, T, dk, dv, tuned=dk == dv and not window, plain=True, masked=bool(window))
    Hq = R * Hkv
    rng = np.random.default_rng(dk + dv + L)
    k = O.round_to_dtype(rng.standard_normal((B, Hkv, T, dk)).astype(np.float32), kvdt)
    v = O.round_to_dtype(rng.standard_normal((B, Hkv, T, dv)).astype(np.float32), kvdt)
    q = O.round_to_dtype(rng.standard_normal((B, Hq, L, dk)).astype(np.float32), kvdt)
    m = create_causal_mask(L, offset=T - L, window_size=window).numpy() if window else None
    want = O.attention_plain(q, k, v, scale=1 / math.sqrt(dk), q_dtype=kvdt, causal=m is None,
                             lengths=lengths, mask=m)
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[kvdt]
    buf = [torch.full((B, Hkv, T + 9, x.shape[-1]), float("nan"), dtype=dt, device=device) for x in (k, v)]
    for b, x in zip(buf, (k, v)):
        b[:, :, :T] = torch.from_numpy(x).to(dt).to(device)
    out = ops.attention_plain(q_tensor(q, kvdt, device), buf[0][:, :, :T], buf[1][:, :, :T], 1 / math.sqrt(dk),
                              m is None, seq_lens=None if lengths is None else torch.tensor(lengths, dtype=torch.int32),
                              mask=None if m is None else torch.from_numpy(m).to(device))
    assert_close(out, want, kvdt, f"plain {kvdt} k{dk} v{dv} L{L} T{T}")
