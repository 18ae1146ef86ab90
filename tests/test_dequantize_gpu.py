"""Dequantize at the sizes where its kernels change: the matrix-core dense one
(from 2048 vectors, 128-vector tiles) and the Hadamard one with four vectors a
lane, against the float64 form of n * R^-1(codebook[idx]).

Dense: d exact piece products added in f32, so (d + 4) 2^-24 of
|codebook[idx]|_1 max|R| <= sqrt(d), times the norm; Hadamard: log2(d) + 3
roundings of values below sqrt(d) max|c| / sqrt(d) each."""
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O
from kaplumba_amd import ops

pytestmark = pytest.mark.gpu


def _case(device, d, bits, rot, B, H, T, cap, norm):
    rng = np.random.default_rng(d + T + bits)
    codec = ops.Codec(d, bits, 1, rotation=rot)
    idx = rng.integers(0, 1 << bits, size=(B, H, T, d))
    words = O.pack_lowbit(idx.astype(np.uint32), bits)
    n = rng.uniform(0.5, 4.0, size=(B, H, T)).astype(np.float16 if norm == torch.float16 else np.float32)
    p = torch.full((B, H, cap, codec.packed_width), -1, dtype=torch.int32, device=device)
    p[:, :, :T] = torch.from_numpy(words.astype(np.uint32).view(np.int32)).to(device)
    nt = torch.full((B, H, cap), float("nan"), dtype=norm, device=device)
    nt[:, :, :T] = torch.from_numpy(n).to(device)
    got = ops.dequantize(p.view(torch.uint32)[:, :, :T], nt[:, :, :T], codec)
    c = torch.from_numpy(codec.codebook.astype(np.float64)).to(device)[torch.from_numpy(idx).to(device)]
    if rot == "dense":
        y = c @ torch.from_numpy(np.array(codec.rot_host, np.float64)).to(device)
        bound = (d + 4) * 2.0 ** -24 * math.sqrt(d)
    else:
        h = torch.ones(1, 1, dtype=torch.float64, device=device)
        while h.shape[0] < d:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        y = (c @ h) / math.sqrt(d) * torch.from_numpy(np.array(codec.rot_host, np.float64)).to(device)
        bound = (math.log2(d) + 3) * 2.0 ** -24 * math.sqrt(d) * float(np.abs(codec.codebook).max())
    want = y * torch.from_numpy(n.astype(np.float64)).to(device)[..., None]
    assert got.shape == (B, H, T, d)
    assert (got.double() - want).abs().max().item() <= bound * 4.0
    if rot == "dense":
        # one chain of sums per order of the piece products, the main one rounded
        # once per 32 terms: 5-9e-8 of the result (all orders in one chain 0.9-2.3e-7,
        # one f32 chain of d terms 1.5-2.9e-7)
        assert ((got.double() - want).norm() / want.norm()).item() <= 6e-8 + 2e-10 * d


@pytest.mark.parametrize("d", [24, 64, 96, 100, 130, 192, 255, 256])
@pytest.mark.parametrize("bits", [1, 2, 3, 4])
def test_dense_many_vectors(device, d, bits):
    _case(device, d, bits, "dense", 2, 3, 683, 700, torch.float16 if bits == 2 else torch.float32)  # 4098 vectors


@pytest.mark.parametrize("d,T", [(32, 21850), (64, 10930), (128, 5470), (256, 2731)])
@pytest.mark.parametrize("bits", [1, 3, 4])
def test_hadamard_many_vectors(device, d, T, bits):
    _case(device, d, bits, "hadamard", 2, 3, T, T + 5, torch.float32)
