"""Error of f32 queries over packed caches where the general path's vector kernel
computes in f32 (masks, dims other than 64 / 128 / 256), against the float64
form: at few and at many query rows per kv head, where 16-bit queries take the
matrix-core kernels.

Mean relative error over seeds: 3.5-5.0e-7 with few rows and 5.1-7.9e-7 with many
in f32; operands in two f16 pieces (22 bits) gave 5.6-9.1e-7 and 6.0-10e-7.  The
bars lie between."""
import math

import pytest
import torch

from kaplumba_amd import ops
from tests.test_norm_range_gpu import attention64, random_side

pytestmark = pytest.mark.gpu


def mean_error(device, d, rot, Hq, Hkv, L, T, masked, seeds):
    total = 0.0
    for seed in range(seeds):
        g = torch.Generator(device=device).manual_seed(100 * seed + d)
        kc, vc = ops.Codec(d, 4, 0, rotation=rot), ops.Codec(d, 4, 1, rotation=rot)
        norm = lambda s: torch.exp(s * torch.randn(Hkv, T, generator=g, device=device))  # noqa: E731
        k_norms, k_words, k_rows = random_side(g, kc, Hkv, T, math.sqrt(d) * norm(0.2), device)
        v_norms, v_words, v_rows = random_side(g, vc, Hkv, T, norm(0.3), device)
        q = torch.randn(1, Hq, L, d, generator=g, device=device)
        keep = torch.arange(T, device=device)[None] <= torch.arange(T - L, T, device=device)[:, None]
        want = attention64(q, 1 / math.sqrt(d), kc, vc, k_rows, v_rows, keep)
        out = ops.attention_packed(q, k_norms, k_words, v_norms, v_words, kc, vc, 1 / math.sqrt(d), not masked,
                                   mask=keep if masked else None)
        total += ((out.double() - want).norm() / want.norm()).item()
    return total / seeds


@pytest.mark.parametrize("d,rot,masked", [(128, "hadamard", True), (256, "hadamard", True), (96, "dense", False)])
def test_few_rows(device, d, rot, masked):
    assert mean_error(device, d, rot, 8, 2, 3, 2111, masked, 12) <= 5.5e-7


@pytest.mark.parametrize("d,rot,masked,bar", [(128, "hadamard", True, 6.2e-7), (256, "hadamard", True, 8.2e-7),
                                              (96, "dense", False, 6.5e-7)])
def test_many_rows(device, d, rot, masked, bar):
    assert mean_error(device, d, rot, 64, 16, 160, 2111, masked, 3) <= bar
