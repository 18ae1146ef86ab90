"""The matrix-core rotation of query rows and merged outputs (tq_rotate.hip),
seen through attention over one or two tokens in f32.

One token: the output is its value n * (c[idx] @ R_V) whatever the query, so
the rotation of the output stands alone.  Two tokens: the weights depend on
the rotated query's scores too.  Every term of a rotation is a product of
pieces that sum to the f32 operands exactly, added in f32: d terms give at
most (d + 4) 2^-24 of the sum of magnitudes, |c[idx]|_1 max|R| <= sqrt(d) per
unit of norm; a score error e moves a weight by at most e / 4."""
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O
from kaplumba_amd import ops
from tests.test_attention_gpu import to_buffers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("qdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("d", [8, 36, 64, 80, 96, 130, 160, 192, 252, 256])
@pytest.mark.parametrize("Hq,L", [(1, 1), (3, 13), (4, 701)])  # 1, 39 and 2804 rows
def test_rotations_of_any_dim(device, T, qdt, d, Hq, L):
    if d in (64, 128, 256) and Hq * L < 64:
        pytest.skip("the tuned kernels rotate these themselves")
    rng = np.random.default_rng(d + L)
    x = rng.standard_normal((2, 1, 1, T, d)).astype(np.float32)
    R = [O.rotation_matrix(d, s) for s in (0, 1)]
    cb = O.beta_codebook(d, 3)
    (kp, kn, _), (vp, vn, _) = (O.quantize_dense(x[i], 3, R[i], cb, "float32") for i in (0, 1))
    q = O.round_to_dtype(rng.standard_normal((1, Hq, L, d)).astype(np.float32), qdt)
    want = O.attention(q, kp, kn, vp, vn, k_bits=3, v_bits=3, k_codebook=cb, v_codebook=cb, rot_kind="dense",
                       k_rot=R[0], v_rot=R[1], scale=1 / math.sqrt(d), q_dtype=qdt, causal=False)
    kn_t, ki, vn_t, vi = to_buffers(kp, kn, vp, vn, device)
    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[qdt]
    out = ops.attention_packed(torch.from_numpy(q).to(dt).to(device), kn_t, ki, vn_t, vi, ops.Codec(d, 3, 0, "dense"),
                               ops.Codec(d, 3, 1, "dense"), 1 / math.sqrt(d), False)
    bound = (d + 4) * 2.0 ** -24 * math.sqrt(d) * float(vn.max())
    if T == 2:
        score = (d + 4) * 2.0 ** -24 * math.sqrt(d) * float(kn.max()) * np.abs(q).max()
        bound += score / 4 * 2 * float(vn.max())
    ulp = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[qdt]
    err = np.abs(out.float().cpu().numpy() - want)
    tol = bound + ulp * np.abs(want) + 2.0 ** -24
    if d not in (64, 128, 256) or Hq * L < 64:
        # the weights of two tokens: f32 in the vector kernel
        assert (err <= tol).all(), (float(err.max()), bound)
    else:
        # the tuned shapes' weights are f16 (2^-11 each, and their sum)
        assert (err <= tol + 2.0 ** -10 * float(vn.max())).all(), (float(err.max()), bound)
