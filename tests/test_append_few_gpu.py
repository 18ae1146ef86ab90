"""The dense-rotation append at dims that are no 64, 128 or 256 (tq_append_few.hip),
keys and values in one call, and few vectors at those dims: every dim class, width pair and input type, vector counts at the
edges of its 16-vector groups.  Bar of test_append_general_gpu: norms bit-exact,
indices equal to the oracle's but within its band of a midpoint (each y is a
sum of exact piece products in f32, no longer than that band's d / 4 + 2 ulps),
nothing written outside the appended rows."""
import numpy as np
import pytest
import torch

from oracle import tq_oracle as O
from kaplumba_amd import ops
from tests.test_append_general_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [8, 40, 64, 72, 96, 128, 160, 192, 248, 256])
@pytest.mark.parametrize("kb,vb", [(3, 3), (4, 2), (1, 3), (2, 1)])
@pytest.mark.parametrize("xdt,B,H,L", [("bf16", 1, 1, 1), ("f16", 2, 3, 5), ("f32", 1, 2, 8), ("bf16", 3, 1, 11)])
def test_few_vectors_keys_and_values(device, d, kb, vb, xdt, B, H, L):
    rng = np.random.default_rng(d + 10 * kb + L)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[xdt]
    # strided input: heads and tokens swapped, as a projection leaves them
    xs = [torch.from_numpy(rng.standard_normal((B, L, H, d)).astype(np.float32)).to(dt).to(device).transpose(1, 2)
          for _ in range(2)]
    codecs = [ops.Codec(d, b, s, rotation="dense") for b, s in ((kb, 0), (vb, 1))]
    cap, off = L + 6, 3
    packed = [torch.full((B, H, cap, c.packed_width), 0x5a5a5a5a, dtype=torch.int32, device=device).view(torch.uint32)
              for c in codecs]
    norms = [torch.full((B, H, cap), -7.0, dtype=torch.float32, device=device) for _ in codecs]
    ops.append_quantize_kv(xs[0], xs[1], codecs[0], codecs[1], packed[0], norms[0], packed[1], norms[1], off)
    for x, c, p, n, b, s in zip(xs, codecs, packed, norms, (kb, vb), (0, 1)):
        gp, gn = p.cpu().numpy().astype(np.uint32), n.cpu().numpy()
        assert _check(x.float().cpu().numpy(), b, d, s, gp[:, :, off:off + L], gn[:, :, off:off + L]) <= 2
        assert (np.delete(gp, np.s_[off:off + L], axis=2) == 0x5a5a5a5a).all()
        assert (np.delete(gn, np.s_[off:off + L], axis=2) == -7.0).all()
        used = d * b % 32
        if used:  # bits past the last coordinate are zero
            assert not (gp[:, :, off:off + L, -1] >> used).any()


def midpoints_on(x, rot, rng, count, off=0):
    """Sorted thresholds (f32) on rotated coordinates of random vectors, ``off`` f32 steps away."""
    u = x.astype(np.float64).reshape(-1, x.shape[-1])
    u = u / np.linalg.norm(u, axis=1, keepdims=True)
    v, i = rng.integers(0, u.shape[0], count), rng.integers(0, u.shape[1], count)
    y = np.einsum("cd,cd->c", u[v], rot.astype(np.float64)[i]).astype(np.float32)
    return np.sort(y + off * np.spacing(y))


@pytest.mark.parametrize("d", [64, 128, 256, 96])
@pytest.mark.parametrize("xdt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("kb,vb", [(4, 4), (4, 2), (3, 4)])
def test_words_do_not_depend_on_the_call(device, d, xdt, kb, vb):
    """The words of a vector on a threshold are the same whether it is appended
    with thousands of others, with few or alone, as one side or both."""
    rng = np.random.default_rng(d + kb)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[xdt]
    H, L = 4, 640
    xs = [torch.from_numpy(rng.standard_normal((1, H, L, d)).astype(np.float32)).to(dt).to(device) for _ in range(2)]
    codecs = [ops.Codec(d, b, s, rotation="dense") for b, s in ((kb, 0), (vb, 1))]

    def buffers(n):
        return [(torch.zeros((1, H, n, c.packed_width), dtype=torch.uint32, device=device),
                 torch.zeros((1, H, n), device=device)) for c in codecs]

    for trial in range(12):
        for c, x in zip(codecs, xs):
            m = midpoints_on(x[:, :, :100].float().cpu().numpy(), np.array(c.rot_host), rng, (1 << c.bits) - 1)
            c.device_tensors(x.device)["midpoints"] = torch.from_numpy(m).to(device)
        whole = buffers(L)
        ops.append_quantize_kv(*xs, *codecs, *whole[0], *whole[1], 0)
        for n in (1, 7, 100):
            part = [x[:, :, :n] for x in xs]
            both, single = buffers(n), buffers(n)
            ops.append_quantize_kv(*part, *codecs, *both[0], *both[1], 0)
            for x, c, s, b, w in zip(part, codecs, single, both, whole):
                ops.append_quantize(x, c, *s, 0)
                for got in (s, b):
                    assert torch.equal(got[0].view(torch.int32), w[0][:, :, :n].view(torch.int32)), (trial, n)
                    assert torch.equal(got[1], w[1][:, :, :n])


def vector_kernel_sums(x, den, rot):
    """y of the vector kernel (tq_append_general.hip) in its own f32 arithmetic: u = x / den, four chains of
    fused adds (coordinates k mod 4 in order), added in pairs.  An 80-bit add of the exact product stands for
    the fused one."""
    u = (x / den[..., None]).astype(np.float32)
    c = []
    for s in range(4):
        acc = np.zeros(u.shape[:-1] + (rot.shape[0],), np.float32)
        for k in range(s, u.shape[-1], 4):
            acc = (u[..., k:k + 1].astype(np.longdouble) * rot[:, k].astype(np.longdouble) + acc).astype(np.float32)
        c.append(acc)
    return (c[0] + c[1]) + (c[2] + c[3])


@pytest.mark.parametrize("d", [8, 40, 96, 192, 248])
@pytest.mark.parametrize("xdt", ["bf16", "f16", "f32"])
def test_ties_are_the_vector_kernels(device, d, xdt):
    """Thresholds placed on coordinates as the vector kernel computes them, and one f32 step below: every index
    is that kernel's, bit for bit.  (Without the branch for ties about a third of the coordinates on a
    threshold come out on the other side.)"""
    rng = np.random.default_rng(d)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[xdt]
    N = 33
    x = torch.from_numpy(rng.standard_normal((1, 1, N, d)).astype(np.float32)).to(dt).to(device)
    codec = ops.Codec(d, 4, 0, rotation="dense")
    p = torch.zeros((1, 1, N, codec.packed_width), dtype=torch.uint32, device=device)
    n = torch.zeros((1, 1, N), device=device)
    ops.append_quantize(x, codec, p, n, 0)
    y = vector_kernel_sums(x.float().cpu().numpy()[0, 0], n.cpu().numpy()[0, 0], np.array(codec.rot_host, np.float32))
    for trial in range(16):
        m = np.sort(rng.choice(y.reshape(-1), 15, replace=False))
        if trial % 2:
            m = np.nextafter(m, np.float32(-np.inf))
        codec.device_tensors(x.device)["midpoints"] = torch.from_numpy(m).to(device)
        ops.append_quantize(x, codec, p, n, 0)
        want = (y[..., None] > m).sum(-1)
        got = O.unpack_lowbit(p.cpu().numpy().astype(np.uint32)[0, 0], 4, d)
        assert np.array_equal(got, want), np.argwhere(got != want)[:4]


@pytest.mark.parametrize("d", [8, 40, 96, 192])
@pytest.mark.parametrize("xdt", ["bf16", "f32"])
@pytest.mark.parametrize("bits", [1, 3, 4])
def test_norms_past_the_range(device, d, xdt, bits):
    """Finite vectors whose norm is infinite: u = x / inf = 0, so every index counts the thresholds below 0."""
    dt = {"bf16": torch.bfloat16, "f32": torch.float32}[xdt]
    x = torch.randn(1, 1, 20, d, generator=torch.Generator().manual_seed(d)).to(dt)
    x[0, 0, 3] *= 2e30
    x[0, 0, 4, 1] = torch.finfo(dt).max
    x[0, 0, 5] = torch.finfo(dt).max
    codec = ops.Codec(d, bits, 0, rotation="dense")
    p = torch.zeros((1, 1, 20, codec.packed_width), dtype=torch.uint32, device=device)
    n = torch.zeros((1, 1, 20), device=device)
    ops.append_quantize(x.to(device), codec, p, n, 0)
    got = O.unpack_lowbit(p.cpu().numpy().astype(np.uint32)[0, 0], bits, d)
    assert torch.isinf(n[0, 0, 3:6]).all()
    assert (got[3:6] == (0.0 > np.array(codec.midpoints)).sum()).all()
    rest = np.r_[0:3, 6:20]
    assert _check(x.float().numpy()[:, :, rest], bits, d, 0, p.cpu().numpy().astype(np.uint32)[:, :, rest],
                  n.cpu().numpy()[:, :, rest]) <= 2
