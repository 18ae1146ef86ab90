"""Routing of attention calls (CPU): workspaces that are as large as the size queries
say, or smaller, and the scratch of the entry point without a workspace."""
import math

import numpy as np

from kaplumba_amd import _lib
from tests import attention_paths as paths

SHAPES = ((16, 8, 256, "dense"), (32, 8, 64, "hadamard"), (32, 8, 128, "hadamard"), (32, 8, 96, "dense"), (8, 1, 128, "hadamard"),
          (28, 4, 192, "dense"), (4, 4, 24, "dense"), (16, 16, 8, "dense"), (4, 4, 512, "dense"))


def problems(seed, count, tokens=200000):
    rng = np.random.default_rng(seed)
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    for Hq, Hkv, d, rot in SHAPES:
        for _ in range(count):
            yield Hq, Hkv, d, rot, log(1, 64), log(1, 1024), log(1, tokens)


def test_the_queried_size_is_enough():
    """A call with the queried size runs, on the kernel that any larger workspace gives."""
    seen = set()
    for Hq, Hkv, d, rot, B, L, T in problems(1, 300):
        for kw in (dict(), dict(mask=_lib.TQ_MASK_BOOL), dict(v_rot="dense"), dict(plain="bf16"), dict(q="f32")):
            got = paths.path(B, Hq, Hkv, L, T, d, k_rot=rot, **kw)
            assert got != paths.TOO_SMALL, (Hq, Hkv, d, B, L, T, kw)
            assert got == paths.path(B, Hq, Hkv, L, T, d, k_rot=rot, workspace=1 << 62, **kw), (Hq, Hkv, d, B, L, T, kw)
            seen.add(got)
    assert seen == {paths.TUNED, paths.TILE, paths.WIDE, paths.NARROW, paths.VECTOR}


def test_static_scratch_gives_the_same_kernel():
    """tq_attention_noalloc's 64 MiB run every problem that it takes on the kernel of a full workspace (the plans
    depend on the problem alone), among them the wide and narrow ones."""
    lib = _lib.load()
    seen = {}
    for Hq, Hkv, d, rot, B, L, T in problems(2, 1500, tokens=20000):
        rc = lib.tq_attention_noalloc(None, _lib.TQ_DTYPE_BF16, B, Hq, Hkv, L, d, 0, 0, 0, 0.1, _lib.TQ_KV_PACKED, 0, None,
                                      None, None, None, 0, 3, 3, None, None, 0, None, None, T, T, None, None, 0, None, None)
        assert rc != _lib.TQ_OK  # null pointers, or no device: nothing is launched
        if rc == _lib.TQ_ERR_WORKSPACE:
            continue
        for kw in (dict(), dict(plain="bf16"), dict(q="f32")):
            full = paths.path(B, Hq, Hkv, L, T, d, k_rot=rot, **kw)
            assert paths.path(B, Hq, Hkv, L, T, d, k_rot=rot, workspace=64 << 20, **kw) == full, (Hq, Hkv, d, B, L, T, kw)
            seen[full] = seen.get(full, 0) + 1
    assert min(seen.get(p, 0) for p in (paths.TUNED, paths.TILE, paths.WIDE, paths.NARROW)) >= 10, seen


def test_a_smaller_workspace_still_runs():
    """Sizes from before the wide and narrow kernels: the kernels of then take the call."""
    # the bytes that the tuned and vector kernels need (rotated queries, split partials): one split of 4000 rows of 64
    B, Hq, Hkv, L, T = 2, 32, 8, 500, 4097
    assert paths.path(B, Hq, Hkv, L, T, 64) == paths.WIDE
    assert paths.path(B, Hq, Hkv, L, T, 64, workspace=17 << 20) == paths.TUNED
    assert paths.path(B, Hq, Hkv, L, T, 64, workspace=1 << 20) == paths.TOO_SMALL
    assert paths.path(8, 32, 8, 1, 6000, 96, k_rot="dense") == paths.NARROW
    small = min(w for w in range(1 << 16, 1 << 24, 1 << 14)
                if paths.path(8, 32, 8, 1, 6000, 96, k_rot="dense", workspace=w) != paths.TOO_SMALL)
    assert paths.path(8, 32, 8, 1, 6000, 96, k_rot="dense", workspace=small) in (paths.VECTOR, paths.NARROW)


def test_f32_queries_keep_the_f32_kernels():
    for kw in (dict(mask=_lib.TQ_MASK_BOOL), dict(mask=_lib.TQ_MASK_ADD_F32), dict(v_rot="dense")):
        for L in (1, 512):
            assert paths.path(1, 32, 8, L, 8192, 64, q="f32", **kw) == paths.VECTOR
            assert paths.path(1, 32, 8, L, 8192, 64, q="f16", **kw) in (paths.WIDE, paths.NARROW)
