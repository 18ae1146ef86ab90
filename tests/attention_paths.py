"""Which kernels serve an attention call, as the library's own routing rule says
(tq_attention_path in kaplumba_amd/csrc/tq_attention.hip): host arithmetic only, so
tests can tell whether a call runs the kernel that they name."""
import ctypes

from kaplumba_amd import _lib

TUNED, TILE, WIDE, NARROW, VECTOR = range(5)
TOO_SMALL = -1


def path(B, Hq, Hkv, L, T, dk, dv=None, *, plain=None, q="bf16", k_rot="hadamard", v_rot=None, mask=0, workspace=None):
    """``plain``: the cache's type, None for a packed cache; ``mask``: a TQ_MASK_* code; ``workspace``: bytes, the
    size query's answer by default."""
    lib = _lib.load()
    fn = lib.tq_attention_path
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_int] * 12 + [ctypes.c_int64] * 2
    dv = dk if dv is None else dv
    v_rot = k_rot if v_rot is None else v_rot
    if workspace is None:
        one = not mask and dv == dk and v_rot == k_rot
        workspace = (lib.tq_attention_workspace_size(B, Hq, Hkv, L, dk, T) if one else
                     lib.tq_attention_general_workspace_size(B, Hq, Hkv, L, dk, dv, T))
    code = {"f32": _lib.TQ_DTYPE_F32, "f16": _lib.TQ_DTYPE_F16, "bf16": _lib.TQ_DTYPE_BF16}
    rot = {"hadamard": _lib.TQ_ROT_HADAMARD, "dense": _lib.TQ_ROT_DENSE}
    return fn(_lib.TQ_KV_PLAIN if plain else _lib.TQ_KV_PACKED, code[q], code[plain] if plain else 0, B, Hq, Hkv, L,
              dk, dv, rot[k_rot], rot[v_rot], mask, T, workspace)
