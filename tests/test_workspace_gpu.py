"""ops.reserve_workspace: the workspace that it sizes is the one that later calls on
the stream use, however the device was named and whatever smaller problem comes."""
import pytest
import torch

from kaplumba_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["cuda", "cuda:0"])
def test_reserved_workspace_is_used(device, name):
    stream = torch.cuda.Stream(device)
    with torch.cuda.stream(stream):
        ops.reserve_workspace(name, 4, 32, 8, 300, 64, 4096)
        key = (torch.device("cuda", 0), stream.cuda_stream)
        reserved = ops._WORKSPACES[key]
        codecs = [ops.Codec(64, 3, s) for s in (0, 1)]
        for B, L, T in ((4, 300, 4096), (1, 300, 4096), (3, 17, 900), (4, 1, 4096)):
            sides = []
            for c in codecs:
                sides += [torch.ones(B, 8, T, device=device),
                          torch.zeros(B, 8, T, c.packed_width, dtype=torch.uint32, device=device)]
            q = torch.ones(B, 32, L, 64, dtype=torch.bfloat16, device=device)
            ops.attention_packed(q, *sides, *codecs, 0.125, L > 1)
            assert ops._WORKSPACES[key] is reserved, (B, L, T)
    stream.synchronize()
