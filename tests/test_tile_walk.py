"""Row numbers of the rotation kernels' tiles near the end of the 32-bit range
(kaplumba_amd/csrc/tq_tiles.h), on the host: a walk that counted rows wrapped
around there, so that its loop read and wrote at negative rows."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "kaplumba_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_tiles_stay_in_range(tmp_path):
    exe = str(tmp_path / "tile_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=undefined", "-I", CSRC,
                    os.path.join(HERE, "csrc", "tile_walk.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=120).stdout
    assert out.strip() == "ok"
