"""bench.py's command-line contract on the CPU: one GPU only (``--gpus N``
above 1, or a multi-rank launch, exits with a message and status 2, before
anything touches a device)."""

import os
import subprocess
import sys

import pytest

from conftest import REPO


@pytest.mark.parametrize("argv, env", [(["--gpus", "2"], {}), (["--gpus", "8", "--steps", "1"], {}),
                                       ([], {"WORLD_SIZE": "2"})])
def test_bench_refuses_more_than_one_gpu(argv, env):
    res = subprocess.run([sys.executable, str(REPO / "bench.py"), *argv], capture_output=True, text=True,
                         env=dict(os.environ, **env), timeout=120, cwd=REPO)
    assert res.returncode == 2, res.stderr
    assert "one GPU only" in res.stderr
    assert res.stdout == ""


def test_small_decode_roofline_follows_the_launches(int_models):
    """The bound of a small decode is that of the kernel that runs, as the
    decode's log names it."""
    import bench
    m = int_models["lossless"]
    head = "chunks 675 cu 256 plan [] leftover 675 "
    fed = bench.small_decode_roofline(m, head + "fed launch steps 2048 seg 256 fed 22+4x16 rt 1", 675, 2048, 0.04096)
    assert fed["roofline_fed"]["kernel"] == "k_decompress_fed<1>"
    assert fed["roofline_fed"]["achieved"] == round(7 * 512 * 512 / 20e-6 / 1e9, 2)
    wide = bench.small_decode_roofline(m, head + "fed launch steps 2048 seg 256 fed 11+4x16 rt 2", 675, 2048, 0.04096)
    assert wide["roofline_fed"]["achieved"] == round((7 * 512 * 512 + 512 * 256) / 20e-6 / 1e9, 2)
    split = bench.small_decode_roofline(m, head + "split launch p8 steps 2048 seg 256 fed 0+0x16 rt 0", 675, 2048, 0.0512)
    assert split["roofline_split"]["achieved"] == round(2490368 / 25e-6 / 1e9, 2)
    for other in (head + "launch steps 2048 seg 256 fed 0+0x16 rt 0",
                  "chunks 40961 cu 256 plan [3,2] leftover 1 fed launch steps 2048 seg 256 fed 1+1x16 rt 1",
                  "chunks 40961 cu 256 rotating launches: rt 4 steps 2048 seg 64 launches 39"):
        n = int(other.split()[1])
        assert bench.small_decode_roofline(m, other, n, 2048, 0.1) == {}
