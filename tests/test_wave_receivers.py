"""The receivers of the packed sweeps on the CPU: tests/host/wave_receivers.cpp
compiles cad_wave_sweep.hip for the host, runs a receiver's 64 lanes in lockstep
and serves each lane's mailbox loads at a time of its own, so a value that is used
without a look at its own sequence number turns up as a stale one.
"""
import subprocess

import pytest

from conftest import PKG_DIR, ROOT

CLANG = "/opt/rocm/lib/llvm/bin/clang++"


@pytest.fixture(scope="module")
def receivers(tmp_path_factory):
    exe = tmp_path_factory.mktemp("wave") / "receivers"
    subprocess.run([CLANG, "-std=c++20", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{PKG_DIR / 'csrc'}", f"-I{ROOT / 'include'}",
                    f'-DWAVE_SOURCE="{PKG_DIR / "csrc" / "cad_wave_sweep.hip"}"',
                    str(ROOT / "tests" / "host" / "wave_receivers.cpp"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("nw", [1, 2])
@pytest.mark.parametrize("way", ["fwd", "bwd"])
@pytest.mark.parametrize("which", ["j", "k"])
def test_receivers_take_only_checked_values(receivers, which, way, nw):
    """Every value that a receiver hands to the walking wave is the producer's of
    this launch, whatever the order in which a load's lanes are served."""
    for seed in range(12):
        r = subprocess.run([receivers, which, way, str(nw), str(seed)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (seed, r.stdout)


@pytest.mark.parametrize("nw", [1, 2])
@pytest.mark.parametrize("way", ["fwd", "bwd"])
def test_ring_space_that_never_comes_sets_the_error_flag(receivers, way, nw):
    """A walking wave that stands still: the K receiver's wait for room in the ring
    ends, and the launch's error flag says so."""
    r = subprocess.run([receivers, "stuck", way, str(nw)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
