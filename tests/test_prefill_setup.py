"""mia_gpu_model_prefill when device memory runs out in its one-time set-up
(no counterpart in the reference, whose prompt is one step per token): the
call fails, leaves nothing behind, never runs a kernel on a missing buffer,
and a later call with memory works. On the CPU: prefill_setup.c runs the
model source over stand-ins of the device calls; on the GPU: an allocation
that fails is reported once, not again by the launches after it."""
import os
import subprocess

import pytest

import motoria_amd as M

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_prefill_setup_without_memory(tmp_path):
    exe = str(tmp_path / "prefill_setup")
    subprocess.run(["gcc", "-std=c99", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "motoria_amd", "host"),
                    "-I" + os.path.join(ROOT, "motoria_amd", "csrc"),
                    os.path.join(HERE, "prefill_setup.c"), "-o", exe, "-lm",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    assert subprocess.run([exe], timeout=60).returncode == 0


@pytest.mark.gpu
def test_failed_allocation_is_reported_once():
    g = M.Gpu()
    try:
        L = M.lib()
        assert not L.mhip_malloc(g.h, 1 << 50)
        assert b"hipMalloc" in L.mhip_error(g.h)
        p = g.malloc(1024)
        g.check(L.mhip_zero(g.h, p, 1024), "launch after a failed allocation")
        g.check(L.mhip_sync(g.h), "sync")
    finally:
        g.close()
