"""Kernels that take more LDS than the default are granted it on every device that is asked, once each
(tests/cpu_kernels/grants_check.cpp): a process with several GPUs calls them on each."""

import subprocess

import pytest

from test_cpu_batch_kernel import CLANG, HERE, _build_harness

pytestmark = pytest.mark.skipif(not CLANG.exists(), reason="host clang++ with sanitizer runtimes not found")


def test_reorthogonalisation_kernels_are_granted_lds_on_each_device():
    bh = _build_harness()
    bh.TARGETS["grants"] = (HERE / "cpu_kernels/grants_check.cpp", "ed_reorth")
    exe = bh.build(name="grants_check", target="grants")

    def ask(*devices):
        r = subprocess.run([str(exe), *devices], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr[-2000:]
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]

    assert ask("0", "1", "0", "1", "3") == [(0, 1, 2), (1, 1, 2), (0, 1, 0), (1, 1, 0), (3, 1, 2)]
    # a device that refuses says nothing of the others
    assert ask("-1", "0", "-1", "1") == [(1, 0, 0), (0, 1, 2), (1, 0, 0), (1, 1, 2)]
