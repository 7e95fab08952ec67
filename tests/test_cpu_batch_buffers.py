"""The batch buffers that grow with the number of frequencies, on the CPU under AddressSanitizer and UBSan
(tests/cpu_kernels/regrow_check.cpp): one batch solved and differentiated at a few frequencies, at more of them and at
a few again, against a fresh batch for each; the same with an allocation that fails on the way."""

import os
import subprocess

import numpy as np
import pytest

from test_cpu_batch_kernel import CLANG, HERE, _build_harness

pytestmark = pytest.mark.skipif(not CLANG.exists(), reason="host clang++ with sanitizer runtimes not found")


@pytest.fixture(scope="module")
def run():
    bh = _build_harness()
    bh.TARGETS["regrow"] = (HERE / "cpu_kernels/regrow_check.cpp", "ed_batch")
    exe = bh.build(name="regrow_check", target="regrow")

    def steps(*script, free=None):
        env = {**os.environ, **({"EMU_FREE_BYTES": str(free)} if free else {})}
        r = subprocess.run([str(exe), *script], capture_output=True, text=True, timeout=300, env=env)
        assert r.returncode == 0, r.stderr[-4000:]
        assert "AddressSanitizer" not in r.stderr and "runtime error" not in r.stderr, r.stderr[-4000:]
        return [(t[0], int(t[1]), np.array(t[2:], dtype=float)) for t in map(str.split, r.stdout.splitlines())]

    return steps


@pytest.fixture(scope="module")
def fresh(run):
    """The gradients of a fresh batch at n frequencies."""
    return {n: run("s%d" % n, "b")[-1][2] for n in (2, 4, 48)}


def test_more_and_fewer_frequencies_on_one_batch(run, fresh):
    got = [r for r in run("s4", "b", "s48", "b", "s4", "b") if r[0] == "grad"]
    for (_, rc, g), n in zip(got, (4, 48, 4)):
        assert rc == 0 and np.isfinite(g).all() and np.array_equal(g, fresh[n])


@pytest.mark.parametrize("before", [(), ("s4", "b")])
@pytest.mark.parametrize("fail", range(9))
def test_failed_allocation_of_a_backward(run, fresh, before, fail):
    """One of the allocations of a backward, the batch's first or one that grows, fails: that call is refused, the next
    one is right."""
    out = run(*before, "s48", "f%d" % fail, "b", "b")
    assert out[-1][1] == 0 and np.array_equal(out[-1][2], fresh[48])


def test_refused_frequencies_leave_the_last_solve(run, fresh):
    """A solve refused for a zero frequency, at more of them than the batch had, does not touch what a backward of the
    solve before it reads."""
    out = run("s2", "z", "b")
    assert out[1][1] != 0 and out[2][1] == 0 and np.array_equal(out[2][2], fresh[2])


@pytest.mark.parametrize("fail", range(2))
def test_failed_allocation_of_a_solve(run, fresh, fail):
    """Nor is a backward of a solve that did not come about taken for one."""
    out = run("s4", "f%d" % fail, "s48", "b", "s48", "b")
    assert out[1][1] != 0 and out[2][1] != 0
    assert out[4][1] == 0 and np.array_equal(out[4][2], fresh[48])


@pytest.mark.parametrize("free", [1500, 4000, 30000])
def test_gradients_do_not_depend_on_the_free_memory(run, fresh, free):
    """With little memory to spare the models of a backward share the job store in turn: the same bits."""
    assert np.array_equal(run("s48", "b", free=free)[-1][2], fresh[48])


@pytest.mark.parametrize("tries", [1, 2, 3])
def test_job_store_is_halved_until_it_can_be_had(run, fresh, tries):
    """The store's allocation fails, and again at half the size: the models share what there is, or the call is refused,
    and the next one is right."""
    out = run("s48", "k%d" % tries, "f2", "b", "b")
    assert out[1][1] == 0 or tries > 1
    assert out[-1][1] == 0 and np.array_equal(out[-1][2], fresh[48])
