"""A batch at its limits, on a HIP runtime without a GPU.

Where its merge runs out of memory, the error is returned and no half-built
merge is left behind: later calls build it anew instead of launching kernels on
descriptors that do not exist.  Where its members have more tasks than one
launch may have, there are several launches.
"""
import os
import subprocess

import hip_stub
import pytest


def test_merge_is_built_anew_after_a_failed_allocation(tmp_path):
    out = hip_stub.run(tmp_path, """
        g = pystrip.Geometry.make(350, 500, 128, 100, 2.0, 10.0, 42.0)
        events = np.zeros((100, 3), np.float32)

        def make():
            b = pystrip.Batch()
            b.add(g, events)
            b.add(g, events)
            return b

        def iterate(b):
            try:
                b.iterate(1)
                return True
            except pystrip.StripMLEMError:
                return False

        b = make()
        before = stub.stub_allocations()
        assert iterate(b)
        allocations = stub.stub_allocations() - before
        b.close()
        result = []
        for k in range(1, allocations + 1):
            b = make()
            stub.stub_fail_in(k)
            failed = not iterate(b)
            stub.stub_fail_in(0)
            stub.stub_clear_launches()
            retried = iterate(b)
            iterate(b)
            result.append([failed, retried,
                           stub.stub_launches(b"batch_", 0, 0),
                           stub.stub_launches(b"batch_", 1, 0)])
            b.close()
    """)
    assert any(failed for failed, *_ in out)
    for k, (failed, retried, launches, without_descriptors) in enumerate(out, 1):
        assert retried, f"allocation {k}: the batch does not recover"
        assert launches > 0 and without_descriptors == 0, \
            f"allocation {k}: launched on a half-built merge"


@pytest.mark.parametrize("backward, waves, tasks", [
    (0, 4, 1000), (0, 4, (1 << 24) + 3), (0, 1, (1 << 26) + 1),
    (1, 1, (1 << 26) + 1), (1, 1, 0)])
def test_no_launch_of_more_work_items_than_a_dispatch_counts(
        tmp_path, backward, waves, tasks):
    # a dispatch counts its work-items in 32 bits; the members' tasks together
    # can be more, and every one of them has to run
    lib = str(tmp_path / "launch.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-shared",
                    "-fPIC", "-x", "hip", "--offload-host-only",
                    *hip_stub.compiler()[3:], os.path.join(
                        hip_stub.HERE, "moment_batch_launch.cpp"),
                    "-o", lib], check=True, capture_output=True, text=True)
    over, items = hip_stub.run(tmp_path, f"""
        ctypes.CDLL(pystrip.LIB_PATH, mode=ctypes.RTLD_GLOBAL)
        assert ctypes.CDLL({lib!r}).launch_tasks({backward}, {waves},
                                                 {tasks}) == 0
        result = [stub.stub_launches(b"moment_", 0, (1 << 32) - 1),
                  stub.stub_work_items(b"moment_")]
    """)
    assert over == 0
    assert items == tasks * waves * 64
