"""A batch whose merge runs out of memory, on a HIP runtime without a GPU: the
error is returned and no half-built merge is left behind, so later calls build
it anew instead of launching kernels on descriptors that do not exist."""
import hip_stub


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
            for _ in range(3):
                last = iterate(b)
            result.append([failed, last,
                           stub.stub_launches(b"batch_", 0, 0),
                           stub.stub_launches(b"batch_", 1, 0)])
            b.close()
    """)
    assert any(failed for failed, *_ in out)
    for k, (failed, last, launches, without_descriptors) in enumerate(out, 1):
        assert last, f"allocation {k}: the batch does not recover"
        assert launches > 0 and without_descriptors == 0, \
            f"allocation {k}: launched on a half-built merge"
