"""A context at its limits, on a HIP runtime without a GPU: what asks about a plan
in the moment form works wherever the same question about lists did."""
import hip_stub

# a few pairs on short lines, which take the moment form: pairs, most bands,
# |tan| (bits), box width, slot rows, groups of two bands and of one, status,
# occupied bins
MOMENTS = """
import struct
stats = struct.pack("<Qiiiiiiii", 40, 2, 0, 20, 64, 3, 2, 0, 0)
stub.stub_effect(b"moment_stats_kernel", 3, stats, len(stats))

def make():
    r = pystrip.Reconstruction(
        pystrip.Geometry.make(250, 700, 61, 37, 5.0, 10.0, 42.0))
    r.set_events(np.zeros((20, 3), np.float32))
    return r
"""


def test_tiling_of_a_moment_plan_wherever_lists_fit(tmp_path):
    out = hip_stub.run(tmp_path, MOMENTS + """
r = make()
result = {"forms": [r.plan_forms()], "same": [], "again": []}
before = stub.stub_allocations()
tiling = (r.band_tiling(), r.band_groups())
allocations = stub.stub_allocations() - before
# asked again: from what was found
assert (r.band_tiling(), r.band_groups()) == tiling
result["repeated"] = stub.stub_allocations() - before - allocations
result["allocations"] = allocations
for k in range(1, allocations + 1):
    r = make()
    r.plan_forms()
    stub.stub_fail_in(k)
    result["same"].append((r.band_tiling(), r.band_groups()) == tiling)
    stub.stub_fail_in(0)
    r.iterate(1)
    result["again"].append(r.plan_forms())
    r.close()
""")
    assert out["forms"] == [[1, 0]]
    assert out["allocations"] > 0 and out["repeated"] == 0
    assert all(out["same"])
    assert all(forms == [1, 0] for forms in out["again"])
