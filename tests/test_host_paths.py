"""What the host code of libawk_hip.so allocates and launches, on a HIP runtime that
only keeps books (fake_hip.py): no GPU, no kernel runs."""
import pytest

import fake_hip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("size", [(4, 6, 8), (5, 7, 9), (5, 6, 9), (3, 3, 3), (1, 1, 1), (128, 128, 128)])
def test_sorted_splat_keys_are_aligned(fake, size):
    """k_radix_hist loads its keys 16 bytes at a time: they start at a multiple of 16 in
    every pass, whatever the parities of the voxel and base cell counts, in the scratch
    of a call and in the LDMM iterator's own buffer."""
    out = fake_hip.run(fake, """
size = %r
p = P(0x4000)
assert lib.awk_splat_sorted(p, p, p, p, p, *size, 1, None, None, None) == 0
assert lib.awk_splat_sorted(p, p, p, p, p, *size, 1, P(0x8000), None, None) == 0
l = P()
assert lib.awk_ldmm_create(ctypes.byref(l), *size, 1.0, 1.0, 1.0, 0.01, 0.01, 0.001, 2, 1.0, 0.1) == 0
assert lib.awk_ldmm_set_gradient(l, 0) == 0
assert lib.awk_ldmm_set_splat(l, 1) == 0
v = (P * 6)(*[0x10000 * (i + 1) for i in range(6)])
assert lib.awk_ldmm_iterate(l, P(0x4000), P(0x8000), v, None, 0, None) == 0
rows = [r for r in log("launch") if "k_radix_hist" in r[1]]
print(len(rows), sum(int(r[-1]) %% 16 != 0 for r in rows))
""" % (size,))
    n, bad = map(int, out.split())
    assert n >= 4 and bad == 0, (n, bad)


@pytest.mark.parametrize("size", [(1, 1, 1 << 26), (1, 1 << 13, 1 << 13), (2, 4096, 4096), (1, 1, (1 << 28) - 1)])
def test_sorted_splat_of_short_rows_launches(fake, size):
    """Volumes of many short rows: every launch stays below 2^32 threads (a block per row
    of one or two voxels does not)."""
    fake_hip.run(fake, """
p = P(0x4000)
rc = lib.awk_splat_sorted(p, p, p, p, p, *%r, 1, None, None, None)
assert rc == 0, lib.awk_last_error()
assert any("k_base_sum" in r[1] for r in log("launch"))
""" % (size,))
