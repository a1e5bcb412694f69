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


# what a handle or call takes, in every way the library allocates
_TAKERS = {
    "gaussian_filter": "assert lib.awk_gaussian_filter(p, q, 96, 96, 96, 1.0, 1.0, 1.0, 2, 2, 2, None) == 0, lib.awk_last_error()",
    "splat": "assert lib.awk_splat(p, q, q, q, q, 96, 96, 96, 0, None) == 0, lib.awk_last_error()",
    "greedy": "assert lib.awk_greedy_create(ctypes.byref(h), 80, 80, 80, *([1.0] * 3), .01, .01, .001, .1) == 0, lib.awk_last_error()",
    "atlas": "assert lib.awk_atlas_create(ctypes.byref(h), 48, 48, 48, *([1.0] * 3), .01, .01, .001, .1, 3) == 0, lib.awk_last_error()",
    "ldmm_atlas": "assert lib.awk_ldmm_atlas_create(ctypes.byref(h), 40, 40, 40, *([1.0] * 3), .01, .01, .001, 3, 1.0, .1, 2, 0) == 0, lib.awk_last_error()",
    "unet": "w = (ctypes.c_float * lib.awk_unet_weight_count())(); assert lib.awk_unet_create(ctypes.byref(h), 64, 64, 64, w, len(w)) == 0, lib.awk_last_error()",
    "unet_trainer": "t = P(); w = (ctypes.c_float * lib.awk_unet_weight_count())(); assert lib.awk_unet_create(ctypes.byref(h), 32, 32, 32, w, len(w)) == 0 and "
                    "lib.awk_unet_trainer_create(ctypes.byref(t), h, w, len(w)) == 0, lib.awk_last_error()",
}


@pytest.mark.parametrize("kept", ["blocks", "scratch"])
@pytest.mark.parametrize("taker", sorted(_TAKERS))
def test_kept_memory_is_given_back(fake, taker, kept):
    """An allocation that fits the device once nothing is kept succeeds while blocks or
    scratch are: what the taker needs is measured in a fresh process, then it runs on a
    device with exactly that much beside what the program itself holds."""
    head = "h, p, q = P(), P(0x4000), P(0x8000)\n"
    need = int(fake_hip.run(fake, head + _TAKERS[taker] + "\nprint(fake.fake_used())"))
    keep = {"blocks": "g = P(); assert lib.awk_greedy_create(ctypes.byref(g), 64, 72, 60, *([1.0] * 3), .01, .01, .001, .1) == 0 and lib.awk_greedy_destroy(g) == 0",
            "scratch": "assert lib.awk_splat(p, q, q, q, q, 64, 72, 60, 0, None) == 0"}[kept]
    fake_hip.run(fake, head + keep + """
assert fake.fake_used() > 1 << 20  # kept
fake.fake_budget(max(%d, fake.fake_used()))
""" % need + _TAKERS[taker])


def test_release_memory(fake):
    fake_hip.run(fake, """
g, p, q = P(), P(0x4000), P(0x8000)
assert lib.awk_greedy_create(ctypes.byref(g), 64, 72, 60, *([1.0] * 3), .01, .01, .001, .1) == 0
live = fake.fake_used()
assert lib.awk_splat(p, q, q, q, q, 64, 72, 60, 0, None) == 0
assert lib.awk_release_memory() == 0 and fake.fake_used() == live
assert lib.awk_greedy_destroy(g) == 0 and fake.fake_used() == live  # kept
assert lib.awk_release_memory() == 0 and fake.fake_used() == 0
""")


@pytest.mark.parametrize("relaxed", [False, True])
def test_eigen_table_is_not_recorded_unmade(fake, relaxed):
    """The first application of an operator with an eigen table allocates and fills it: a
    capture refuses that also where a kept block has the size, a relaxed one records it,
    and either way the next call outside makes the table."""
    fake_hip.run(fake, """
relaxed = %r
def op():
    k = P()
    assert lib.awk_fluid_kernel_create(ctypes.byref(k), 24, 24, 24, 1.0, 1.0, 1.0, .02, .01, .01, 0.5, 0) == 0
    return k
def tables():
    return sum("k_eigen_table" in r[1] for r in log("launch"))
p = P(0x4000)
a, b = op(), op()
assert lib.awk_fluid_kernel_apply(a, p, p, p, 1, None) == 0
assert lib.awk_fluid_kernel_destroy(a) == 0
fake.fake_clear()
fake.fake_capture(2 if relaxed else 1)
rc = lib.awk_fluid_kernel_apply(b, p, p, p, 1, None)
fake.fake_capture(0)
assert (rc == 0) == relaxed and tables() == int(relaxed), (rc, tables())
assert lib.awk_fluid_kernel_apply(b, p, p, p, 1, None) == 0
assert tables() == 1 + int(relaxed)
fake.fake_capture(1)
assert lib.awk_fluid_kernel_apply(b, p, p, p, 1, None) == 0  # with its table it may be captured
assert tables() == 1 + int(relaxed)
""" % relaxed)


def test_weight_gradient_stream_is_joined_on_every_exit(fake):
    """Whichever launch of a training step fails, the caller's stream waits for what was
    put on the weight gradients' stream: the next call may overwrite what they read."""
    out = fake_hip.run(fake, """
w = (ctypes.c_float * lib.awk_unet_weight_count())()
net, t = P(), P()
assert lib.awk_unet_create(ctypes.byref(net), 16, 16, 16, w, len(w)) == 0
assert lib.awk_unet_trainer_create(ctypes.byref(t), net, w, len(w)) == 0
p, s = P(0x4000), 0x77770
u = (P * 3)(0x4000, 0x8000, 0xc000)
def step():
    fake.fake_clear()
    rc = lib.awk_unet_trainer_step(t, p, p, u, 1e-3, p, P(s))
    rows = log()
    side = [i for i, r in enumerate(rows) if r[0] == "launch" and r[5] != str(s)]
    if not side:
        return rc, len([r for r in rows if r[0] == "launch"]), True
    st = rows[side[-1]][5]
    after = rows[side[-1] + 1:]
    rec = [i for i, r in enumerate(after) if r[0] == "record" and r[2] == st]
    joined = any(r[0] == "wait" and r[1] == str(s) and r[2] == after[i][1] for i in rec for r in after[i:])
    return rc, len([r for r in rows if r[0] == "launch"]), joined
rc, n, joined = step()
assert rc == 0 and joined, (rc, joined)
bad = []
for k in range(n):
    fake.fake_fail(b"k_", k)
    rc, _, joined = step()
    assert rc != 0, k
    if not joined:
        bad.append(k)
fake.fake_fail(b"", 0)
assert step()[0] == 0
print(n, len(bad))
""")
    n, bad = map(int, out.split())
    assert n > 50 and bad == 0, (n, bad)


_MAKERS = dict({k: v for k, v in _TAKERS.items() if k not in ("splat", "gaussian_filter")},
               fluid="assert lib.awk_fluid_kernel_create(ctypes.byref(h), 24, 24, 24, 1.0, 1.0, 1.0, .02, .01, .01, 1.0, 0) == 0",
               ldmm="assert lib.awk_ldmm_create(ctypes.byref(h), 16, 16, 16, 1.0, 1.0, 1.0, .01, .01, .001, 2, 1.0, .1) == 0",
               gradients=_TAKERS["unet_trainer"] + "\nu = (P * 3)(1 << 16, 2 << 16, 3 << 16); l = ctypes.c_double()\n"
                         "assert lib.awk_unet_trainer_gradients(t, p, q, u, w, ctypes.byref(l)) == 0")


@pytest.mark.parametrize("maker", sorted(_MAKERS))
def test_handles_are_ready_for_any_stream(fake, maker):
    """A handle is made on the null stream and used on the caller's, which need not wait for
    it: what the creation clears has been waited for when it returns."""
    fake_hip.run(fake, "h, p, q = P(), P(0x4000), P(0x8000)\n" + _MAKERS[maker] + """
kinds = [r[0] for r in log() if r[0] in ("memset", "sync")]
assert "memset" not in kinds or kinds[-1] == "sync", kinds[-6:]
""")


def test_a_reported_error_is_not_reported_again(fake):
    """A call that fails returns its error; the next one, which does not, returns none."""
    fake_hip.run(fake, """
h, p, q = P(), P(0x4000), P(0x8000)
fake.fake_budget(1 << 20)
assert lib.awk_splat(p, q, q, q, q, 96, 96, 96, 0, None) != 0
assert lib.awk_splat(p, q, q, q, q, 16, 16, 16, 0, None) == 0, lib.awk_last_error()
assert lib.awk_greedy_create(ctypes.byref(h), 80, 80, 80, *([1.0] * 3), .01, .01, .001, .1) != 0
assert lib.awk_hfield_set_to_identity(p, p, p, 16, 16, 16, None) == 0, lib.awk_last_error()
""")


_DESTROY = {"fluid": "awk_fluid_kernel_destroy", "greedy": "awk_greedy_destroy", "ldmm": "awk_ldmm_destroy"}


@pytest.mark.parametrize("maker", sorted(_DESTROY))
def test_destroying_leaves_a_relaxed_capture_valid(fake, maker):
    """Freeing memory is allowed while a relaxed capture runs; waiting for the device is not."""
    fake_hip.run(fake, "h, p, q = P(), P(0x4000), P(0x8000)\n" + _MAKERS[maker] + """
fake.fake_clear()
fake.fake_capture(2)
assert lib.%s(h) == 0
fake.fake_capture(0)
assert not log("invalidated")
""" % _DESTROY[maker])


@pytest.mark.parametrize("maker", sorted(_DESTROY))
def test_destroying_needs_no_host_memory(fake, maker):
    """A handle's blocks are put away without allocating: nothing is thrown through the C entry."""
    fake_hip.run(fake, """
h, p, q = P(), P(0x4000), P(0x8000)
handles = []
for i in range(5):
    h = P()
    %s
    handles.append(h)
for h in handles:
    fake.fake_no_host_memory(1)
    rc = lib.%s(h)
    fake.fake_no_host_memory(0)
    assert rc == 0
assert lib.awk_release_memory() == 0 and fake.fake_used() == 0
""" % (_MAKERS[maker], _DESTROY[maker]))


# calls after which work on the handle's buffers may be under way on stream s
_USES = {
    ("fluid", "apply"): "assert lib.awk_fluid_kernel_apply(h, p, p, p, 1, s) == 0",
    ("greedy", "iterate"): "v = (P * 3)(1 << 16, 2 << 16, 3 << 16); assert lib.awk_greedy_iterate(h, p, q, v, v, None, None, None, s) == 0",
    ("greedy", "set_step"): "assert lib.awk_greedy_set_step(h, 0.5, s) == 0",
    ("greedy", "get_flags"): "assert lib.awk_greedy_get_flags(h, ctypes.byref(ctypes.c_uint()), 1, s) == 0",
    ("ldmm", "iterate"): "v = (P * 6)(*[(i + 1) << 16 for i in range(6)]); assert lib.awk_ldmm_iterate(h, p, q, v, None, 0, s) == 0",
}


@pytest.mark.parametrize("maker,use", sorted(_USES))
def test_blocks_are_put_away_after_their_streams(fake, maker, use):
    """A block is put away once the work on it is done: behind a wait for the device (the free
    of a small block) where its handle used a stream of its own, or for the null stream."""
    fake_hip.run(fake, """
p, q = P(0x4000), P(0x8000)
for s, waits in ((P(0x77770), ("free",)), (None, ("free", "sync"))):
    h = P()
    %s
    %s
    fake.fake_clear()
    assert lib.%s(h) == 0
    kinds = [r[0] for r in log()]
    assert kinds and kinds[0] in waits, kinds
""" % (_MAKERS[maker], _USES[(maker, use)], _DESTROY[maker]))
