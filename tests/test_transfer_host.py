"""Host side of the large field transfers, on a HIP runtime without a GPU (_fakehip)."""
from _fakehip import run

OPEN = """
c = M.Case(make_case_dir(d2(nx=723, ny=725, btype=3)), heat_transfer=False, device=0)
a = np.random.default_rng(1).standard_normal(c._shape("U"))
"""


def test_transfers_do_not_depend_on_the_current_device(tmp_path):
    """A case on device 0 while the caller's current device is 1: no event of another device is
    recorded on the case's stream, and the caller's device stays."""
    print(run(tmp_path, OPEN + """
device.value = 1
c.set("U", a)
c.get("U")
assert device.value == 1
"""))


def test_without_pinned_memory_fields_go_through_pageable_copies(tmp_path):
    print(run(tmp_path, OPEN + """
pinned_fails.value = 1
c.set("U", a)
assert np.array_equal(c.get("U"), a)
pinned_fails.value = 0
c.set("U", a)
c.close()
"""))


def test_a_transfer_that_cannot_start_threads_copies_by_itself(tmp_path):
    """Worker threads fail to start for want of memory as well as of threads."""
    print(run(tmp_path, OPEN + """
c.set("U", a)
new_limit.value = 20
c.set("U", a)
c.get("U")
new_limit.value = 0
"""))
