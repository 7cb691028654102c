"""A wave's chunk of miss records passes between its lanes through LDS with no
barrier between; a plain read there may be answered by a value the lane read
before.  That shows in no run until a compiler takes the freedom, so the
source is held to it: every access of a wave's slot is atomic."""

import os
import re

from conftest import PKG


def source(name):
    with open(os.path.join(PKG, "csrc", name)) as f:
        return re.sub(r"//[^\n]*", "", f.read())


def test_every_access_of_a_waves_slot_is_atomic():
    kernel = source("walk_kernel.inc")
    # (one level of brackets inside the index: readfirstlane(...))
    uses = re.findall(r"ml->wave\s*\[(?:[^\[\]])*\]\s*([^;{]{0,12})", kernel)
    assert len(uses) >= 5
    for after in uses:
        assert re.match(r"\.(load\(\)|store\()", after), after


def test_a_slot_is_accessed_by_its_members_alone():
    text = source("walk.hpp")
    body = re.search(r"struct MissSlot \{(.*?)\n\};", text, re.S).group(1)
    assert "__hip_atomic_load(&at" in body and "__hip_atomic_store(&at" in body
    assert re.search(r"private:\s*unsigned long long at;\s*$", body)
