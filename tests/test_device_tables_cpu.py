"""What the planner keeps for a device (buffers, pinned tables, constants, events) is found by the device's own number:
a table indexed by part of it gives one device another's memory where a node shows more devices than the table has
places, and a growing array of owners frees what it moves when a thread takes a second device.  One GPU shows neither, so
the sources are read."""
import re

from limbforge_amd import build


def sources():
    return {p.name: p.read_text() for p in sorted(build.CSRC.glob("*.hip")) + sorted(build.CSRC.glob("*.hpp"))}


def test_no_table_is_indexed_by_part_of_a_device_number():
    for name, text in sources().items():
        assert not re.search(r"\[\s*\w*dev(ice)?\w*\s*[&%]", text), name


def test_per_device_owners_do_not_move():
    for name, text in sources().items():
        assert not re.search(r"thread_local\s+std::vector<std::pair<int,", text), name
