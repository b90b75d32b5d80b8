"""Host logic shared with kernels and launches, checked on the CPU: each check
is a small program over the library's own headers."""

from util import run_host_check


def test_tap_walks_read_written_entries(tmp_path):
    """The sparse convs' loaders read the list of active taps only where a tap
    is listed."""
    assert run_host_check("tap_walk_check.hip", tmp_path) == "ok\n"
