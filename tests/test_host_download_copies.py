"""Copies of results into the caller's memory, on the CPU (host memory in the
place of the GPU): the paths that only a failure or odd arguments reach."""

import pytest

import hostbuild


@pytest.mark.parametrize("what", ["sizes", "no_pinned_memory", "no_threads", "one_thread", "same_array", "pinned"])
def test_copies(what):
    hostbuild.run("download_copies", what)
