"""Boxes where memory can be pinned and where it cannot (the step report and the
download ring are pinned when they can be)."""

import pytest

import hostbuild


@pytest.mark.parametrize("pinned", ["some", "none"])
def test_box_without_pinned_memory(pinned):
    hostbuild.run("no_pinned_memory", pinned)
