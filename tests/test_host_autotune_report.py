"""The ensemble tuner's report against the tiling it keeps."""

import hostbuild


def test_report_names_the_kept_tiling():
    hostbuild.run("autotune_report")
