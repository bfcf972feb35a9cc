"""Uses of a network after its workspace could not be allocated."""

import hostbuild


def test_workspace_that_could_not_grow():
    hostbuild.run("net_workspace")
