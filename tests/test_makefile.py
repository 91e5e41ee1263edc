"""A change of any header rebuilds every object: structs of the headers cross them."""

from __future__ import annotations

import shutil
import subprocess

import pytest

from research_amd import build

OBJECTS = [name for name in build.SOURCE_FILES if name.endswith(".hip")]


@pytest.mark.skipif(shutil.which("make") is None, reason="needs make")
@pytest.mark.parametrize("header", sorted(path.name for path in build.source_dir().glob("*.hpp")))
def test_a_header_rebuilds_every_object(header):
    assert header in build.SOURCE_FILES  # ... and is part of what the manifest records
    out = subprocess.run(["make", "-n", "-W", header, f"OUTDIR={build.cache_dir().as_posix()}", "all"], cwd=build.source_dir(),
                         capture_output=True, text=True, check=True).stdout
    for source in OBJECTS:
        assert f" {source} -o " in out, f"{source} does not depend on {header}"
