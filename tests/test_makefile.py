"""csrc/Makefile builds the library without Python: from the same sources as _build.py."""
import os
import re

from ringattention_amd import _build


def test_the_makefile_names_every_source():
    with open(os.path.join(_build.CSRC, "Makefile")) as f:
        text = f.read().replace("\\\n", " ")
    assert set(re.search(r"^SOURCES = (.*)$", text, re.M).group(1).split()) == set(_build.SOURCES)
