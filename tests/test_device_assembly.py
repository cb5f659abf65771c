"""Inline assembly of the kernels, read from the sources: what the compiler has to be told."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rmlx_amd", "csrc")


def _statements():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        for m in re.finditer(r"\basm(?:\s+volatile)?\s*\((.*?)\);", open(path).read(), re.S):
            yield os.path.basename(path), m.group(1).replace("\\n", "\n").replace("\\t", "\t")


def test_statements_that_write_m0_say_so():
    writers = [(name, text) for name, text in _statements() if re.search(r"\bs_\w+ m0,", text)]
    assert len(writers) >= 4
    for name, text in writers:
        assert '"m0"' in text, (name, text)


def test_direct_loads_into_lds_set_m0_in_their_own_statement():
    loads = [(name, text) for name, text in _statements() if re.search(r"buffer_load_\w+ .*\blds\b", text)]
    assert len(loads) >= 4
    for name, text in loads:
        assert re.search(r"\bs_\w+ m0,", text), (name, text)
