"""build()'s source list: one file for the library and for its sanitizer build,
whatever list the latter's Makefile holds itself."""
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cngpt_amd", "csrc")
sys.path.insert(0, ROOT)

import __graft_entry__ as entry  # noqa: E402


def units(out):
    return {w for w in re.findall(r"([\w]+\.(?:hip|cpp|c)) -o ", out)}


def test_every_source_is_listed():
    listed = {f for v in entry._sources() for f in v.split("=")[1].split()}
    here = {f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp", ".c"))}
    assert listed == here - {"cngpt_cli.c"}  # (linked into the command only)


def test_sanitizer_build_takes_the_library_sources(tmp_path):
    listed = {f for v in entry._sources() for f in v.split("=")[1].split()}
    asan = os.path.join(ROOT, "tests", "asan")
    run = lambda *a: subprocess.run(["make", "-nB", *a], capture_output=True, text=True, check=True).stdout
    assert units(run("-C", asan)) == listed
    # a Makefile with a shorter list of its own, as one from before a source was added
    with open(os.path.join(asan, "Makefile")) as f:
        old = f.read().replace("include $(SRC)/sources.mk",
                               "HIP_SRC := gemm.hip\nCPP_SRC := cngpt_hip.cpp\nC_SRC := fast.c")
    stale = tmp_path / "Makefile"
    stale.write_text(old)
    assert units(run("-C", asan, "-f", str(stale))) == {"gemm.hip", "cngpt_hip.cpp", "fast.c"}
    assert units(run("-C", asan, "-f", str(stale), *entry._sources())) == listed
