"""Where the fused step's kernels wait for memory, read from the built library's own machine code.

A boundary node's operator list is loaded ahead of the node's pull so that both are under way together.
Whether they are is the compiler's doing: it has twice put a wait for the list between the two, which
shows in no result and costs a small grid's step a memory round trip."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "panslbm2_amd", "libpanslbm2_hip.so")
TOOLS = "/opt/rocm/llvm/bin"
OBJDUMP, READELF = (os.path.join(TOOLS, t) for t in ("llvm-objdump", "llvm-readelf"))


def _out(*cmd):
    return subprocess.run(cmd, check=True, stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True).stdout


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    if not all(os.path.exists(p) for p in (LIB, OBJDUMP, READELF)):
        pytest.skip("library not built, or no LLVM tools")
    d = tmp_path_factory.mktemp("code")
    lib = shutil.copy(LIB, d)  # the code objects are written beside it
    _out(OBJDUMP, "--offloading", lib)
    objects = [os.path.join(d, f) for f in os.listdir(d) if "gfx950" in f]
    assert objects
    return {o: _out(READELF, "--symbols", "--wide", o) for o in objects}


def _kernel(objects, prefix):
    for o, symbols in objects.items():
        m = re.search(r"FUNC .* (%s\w*)$" % prefix, symbols, re.M)
        if m:
            return _out(OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + m.group(1), o).splitlines()
    raise AssertionError("no kernel " + prefix)


@pytest.mark.parametrize("la,lb,nc", [("4D2Q9", "4D2Q5", 14), ("5D3Q15", "4D3Q7", 22)], ids=["2d", "3d"])
@pytest.mark.parametrize("body", ["6ADBody", "7AADBody"], ids=["fwd", "adj"])
def test_pull_is_under_way_before_the_operator_list_is_waited_for(code_objects, la, lb, nc, body):
    lb_again = "S2_"
    code = _kernel(code_objects, "_ZN3lbm15k_collide_fusedINS_%sENS_%sENS_%sIS1_%sdEEdE" % (la, lb, body, lb_again))
    # the list: a node's header and values, 16 bytes at a time from one address
    at = max(i for i, x in enumerate(code[:len(code) // 3])
             if "global_load_dwordx4" in x and re.search(r"off offset:(16|32)\b", x))
    loads = 0
    for x in code[at + 1:]:
        if "s_waitcnt" in x and "vmcnt" in x:
            break
        loads += "global_load_dwordx2" in x
    assert loads >= nc, "%d of %d populations are loaded before the first wait after the list's loads" % (loads, nc)
