"""Promises that kernels make to the compiler, read from the device IR of this package's own
sources (compiled here for gfx950; no GPU is needed)."""
import os
import re
import subprocess

import pytest

from catboost_rs_amd import build as B


@pytest.fixture(scope="module")
def ir(tmp_path_factory):
    """Device IR, with argument names, of the kernels that the wrapper names."""
    d = tmp_path_factory.mktemp("ir")
    src, out = d / "k.hip", d / "k.ll"
    src.write_text('#include "kernels.hpp"\n'
                   "namespace cbh { auto* leaf_values = &leaf_values_kernel<1>; }\n"
                   "void* referenced() { return (void*)cbh::leaf_values; }\n")
    cmd = [B.HIPCC, "-x", "hip"] + B.DEVICE + B.COMMON + ["-I", B.CSRC, "--cuda-device-only", "-fno-discard-value-names",
                                                          "-S", "-emit-llvm", str(src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out.read_text()


def _arguments(ir, kernel):
    """Attributes of a kernel's arguments by name."""
    line, = [l for l in ir.splitlines() if l.startswith("define") and kernel in l]
    args = line[line.index("("):]
    return {m.group(2): m.group(1).split() for m in re.finditer(r"ptr addrspace\(1\) ([^%]*)%(\w+?)(?:\.coerce)?[,)]", args)}


def test_leaf_values_publishes_what_it_stored(ir):
    """With one output the kernel stores the leaf values into the tree's result block and then copies
    the whole block to the host, so neither pointer may claim that nothing else reaches its
    memory: with that claim the copy may be moved ahead of the stores, and the caller would get the
    leaf values of the tree before."""
    args = _arguments(ir, "leaf_values_kernelILi1E")
    assert {"raw", "out", "host"} <= set(args)
    assert "noalias" not in args["raw"]
    assert "noalias" not in args["out"]
