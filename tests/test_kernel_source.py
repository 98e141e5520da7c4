"""Checks of the kernels' source text."""

import glob
import os
import re

import ludwig_amd

CSRC = os.path.join(os.path.dirname(ludwig_amd.__file__), "csrc")


def test_inline_assembly_writes_no_register_behind_the_compiler():
    # a register written by name inside an asm text is neither operand nor,
    # for the reserved ones, a clobber the compiler honours
    found = 0
    for path in glob.glob(os.path.join(CSRC, "*")):
        text = open(path).read()
        for m in re.finditer(r'asm\s+volatile\s*\(\s*((?:"[^"]*"\s*)+)', text):
            found += 1
            for ins in re.split(r"\\n|\\t|;", "".join(re.findall(r'"([^"]*)"', m.group(1)))):
                dst = re.match(r"\s*[sv]_\w+\s+(m0|vcc\w*|exec\w*|[sv]\d+|[sv]\[\d)", ins)
                assert not dst, (os.path.basename(path), ins)
    assert found >= 2
