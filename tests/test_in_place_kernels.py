"""The reductions that run in place (the FP64 form puts its reflectors over H(k), the
blocked kernel leaves the trailing block for the next one where it was) take input and
reflectors as pointers that may overlap, and the grids of the complex64 chain their
hand-over block too: none may be declared __restrict__, which would let the compiler move
a load of the matrix past a store."""
from __future__ import annotations

import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ultimateepm_amd", "csrc")


@pytest.mark.parametrize("source,kernel", [("tridiag_grid.hpp", "tridiag_reg_kernel"), ("tridiag_row.hpp", "tridiag_row_kernel"),
                                           ("tridiag_strip.hpp", "tridiag_strip_kernel"),
                                           ("tridiag_blocked.hip", "tridiag_blocked_kernel")])
def test_input_and_reflectors_may_overlap(source, kernel):
    with open(os.path.join(CSRC, source)) as f:
        text = f.read()
    args = re.search(r"\bvoid " + kernel + r"\((.*?)\)\s*\{", text, re.S).group(1)
    for name in ("Hin", "Vout") + (("Bout",) if kernel == "tridiag_reg_kernel" else ()):
        arg = [a for a in args.split(",") if re.search(r"\b" + name + r"$", a.strip())]
        assert len(arg) == 1, (kernel, name, args)
        assert "__restrict__" not in arg[0], (kernel, arg[0])
