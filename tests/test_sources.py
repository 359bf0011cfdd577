"""Properties of the kernel sources that a run does not show."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "nanopd_amd" / "csrc"


@pytest.mark.parametrize("src", sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")),
                         ids=lambda p: p.name)
def test_inline_asm_that_writes_m0_says_so(src):
    """m0 is the compiler's too (indexed moves, its own direct-to-LDS loads): a
    statement that writes it has to name it as clobbered."""
    for stmt in re.findall(r"asm volatile\((.*?)\);", src.read_text(), flags=re.S):
        if re.search(r"\bs_mov_b32 m0\b", stmt):
            assert '"m0"' in stmt.rsplit(":", 1)[1], stmt


@pytest.mark.parametrize("src", sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")),
                         ids=lambda p: p.name)
def test_no_bit_cast_of_a_vector_element(src):
    """__builtin_bit_cast(T, v[i]) reads element 0 of an ext_vector whatever i
    is: the element goes through a variable of its own first."""
    assert not re.findall(r"__builtin_bit_cast\([^,()]*,\s*[\w.]+(?:\[[^\]]*\])+\s*\)", src.read_text())
