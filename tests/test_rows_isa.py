"""Row kernels whose streams are never read past the caches keep to loads and stores of their own types."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "csrc" / "kernels"


def test_plain_vectors_are_not_built_for_the_nontemporal_ones():
    """The nontemporal builtins want vector types of their own; where they are not used, loads as those types changed the compiler's
    order in kernels that had nothing to gain (4800 and 16 000 rows of 4096 of a recurrence 5 and 7 % slower)."""
    src = (CSRC / "rows.h").read_text()
    for name in ("row_f4", "row_u2"):
        for line in src.splitlines():
            if name in line and not line.startswith("typedef"):
                assert "__builtin_nontemporal" in line, line
    assert len(re.findall("__builtin_nontemporal", src)) == 4


def test_streams_past_the_caches_do_not_fit_them():
    """x (4 bytes a value), a product's 4 and two 16-bit rows' of a gated norm are 256 MB together where x goes past them."""
    past = int(re.search(r"PAST_BYTES = (\d+)ll << 20", (CSRC / "rows.h").read_text()).group(1))
    assert past * (4 + 4 + 2 + 2) / 4 >= 256
