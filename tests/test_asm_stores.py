"""Inline assembly of the kernels: a store of more than eight bytes reads its registers over several cycles.  The compiler keeps two wait states between its own stores and
an instruction that overwrites their data, but does not look inside a statement of ours, so the statement has to end with them."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parent.parent / "qserve_amd" / "csrc"


def _wait_states_behind_stores(text):
    """-> for every wide store in an asm statement, the wait states behind it in that statement"""
    for body in re.findall(r'asm\s*(?:volatile)?\s*\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', text):
        lines = [x.strip() for x in "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', body)).replace("\\t", " ").split("\\n")]
        for i, x in enumerate(lines):
            if re.match(r"(global|flat|buffer)_store_(dwordx[34]|b96|b128)", x):
                yield sum(int(y.split()[1]) + 1 if y.startswith("s_nop") else 1 for y in lines[i + 1:] if y)


def test_wide_stores_end_with_two_wait_states():
    found = {p.name: list(_wait_states_behind_stores(p.read_text())) for p in sorted(CSRC.rglob("*")) if p.suffix in (".hip", ".h")}
    assert sum(map(len, found.values())) >= 6
    assert {n: w for n, w in found.items() if any(x < 2 for x in w)} == {}
