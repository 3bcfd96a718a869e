"""Checks of the kernel sources themselves, for faults that no run shows reliably."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "xreg_amd" / "csrc"


def test_waits_order_memory():
    """A wait written as inline assembly orders the memory accesses around it only if it says so: without
    a "memory" clobber the compiler may read LDS that is still being filled ahead of the wait."""
    waits = [(p.name, m.group(0)) for p in sorted(CSRC.glob("*.h*"))
             for m in re.finditer(r'asm\s+(?:volatile\s*)?\([^;]*?s_waitcnt[^;]*;', p.read_text())]
    assert len(waits) >= 2
    assert [w for w in waits if '"memory"' not in w[1]] == []
