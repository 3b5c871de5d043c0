"""Rules on the kernels' sources that no run would notice broken."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "clgpu_amd" / "csrc"


def test_matrix_instructions_are_builtins():
    """An MFMA in an asm statement hides its latency: the compiler then neither waits between a write
    of its operands and it, nor between it and a read of its sum."""
    for path in sorted(CSRC.iterdir()):
        for statement in re.findall(r"\basm\b[^;]*;", path.read_text()):
            assert "mfma" not in statement, (path.name, statement)
