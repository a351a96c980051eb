"""The direct loads into LDS take their place there from m0, which the compiler uses for work of its own: wherever the sources
write such a load by hand, the statement that holds it sets m0 first (here without a GPU)."""
import re
from pathlib import Path

import llm_inference_lab_amd

CSRC = Path(llm_inference_lab_amd.__path__[0]) / "csrc"


def statements(text):
    """The texts of every inline assembly statement, its pieces joined."""
    for match in re.finditer(r"asm\s+volatile\s*\(", text):
        depth, end = 1, match.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[end], 0)
            end += 1
        body = text[match.end():end - 1]
        code = re.match(r'(?:\s*"(?:[^"\\]|\\.)*")+', body)
        yield (code.group(0) if code else ""), body


def test_a_statement_with_a_load_into_lds_sets_m0_itself():
    loads = 0
    for path in sorted(CSRC.glob("*.hip")):
        for code, body in statements(path.read_text()):
            if "load_lds" in code:
                loads += 1
                assert "s_mov_b32 m0" in code.split("global_load_lds")[0], f"{path.name}: {code}"
                assert '"m0"' in body, f"{path.name}: m0 is not named as overwritten: {code}"
    assert loads >= 3
