"""The kernels hold no instruction in inline assembly.  The compiler keeps the wait states between dependent instructions
(a v_readlane and a vector instruction that reads its scalar result, among others) for the instructions that it emits, not
for those inside an asm statement, so one there is right only by what happens to stand before it.  Empty asm statements,
which pin a value, are not meant."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parent.parent / "surfaceonlydeformables_amd" / "csrc"


def test_asm_statements_are_empty():
    files = [p for p in CSRC.iterdir() if p.suffix in (".hip", ".hpp", ".cpp")]
    assert files
    for p in files:
        for m in re.finditer(r"\basm\b(?:\s+(?:volatile|goto|inline))*\s*\(\s*(R?\"[^\"]*\")", p.read_text()):
            assert m[1] == '""', (p.name, m[0])
