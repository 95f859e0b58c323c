"""A rule on the kernels' sources, checked without a GPU.

The compiler puts the wait states that a matrix instruction's result needs in front of the vector
instructions that it emits itself, and none in front of those inside an asm statement, whose operands'
origin it does not look at. A vector ALU instruction in inline assembly can therefore read scores that an
MFMA has not written yet, with no error. Sources hold none, but for the lane maxima of row16_max4,
whose operands are results of vector instructions on the far side of a barrier."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "in-c-test_amd", "csrc")
ALLOWED = {"v_max_f32_dpp"}


def asm_statements(text):
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"\basm\b(?:\s+volatile)?\s*\(", text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        template = re.match(r"(?:\s*\"(?:[^\"\\]|\\.)*\")*", text[m.end():i]).group(0)
        yield "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", template)).replace("\\n", "\n").replace("\\t", " ")


def test_no_vector_alu_instruction_in_inline_asm():
    seen = 0
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h", ".cpp")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            for template in asm_statements(f.read()):
                seen += 1
                ops = {line.split()[0] for line in template.splitlines() if line.split()}
                bad = {op for op in ops if op.startswith("v_")} - ALLOWED
                assert not bad, (name, template)
    assert seen >= 10  # the parser finds the statements
