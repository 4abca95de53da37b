"""Hand-written loads that land in LDS: what the compiler would see to, were it not for the asm block."""
import re
from pathlib import Path

SOURCES = sorted((Path(__file__).resolve().parent.parent / "hqmq_amd").glob("csrc*/*.h*"))


def _asm_blocks(text):
    for m in re.finditer(r"\basm\b[^;]*?\(\s*((?:\"(?:[^\"\\]|\\.)*\"|//[^\n]*|\s)+)", text):
        code = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", re.sub(r"//[^\n]*", "", m.group(1))))
        yield [line.strip() for line in re.split(r"\\n|\\t", code) if line.strip()]


def test_a_wait_state_between_m0_and_the_load_that_reads_it():
    """A scalar write of m0 needs one wait state before a load to LDS reads it."""
    seen = 0
    for path in SOURCES:
        for block in _asm_blocks(path.read_text()):
            for line, behind in zip(block, block[1:] + [""]):
                if re.match(r"s_\w+ m0\b", line):
                    seen += 1
                    assert behind.startswith("s_nop"), (path.name, block)
    assert seen >= 4        # attention_fast.hip and read_probes.hip have them


def test_waits_by_count_only_where_the_loads_are_written_by_hand():
    """attn_lds_kernel writes every load it counts; in attn_fast_kernel their number is the compiler's choice, so it may not wait by count."""
    text = next(p for p in SOURCES if p.name == "attention_fast.hip").read_text()
    fast, lds = text.index("void attn_fast_kernel("), text.index("void attn_lds_kernel(")
    bodies = [text[fast:lds], text[lds:text.index("template <", text.index("\n}\n", lds))]]
    bodies[0] = bodies[0][:bodies[0].index("\n}\n")]
    assert "land_tables" in bodies[0] and "land_tables" in bodies[1]
    assert not re.search(r"wait_(vm|groups)\b|s_waitcnt\b", bodies[0])
    assert re.search(r"wait_groups\(", bodies[1])


def test_prefill_waits_for_every_load_before_the_tables_are_read():
    """attn_prefill_kernel's loads are the compiler's beside the landing ones, so it waits for all of them, in every wavefront and before the first
    barrier that the tables are read behind."""
    text = next(p for p in SOURCES if p.name == "attention_prefill.hip").read_text()
    body = text[text.index("void attn_prefill_kernel("):text.index("// Launch plan")]
    assert re.findall(r"wait_vm<\s*(\w+)\s*>|wait_groups|vmcnt", body) == ["0"] and body.count("land_tables<") == 1
    landed, waited = body.index("if (land) land_tables<8>("), body.index("if (land) {\n            wait_vm<0>();")
    met = body.index("if (it == 0) tables();\n    __syncthreads();")
    assert landed < waited < met and "__syncthreads" not in body[landed:met] and body.index("for (int it = 0;") < met
    assert "int64_t rows = gx;" in text and "per <= gx" in text        # at most as many rows as column blocks: the first round is every block's
