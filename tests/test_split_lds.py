"""The LDS words through which a workgroup's waves agree on the split: read
after auto_split's only barrier with no barrier behind the reads, so no other
code may write them.  Shown on the source (a lost race leaves no trace that a
test on the device could rely on)."""
import re
from pathlib import Path

SRC = (Path(__file__).resolve().parents[1] / "cast_amd" / "csrc" / "tree_attn.hip").read_text()


def _body(head):
    """The brace-balanced body that follows the first match of head."""
    m = re.search(head, SRC)
    assert m, head
    i = SRC.index("{", m.end() - 1)
    depth = 0
    for j in range(i, len(SRC)):
        depth += {"{": 1, "}": -1}.get(SRC[j], 0)
        if depth == 0:
            return SRC[i:j + 1]
    raise AssertionError(head)


def test_the_split_choice_owns_its_lds():
    body = _body(r"__device__ void auto_split\(")
    before, after = body.split("__syncthreads();")         # exactly one barrier
    own = re.findall(r"__shared__ [^;]*?(\w+)\[\d+\];", before)
    assert own == ["fit"]                                    # declared here: no other function can name it
    assert len(re.findall(r"\bfit\[[^]]*\] =[^=]", before)) == 1
    assert re.findall(r"\bfit\b", after) and not re.search(r"\bfit\[[^]]*\] =[^=]", after)
    assert not re.search(r"\bauto_split\([^)]*(pack_hi|fit|skr|Ks|Vt)", SRC)   # and no LDS is passed in
