"""What the C header says about names that other files define."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minife_amd", "csrc")


def header_comment(before):
    """The comment in front of a declaration, in one line."""
    with open(os.path.join(ROOT, "include", "minife_hip.h")) as f:
        text = f.read()
    at = text.index(before)
    return re.sub(r"\s*\n \*\s*", " ", text[text.rindex("/*", 0, at):at])


def test_batch_phases_are_the_ones_the_header_describes():
    """Batch.PHASES names the columns that mfe_batch_timing fills, in their order."""
    import minife_amd
    doc = header_comment("int mfe_batch_timing(")
    at = [re.search(rf"\b{name}\b", doc) for name in minife_amd.Batch.PHASES]
    assert len(at) == 6 and all(at), list(zip(minife_amd.Batch.PHASES, at))
    assert [a.start() for a in at] == sorted(a.start() for a in at)


def test_environment_variables_are_documented():
    """Every environment variable that the library reads is described in its header."""
    with open(os.path.join(ROOT, "include", "minife_hip.h")) as f:
        text = f.read()
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as f:
            for var in re.findall(r'getenv\("(\w+)"\)', f.read()):
                assert var in text, (name, var)
