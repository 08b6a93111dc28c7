"""The library's make rules, run with a stand-in for the compiler: what is compiled again after an edit of a header, and
where the compiler's list of an object's headers is missing."""
import os
import shutil
import subprocess
import sys
import time

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sable_amd", "csrc")

# notes the object, writes it, and lists its headers as the compiler would
COMPILER = """#!%s
import os, sys
args = sys.argv[1:]
out = args[args.index("-o") + 1]
if "-c" in args:
    open("compiled.txt", "a").write(out + "\\n")
    if "-MMD" in args:
        open(out[:-2] + ".d", "w").write("%%s: %%s field.hpp\\nfield.hpp:\\n" %% (out, args[args.index("-c") + 1]))
open(out, "w").write("")
"""


@pytest.fixture(scope="module")
def tree(tmp_path_factory):
    """A copy of the sources, built once; run() makes the library again and returns the objects it compiled."""
    root = tmp_path_factory.mktemp("build")
    csrc = root / "sable_amd" / "csrc"
    keep = lambda d, names: [n for n in names if n == "gen" or n.endswith((".o", ".d"))]  # noqa: E731
    shutil.copytree(CSRC, csrc, ignore=keep)
    shutil.copytree(os.path.join(CSRC, "..", "..", "include"), root / "include")
    compiler = root / "compiler"
    compiler.write_text(COMPILER % sys.executable)
    compiler.chmod(0o755)

    def run():
        log = csrc / "compiled.txt"
        if log.exists():
            log.unlink()
        subprocess.run(["make", "-s", "-j4", "HIPCC=%s" % compiler], cwd=csrc, check=True, timeout=300,
                       env={k: v for k, v in os.environ.items() if k not in ("MAKEFLAGS", "MAKELEVEL")})
        return set(log.read_text().split()) if log.exists() else set()

    run.csrc, run.first = csrc, run()
    return run


# seconds of age: the sources, then what each step of the build made from the one before
AGES = [("stmtgen", 190), (".hip", 180), (".inc", 180), (".stamp", 170), (".d", 160), (".o", 150), (".objects", 140)]


def age(csrc):
    """Everything as it is, but made minutes ago."""
    now = time.time()
    for folder, _, names in os.walk(csrc):
        for n in names:
            made = [a for end, a in AGES if n.endswith(end)]
            old = 200 if not made or (n.endswith(".hip") and folder == str(csrc)) else made[0]
            os.utime(os.path.join(folder, n), (now - old, now - old))
    os.utime(csrc.parent / "libexacta_hip.so", (now - 130, now - 130))


def test_a_build_that_is_up_to_date_compiles_nothing(tree):
    assert {"context.o", "interp_r4.o", "interp_t8.o", "prover.o", "gen/stmt0.o"} <= tree.first
    age(tree.csrc)
    assert tree() == set()


@pytest.mark.parametrize("name", ["commit", "prover", "interp_t4", "gen/stmt3"])
def test_an_object_without_its_list_of_headers_is_compiled_again(tree, name):
    age(tree.csrc)
    os.unlink(tree.csrc / (name + ".d"))
    assert tree() == {name + ".o"}
    assert (tree.csrc / (name + ".d")).exists()


def test_an_edited_header_reaches_every_object_that_lists_it(tree):
    age(tree.csrc)
    at = time.time() - 40
    os.utime(tree.csrc / "field.hpp", (at, at))
    assert tree() >= {o for o in tree.first if o.startswith(("gen/", "interp_")) or o in ("commit.o", "prover.o")}
