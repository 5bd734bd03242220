"""CPU check of the kernels' sources: a word array in LDS is written and read as words.  The compiler may take
an 8-byte access to it for an access to something else (strict aliasing) and move it past the words' own."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "trianglecount_amd", "csrc")
WORDS = re.compile(r"__shared__\s+(?:__align__\(\d+\)\s+)?uint32_t\s+([^;]*);")
MEMBERS = re.compile(r"struct \w*(?:Lds|Shared)\w* \{(.*?)\n\};", re.S)
WIDE = r"\(\s*(?:const\s+)?(?:uint64_t|unsigned long long)\s*\*\s*\)\s*\(?\s*(?:\w+(?:\.|->))*(\w+)"


def _names(decl):
    return re.findall(r"(\w+)\s*(?:\[[^\]]*\])*\s*(?:,|$)", decl.strip())


def test_lds_words_are_accessed_as_words():
    found = []
    for path in sorted(glob.glob(CSRC + "/*.h") + glob.glob(CSRC + "/*.hip")):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        names = {n for d in WORDS.findall(text) for n in _names(d)}
        for h in [path] + [os.path.join(CSRC, i) for i in re.findall(r'#include "(\w+\.h)"', text)]:
            if os.path.exists(h):
                for body in MEMBERS.findall(re.sub(r"//[^\n]*", "", open(h).read())):
                    names |= {n for d in re.findall(r"uint32_t\s+([^;]*);", body) for n in _names(d)}
        names |= {p for p, a in re.findall(r"uint32_t \*(\w+) = (\w+)", text) if a in names}
        found += [f"{os.path.basename(path)}: {n}" for n in re.findall(WIDE, text) if n in names]
    assert not found, found
