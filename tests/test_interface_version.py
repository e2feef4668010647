"""The interface version of the kernel library goes up with its entry points: the package refuses a library of another version by saying so,
where one that lacks an entry point, or takes other arguments, would fail at some later call or not at all."""
import hashlib
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# version -> the first of the digest of csrc/api.h's declarations (comments and spaces aside).  An entry point that is added, taken away
# or given other arguments needs a new version in csrc/runtime.hip and kernels/__init__.py, and a line here.
DECLARATIONS = {20: "1e1b23230576f9ec", 21: "19b0612161b5bb86", 22: "24410fd5ad499510", 23: "40662c18965df9ba", 24: "f920d1abedef5fa6",
                25: "5d11631c9e87062c", 26: "b420149118ad7001"}


def declarations(text: str) -> str:
    text = re.sub(r"//[^\n]*|/\*.*?\*/", " ", text, flags=re.S)
    found = sorted(" ".join(d.split()) for d in re.findall(r"\b[\w \*]+\bfllm_\w+\s*\([^;{]*\)\s*;", text))
    assert len(found) > 50
    return hashlib.sha256("\n".join(found).encode()).hexdigest()[:16]


def source(*path: str) -> str:
    with open(os.path.join(ROOT, "fllm_amd", *path)) as fh:
        return fh.read()


def test_the_version_is_that_of_the_entry_points():
    version = int(re.search(r"fllm_abi_version\(void\) \{ return (\d+); \}", source("csrc", "runtime.hip")).group(1))
    assert int(re.search(r"^ABI_VERSION = (\d+)$", source("kernels", "__init__.py"), re.M).group(1)) == version
    assert declarations(source("csrc", "api.h")) == DECLARATIONS.get(version)
