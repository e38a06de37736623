"""Audit the gfx950 assembly of libsigcomp_hip: which instructions reach memory.

Kernels here read memory through vector and scalar loads and write it through
vector stores only.  The audit recompiles the library to assembly and lists
its scalar instructions and its memory instructions; any that is not named
below fails the build, to be looked at before it is added.
"""

import re
import sys
import tempfile
from pathlib import Path

# scalar instructions: loads, arithmetic, comparisons, moves, branches, waits
SCALAR = re.compile(
    r"s_(?:load_dword(?:x\d+)?"
    r"|(?:abs|add|addc|addk|and|andn2|ashr|bfe|bfm|brev|cselect|ff1|lshl|lshr|max|min|mov|movk|mul|mul_hi|mulk"
    r"|nor|not|or|orn2|sext|sub|subb|xnor|xor)_[iu]?b?\d+(?:_[bi]\d+)?"
    r"|(?:and|andn2|or)_saveexec_b64|bit(?:cmp|set)[01]_b(?:32|64)|cmpk?_(?:eq|ge|gt|le|lg|lt)_[iu](?:32|64)"
    r"|c?branch(?:_\w+)?|barrier|endpgm|getpc_b64|setpc_b64|swappc_b64|nop|sleep|waitcnt)")
# vector memory and LDS instructions
VECTOR = re.compile(
    r"(?:global|buffer|scratch)_(?:load|store)_(?:dword(?:x[234])?|[us]?byte|[us]?short)"
    r"|ds_(?:read|write)2?(?:st64)?_[bui]\d+|ds_(?:bpermute_b32|max_i32|or_b32)")
MEMORY = re.compile(r"(?:global|buffer|scratch|flat|image|tbuffer|ds)_")


def check(asm: str) -> None:
    """RuntimeError when an instruction of `asm` is not one of the above."""
    names = set(re.findall(r"^[ \t]+([a-z][a-z0-9_]*)(?=[ \t\n])", asm, re.M))
    other = sorted(n for n in names if n.startswith("s_") and not SCALAR.fullmatch(n))
    other += sorted(n for n in names if MEMORY.match(n) and not VECTOR.fullmatch(n))
    if other:
        raise RuntimeError(f"instructions in device code that isa_audit does not list: {other}")


def audit() -> None:
    sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
    from sigcomp_amd.build import device_asm
    with tempfile.TemporaryDirectory() as tmp:
        asm = device_asm(Path(tmp) / "sc.s").read_text()
    check(asm)
    n_mfma = len(re.findall(r"v_mfma_i32_32x32x32_i8", asm))
    print(f"isa audit ok ({n_mfma} int8 MFMA instructions, memory written by vector stores only)")


if __name__ == "__main__":
    audit()
