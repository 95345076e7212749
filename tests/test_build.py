"""The HIP libraries: no execution path without them, and clear errors on the way to them."""

import re
import struct
import subprocess
from pathlib import Path

import pytest

from clockwork_amd import ops
from clockwork_amd.csrc import build


def test_head_sizes_outside_the_kernels_range_are_refused_by_name():
    for hd in (8, 24, 272):
        with pytest.raises(ValueError, match="head sizes in steps of 16"):
            build.library_path("attention", hd)
    with pytest.raises(KeyError):
        build.library_path("no_such_library")


def test_a_library_that_cannot_be_built_is_an_error_not_a_fallback(monkeypatch):
    """Nothing is built and there is no compiler: the first op that needs a library raises."""
    monkeypatch.setattr(build, "_find_built", lambda name, head_dim: None)
    monkeypatch.setenv("HIPCC", "/nonexistent/hipcc")
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    monkeypatch.setattr(build.Path, "exists", lambda self: False)
    monkeypatch.setattr(ops, "_libs", {})
    with pytest.raises(RuntimeError, match="hipcc was not found"):
        ops._load("core")


def test_a_library_that_does_not_load_is_an_error(monkeypatch, tmp_path):
    broken = tmp_path / "core-broken.so"
    broken.write_bytes(b"not a shared object")
    monkeypatch.setattr(build, "ensure_built", lambda name, head_dim=None: broken)
    monkeypatch.setattr(ops, "_libs", {})
    with pytest.raises(ops.KernelError, match="cannot load the HIP library"):
        ops._load("core")


def test_the_digest_follows_the_source_and_the_flags(monkeypatch):
    before = build.library_path("core").name
    monkeypatch.setattr(build, "FLAGS", build.FLAGS + ["-DSOMETHING_ELSE"])
    assert build.library_path("core").name != before


def test_the_target_rules_xnack_out_unless_told_otherwise(monkeypatch):
    monkeypatch.delenv("CLOCKWORK_AMD_ARCH", raising=False)
    assert build.target_arch() in ("gfx950:xnack-", "gfx950")  # the latter only on a card with XNACK on
    monkeypatch.setenv("CLOCKWORK_AMD_ARCH", "gfx950")
    assert build.target_arch() == "gfx950"
    assert "--offload-arch" not in " ".join(build.FLAGS)  # the target is added per compile


def _assembly_statements(text: str):
    """The inline assembly of a source, statement by statement."""
    for found in re.finditer(r"\basm\s+(?:volatile\s*)?\(", text):
        depth, at, quoted = 1, found.end(), False
        while depth:
            c = text[at]
            if c == "\\":
                at += 1
            elif c == '"':
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            at += 1
        yield text[found.start() : at]


def test_inline_assembly_names_the_scalar_register_that_it_writes():
    """The compiler keeps values in m0 of its own (LDS loads, lane writes, registers chosen at run time): a statement
    that writes it has to say so."""
    statements = [a for path in sorted(build.CSRC.glob("*.h*")) for a in _assembly_statements(path.read_text())]
    writers = [a for a in statements if re.search(r"\bs_\w+ m0\b", a)]
    assert len(statements) > len(writers) >= 3
    assert [a for a in writers if '"m0"' not in a] == []


def test_no_limit_of_lds_follows_the_launches():
    """A limit that is raised to what a launch takes, and remembered, may be lowered again by a thread that remembers an
    older one: kernels whose launches differ in LDS are allowed their most at once."""
    for path in sorted(build.CSRC.glob("*.h*")):
        assert re.findall(r"\bstatic\s+(?!bool\b)\w+\s+raised\b.*", path.read_text()) == [], path.name

    # (the kernels that raise theirs at every launch are older than this rule; no new ones)
    launches = (build.CSRC / "sink_attention.hip").read_text()
    assert not re.search(r"hipFuncSetAttribute\(\(const void\*\)sink_decode_runs_beside_kernel", launches)


LLVM = Path("/opt/rocm/llvm/bin")


def _code_objects(path: Path):
    """The ELF files for the GPU inside a built library."""
    data, mark = path.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(mark)
    while at >= 0:
        (count,), entry = struct.unpack_from("<Q", data, at + len(mark)), at + len(mark) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"amdgcn" in data[entry + 24 : entry + 24 + length] and size:
                yield data[at + offset : at + offset + size]
            entry += 24 + length
        at = data.find(mark, at + 1)


def _llvm(tool: str, library: str, tmp_path, *options) -> str:
    out = []
    for i, code in enumerate(_code_objects(build.ensure_built(library))):
        file = tmp_path / f"{library}{i}.co"
        file.write_bytes(code)
        out.append(subprocess.run([LLVM / tool, *options, file], capture_output=True, text=True, check=True).stdout)
    assert out
    return "\n".join(out)


def _instructions(library: str, tmp_path, pattern: str) -> dict:
    """Kernels whose names match -> their instructions in order."""
    found = {}
    for part in re.split(r"\n(?=[0-9a-f]+ <)", _llvm("llvm-objdump", library, tmp_path, "-d", "--no-show-raw-insn")):
        head = re.match(r"[0-9a-f]+ <(\S+)>:", part)
        if head and re.search(pattern, head.group(1)):
            found[head.group(1)] = [line.split("//")[0].strip() for line in part.split("\n")[1:] if line.strip()]
    return found


def _registers(operands: str) -> set:
    out = {(kind, n) for kind, first, last in re.findall(r"\b([av])\[(\d+):(\d+)\]", operands) for n in range(int(first), int(last) + 1)}
    return out | {(kind, int(n)) for kind, n in re.findall(r"\b([av])(\d+)\b", operands)}


def test_products_written_in_assembly_wait_for_their_operands(tmp_path):
    """The compiler does not see that they are products. In the code as built: a tile's first ones begin with a zero of
    their own; no vector instruction writes an operand less than two states before the product that reads it, and none
    looks at a result less than twelve states behind the product that writes it (8 passes of 16 x 16 x 32)."""
    kernels = _instructions("gemm_tile", tmp_path, r"gemm_wide_bf16_kernelILi\d+ELi8ELi9E")
    assert len(kernels) >= 2
    for name, code in kernels.items():
        products = [i for i, x in enumerate(code) if x.startswith("v_mfma")]
        assert sum(code[i].endswith(", 0") for i in products) == 72, name
        for i in products:
            result, *operands = code[i].split(None, 1)[1].split(", ")
            written, read = _registers(result), set().union(*map(_registers, operands))
            states = 0
            for x in reversed(code[max(0, i - 4) : i]):
                if states >= 2:
                    break
                if x.startswith("s_nop"):
                    states += int(x.split()[1]) + 1
                    continue
                assert not (x.startswith("v_") and not x.startswith("v_mfma") and _registers(x.split(None, 1)[1].split(", ")[0]) & read), (name, x, code[i])
                states += 1
            states = 0
            for x in code[i + 1 : i + 13]:
                if states >= 12:
                    break
                if x.startswith("s_nop"):
                    states += int(x.split()[1]) + 1
                    continue
                assert x.startswith(("s_", "v_mfma")) or not _registers(x) & written, (name, code[i], x)
                states += 1


def test_the_wide_tiles_keep_everything_in_registers(tmp_path):
    """What a tile's end fetches back from scratch waits for the loads of the next tile that are in flight."""
    kernels = re.split(r"\n\s+- \.agpr_count", _llvm("llvm-readelf", "gemm_tile", tmp_path, "--notes"))[1:]
    wide = [k for k in kernels if "gemm_wide_bf16_kernel" in k]
    assert len(wide) > 30
    for kernel in wide:
        found = dict(re.findall(r"\.(name|vgpr_spill_count|private_segment_fixed_size):\s+(\S+)", kernel))
        assert found["vgpr_spill_count"] == found["private_segment_fixed_size"] == "0", found
