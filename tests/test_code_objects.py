"""What the compiler made of the kernels, read from the gfx950 code objects of
the library built here: properties that results do not show (cache hints,
registers spilled to memory)."""

import os
import re
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"

pytestmark = pytest.mark.skipif(not os.path.exists(LLVM + "/llvm-objdump"),
                                reason="ROCm's LLVM tools are not installed")


def _run(*cmd):
    return subprocess.run(cmd, check=True, capture_output=True, text=True).stdout


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled kernel name: (mangled name, code object path)}"""
    from mojodgl import _lib

    _lib.lib()
    tmp = tmp_path_factory.mktemp("code")
    fat = str(tmp / "fatbin")
    _run(LLVM + "/llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, _lib.LIB,
         os.devnull)
    data = open(fat, "rb").read()
    at = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)]
    names = {}
    for i, start in enumerate(at):
        def word(o):
            return int.from_bytes(data[start + o:start + o + 8], "little")

        o = 32
        for _ in range(word(24)):
            off, size, length = word(o), word(o + 8), word(o + 16)
            target = data[start + o + 24:start + o + 24 + length].decode()
            o += 24 + length
            if "gfx950" not in target:
                continue
            path = str(tmp / "code{}".format(i))
            open(path, "wb").write(data[start + off:start + off + size])
            mangled = [line.split()[-1] for line in _run(LLVM + "/llvm-readelf", "-sW",
                                                         path).splitlines() if " FUNC " in line]
            plain = _run("c++filt", *mangled).splitlines() if mangled else []
            names.update(zip(plain, ((m, path) for m in mangled)))
    assert names
    return names


def _named(kernels, pattern):
    got = {k: v for k, v in kernels.items() if re.match("void mdgl::" + pattern, k)}
    assert got, pattern
    return got


def _asm(kernel):
    return _run(LLVM + "/llvm-objdump", "-d", "--no-show-raw-insn",
                "--disassemble-symbols=" + kernel[0], kernel[1])


@pytest.mark.parametrize("pattern", [
    # copy_e and mul with both operands contiguous; sum, and max
    r"gspmm_kernel<float, 6, 0, 4, 0, \d>", r"gspmm_kernel<double, 6, 0, 2, 0, \d>",
    r"gspmm_kernel<float, 2, 0, 4, 0, \d>", r"gspmm_kernel<double, 2, 1, 2, 0, \d>"])
def test_edge_rows_stream_past_the_caches(kernels, pattern):
    """Wide edge rows are read once per edge: the loads of a batch of eight carry
    the non-temporal hint, so that they leave the source rows, read again, in the
    caches. Narrow ones, which share lines, do not (path 7 beside path 0)."""
    near = re.sub(r"0, (\\d>)$", r"7, \1", pattern)
    for paths, hints in ((pattern, True), (near, False)):
        for name, kernel in _named(kernels, paths).items():
            rows = re.findall(r"global_load_dwordx4 .*", _asm(kernel))
            hinted = sum(bool(re.search(r"\bnt\b", r)) for r in rows)
            assert (hinted >= 8) if hints else (rows and hinted == 0), name


def _notes(kernel):
    """The kernel's entry in its code object's metadata."""
    notes = _run(LLVM + "/llvm-readelf", "--notes", kernel[1])
    return next(e for e in notes.split("- .agpr_count")
                if re.search(r"\.name: +" + re.escape(kernel[0]) + r"\s", e))


def test_dots_of_whole_vectors_keep_eight_wavefronts(kernels):
    """64 registers at most: eight wavefronts per SIMD wait for their rows."""
    (kernel,) = _named(kernels, r"gsddmm_dot_kernel<float, 4, 0>").values()
    assert int(re.search(r"\.vgpr_count: +(\d+)", _notes(kernel)).group(1)) <= 64


@pytest.mark.parametrize("pattern", [r"grouped_tn_(tile_)?kernel<", r"grouped_gemm_any_kernel<"])
def test_grouped_products_keep_their_registers(kernels, pattern):
    """No instance spills: three steps of a 64 x 64 tile of doubles did, two
    groups of four rows each, and one column block at five wavefronts per SIMD."""
    for name, kernel in _named(kernels, pattern).items():
        assert re.search(r"\.private_segment_fixed_size: 0\b", _notes(kernel)), name
