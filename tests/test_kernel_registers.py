"""Scratch memory of the grouped GEMM kernels that hold a wave's whole register file, from the code object's own notes: a register that is
spilled around a tile boundary is reloaded behind a wait that drains the LDS-DMA stream."""
import os
import re
import struct
import subprocess

import pytest

from fast_moe_amd.kernels.hip import _lib

TOOLS = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """Demangled kernel name -> bytes of scratch per lane."""
    if not os.path.exists(os.path.join(TOOLS, "llvm-readelf")):
        pytest.skip("no llvm-readelf")
    tmp = tmp_path_factory.mktemp("notes")
    bundle = str(tmp / "fatbin")
    subprocess.run([f"{TOOLS}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", _lib.LIB_PATH, str(tmp / "rest")], check=True)
    data, found = open(bundle, "rb").read(), {}
    for start in (m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):
        count, at = struct.unpack_from("<Q", data, start + 24)[0], start + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" not in target or not size:
                continue
            (tmp / "co").write_bytes(data[start + offset:start + offset + size])
            notes = subprocess.run([f"{TOOLS}/llvm-readelf", "--notes", str(tmp / "co")], capture_output=True, text=True, check=True).stdout
            for kernel in notes.split("- .agpr_count")[1:]:
                name, size_ = (re.search(rf"\.{key}:\s+(\S+)", kernel).group(1) for key in ("name", "private_segment_fixed_size"))
                found[name] = int(size_)
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.split("\n")
    return {n.split("(fmoe::")[0].replace("fmoe::", ""): v for n, v in zip(names, found.values())}


# ring kernels: <configuration, e4m3, epilogue, wtr, kwin, xtr, msc, ktail>; streaming ones: <e4m3, epilogue, msc>
@pytest.mark.parametrize("pattern,most", [
    (r"ring_kernel<RingCfg<256, 256, 2, 4, [124], 2>, true, \d, false, false, false, (true|false), false>", 0),     # scales in the MFMAs or divided out
    (r"ring_kernel<(Mfma16<)?RingCfg<256, 256, 2, 4, [124], 2>( >)?, false, \d, false, false, false, false, (true|false)>", 0),
    (r"ring_kernel<(Mfma16<)?RingSplitCfg<[14]>( >)?, false, ", 20),
    (r"ring_kernel<RingCfg<256, 256, 2, 4, 0, 2>, true, [02], ", 0),
    (r"ring_kernel<RingCfg<256, 256, 2, 4, 0, 2>, true, 1, ", 24),
    (r"ring_kernel<RingCfg<256, 256, 2, 4, 4, 2>, true, \d, false, false, false, (true|false), true>", 32),         # K tails
    (r"ring_kernel<RingSplitCfg<1>, true, ", 40),
    (r"stream_kernel<1, [02], ", 0),
    (r"grouped_wgrad_kernel<", 0),
    (r"stream_kernel<1, 1, ", 44),
])
def test_scratch_of_the_kernels_that_fill_the_register_file(scratch, pattern, most):
    kernels = {n: v for n, v in scratch.items() if re.search(pattern, n)}
    assert kernels, "no such kernel"
    assert not {n: v for n, v in kernels.items() if v > most}
