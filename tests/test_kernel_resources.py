"""What the built kernels take of a compute unit, as the code objects in the
library state it: registers and LDS, which bound how many wavefronts the launch
rules may count on, and spills."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "qkxtm_mpi_amd", "libqkx_hip.so")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 code objects of every offload bundle in the library."""
    at = 0
    while (at := blob.find(MAGIC, at)) >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, tlen = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24: p + 24 + tlen] and size:
                yield blob[at + off: at + off + size]
            p += 24 + tlen
        at += len(MAGIC)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    found = {}
    f = tmp_path_factory.mktemp("co") / "code.elf"
    for co in _code_objects(open(LIB, "rb").read()):
        f.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for k in notes.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name: +(\S+)", k[k.rindex(".group_segment_fixed_size"):]).group(1)
            found[name] = {w: int(re.search(rf"\.{w}: +(\d+)", k).group(1))
                           for w in ("vgpr_count", "vgpr_spill_count", "group_segment_fixed_size")}
    assert found
    return found


def named(kernels, part):
    ks = {n: k for n, k in kernels.items() if part in n}
    assert ks, part
    return ks


def test_batched_direction_step_occupancy(kernels):
    """Four wavefronts per SIMD at least: 128 of its 512 registers."""
    for n, k in named(kernels, "cgb_dir_kernel").items():
        assert k["vgpr_count"] <= 128 and k["vgpr_spill_count"] == 0, (n, k)


def test_weight_gradient_lds(kernels):
    """One sum buffer for all path groups, sized by the launch: nothing static, so
    that the eight 64-thread workgroups which the launch rule counts on per CU
    (160 KB of LDS) are resident whatever the hidden channels."""
    for n, k in named(kernels, "net_wgrad_kernel").items():
        assert k["group_segment_fixed_size"] * 8 <= 160 * 1024, (n, k)


def test_learned_kernels_do_not_spill(kernels):
    """The network's layers and gradients keep their sums in registers."""
    for part in ("net_wgrad_kernel", "net_expand_kernel", "net_contract_kernel", "eo_hidden_kernel", "eo_out_kernel"):
        for n, k in named(kernels, part).items():
            assert k["vgpr_spill_count"] == 0, (n, k)
