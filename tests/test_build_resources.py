"""What the compiler made of the chain kernels, read from the built library's own metadata (no GPU): the persistent chain
kernels run 12 waves per CU at 168 registers a lane, and a register spilled around their out-of-line ops is paid for by every
chain, whether it holds such an op or not (chains of 5 rows lost 15% to 6 more of them)."""
import re
import shutil
import struct
import subprocess

from p0pc0rn_amd import capi

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
# most spilled registers per kernel <M, q8>; the q8 instantiations of M > 1 are left out (they hold both arithmetics)
LIMITS = {"q4_chain_pipe_kernelILi1ELb0EE": 0, "q4_chain_pipe_kernelILi1ELb1EE": 0, "q4_chain_pipe_kernelILi2ELb0EE": 0,
          "q4_chain_pipe_kernelILi3ELb0EE": 0, "q4_chain_pipe_kernelILi4ELb0EE": 0, "q4_chain_pipe_kernelILi5ELb0EE": 3,
          "q4_chain_wide_kernelILi8EE": 5, "q4_chain_wide_kernelILi16EE": 5}


def _spills(tmp_path):
    data = open(capi.LIB_PATH, "rb").read()
    out, at = {}, data.find(MAGIC)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idl = struct.unpack_from("<QQQ", data, p)
            ident = data[p + 24:p + 24 + idl].decode()
            p += 24 + idl
            if "gfx950" in ident and size:
                f = tmp_path / "code.elf"
                f.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
                for name, spill in re.findall(r"\.name: +(_ZN2p0\S+).*?\.vgpr_spill_count: +(\d+)", notes, re.S):
                    out[re.sub(r"^_ZN2p0\d+", "", name)] = int(spill)
        at = data.find(MAGIC, at + 1)
    return out


def test_chain_kernels_spill_no_more_registers(tmp_path):
    got = _spills(tmp_path)
    assert len(got) > 50
    for kernel, most in LIMITS.items():
        hit = [v for k, v in got.items() if k.startswith(kernel)]
        assert len(hit) == 1 and hit[0] <= most, (kernel, hit, most)
