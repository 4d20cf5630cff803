"""Kernels whose registers have to hold what they keep there, or leave room for another block: what the compiler gave them, as the
built library says. Needs no GPU."""

import re
import subprocess
from pathlib import Path

import pytest

from qwen3_runtime_amd.ops import build

TOOLS = Path("/opt/rocm/llvm/bin")


def metadata(name, tmp_path, field="private_segment_fixed_size"):
    """A figure of every kernel by its mangled name (bytes of scratch a lane, vgpr_count), from the metadata of a library's gfx950 code objects."""
    so = build.build_library(name)
    subprocess.run([TOOLS / "llvm-objcopy", f"--dump-section=.hip_fatbin={tmp_path}/all", so, tmp_path / "rest"], check=True)
    whole = (tmp_path / "all").read_bytes()
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", whole)]  # one bundle a source file
    found = {}
    for at, end in zip(starts, starts[1:] + [len(whole)]):
        (tmp_path / "bundle").write_bytes(whole[at:end])
        subprocess.run([TOOLS / "clang-offload-bundler", "--unbundle", "--type=o", f"--input={tmp_path}/bundle", f"--output={tmp_path}/object",
                        f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}"], check=True)
        notes = subprocess.run([TOOLS / "llvm-readelf", "--notes", tmp_path / "object"], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            found[re.search(r"\.name:\s+(\S+)", kernel)[1]] = int(re.search(rf"\.{field}:\s+(\d+)", kernel)[1])
    return found


# One-kernel decode steps ask for the token's own head in front of the keys: with both blocks of keys behind it heads of 256 had 404 bytes of
# scratch a lane and were a third slower. What is left there is 88.
@pytest.mark.skipif(not (TOOLS / "llvm-readelf").exists(), reason="needs the compiler's tools")
@pytest.mark.parametrize("library,most", [("attn_bf16_d64", 0), ("attn_bf16_d128", 0), ("attn_bf16_d192", 0), ("attn_bf16_d256", 96)])
def test_decode_attention_keeps_a_token_in_registers(library, most, tmp_path):
    decode = {k: v for k, v in metadata(library, tmp_path).items() if "attention_bf16_decode_kernel" in k}
    assert len(decode) >= 8 and max(decode.values()) <= most, decode


# a block of the router's choice has 16 waves: two share a compute unit's four SIMDs with up to 64 registers a lane
@pytest.mark.skipif(not (TOOLS / "llvm-readelf").exists(), reason="needs the compiler's tools")
def test_two_blocks_of_the_routers_choice_share_a_compute_unit(tmp_path):
    for_many = {k: v for k, v in metadata("core", tmp_path, "vgpr_count").items() if "route_top_lanes_kernel" in k and "Li1ELi4E" in k}
    assert len(for_many) == 2 and max(for_many.values()) <= 64, for_many
