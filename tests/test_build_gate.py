"""The build stops when a kernel that issues its loads by hand spills or uses scratch memory (no GPU)."""
import re
import subprocess
from pathlib import Path

import pytest

from dlcompiler_amd.build import ARCH, CSRC_DIR, HIPCC, OBJ_DIR, check_hand_scheduled, kernel_resources

# kernels that run the helpers of inline-assembly loads, or the key walk of the paged decode kernels, which
# looks pages up with hand-issued scalar loads
KERNELS = ["moe_gemm_kernel", "moe_stream_kernel", "prefill_attn_kernel", "paged_decode_split_kernel",
           "paged_decode_direct_kernel"]


@pytest.mark.parametrize("kernel", KERNELS)
def test_spills_and_scratch_are_refused(kernel):
    name = f"_ZN3dlb12_GLOBAL__N_1{len(kernel)}{kernel}ILi0EEEv"
    assert not check_hand_scheduled({name: {"scratch_bytes": 0, "vgpr_spills": 0}})
    assert check_hand_scheduled({name: {"scratch_bytes": 8, "vgpr_spills": 0}})
    assert check_hand_scheduled({name: {"scratch_bytes": 0, "vgpr_spills": 1}})
    assert check_hand_scheduled({name: {"scratch_bytes": 0}})
    assert check_hand_scheduled({}, f"void {kernel}(")


def test_every_kernel_with_hand_issued_loads_is_named():
    """Sources that issue loads by hand hold no kernel outside the gate but these, which use ordinary loads."""
    ordinary = {"prefill_combine_kernel", "paged_decode_combine_kernel", "quant_fp8_group128_kernel",
                "moe_topk_sum_kernel"}
    for src in CSRC_DIR.glob("*.hip"):
        text = src.read_text()
        if re.search(r"dma\d+_global_to_lds|s_load_dword|buffer_of\(", text):
            assert set(re.findall(r"void (\w+_kernel)\(", text)) - ordinary <= set(KERNELS), src.name


def test_short_head_dims_keep_their_waves():
    """128-row prefill workgroups of 64 dims: three per CU, so 512 / 3 registers in steps of 8."""
    reports = [r for name, r in kernel_resources().items()
               if re.search(r"prefill_attn_kernelILi\dELi64ELi\dELb\dELi4E", name)]
    assert reports and all(r["occupancy"] >= 3 and r["vgprs"] <= 168 for r in reports)


def test_the_build_reports_every_gated_kernel():
    built = kernel_resources()
    for kernel in KERNELS:
        reports = [r for name, r in built.items() if kernel in name]
        assert reports and all(r["scratch_bytes"] == r["vgpr_spills"] == 0 for r in reports), kernel


def test_no_instance_that_no_dispatch_reaches():
    """Grouped GEMM with few rows: 16-row tiles split K over one column wave, taller ones over two."""
    shapes = {m.groups() for m in (re.search(r"moe_stream_kernelILb\dELi\dELi\dELi\dELi(\d)ELi(\d)ELi(\d)E", name)
                                   for name in kernel_resources()) if m}
    assert shapes == {("4", "1", "1"), ("4", "2", "1"), ("1", "4", "1"), ("4", "1", "2"), ("2", "2", "2"),
                      ("4", "1", "4"), ("2", "2", "4"), ("4", "1", "8")}


@pytest.mark.parametrize("source", ["moe_fp8", "moe_stream", "paged_decode", "prefill_attn"])
def test_pipelined_loads_are_global(source, tmp_path):
    """A flat load counts as an LDS operation too: the next wait for LDS waits for every load in flight."""
    tools = Path(HIPCC).resolve().parent.parent / "llvm" / "bin"
    fat, code = tmp_path / "fat", tmp_path / "code"
    subprocess.run([tools / "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", OBJ_DIR / f"{source}.o",
                    tmp_path / "unused"], check=True)
    subprocess.run([tools / "clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--output={code}",
                    f"--targets=hipv4-amdgcn-amd-amdhsa--{ARCH}"], check=True)
    text = subprocess.run([tools / "llvm-objdump", "-d", code], check=True, capture_output=True, text=True).stdout
    assert "global_load" in text or "buffer_load" in text
    flat = {block.split(">", 1)[0] for block in re.split(r"^[0-9a-f]+ <", text, flags=re.M) if "flat_load" in block}
    assert not flat, flat
