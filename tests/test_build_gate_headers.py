"""The build's checks look at a source together with the headers it includes, and at the code of kernels whose order of loads
and stores is by hand (no GPU)."""
import re
import subprocess
from pathlib import Path

import pytest

from dlcompiler_amd.build import ARCH, CSRC_DIR, HIPCC, OBJ_DIR, check_hand_scheduled, text_with_headers
from test_build_gate import KERNELS


def test_every_kernel_with_hand_issued_loads_is_named():
    """Sources and headers that issue loads by hand define no kernel outside the gate but these, which use ordinary loads."""
    ordinary = {"prefill_combine_kernel", "paged_decode_combine_kernel", "quant_fp8_group128_kernel",
                "moe_topk_sum_kernel"}
    named = set()
    for src in [*CSRC_DIR.glob("*.hip"), *CSRC_DIR.glob("*.h")]:
        text = src.read_text()
        if re.search(r"dma\d+_global_to_lds|s_load_dword|buffer_of\(", text):
            found = set(re.findall(r"__global__[^;{]*void (\w+_kernel)\(", text)) - ordinary
            assert found <= set(KERNELS), src.name
            named |= found
    assert named == set(KERNELS)


@pytest.mark.parametrize("source,kernels", [("moe_fp8", {"moe_gemm_kernel"}), ("moe_stream", {"moe_stream_kernel"}),
                                            ("paged_decode", {"paged_decode_split_kernel", "paged_decode_direct_kernel"}),
                                            ("prefill_attn", {"prefill_attn_kernel"}),
                                            ("prefill_attn_cap", {"prefill_attn_kernel"}),
                                            ("silu_and_mul", set())])
def test_missing_reports_stop_the_build(source, kernels):
    """Kernels count as a source's where it or a header of its defines them, comments aside."""
    text = re.sub(r"//.*", "", text_with_headers(CSRC_DIR / f"{source}.hip"))
    assert {m.split(":")[0] for m in check_hand_scheduled({}, text)} == kernels
    assert not check_hand_scheduled({}, "// " + " ".join(KERNELS))


def _code_of(source, tmp_path):
    """The assembly of each function that an object built here holds."""
    tools = Path(HIPCC).resolve().parent.parent / "llvm" / "bin"
    fat, code = tmp_path / "fat", tmp_path / "code"
    subprocess.run([tools / "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", OBJ_DIR / f"{source}.o",
                    tmp_path / "unused"], check=True)
    subprocess.run([tools / "clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--output={code}",
                    f"--targets=hipv4-amdgcn-amd-amdhsa--{ARCH}"], check=True)
    text = subprocess.run([tools / "llvm-objdump", "-d", code], check=True, capture_output=True, text=True).stdout
    return dict(block.split(">", 1) for block in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:])


def test_capped_prefill_loads_are_global(tmp_path):
    """A flat load counts as an LDS operation too: the next wait for LDS waits for every load in flight."""
    code = _code_of("prefill_attn_cap", tmp_path)
    assert any("global_load" in text or "buffer_load" in text for text in code.values())
    flat = {name for name, text in code.items() if "flat_load" in text}
    assert not flat, flat


def test_gate_up_waits_for_its_slots_alone(tmp_path):
    """fp8 gate_up GEMM: the first activations' addresses (which one 16-byte LDS store parks) wait for the routing slots.  A
    copy into LDS in front of them, which the compiler does not count, would have that wait cover the first weights."""
    gated = {name: text for name, text in _code_of("moe_fp8", tmp_path).items() if "moe_gemm_kernelILb1E" in name}
    assert gated
    for name, text in gated.items():
        start = text[:text.index("ds_write_b128")]
        slots, weights = start.rindex("global_load_dword "), start.index("global_load_dwordx4")
        assert slots < weights and "global_load_lds" not in start, name
        assert min(int(n) for n in re.findall(r"vmcnt\((\d+)\)", start[weights:])) >= 4, name


def test_down_gemm_stores_past_the_caches_too(tmp_path):
    """fp8 down GEMM: slot rows go through the caches where the sum over the slots follows, past them where it is called
    alone.  (Both stores on either side of a condition, the compiler would make them one.)"""
    down = {name: text for name, text in _code_of("moe_fp8", tmp_path).items() if "moe_gemm_kernelILb0E" in name}
    assert down
    for name, text in down.items():
        stores = re.findall(r"global_store_dwordx4 .*", text)
        past = [" nt" in store.split("//")[0] for store in stores]
        assert any(past) and not all(past), name


def test_routing_weights_of_a_token_are_asked_for_together(tmp_path):
    """Renormalised weights: a loop that loads, waits and adds is a chain of as many loads as a token has slots."""
    for source, kernel in (("moe_fp8", "moe_gemm_kernelILb0E"), ("moe_stream", "moe_stream_kernelILb0E")):
        down = {name: text for name, text in _code_of(source, tmp_path).items() if kernel in name}
        assert down
        for name, text in down.items():
            runs = re.split(r"s_waitcnt[^\n]*vmcnt|s_cbranch", text)
            assert max(len(re.findall(r"global_load_dword ", run)) for run in runs) >= 8, name
