"""CPU: properties of the code that the compiler makes of single kernels which no result shows for certain: how two waves
order what they hand to each other without a barrier, and what a kernel needs of the registers that other waves could use."""
import importlib
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")


def compile_kernels(tmp_path, header, kernels):
    """{kernel (its mangled name): (its instructions and labels, its register figures)} of explicit instantiations."""
    build = importlib.import_module("ttt-rs_amd.build")
    src, asm = tmp_path / "kernels.hip", tmp_path / "kernels.s"
    src.write_text(f'#include "{header}"\nnamespace ttt {{\n' + "".join(f"template __global__ void {k};\n" for k in kernels) + "}\n")
    subprocess.run([HIPCC, *build.HIPCC_FLAGS, "-I", os.path.join(build.HERE, "csrc"), "--cuda-device-only", "-S", "-o", str(asm),
                    str(src)], check=True, capture_output=True)
    bodies, figures, func = {}, {}, None
    meta = {}
    for line in asm.read_text().splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            func = bodies.setdefault(m.group(1), [])
        elif line.startswith(".Lfunc_end"):
            func = None
        elif func is not None and line.split(";")[0].strip():
            func.append(line.split(";")[0].strip())
        m = re.match(r"[\s-]+\.(name|vgpr_count|vgpr_spill_count|wavefront_size):\s+(\S+)", line)
        if m:
            meta[m.group(1)] = m.group(2)
            if m.group(1) == "wavefront_size":
                figures[meta["name"]] = {k: int(v) for k, v in meta.items() if k != "name"}
    assert len(figures) == len(kernels)
    return {k: (bodies[k], figures[k]) for k in figures}


def scan_loop(body):
    """The instructions of the loop over the mini-batches: the shortest of the loops with the most matrix instructions
    (branches back from blocks that the compiler moved behind the loop span it as well)."""
    at = {s[:-1]: i for i, s in enumerate(body) if s.endswith(":")}
    loops = [body[at[m.group(1)]:i] for i, s in enumerate(body)
             if (m := re.match(r"s_c?branch\w*\s+(\.LBB\w+)", s)) and at.get(m.group(1), i) < i]
    return min(loops, key=lambda loop: (-sum(s.startswith("v_mfma") for s in loop), len(loop)))


def test_mlp_pair_hands_a2_over_in_lds(tmp_path):
    """Wave 2 of the TTT-MLP forward on a pair of CUs sums A2 as soon as a counter per wave says that every wave's partial
    block is written, with no barrier between.  That holds if block and counter are both LDS instructions: a FLAT access to the
    counter takes another path than the block, in an order that nothing guarantees."""
    for name, (body, _) in compile_kernels(tmp_path, "ttt_mlp_fwd_cl2.hip.h", [
            f"ttt_mlp_fwd_cl2_kernel<BF16, {d}>(Problems<MlpFwdArgs>)" for d in (96, 128)]).items():
        flat = [s for s in body if s.startswith("flat_")]
        assert not flat, f"{name}: {flat}"


def test_linear_backward_reloads_nothing_in_its_loop(tmp_path):
    """head_dim 128, bf16 I/O with f32 row-major checkpoints, and head_dim 64, f32 I/O from sparse checkpoints: the kernels
    that sit at the limit of their registers.  A value spilled inside the loop is reloaded behind every load and store of the
    wave that is in flight."""
    for name, (body, _) in compile_kernels(tmp_path, "ttt_linear_bwd_mw.hip.h", [
            f"ttt_linear_bwd_mw_kernel<{k}>(LinearBwdArgs)" for k in (
                "BF16, 128, 4, false, false, false, false", "F32, 64, 4, true, false, true, true")]).items():
        reloads = [s for s in scan_loop(body) if s.startswith("scratch_load")]
        assert not reloads, f"{name}: {reloads}"


def test_mlp_forward_d32_leaves_room_for_a_second_workgroup(tmp_path):
    """Eight waves, two a SIMD: a CU takes two workgroups if a wave needs at most a quarter of a SIMD's 512 registers."""
    for name, (body, figures) in compile_kernels(tmp_path, "ttt_mlp_fwd_rr.hip.h", [
            f"ttt_mlp_fwd_rr_kernel<BF16, 32, {save}>(Problems<MlpFwdArgs>)" for save in ("false", "true")]).items():
        assert figures["vgpr_count"] <= 128 and figures["vgpr_spill_count"] == 0, f"{name}: {figures}"


def test_mlp_backward_reads_its_look_ahead_from_lds(tmp_path):
    """The look-ahead at the partner's counter is copied to LDS to spare a trip through the vector memory path: its reader may
    not take that path either."""
    for name, (body, _) in compile_kernels(tmp_path, "ttt_mlp_bwd_rp.hip.h", [
            f"ttt_mlp_bwd_rp_kernel<{d}>(MlpBwdRpArgs)" for d in (32, 64)]).items():
        flat = [s for s in body if s.startswith("flat_")]
        assert not flat, f"{name}: {flat}"


def test_linear_adam_keeps_no_addresses_through_its_loop(tmp_path):
    """f32 I/O, head_dim 64: state, moments and rows fill the registers, and what is spilled besides is spilled around the loop.  The
    addresses of the initial state, 32 registers, were kept from the prologue for the final state (44 to 63 spilled, now 18 to 36)."""
    for name, (_, figures) in compile_kernels(tmp_path, "ttt_linear_fwd_sk.hip.h", [
            f"ttt_linear_adam_fwd_kernel<F32, 64, 4, {k}, 2>(LinearFwdArgs, AdamArgs)" for k in (
                "2, true, 5, false", "1, true, 0, true", "1, false, 0, true")]).items():
        assert figures["vgpr_spill_count"] <= 40, f"{name}: {figures}"
