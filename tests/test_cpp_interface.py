"""The C++ operator interface (include/core, include/ops, include/optim) over the C-ABI.

CPU part: every header of the interface is self-contained C++20 and the set declares the functions
the reference's callers use, in the reference's argument order. GPU part: the compiled test program
replays the reference tests' known answers through that interface (tests/cpp/ops_interface_test.cpp).
"""
import os
import pathlib
import re
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
INCLUDE = ROOT / "include"
HEADERS = sorted(p.relative_to(INCLUDE).as_posix() for p in INCLUDE.rglob("*.h") if p.parent != INCLUDE)

# name -> leading parameter names, as declared by the reference (include/ops/**, include/optim/adamw.h)
REFERENCE_SIGNATURES = {
    "rmsnorm_backward": ["grad_input", "grad_weight", "grad_output", "input", "weight", "epsilon", "stream"],
    "rope_backward": ["grad_query", "grad_key", "grad_rotated_query", "grad_rotated_key", "cos_cache", "sin_cache",
                      "stream", "rope_options"],
    "linear_backward": ["grad_input", "grad_weight", "grad_bias", "grad_output", "input", "weight"],
    "embedding_backward": ["grad_weight", "grad_output", "device_token_ids", "token_count", "stream", "options"],
    "cross_entropy_forward_backward": ["loss", "gradient", "logits", "device_targets", "target_count", "stream",
                                       "gradient_scale"],
    "cut_cross_entropy_forward_backward": ["loss", "input_gradient", "classifier_gradient", "input", "classifier",
                                           "device_targets", "target_count", "stream"],
    "flash_gqa_attention_backward_with_lse": ["grad_query", "grad_key", "grad_value", "grad_output", "output",
                                              "logsumexp", "query", "key", "value", "stream", "options",
                                              "accumulate_grads"],
    "flash_gqa_attention_backward": ["grad_query", "grad_key", "grad_value", "grad_output", "query", "key", "value",
                                     "stream", "options", "accumulate_grads"],
    "adamw_step": ["parameter", "gradient", "state", "options", "stream"],
    "adamw_step_many_async": ["entries", "options", "workspace", "stream"],
}


@pytest.mark.parametrize("header", HEADERS)
def test_header_is_self_contained(header, tmp_path):
    compiler = shutil.which("g++")
    if compiler is None or not pathlib.Path("/opt/rocm/include/hip/hip_runtime_api.h").exists():
        pytest.skip("needs g++ and the HIP runtime headers")
    source = tmp_path / "unit.cpp"
    source.write_text(f'#include "{header}"\nint main() {{ return 0; }}\n')
    proc = subprocess.run([compiler, "-std=c++20", "-fsyntax-only", "-D__HIP_PLATFORM_AMD__", f"-I{INCLUDE}",
                           "-I/opt/rocm/include", str(source)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]


def test_signatures_follow_the_reference_order():
    text = "\n".join((INCLUDE / h).read_text() for h in HEADERS)
    for name, want in REFERENCE_SIGNATURES.items():
        match = re.search(r"inline\s+(?:void|bool)\s+" + name + r"\s*\(([^)]*)\)", text)
        assert match, f"{name} is not declared"
        params = [re.sub(r"\s*=.*", "", p).strip().split()[-1].lstrip("&*") for p in match.group(1).split(",")]
        params = [p for p in params if p not in ("GemmContext&",)]
        named = [p for p in params if re.fullmatch(r"[a-z_]+", p)]
        assert named[: len(want)] == want[: len(named)] or named == want, (name, named, want)


@pytest.mark.gpu
def test_interface_program_replays_reference_known_answers():
    binary = ROOT / "tests" / "cpp" / "ops_interface_test.bin"
    assert binary.exists(), "build it with `python -m cgpt_amd.build` (there is no fallback)"
    proc = subprocess.run([str(binary)], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "0 failure(s)" in proc.stdout


@pytest.mark.gpu
def test_token_batches_upload_through_the_data_header():
    """tests/cpp/data_upload_test.cpp: data::Batch / data::DeviceBatch / data::upload_batch
    (include/data/dataset_loader.h) over the library's upload entry points: alternating page-locked batches arrive
    bit for bit, device buffers keep their address, shape mismatches throw, copies are deep, moves carry the
    pending upload."""
    binary = ROOT / "tests" / "cpp" / "data_upload_test.bin"
    assert binary.exists(), "build it with `python -m cgpt_amd.build` (there is no fallback)"
    proc = subprocess.run([str(binary)], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "0 failure(s)" in proc.stdout


@pytest.mark.gpu
def test_callers_of_the_headers_reproduce_the_library_step():
    """tests/cpp/block_backward_test.cpp: the wrappers accept the reference's argument lists (compile-time), and
    the library's own table of operator calls (the step as the reference's call sequence, CGPTX_FUSE=0), made
    through include/ops/** eagerly and from a HipGraph capture, gives the library step's gradients bit for bit."""
    binary = ROOT / "tests" / "cpp" / "block_backward_test.bin"
    assert binary.exists(), "build it with `python -m cgpt_amd.build` (there is no fallback)"
    proc = subprocess.run([str(binary)], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "0 failure(s)" in proc.stdout


@pytest.mark.gpu
def test_projections_of_a_small_block_share_exact_launches():
    """tests/cpp/gemm_group_test.cpp: the forward projections of q, k and v as one launch, and their four gradients as one whose
    input gradient reads three buffers; ragged rows and segments that end inside a K tile, exact on whole numbers."""
    binary = ROOT / "tests" / "cpp" / "gemm_group_test.bin"
    assert binary.exists(), "build it with `python -m cgpt_amd.build` (there is no fallback)"
    proc = subprocess.run([str(binary)], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "\n0 failure(s)" in proc.stdout


def run_plan_test(mode, **environment):
    binary = ROOT / "tests" / "cpp" / "gemm_plan_test.bin"
    assert binary.exists(), "build it with `python -m cgpt_amd.build` (there is no fallback)"
    proc = subprocess.run([str(binary), mode], capture_output=True, text=True, timeout=120, env={**os.environ, **environment})
    assert proc.returncode == 0, proc.stdout[-4000:] + proc.stderr
    assert proc.stdout.endswith("\n0 failure(s)\n") or proc.stdout == "0 failure(s)\n"


def test_a_pinned_tile_size_is_one_that_the_call_has():
    """tests/cpp/gemm_plan_test.cpp: with CGPTX_GEMM_TILE=192 fp32 calls, and those that add a bias, are planned for tiles they have
    kernels of (fp32 results once lacked three quarters of their elements)."""
    run_plan_test("pinned", CGPTX_GEMM_TILE="192")


def test_fp32_gradients_that_share_a_launch_have_no_longer_chains():
    """tests/cpp/gemm_plan_test.cpp: q's, k's and v's gradients in fp32 join only where no sum becomes a longer chain of additions
    than it is in the launches they stand for (the rounding error of a chain grows with its length)."""
    run_plan_test("chains")


def test_launches_that_meet_on_a_tile_counter_leave_it_at_zero():
    """tests/cpp/gemm_plan_test.cpp: the shares by which the K slices of a tile count themselves, in random orders of arrival, alone
    and with other launches between (counting by ones, two such launches left every later one on the stream with a wrong count)."""
    run_plan_test("counters")


def test_tiles_of_192_columns_take_what_their_epilogue_serves():
    """tests/cpp/gemm_plan_test.cpp: a residual or an fp32 addend that does not lie in whole aligned chunks keeps a call on square
    tiles (on 256 x 192 ones it would end in an error)."""
    run_plan_test("narrow")


def test_calls_on_oblong_tiles_keep_their_bits_and_have_a_kernel():
    """Oblong tiles replace large square ones of calls that are one sum over K, stored as it is or with a residual."""
    run_plan_test("oblong")


def test_predictions_that_stop_short_decide_as_whole_ones():
    """tests/cpp/gemm_plan_test.cpp: what both gradients of a projection take in one launch, predicted only as far as the answer
    can matter."""
    run_plan_test("predictions")


def test_a_steps_dense_loss_streams_long_rows_in_vectors():
    """tests/cpp/gemm_plan_test.cpp: the gradient of more logits than the registers hold lies in rows like the logits' own (in rows padded
    for the contractions, an odd vocabulary's were read and written element by element)."""
    run_plan_test("loss_rows")


def test_pairs_on_oblong_tiles_are_those_that_gain():
    """tests/cpp/gemm_plan_test.cpp: gradients that lost up to a fifth on oblong tiles, or apart because of them, share a launch of 128 x 128
    ones, and the ragged shapes of tests/test_gpu_linear.py reach every tile."""
    run_plan_test("oblong_pairs")


def test_a_step_of_many_tokens_holds_no_memory_for_their_groups():
    """tests/cpp/gemm_plan_test.cpp: a step's tokens by id have memory of their own only where they are grouped beside their lookup."""
    run_plan_test("token_groups")


def test_shapes_that_are_there_for_oblong_tiles_reach_them():
    """tests/cpp/gemm_plan_test.cpp: the shapes whose values tests/test_gpu_linear.py and tests/cpp/gemm_group_test.cpp check on oblong tiles are
    planned for those tiles (11871 x 352 x 1024, once meant for 192 x 256, is not)."""
    run_plan_test("oblong_shapes")
