"""What the host code enqueues and allocates (tests/cpp/host_routes.cpp), on the CPU: the library's host source over stand-ins
for the HIP runtime that record launches and allocations."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
CHECKS = ["ffn_scratch_stays", "ffn_slices_are_left_where_there_is_room", "outputs_over_the_activations",
          "runs_of_weight_tiles", "own_images", "scratch_of_graphs_stays"]
CHECKS += ["elements_take_the_f32_kernels", "decoded_weights_scratch"]
CHECKS += ["elements_take_the_f32_experts", "experts_scratch_is_reserved", "experts_line_has_no_edges", "experts_take_the_faster_form", "experts_without_room_take_the_jobs", "token_kernels_are_reached", "experts_workgroups_by_option"]


@pytest.fixture(scope="module")
def program():
    r = subprocess.run(["make", "-C", CPP, "host_routes"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return os.path.join(CPP, "host_routes")


@pytest.mark.parametrize("check", CHECKS)
def test_host_routes(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
