"""Host code of the plans on the CPU: the library's entry points over a HIP
runtime that allocates host memory and runs no kernel (tests/host), so that
what is launched, cleared and allocated can be looked at where running it
could fault a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "tests", "host")
PKG = os.path.join(ROOT, "ceemdan-gpu_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def driver(icm, tmp_path_factory):
    if not shutil.which("g++") or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no host compiler or HIP headers")
    icm.lib()   # says so if the library is not built
    d = tmp_path_factory.mktemp("host")
    flags = ["-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-w"]
    fake, exe = d / "libfake_hip.so", d / "plan_driver"
    subprocess.run(["g++", *flags, "-shared", "-fPIC", os.path.join(HOST, "fake_hip.cpp"), "-o",
                    str(fake)], check=True)
    # the fake runtime first: its definitions are the ones found
    subprocess.run(["g++", *flags, os.path.join(HOST, "plan_driver.cpp"), "-o", str(exe),
                    "-Wl,--no-as-needed", str(fake), f"-L{PKG}", "-liceemdan_mi355x",
                    f"-Wl,-rpath,{d}:{PKG}:{ROCM}/lib", f"-Wl,-rpath-link,{ROCM}/lib"], check=True)

    def run(name, **env):
        base = {k: v for k, v in os.environ.items() if not k.startswith("ICM_")}
        p = subprocess.run([str(exe), name], capture_output=True, text=True, timeout=300,
                           env=dict(base, **env))
        assert p.returncode == 0 and p.stdout == f"{name} ok\n", (p.returncode, p.stdout, p.stderr[-2000:])
    return run


def test_staged_forward_that_changes_path_has_clear_control_words(driver):
    """icm_set_profiling, icm_set_tuning or icm_set_trace between
    icm_forward_begin (or icm_state_load) and icm_forward_stages moves the
    remaining stages from the stage kernel to the launches per step, whose
    window lists are indexed by counters that must start at zero."""
    driver("staged_switch")


def test_stage_kernel_grid_fits_a_launch(driver):
    """Plans of up to 2^28 tiles, of any length that the stage kernel takes."""
    driver("stage_grid")


def test_plan_keeps_to_its_estimate_and_budget(driver):
    """The stage kernel's scratch is in icm_plan_bytes and within
    ICM_MEMORY_BUDGET; a budget that holds the rest of the plan is enough."""
    driver("budget")


def test_backward_buffers_in_place_of_scratch_are_counted_once(driver):
    driver("backward_room", ICM_WHOLE_STAGES="1")


@pytest.mark.parametrize("what", ["record_room", "trace_room"])
def test_records_and_traces_in_place_of_scratch(driver, what):
    """The records of a backward that sifts again, and traces, where memory
    holds them only without the stage kernel's scratch."""
    driver(what, ICM_WHOLE_STAGES="1")


def test_default_tuning_given_back_keeps_the_stage_kernel(driver):
    driver("tuning_round_trip")


def test_few_long_series_launch_step_by_step(driver):
    """Series of 56 tiles and up, too few for a workgroup each to be ahead at
    their number of rows; nothing is tuned on either path."""
    driver("few_series")


def test_long_series_of_few_rows_launch_step_by_step(driver):
    """FP64 series of 95 tiles and up, too many for launches without tuning, in
    a decomposition whose dense first stages weigh most."""
    driver("few_rows")


def test_noise_of_uneven_lengths_launches_few_idle_workgroups(driver):
    driver("noise_groups")


def test_samples_past_the_caches_only_where_they_do_not_fit(driver):
    driver("past_caches")
