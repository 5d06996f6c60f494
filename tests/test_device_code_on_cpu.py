"""Index arithmetic of the per-tile step kernels on lattices of any side up to 65535, by
running them on the CPU (tests/cpp/cpu_hip) over sparse memory: every cell of the first
and the last tile is written, nothing else is, and nothing outside the fields is read.
And, the same way, the LDS that the consumers' launches take, the accept estimates of the
FP64 samplers, the staged downloads' failures, the operators' kept scratch, the lanes of
runs and the default steps' choice of kernel.  No GPU needed."""
import concurrent.futures as cf
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")
CLANG = "/opt/rocm/llvm/bin/clang++"


def compile_cpu(src, exe, *extra):
    """Compile a source of the library, or of tests/cpp, for the CPU through cpu_hip."""
    r = subprocess.run([CLANG, "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I", os.path.join(CPP, "cpu_hip"),
                        "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "trophic_maelstorm_amd", "csrc"),
                        os.path.join(CPP, src), "-pthread", "-o", str(exe), *extra], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(exe)


UNITS = ["tm_kernels_f64.hip", "tm_kernels_f32.hip", "tm_ensemble.hip", "tm_frames.hip", "tm_consumers.hip", "tm_movement.hip",
         "tm_api.cpp", "tm_io.cpp", "tm_hostcopy.hip", "tm_groups.hip"]


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    """Objects of the whole library for the CPU."""
    d = tmp_path_factory.mktemp("units")

    def unit(u):
        obj = d / (u.split(".")[0] + ".o")
        lds = {"tm_consumers.hip": 1, "tm_movement.hip": 2}.get(u, 0)
        return compile_cpu("cpu_unit.cpp", obj, "-c", "-x", "c++", f'-DUNIT="{u}"', f"-DLDS={lds}")

    with cf.ThreadPoolExecutor(8) as ex:
        return list(ex.map(unit, UNITS))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return compile_cpu("kernel_indices.cpp", tmp_path_factory.mktemp("cpu") / "kernel_indices")


# 37837 and 37839 lie on either side of 3 L^2 = 2^32, 46339 and 46343 of 2 L^2 = 2^32
SIDES = [1, 5, 33, 64, 4097, 37837, 37839, 46339, 46343, 65534, 65535]


@pytest.mark.parametrize("kernel", ["frame", "part", "tile", "veg"])
def test_tiles_read_and_write_their_cells_only(exe, kernel):
    r = subprocess.run([exe, kernel, *map(str, SIDES)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_consumer_launches_opt_in_to_their_lds(tmp_path):
    exe = compile_cpu("consumer_lds.cpp", tmp_path / "consumer_lds")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_accept_estimates_as_compiled(tmp_path):
    """ptrs_estimate and gamma_estimate from the source the kernels are built of, with
    v_log_f32 and v_rcp_f32 an ulp off either way, near equality and far from it."""
    exe = compile_cpu("accept_estimates.cpp", tmp_path / "accept_estimates")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_staged_download_reports_failures(tmp_path):
    """A device copy that never lands is an error, not an endless wait; the caller's
    current device stays."""
    exe = compile_cpu("hostcopy.cpp", tmp_path / "hostcopy")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_operators_scratch_is_given_back_by_device(tmp_path):
    exe = compile_cpu("workspace.cpp", tmp_path / "workspace")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stderr)


def test_lanes_are_measured_again_after_a_busy_start(tmp_path):
    exe = compile_cpu("run_lanes.cpp", tmp_path / "run_lanes")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


RULES = [
    ("tm_kernels_f64.hip", "dp_variants_f64", "dp_f64_64x32_t256_x8aq_w6",
     [(1280, "dp_part_kernel<double, 64, 32, 1>"), (1281, "dp_step_kernel")]),
    ("tm_kernels_f32.hip", "dp_variants_f32", "dp_f32_128x24_t256_x8aq",
     [(384, "dp_part_kernel<float, 128, 24, 1>"), (385, "dp_part_kernel<float, 128, 24, 3>"),
      (1152, "dp_part_kernel<float, 128, 24, 3>"), (1153, "dp_step_kernel")]),
    ("tm_movement.hip", "fke2_variants_f64", "fke2_f64_t256",
     [(3072, "fke_head_kernel<SP, true>"), (3073, "fke_head_kernel<SP, false>")]),
    ("tm_movement.hip", "fke3_variants_f64", "fke3_f64_t256",
     [(3072, "fke_head_kernel<SP, true>"), (3073, "fke_head_kernel<SP, false>")]),
]


@pytest.mark.parametrize("unit,table,variant,edges", RULES, ids=[r[1] for r in RULES])
def test_size_rules_hold_for_the_batch(tmp_path, unit, table, variant, edges):
    """A batch in two instance groups takes the kernel of the whole batch's size."""
    exe = compile_cpu("size_rules.cpp", tmp_path / "size_rules", f'-DUNIT="{unit}"', f"-DTABLE={table}",
                      *(["-DMOVE"] if unit == "tm_movement.hip" else []))
    r = subprocess.run([exe, variant, *[str(n) for n, _ in edges]], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    got = r.stdout.split("\n")[:-1]
    for k, (n, want) in enumerate(edges):
        assert want in got[2 * k] and want in got[2 * k + 1], (n, got[2 * k:2 * k + 2])


def test_short_runs_stay_on_their_stream(tmp_path, library):
    exe = compile_cpu("run_streams.cpp", tmp_path / "run_streams", *library)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_consumer_batch_without_its_scratch(tmp_path, library):
    exe = compile_cpu("consumer_memory.cpp", tmp_path / "consumer_memory", *library)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stderr)
