"""CPU checks of host code inside the HIP sources: a check program includes the source, is compiled for the host alone
(no device code, no GPU involved) and reports OK."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build_and_run(tmp_path, name, *args):
    exe = tmp_path / name
    subprocess.check_call(["hipcc", "--offload-host-only", "-x", "hip", "-std=c++17", "-O0", "-Wno-unused-result",
                           os.path.join(ROOT, "tests", name + ".cpp"), "-o", str(exe),
                           "-Wl,--unresolved-symbols=ignore-all", "-lpthread"])
    p = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and "OK" in p.stdout, p.stdout + p.stderr
    return p.stdout


def test_graph_key_tells_every_argument_apart(tmp_path):
    build_and_run(tmp_path, "graph_key_check")


def test_linsolver_after_a_failed_graph_build(tmp_path):
    build_and_run(tmp_path, "linsolve_graph_check")


def test_host_copies_follow_the_null_stream(tmp_path):
    build_and_run(tmp_path, "host_copies_check", "null-stream")


def test_host_copies_of_overlapping_arrays_in_order(tmp_path):
    build_and_run(tmp_path, "host_copies_check", "overlap")


def test_host_copies_short_of_memory(tmp_path):
    build_and_run(tmp_path, "host_copies_check", "memory")


def test_linsolver_form_follows_rows_and_nonzeros(tmp_path):
    build_and_run(tmp_path, "linsolve_graph_check", "form")


def test_linsolver_short_solves_build_no_graph(tmp_path):
    build_and_run(tmp_path, "linsolve_graph_check", "short")
