"""Host code of the library against a model of the runtime (host_model/):
orderings between threads and the lifetime of graphs, which a device gets
wrong only now and then.  Built with the address sanitizer on host code."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "granular_gpu_amd" / "csrc"
HERE = Path(__file__).resolve().parent / "host_model"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")


def _run(tmp_path, program, sources):
    """Links `program` with the host parts of the library's `sources` and the
    model, runs it."""
    common = [HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-g", "-std=c++17", "-ffp-contract=off",
              "-Wno-unused-command-line-argument", "-Xarch_host", "-fsanitize=address",
              f"-I{ROOT / 'include'}", f"-I{CSRC}", f"-I{HERE}"]
    objs = []
    for src in [HERE / "runtime.cpp", HERE / program, *(CSRC / s for s in sources)]:
        objs.append(tmp_path / (src.stem + ".o"))
        subprocess.run([*common, "-x", "hip", "-c", str(src), "-o", str(objs[-1])], check=True)
    exe = tmp_path / "run"
    # (device code is not linked: the images that the objects register are
    # left undefined)
    subprocess.run(["/opt/rocm/llvm/bin/clang++", "-Xarch_host", "-fsanitize=address",
                    "-Wl,--unresolved-symbols=ignore-all", *map(str, objs), "-o", str(exe),
                    "-lpthread"], check=True)
    # (what the library keeps for the life of the process is no leak)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120,
                       env={"ASAN_OPTIONS": "detect_leaks=0"})
    print(r.stdout, r.stderr)
    return r


def test_concurrent_learned_calls_wait_for_their_own_streams(tmp_path):
    r = _run(tmp_path, "side_stream.cpp", ["mlp.hip"])
    assert r.returncode == 0, r.stdout + r.stderr


def test_graphs_are_not_released_with_launches_in_flight(tmp_path):
    r = _run(tmp_path, "graphs.cpp", ["batch.hip", "scenes.hip"])
    assert r.returncode == 0, r.stdout + r.stderr


def test_quantised_list_test_loses_no_pair(tmp_path):
    r = _run(tmp_path, "list_quant.cpp", [])
    assert r.returncode == 0, r.stdout + r.stderr
