"""Host side of large results, on the CPU: the copies of pieces that arrive one
after the other (abyss_amd/csrc/regf_pack.cpp), plain and under
ThreadSanitizer, driven by tests/harness/copy_check.cpp."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DRIVER = os.path.join(ROOT, "tests", "harness", "copy_check.cpp")
PACK = os.path.join(ROOT, "abyss_amd", "csrc", "regf_pack.cpp")

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")


@pytest.fixture(scope="module", params=["", "thread"])
def driver(request, tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("copy") / "copy_check")
    san = [f"-fsanitize={request.param}"] if request.param else []
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", *san, DRIVER, PACK, "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("what", ["pieces", "pool"])
def test_copies_of_arriving_pieces(driver, what):
    p = subprocess.run([driver, what], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, TSAN_OPTIONS="halt_on_error=1"))
    print(p.stdout[-1000:], p.stderr[-2000:])
    assert p.returncode == 0 and "OK: 0 failure(s)" in p.stdout


def test_pool_of_a_process_that_cannot_start_more_threads(tmp_path):
    exe = str(tmp_path / "copy_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", DRIVER, PACK, "-o", exe],
                   check=True)
    p = subprocess.run([exe, "few"], capture_output=True, text=True, timeout=100)
    print(p.stdout[-1000:], p.stderr[-2000:])
    assert p.returncode == 0 and "OK: 0 failure(s)" in p.stdout
