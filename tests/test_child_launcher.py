"""The launcher of the GPU tests' child processes returns and raises what
subprocess.run does."""
import subprocess
import sys

import pytest

from child_launcher import Launcher


@pytest.fixture
def launcher():
    made = Launcher()
    yield made
    made.close()


def py(code):
    return [sys.executable, "-c", code]


def test_returns_what_subprocess_run_does(launcher, tmp_path):
    code = "import os, sys; print(os.getcwd(), sys.argv[1]); print('e', file=sys.stderr); sys.exit(3)"
    for kw in (dict(text=True), dict()):
        kw.update(capture_output=True, timeout=60, cwd=tmp_path)
        a, b = (run([*py(code), tmp_path], **kw) for run in (launcher.run, subprocess.run))
        assert (a.returncode, a.stdout, a.stderr) == (b.returncode, b.stdout, b.stderr) and a.returncode == 3


def test_raises_what_subprocess_run_does(launcher):
    with pytest.raises(subprocess.TimeoutExpired):
        launcher.run(py("import time; time.sleep(60)"), capture_output=True, timeout=1)
    with pytest.raises(subprocess.CalledProcessError):
        launcher.run(py("raise SystemExit(1)"), capture_output=True, check=True)
    with pytest.raises(FileNotFoundError):
        launcher.run(["/nonexistent"], capture_output=True)
    assert launcher.run(py(""), capture_output=True).returncode == 0
