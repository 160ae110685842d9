"""Starts the GPU tests' child processes from a helper process made before the
test process touches the GPU.

The GPU test process has ended with a segmentation fault, on two runs of many,
at the test that launches its first child process; why is not known.  Until it
is, no child is launched from a process that uses the GPU: the helper, which
never does, takes the command line over a pipe, runs it and sends back what
subprocess.run returns.
"""
import base64
import json
import subprocess
import sys

SERVER = r"""
import base64, json, subprocess, sys
for line in sys.stdin:
    q = json.loads(line)
    try:
        r = subprocess.run(q["args"], cwd=q["cwd"], env=q["env"], timeout=q["timeout"], capture_output=True)
        a = dict(code=r.returncode, out=r.stdout, err=r.stderr)
    except subprocess.TimeoutExpired as e:
        a = dict(expired=True, out=e.stdout or b"", err=e.stderr or b"")
    except OSError as e:
        a = dict(errno=e.errno, text=str(e), out=b"", err=b"")
    a["out"], a["err"] = (base64.b64encode(a[k]).decode() for k in ("out", "err"))
    print(json.dumps(a), flush=True)
"""


class Launcher:
    def __init__(self):
        self.helper = subprocess.Popen([sys.executable, "-u", "-c", SERVER], stdin=subprocess.PIPE,
                                       stdout=subprocess.PIPE, text=True)

    def run(self, args, *, capture_output=False, text=False, timeout=None, check=False, cwd=None, env=None):
        """subprocess.run of the arguments the tests use."""
        if not capture_output:
            raise ValueError("the launcher returns the output, it does not show it")
        args = [str(a) for a in args]
        self.helper.stdin.write(json.dumps(dict(args=args, cwd=cwd and str(cwd), env=env, timeout=timeout)) + "\n")
        self.helper.stdin.flush()
        line = self.helper.stdout.readline()
        if not line:
            raise RuntimeError("the helper process has ended")
        a = json.loads(line)
        out, err = base64.b64decode(a["out"]), base64.b64decode(a["err"])
        if text:
            out, err = out.decode(), err.decode()
        if a.get("expired"):
            raise subprocess.TimeoutExpired(args, timeout, out, err)
        if "errno" in a:
            raise OSError(a["errno"], a["text"])
        r = subprocess.CompletedProcess(args, a["code"], out, err)
        if check:
            r.check_returncode()
        return r

    def close(self):
        self.helper.stdin.close()
        self.helper.wait(10)
        self.helper.stdout.close()
