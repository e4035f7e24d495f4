"""Starts programs for the test process from a process that never uses the GPU.

A process that has loaded the HIP runtime starts no other program itself: its
GPU test run has ended in a segmentation fault inside subprocess.Popen.  The
Launcher is started before the runtime is loaded and offers subprocess.run's
interface, as far as the tests use it; it ends with the test process (its
standard input closes).
"""
import json
import subprocess
import sys


class Launcher:
    TimeoutExpired = subprocess.TimeoutExpired

    def __init__(self):
        self._p = subprocess.Popen([sys.executable, "-u", __file__], stdin=subprocess.PIPE, stdout=subprocess.PIPE,
                                   text=True)

    def run(self, args, cwd=None, capture_output=True, text=True, timeout=None):
        if not (capture_output and text):
            raise ValueError("the launcher returns captured text only")
        args = [str(a) for a in args]
        self._p.stdin.write(json.dumps([args, cwd and str(cwd), timeout]) + "\n")
        self._p.stdin.flush()
        answer = self._p.stdout.readline()
        if not answer:
            raise RuntimeError("the launcher has ended")
        kind, *rest = json.loads(answer)
        if kind == "timeout":
            raise subprocess.TimeoutExpired(args, timeout)
        if kind == "error":
            raise OSError(rest[0])
        return subprocess.CompletedProcess(args, *rest)

    def close(self):
        self._p.stdin.close()
        self._p.wait(timeout=60)
        self._p.stdout.close()


def serve():
    for line in iter(sys.stdin.readline, ""):
        args, cwd, timeout = json.loads(line)
        try:
            r = subprocess.run(args, cwd=cwd, stdin=subprocess.DEVNULL, capture_output=True, text=True,
                               timeout=timeout)
            answer = ["done", r.returncode, r.stdout, r.stderr]
        except subprocess.TimeoutExpired:
            answer = ["timeout"]
        except OSError as e:
            answer = ["error", str(e)]
        print(json.dumps(answer), flush=True)


if __name__ == "__main__":
    serve()
