"""The served form's host logic over a runtime that runs nothing (no GPU): many
requests through one server, and a device that stops, which has to end in
errors and not in a server that hangs."""
import os
import re
import shutil
import signal
import subprocess
import time

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "..", "miniaero_amd", "libminiaero_amd.so")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not all(shutil.which(t) for t in ("g++", "nm", "readelf")):
        pytest.skip("g++ and binutils needed")
    tmp = tmp_path_factory.mktemp("stub")

    def run(*cmd):
        return subprocess.run(cmd, check=True, capture_output=True, text=True).stdout

    # the runtime under its own name, with the symbol versions the library asks for
    name = re.search(r"\[(libamdhip64\.so[^\]]*)\]", run("readelf", "-d", LIB)).group(1)
    versions = {}
    for sym, ver in re.findall(r" U (\S+)@(hip_\S+)", run("nm", "-D", "-u", "--with-symbol-versions", LIB)):
        versions.setdefault(ver, []).append(sym)
    (tmp / "map").write_text("".join("%s { global: %s; };\n" % (v, "; ".join(s)) for v, s in versions.items()))
    checks = os.path.join(HERE, "host_checks")
    run("g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", os.path.join(checks, "hip_stub.cpp"),
        "-Wl,--version-script=" + str(tmp / "map"), "-Wl,-soname," + name, "-o", str(tmp / name))
    exe = str(tmp / "server_check")
    run("g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(HERE, "..", "include"),
        os.path.join(checks, "server_check.cpp"), "-Wl,--unresolved-symbols=ignore-in-shared-libs",
        "-L", os.path.dirname(LIB), "-lminiaero_amd", "-o", exe)

    def go(what, meanwhile=None, **env):
        r = subprocess.Popen([exe, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                             env=dict(os.environ, LD_LIBRARY_PATH=str(tmp) + ":" + os.path.dirname(LIB), **env))
        try:
            if meanwhile:
                meanwhile(r)
            out = r.communicate(timeout=100)[0]
        finally:
            r.kill()
        print(out)
        assert r.returncode == 0, out
        return out
    return go


def test_requests_through_one_server(check):
    check("80")


def test_a_process_that_was_stopped_has_lost_nothing(check):
    """Time in which the process does not run is not a wait on the device."""
    def stop_and_continue(p):
        for _ in range(2):
            time.sleep(0.7)
            p.send_signal(signal.SIGSTOP)
            time.sleep(1.5)
            p.send_signal(signal.SIGCONT)
    check("pause", meanwhile=stop_and_continue)


def test_planning_takes_one_thread_a_request(check):
    """ma_server_config.setup_threads is how many host threads plan requests."""
    check("threads")


@pytest.mark.parametrize("kind,after,says", [
    ("event", 0, "a step"), ("event", 40, "a step"),   # (a table's upload event may be the one that stops)
    ("sync", 0, "building a case"), ("sync", 100, "building a case|copying a result back")])
def test_a_device_that_stops_fails_the_requests(check, kind, after, says):
    out = check("stall", STUB_STALL=kind, STUB_AFTER=str(after))
    assert re.search(says + "|queueing steps", out), out
