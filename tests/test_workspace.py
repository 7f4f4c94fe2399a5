"""The hand-over of the MSM workspaces that contexts keep between calls, on the
host alone: small C++ programs over the library's own header and symbols, their
buffers borrowed from the host, so that nothing touches a GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "zyklop_amd")


def run(tmp_path, body):
    """Compile body after the workspace header, run it; its printed line."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("#include <chrono>\n#include <cstdio>\n#include <thread>\n#include \"msm.hpp\"\n" + body)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I", os.path.join(LIB, "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o",
                           str(exe), "-L", LIB, "-lzkp", "-L/opt/rocm/lib", "-lamdhip64", "-lpthread",
                           "-Wl,-rpath," + LIB, "-Wl,-rpath,/opt/rocm/lib"])
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    return res.stdout.strip()


def test_call_local_workspace_is_never_taken_back(tmp_path):
    """While a thread takes a context's workspace back, a call on the context
    works in one of its own, which threads that take workspaces back leave
    alone: its buffers are still there after a while, every time."""
    out = run(tmp_path, r"""
int main() {
    zk::KeptWorkspace kept;
    kept.busy = true;   // being taken back, as seen by a call that starts now
    std::atomic<bool> stop{false};
    std::thread t[3];
    for (auto& x : t) x = std::thread([&] { while (!stop) zk::release_idle_workspaces(); });
    char mark;
    long lost = 0, n = 0;
    const auto t0 = std::chrono::steady_clock::now();
    while (std::chrono::steady_clock::now() - t0 < std::chrono::seconds(1)) {
        zk::WorkspaceUse use(kept, nullptr);
        if (use.w == &kept) return 2;
        use.w->p29.borrow(&mark, 1);
        void* const volatile& p = use.w->p29.p;
        for (int i = 0; i < 200; i++)
            if (p != &mark) { lost++; break; }
        use.w->p29.release();
        n++;
    }
    stop = true;
    for (auto& x : t) x.join();
    if (!kept.busy) return 3;
    printf("%s", n < 1000 ? "too few" : lost ? "lost" : "ok");
    return 0;
}
""")
    assert out == "ok"


def test_kept_workspace_is_taken_back_between_calls_only(tmp_path):
    """The kept workspace serves one call at a time, survives a take-back while
    in use, and gives its buffers up when idle."""
    out = run(tmp_path, r"""
int main() {
    zk::KeptWorkspace kept;
    char mark;
    {
        zk::WorkspaceUse use(kept, nullptr);
        if (use.w != &kept || !kept.busy) return 2;
        use.w->p29.borrow(&mark, 1);
        zk::release_idle_workspaces();
        if (kept.p29.p != &mark) return 3;
        zk::WorkspaceUse other(kept, nullptr);
        if (other.w == &kept) return 4;
    }
    if (kept.busy || kept.p29.p != &mark) return 5;
    zk::release_idle_workspaces();
    if (kept.busy || kept.p29.p) return 6;
    try {
        zk::WorkspaceUse use(kept, nullptr);
        use.w->p29.borrow(&mark, 1);
        throw 1;
    } catch (int) {}
    if (kept.busy || kept.p29.p) return 7;   // a failed call leaves nothing behind
    printf("ok");
    return 0;
}
""")
    assert out == "ok"


def test_take_back_is_per_device(tmp_path):
    """Memory needed on one device leaves the workspaces of another alone; idle
    bytes count what a finished call left, not what a running one holds."""
    out = run(tmp_path, r"""
int main() {
    zk::KeptWorkspace a(0), b(1);
    char mark;
    zk::KeptWorkspace* both[2] = {&a, &b};
    for (int d = 0; d < 2; d++) {
        zk::WorkspaceUse use(*both[d], nullptr);
        use.w->p29.borrow(&mark, 100 + d);
        if (zk::idle_workspace_bytes(d) != 0) return 2;
    }
    if (zk::idle_workspace_bytes(0) != 100 || zk::idle_workspace_bytes(1) != 101) return 3;
    zk::release_idle_workspaces(1);
    if (a.p29.p != &mark || b.p29.p) return 4;
    if (zk::idle_workspace_bytes(0) != 100 || zk::idle_workspace_bytes(1) != 0) return 5;
    zk::release_idle_workspaces();
    if (a.p29.p || zk::idle_workspace_bytes() != 0) return 6;
    printf("ok");
    return 0;
}
""")
    assert out == "ok"


def test_context_may_outlive_the_librarys_statics(tmp_path):
    """A program that frees its context in an exit handler it registered before
    its first use of the library: the list of kept workspaces is still there
    (freed memory is overwritten, so a list that is gone shows)."""
    os.environ["MALLOC_PERTURB_"] = "165"
    try:
        out = run(tmp_path, r"""
#include <cstdlib>
static zk::KeptWorkspace *a, *b;
int main() {
    atexit([] { delete a; zk::release_idle_workspaces(); delete b; printf("ok"); });
    a = new zk::KeptWorkspace;
    b = new zk::KeptWorkspace;
    return 0;
}
""")
    finally:
        del os.environ["MALLOC_PERTURB_"]
    assert out == "ok"
