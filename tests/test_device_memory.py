"""What an MSM call does where device memory is short, through the C ABI on the
host alone: the HIP runtime's calls are those of host_hip.hpp, with a limit on
the bytes, and no kernel runs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "zyklop_amd")


def run(tmp_path, body):
    """Compile body, run it; its printed line."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include "host_hip.hpp"\n#include <stdio.h>\n#include <vector>\n#include "zk_abi.h"\n' + body)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I", os.path.join(ROOT, "tests"), "-I", os.path.join(ROOT, "include"), str(src), "-o",
                           str(exe), "-L", LIB, "-lzkp", "-L/opt/rocm/lib", "-lamdhip64",
                           "-Wl,-rpath," + LIB, "-Wl,-rpath,/opt/rocm/lib"])
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    return res.stdout.strip()


def test_kept_buffers_never_cost_a_call_its_memory(tmp_path):
    """A call that fits into the device memory when nothing is kept fits after
    any other call on the context too: buffers kept for another shape make way.
    One that does not fit is still refused, and leaves nothing allocated."""
    out = run(tmp_path, r"""
static int msm(zk_ctx* c, bool g2, size_t n, int window) {
    static std::vector<char> pts((size_t)1 << 23), sc((size_t)1 << 22);
    uint64_t out[16];
    int inf = 0;
    return g2 ? zk_msm_g2_device(c, pts.data(), sc.data(), n, window, out, &inf)
              : zk_msm_g1_device(c, pts.data(), sc.data(), n, window, out, &inf);
}
int main() {
    struct { bool g2; size_t n; int window; } shape[] = {
        {false, 100000, 0}, {true, 500, 14}, {true, 60000, 8}, {false, 300, 16}, {false, 2000, 4}, {true, 2000, 4}};
    for (auto& after : shape)
        for (auto& before : shape) {
            const size_t all = (size_t)1 << 40;
            host_hip::limit = all;
            zk_ctx* c = nullptr;
            if (zk_ctx_create(0, &c)) return 2;
            const size_t base = host_hip::used;
            if (msm(c, after.g2, after.n, after.window)) return 3;
            const size_t need = host_hip::used - base;   // what the call takes alone
            zk_ctx_destroy(c);
            if (zk_ctx_create(0, &c)) return 2;
            if (msm(c, before.g2, before.n, before.window)) return 3;
            host_hip::limit = base + need > host_hip::used ? base + need : host_hip::used;
            if (msm(c, after.g2, after.n, after.window)) { printf("refused: %s", zk_last_error()); return 0; }
            host_hip::limit = base + 4096;
            const int rc = msm(c, true, 130000, 0);
            if (rc != ZK_E_NOMEM) { printf("not refused: %d", rc); return 0; }
            if (host_hip::used != base) { printf("%zu bytes left", host_hip::used - base); return 0; }
            zk_ctx_destroy(c);
            if (host_hip::used != 0) { printf("%zu bytes leaked", host_hip::used); return 0; }
        }
    printf("ok");
    return 0;
}
""")
    assert out == "ok"


def test_parts_of_a_bucket_give_way(tmp_path):
    """An MSM on its own accumulates a bucket in more parts than one in a proof;
    where those parts' memory is not there it takes the proof's."""
    out = run(tmp_path, r"""
int main() {
    static char pts[64], sc[64];
    uint64_t out[8];
    int inf = 0;
    zk_ctx* c = nullptr;
    if (zk_ctx_create(0, &c)) return 2;
    const size_t base = host_hip::used;
    if (zk_msm_g1_device(c, pts, sc, 100000, 0, out, &inf)) return 3;
    const size_t need = host_hip::used - base;
    zk_ctx_destroy(c);
    if (zk_ctx_create(0, &c)) return 2;
    host_hip::limit = base + need - need / 8;
    if (zk_msm_g1_device(c, pts, sc, 100000, 0, out, &inf)) { printf("refused: %s", zk_last_error()); return 0; }
    host_hip::limit = base + need / 8;
    if (zk_msm_g1_device(c, pts, sc, 100000, 0, out, &inf) != ZK_E_NOMEM) { printf("not refused"); return 0; }
    zk_ctx_destroy(c);
    printf("ok");
    return 0;
}
""")
    assert out == "ok"


def test_workspace_is_given_back_on_request(tmp_path):
    """Memory that a context keeps can be had back by a program whose other
    allocators share the device; the next call allocates again."""
    out = run(tmp_path, r"""
int main() {
    static char pts[64], sc[64];
    uint64_t out[8];
    int inf = 0;
    zk_ctx* c = nullptr;
    if (zk_ctx_create(0, &c)) return 2;
    const size_t base = host_hip::used;
    for (int i = 0; i < 2; i++) {
        if (zk_msm_g1_device(c, pts, sc, 5000, 0, out, &inf)) return 3;
        if (host_hip::used == base) { printf("nothing kept"); return 0; }
        if (zk_msm_free_workspace(c) || host_hip::used != base) { printf("not given back"); return 0; }
    }
    if (zk_msm_free_workspace(c) || zk_msm_free_workspace(nullptr) != ZK_E_ARG) return 4;
    zk_ctx_destroy(c);
    printf("ok");
    return 0;
}
""")
    assert out == "ok"
