"""The server's batch bookkeeping (lbm3_amd/csrc/batch.hpp) on the CPU: a small
C++ program steps requests of two storage types on a model of the device, whose
parity and iteration follow from the ticks as in k_multi_step, while uploads or
launches of the second type fail.  Every request must take exactly its steps,
each at the parity and iteration its own history gives."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "batch.hpp"
using namespace lbm3;

struct Request { int kind, done, steps, flip, iter, pending, stepped; };   // stepped: by the model of the device
struct Desc { Request *r; int tick0, flip0, iter0; };

struct Model {
    Batch b;
    std::vector<Desc> D;
    int failUploads = 0, failLaunches = 0;
    int step(std::vector<Request *> &active)
    {
        return step_batch(
            b, active,
            [&](const std::vector<Request *> &run) {
                if (failUploads > 0) { --failUploads; return -3; }
                D.clear();
                for (Request *r : run) D.push_back({r, b.tick - r->done, (r->flip + r->done) & 1, r->iter - r->done});
                return 0;
            },
            [&](int n, int tick) {
                if (failLaunches > 0) { --failLaunches; return -4; }
                if (n != (int)D.size()) { std::printf("%d requests, tables of %zu\n", n, D.size()); std::exit(1); }
                for (Desc &d : D) {
                    const int age = tick - d.tick0;
                    // parity, iteration and whether a condition is pending: the step before left them
                    if (((d.flip0 + age) & 1) != (d.r->stepped & 1) || d.iter0 + age != d.r->stepped || (age > 0) != (d.r->stepped > 0)) {
                        std::printf("kind %d step %d: age %d\n", d.r->kind, d.r->stepped, age);
                        std::exit(1);
                    }
                    ++d.r->stepped;
                }
                return 0;
            },
            [&](Request *r) { r->flip ^= 1; ++r->iter; });
    }
};

// a server step: the types in order, up to the first that fails; retirement only if none did
static int server_step(Model (&m)[2], std::vector<Request *> &active)
{
    std::vector<Request *> groups[2];
    for (Request *r : active) groups[r->kind].push_back(r);
    for (int k = 0; k < 2; ++k)
        if (const int rc = m[k].step(groups[k])) return rc;
    std::vector<Request *> still;
    for (Request *r : active) {
        if (r->done >= r->steps) m[r->kind].b.stale = true;
        else still.push_back(r);
    }
    active.swap(still);
    return 0;
}

int main()
{
    std::srand(7);
    for (int trial = 0; trial < 2000; ++trial) {
        Model m[2];
        std::vector<Request> all(6);
        std::vector<Request *> active;
        size_t next = 0;
        int failures = 0;
        for (Request &r : all) r = {std::rand() % 2, 0, 1 + std::rand() % 6, 0, 0, 0, 0};
        for (int call = 0; next < all.size() || !active.empty(); ++call) {
            if (next < all.size() && std::rand() % 2) { m[all[next].kind].b.stale = true; active.push_back(&all[next++]); }
            const int k = std::rand() % 8;
            if (k < 2) m[k].failUploads = 1 + std::rand() % 2;
            else if (k < 4) m[k - 2].failLaunches = 1;
            failures += server_step(m, active) != 0;
            if (call > 1000) { std::printf("does not drain\n"); return 1; }
        }
        for (Request &r : all)
            if (r.stepped != r.steps || r.done != r.steps) { std::printf("%d of %d steps\n", r.stepped, r.steps); return 1; }
    }
    std::printf("ok\n");
    return 0;
}
"""


def test_a_type_that_fails_leaves_the_others_in_step(tmp_path):
    src = tmp_path / "batches.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "batches"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "lbm3_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
