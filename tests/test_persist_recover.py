"""What a solve does with the state of a persistent launch in which one workgroup
gave up while the others came to its end (clsparse_amd/csrc/cg_state.hpp,
bicg_state.hpp), on the CPU: the recovered state goes on, and from the iterations
before that launch."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r'''
#include <cstdio>
#include "cg_state.hpp"
#include "bicg_state.hpp"
#define CHECK(x) do { if (!(x)) { std::printf("%s\n", #x); bad = 1; } } while (0)
int main() {
  int bad = 0;
  CgDevState a{};
  a.norm_ref = 3.0; a.rel_tol = 1e-8; a.abs_tol = 1e-9; a.max_iters = 500; a.crit = kCritL2; a.cur_res = 0.25;
  a.failed = a.done = a.converged = a.stop = a.pending = 1;
  a.n_iters = 99; a.iter = 100; a.first = 0; a.init_res = 0.25;  // init_res: of the set-up from the x left
  cg_recover(a, 1.5, 64);
  CHECK(!a.failed && !a.done && !a.converged && !a.stop && !a.pending && a.first == 1);
  CHECK(a.iter == 64 && a.n_iters == 0 && a.init_res == 1.5 && a.cur_res == 0.25);
  CHECK(a.norm_ref == 3.0 && a.rel_tol == 1e-8 && a.abs_tol == 1e-9 && a.max_iters == 500 && a.crit == kCritL2);
  BiDevState b{};
  b.norm_b = 3.0; b.rel_tol = 1e-8; b.abs_tol = 1e-9; b.max_iters = 500; b.n_prior = 7; b.cur_res = 0.25; b.precond = 1;
  b.failed = b.done = b.converged = 1;
  b.stop_kind = 1; b.n_iters = 99; b.iter = 99; b.init_res = 0.25;
  bi_recover(b, 1.5, 0);
  CHECK(!b.failed && !b.done && !b.converged && b.stop_kind == 0);
  CHECK(b.iter == 0 && b.n_iters == 0 && b.init_res == 1.5 && b.cur_res == 0.25);
  CHECK(b.norm_b == 3.0 && b.n_prior == 7 && b.max_iters == 500 && b.precond == 1);
  CHECK(!bi_finished(&b, b.cur_res, b.iter));
  std::printf(bad ? "FAIL\n" : "OK\n");
  return bad;
}
'''


def test_recovered_state_goes_on(tmp_path):
    src = tmp_path / "recover.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "recover"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "clsparse_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
