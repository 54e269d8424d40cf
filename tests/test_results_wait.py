"""The host's wait for reduction results (csrc/lmm_results.h), which polls
entries of pinned memory and falls back to the stream synchronisation: a
program built with the host compiler plays the kernels and the
synchronisation, so both fallbacks and the failures are reached without a GPU.
On the GPU, solves that never poll (LMM_POLL_US=0) give the same bits."""
import os
import shutil
import subprocess

import pytest

from lowmachmixtures_amd import problems as P
from lowmachmixtures_amd import stokes as S
from tests.helpers import bit_equal

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lowmachmixtures_amd", "csrc")

SRC = r"""
#include <cstdio>
#include <cstring>
#include "lmm_results.h"
using lmm::HostResults;
static int bad = 0;
#define CHECK(c) do { if (!(c)) { bad++; printf("line %d: %s\n", __LINE__, #c); } } while (0)
int main() {
  double h[8];
  int syncs = 0;
  auto never = [&] { syncs++; return false; };
  auto idle = [&] { syncs++; return true; };
  HostResults r;

  // written by another thread: found by the poll, whichever entry is first
  r.arm(h, 3);
  std::thread t([&] {
    for (int q = 2; q >= 0; q--) __atomic_store_n((uint64_t *)(h + q), q + 1u, __ATOMIC_RELEASE);
  });
  CHECK(r.wait(60000000, never) && syncs == 0);
  t.join();

  // nothing armed: a synchronisation
  syncs = 0;
  CHECK(r.wait(1000, idle) && syncs == 1);

  // time-out, and a limit of zero: synchronised, then written
  for (long limit : {0L, 1L}) {
    syncs = 0;
    r.arm(h, 2);
    CHECK(r.wait(limit, [&] { syncs++; h[0] = h[1] = 7.0; return true; }) && syncs == 1 && h[1] == 7.0);
  }

  // armed twice: the first write does not end the wait
  syncs = 0;
  r.arm(h, 1);
  r.arm(h, 1);
  h[0] = 1.0;
  CHECK(r.wait(60000000, [&] { syncs++; h[0] = 2.0; return true; }) && syncs == 1 && h[0] == 2.0);

  // the synchronisation fails, or succeeds and leaves an entry unwritten
  r.arm(h, 2);
  h[0] = 1.0;
  CHECK(!r.wait(1, never));
  r.arm(h, 2);
  h[0] = 1.0;
  CHECK(!r.wait(1, idle));
  r.arm(h, 1);
  r.arm(h, 1);
  CHECK(!r.wait(1, idle));

  // a failed wait leaves nothing armed
  syncs = 0;
  r.arm(h, 1);
  h[0] = 3.0;
  CHECK(r.wait(60000000, never) && syncs == 0);

  // results that are not finite are results
  r.arm(h, 3);
  h[0] = __builtin_nan("");
  h[1] = -__builtin_inf();
  h[2] = h[1] - h[1];
  CHECK(r.wait(60000000, never) && syncs == 0);
  return bad;
}
"""


def test_wait_and_its_fallbacks(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "w.cpp", tmp_path / "w"
    src.write_text(SRC)
    subprocess.run([gxx, "-std=c++17", "-O2", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("dim,n,prec,cycles", [(2, (64, 64), "fp64", 2), (3, (32, 32, 32), "fp64", 1),
                                               (3, (32, 32, 32), "fp32_mg", 1)])
def test_never_polling_gives_the_same_bits(dim, n, prec, cycles, monkeypatch):
    pb = P.small_problem(dim, n, visc_type=-1, seed=23, contrast=20.0)
    b_u = P.rhs_from_noise_host(pb)
    out = []
    for us in (None, "0"):
        if us is not None:
            monkeypatch.setenv("LMM_POLL_US", us)
        with S.Context(dim, pb.n, pb.dx, visc_type=-1, precision={"fp64": S.FP64, "fp32_mg": S.FP32_MG}[prec],
                       mg_max_vcycles=cycles, stag_mg_max_vcycles=cycles) as ctx:
            dp = S.DeviceProblem(ctx, pb, rhs=b_u)
            _, info = dp.solve()
            out.append((info["total_iter"], dp.solution()))
    assert out[0][0] == out[1][0]
    assert bit_equal(out[0][1][0], out[1][1][0]) and bit_equal(out[0][1][1], out[1][1][1])
