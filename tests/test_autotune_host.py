"""The autotuner's choice, on the host alone: tc_autotune compiled with a predictor launch and an
event timer that stand in for the device's.  It keeps the shape in force where no candidate is
quicker, takes a quicker one, and leaves the correction's shape, which it does not time, as it is."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "simpletcsolver_amd", "csrc")

STANDIN = r"""
#include <stdio.h>
#include <stdlib.h>
#include <hip/hip_runtime_api.h>
#include "tcstep.h"
#include "host/tc_internal.h"
#include "host/tc_kernels.h"

static int g_kb, g_ty, g_qkb, g_qty;
static float g_quick;

hipError_t hipSetDevice(int d){ return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t * e){ *e = NULL; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s){ return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e){ return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e){ return hipSuccess; }
/* every shape takes 1 ms a launch, one of them g_quick */
hipError_t hipEventElapsedTime(float * ms, hipEvent_t a, hipEvent_t b){
  *ms = 3.f * (g_kb == g_qkb && g_ty == g_qty ? g_quick : 1.f);
  return hipSuccess;
}
int tck_launch_predict(const tc_geom_t * g, const tc_coef_t * c, const tc_flags_t * f, const double * const * cur,
    const double * p, double * const * nxt, void * const * dlt, const void * const * sb, void * const * sa,
    const float * const * corr, const double * dt, int rk, int final_here, int mixed, int kb, int ty, int window,
    hipStream_t stream){
  g_kb = kb;
  g_ty = ty;
  return 0;
}

/* arguments: nz, the predictor's shape, the correction's, the quick shape and its time; prints the
 * shapes after tuning and what the call returned */
int main(int argc, char ** argv){
  tc_solver_t * s = calloc(1, sizeof(*s));
  s->p.nz = atoi(argv[1]);
  s->tune[TC_TUNE_PREDICT][0] = atoi(argv[2]); s->tune[TC_TUNE_PREDICT][1] = atoi(argv[3]);
  s->tune[TC_TUNE_CORRECT][0] = atoi(argv[4]); s->tune[TC_TUNE_CORRECT][1] = atoi(argv[5]);
  g_qkb = atoi(argv[6]); g_qty = atoi(argv[7]); g_quick = (float)atof(argv[8]);
  int kb, ty;
  double ms;
  if(tc_autotune(s, 3, &kb, &ty, &ms)) return 1;
  printf("%d %d %d %d %d %d %.2f\n", s->tune[TC_TUNE_PREDICT][0], s->tune[TC_TUNE_PREDICT][1],
      s->tune[TC_TUNE_CORRECT][0], s->tune[TC_TUNE_CORRECT][1], kb, ty, ms);
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("gcc") or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("no C compiler or HIP headers")
    d = tmp_path_factory.mktemp("autotune")
    src, exe = d / "standin.c", d / "standin"
    src.write_text(STANDIN)
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT}/include", f"-I{CSRC}", f"-I{CSRC}/host", str(src), f"{CSRC}/host/tc_solver.c",
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(exe), "-lm"], check=True)
    return lambda *a: subprocess.run([str(exe), *map(str, a)], check=True, capture_output=True, text=True).stdout.split()


@pytest.mark.parametrize("nz,shape,correct", [(256, (24, 4), (8, 4)), (32, (1, 4), (1, 4)), (105, (12, 4), (2, 4)), (6, (6, 4), (4, 4))])
def test_the_shape_in_force_stays_where_it_is_the_quickest(program, nz, shape, correct):
    got = program(nz, *shape, *correct, *shape, 0.9)
    assert got == [str(v) for v in (*shape, *correct, *shape)] + ["0.90"]


@pytest.mark.parametrize("nz,shape,correct", [(256, (24, 4), (8, 4)), (32, (1, 4), (1, 4))])
def test_a_tie_changes_nothing(program, nz, shape, correct):
    assert program(nz, *shape, *correct, 99, 4, 0.5) == [str(v) for v in (*shape, *correct, *shape)] + ["1.00"]


@pytest.mark.parametrize("quick", [(2, 1), (8, 4), (16, 2), (32, 4)])
def test_a_quicker_candidate_is_taken_for_the_predictor_alone(program, quick):
    assert program(256, 24, 4, 14, 4, *quick, 0.5) == [str(v) for v in (*quick, 14, 4, *quick)] + ["0.50"]


def test_candidates_deeper_than_the_grid_are_left_out(program):
    assert program(10, 6, 4, 2, 4, 16, 4, 0.5) == ["6", "4", "2", "4", "6", "4", "1.00"]
