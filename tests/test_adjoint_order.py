"""The force sweep (csrc/adjoint.hip) computes the same bits in whatever order its threads reach a
barrier.  The sweep's source up to its first kernel is compiled for the CPU, with a coroutine per
thread: between two barriers the threads run one after the other, once in ascending and once in
descending order, so any two accesses to LDS that no barrier orders give different results.  Stored
(k = 1) and recomputed (k > 1) slices, W_0 written early or not, over the forms that the sizes select:
one site per thread with the next slice's S built ahead, without, fp64 at four columns, two sites."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "electron-phonon-hmc_amd", "csrc")

# the declarations that internal.h and the sweep's body name
HIP_RUNTIME = r"""
#pragma once
#include <cmath>
#include <cstdlib>
#include <algorithm>
#define __host__
#define __device__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
using std::fma;
using std::max;
using std::min;
typedef int hipError_t;
typedef struct hipStream *hipStream_t;
typedef struct hipEvent *hipEvent_t;
typedef struct hipGraph *hipGraph_t;
typedef struct hipGraphExec *hipGraphExec_t;
struct double2 { double x, y; };
struct double4 { double x, y, z, w; };
struct int4 { int x, y, z, w; };
struct Dim { unsigned x = 0, y = 0, z = 0; };
extern Dim threadIdx;
void __syncthreads();
"""

DRIVER = r"""
#include "sweep.h"
#include <cstdio>
#include <cstring>
#include <functional>
#include <random>
#include <ucontext.h>
Dim threadIdx;
namespace ephmc { alignas(16) unsigned char smem_raw[160 * 1024]; }
static ucontext_t sched;
static std::vector<ucontext_t> fib;
static std::vector<char> done;
static unsigned cur;
static std::function<void()> body;
static void entry(){ body(); done[cur] = 1; swapcontext(&fib[cur], &sched); }
void __syncthreads(){ const unsigned me = cur; swapcontext(&fib[me], &sched); threadIdx.x = me; }

static void run(unsigned n, bool descending)
{
	constexpr size_t STACK = 96 * 1024;
	std::vector<char> stack(STACK * n);
	fib.assign(n, ucontext_t());
	done.assign(n, 0);
	std::memset(ephmc::smem_raw, 0, sizeof(ephmc::smem_raw));
	for(unsigned t = 0; t < n; t++){
		getcontext(&fib[t]);
		fib[t].uc_stack.ss_sp = stack.data() + STACK * t;
		fib[t].uc_stack.ss_size = STACK;
		fib[t].uc_link = nullptr;
		makecontext(&fib[t], entry, 0);
	}
	for(unsigned left = n; left;){
		for(unsigned i = 0; i < n; i++){
			const unsigned t = descending ? n - 1 - i : i;
			if(done[t]) continue;
			cur = t;
			threadIdx.x = t;
			swapcontext(&sched, &fib[t]);
			if(done[t]) left--;
		}
	}
}

template <typename R, int C, int BT, int S, int DEG>
static bool same(unsigned l1, unsigned l2, int nt, int direct, int early)
{
	using namespace ephmc;
	const unsigned ns = l1 * l2;
	std::mt19937_64 rng(l1 * 100 + DEG);
	std::normal_distribution<double> g;
	auto draw = [&](size_t n, double s){ std::vector<R> v(n); for(R &e : v) e = (R)(s * g(rng)); return v; };
	std::vector<int> nb(6 * (size_t)ns);
	for(unsigned i = 0; i < ns; i++){
		const unsigned x = i % l1, y = i / l1, xp = (x + 1) % l1, xm = (x + l1 - 1) % l1, yp = (y + 1) % l2, ym = (y + l2 - 1) % l2;
		const unsigned v[6] = {y * l1 + xp, y * l1 + xm, yp * l1 + x, ym * l1 + x, yp * l1 + xm, ym * l1 + xp};
		for(int d = 0; d < 6; d++) nb[(size_t)d * ns + i] = (int)v[d];
	}
	const std::vector<R> coef = draw((size_t)nt * 6 * ns, 0.2), ck = draw((size_t)nt * ns * ns, 1);
	std::vector<double> w0((size_t)ns * ns);
	for(double &e : w0) e = g(rng);
	AdjArgs<R> a{};
	a.coef = coef.data();
	a.nb = nb.data();
	a.mu = (R)-0.1;
	a.ns = ns;
	a.deg = DEG;
	for(int q = 0; q <= DEG; q++) a.cm[q] = (R)(1.0 / (q + 1));
	a.np = DEG / 2;
	for(int p = 0; p < a.np; p++){ a.a_lin[p] = (R)0.5; a.a_quad[p] = (R)0.25; a.cplx[p] = 1; }
	a.ck = ck.data();
	a.direct = direct;
	a.w0_early = early;
	a.seg_stride = nt * C * ns;
	a.w_init = w0.data();
	a.nwg = (ns + C - 1) / C;
	a.tau_b = 0;
	a.tau_e = nt;
	const unsigned bx = a.nwg - 1;                  // the last workgroup, where columns may be missing
	std::vector<R> out[2][2];
	for(int o = 0; o < 2; o++){
		std::vector<R> seg((size_t)(bx + 1) * a.seg_stride), part((size_t)nt * a.nwg * 3 * ns), w((size_t)ns * ns);
		a.seg = seg.data();
		a.partial = part.data();
		a.wbuf = w.data();
		body = [&]{ adjoint_body<R, C, BT, S, DEG>(a, bx, BT); };
		run(BT, o == 1);
		out[o][0] = part;
		out[o][1] = w;
	}
	double sum = 0;
	for(R v : out[0][0]) sum += std::fabs((double)v);
	return sum > 0 && std::isfinite(sum) && out[0][0] == out[1][0] && out[0][1] == out[1][1];
}

int main()
{
	int bad = 0;
	for(int direct = 0; direct < 2; direct++)
		for(int early = 0; early < 2; early++){
#define CASE(R, C, BT, S, DEG, L1, L2, NT) do {                                                    \
				const bool ok = same<R, C, BT, S, DEG>(L1, L2, NT, direct, early);                     \
				printf("%s %d columns, %d threads, %d sites each, degree %d, %s, W_0 %s: %s\n", #R, C, BT, S, DEG, \
					direct ? "stored" : "recomputed", early ? "early" : "in place", ok ? "same" : "ORDER MATTERS"); \
				bad += !ok;                                                                            \
			} while(0)
			CASE(double, 1, 256, 1, 4, 11, 13, 5);
			CASE(float, 2, 256, 1, 2, 9, 9, 4);
			CASE(double, 2, 512, 1, 6, 19, 15, 3);
			CASE(float, 4, 512, 1, 4, 19, 15, 3);
			CASE(float, 4, 1024, 1, 4, 27, 19, 3);
			CASE(double, 4, 1024, 1, 4, 27, 19, 3);
			CASE(double, 2, 1024, 1, 8, 27, 19, 3);
			CASE(float, 2, 1024, 2, 4, 41, 25, 3);
			CASE(double, 2, 1024, 2, 4, 41, 25, 3);
		}
	return bad != 0;
}
"""


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    d = tmp_path_factory.mktemp("sweep")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP_RUNTIME)
    with open(os.path.join(CSRC, "adjoint.hip")) as f:
        text = f.read()
    head = text[:text.index("\ntemplate <typename R, int C, int BT, int S, int DEG>\n__global__")]
    assert "adjoint_body(" in head
    (d / "sweep.h").write_text(head.replace('"internal.h"', '"%s"' % os.path.join(CSRC, "internal.h")) + "\n}\n")
    (d / "t.cpp").write_text(DRIVER)
    exe = d / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-I" + str(d), str(d / "t.cpp"), "-o", str(exe)], check=True)
    return str(exe)


def test_sweep_does_not_depend_on_thread_order(prog):
    r = subprocess.run([prog], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
