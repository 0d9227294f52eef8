// correlator.hip -- current-current correlator of a measured configuration, replacing
// cc_correlator (organic_dense_matrix.c:451-524) on the GPU (FP64).
//
// Transfer matrices (same storage convention as the reference, column-major chunks):
//   R_t0[tau] = B_tau ... B_{nt-1} M_hat^{-1}          (slots 0..nt-1, built slice by slice
//               from nt-1 down to 0; slot tau keeps the state after slice tau)
//   R_0t[tau] = B_{tau-1} ... B_0 (M_hat^{-1})^T        (used at tau before slice tau is applied)
// and for every tau and pair of bond directions (a, b)
//   g_ab(tau) = 1/N sum_{i,j} chi_ia chi_jb [R_t0[j*N+i] R_0t[jb*N+ia] + R_t0[jb*N+ia] R_0t[j*N+i]
//                                        - R_t0[jb*N+i] R_0t[j*N+ia] - R_t0[j*N+ia] R_0t[jb*N+i]]
// with ia = nb(i, 2a), jb = nb(j, 2b), chi_ia = t_a - kappa_a x[0][i][a], chi_jb from slice tau.
// With the antisymmetric current matrices J_a = sum_i chi_ia (|i><ia| - |ia><i|) of slice 0 and J'_b of
// slice tau, and R_0t as the row-indexed Q[j][i] = R_0t[j*N+i], that sum is
//   g_ab(tau) = -1/N sum_{i,j} (J_a R_t0)[i][j] (J'_b Q)[j][i]:
// two neighbours of i in R_t0's column j per a, two neighbours of j in Q's rows per b, then nine
// products, in place of four products of gathered entries for each of the nine (a, b).
// One launch covers every tau.  A workgroup takes up to CC_L sites j of a lattice row (of several rows
// where rows are short) and walks them in order: R_t0's column goes through LDS for the neighbours in
// i, the rows of Q slide along in registers (three new ones per j), all loaded one j ahead.  Block
// sums per (tau, workgroup), then a fixed-order pass per tau.
#include "internal.h"
#include "alloc_group.h"
#include <mutex>

namespace ephmc {

constexpr unsigned CC_L = 32;  // sites j of one lattice row per workgroup
constexpr unsigned CC_J = 8;   // (sizes the block sums: at least this many sites j per workgroup)

// block sums of one correlator call: at most [nt][ceil(N/CC_J)][9]
static size_t cc_partials(unsigned ns, unsigned nt)
{
	return (size_t)nt * ((ns + CC_J - 1) / CC_J) * 9;
}

// workgroups per slice: pieces of a lattice row times row groups, with at least CC_J sites j each
// (but for the last), so no more than ceil(N / CC_J)
struct CcShape { unsigned pieces, len, rows, groups; };

static CcShape cc_shape(const ephmc_ctx *c)
{
	CcShape s;
	s.pieces = (c->l1 + CC_L - 1) / CC_L;
	s.len = (c->l1 + s.pieces - 1) / s.pieces;
	s.rows = c->l1 < CC_J ? (CC_J + c->l1 - 1) / c->l1 : 1;
	s.groups = (c->l2 + s.rows - 1) / s.rows;
	return s;
}

// R_t0 and R_0t (store values each) and the result block (res values), all or none
static int cc_alloc(ephmc_ctx *c, size_t store, size_t res)
{
	if(c->d_Rt0) (void)hipFree(c->d_Rt0);
	if(c->d_R0t) (void)hipFree(c->d_R0t);
	if(c->d_ccg) (void)hipFree(c->d_ccg);
	void **ptrs[3] = {(void **)&c->d_Rt0, (void **)&c->d_R0t, (void **)&c->d_ccg};
	const size_t bytes[3] = {store * sizeof(double), store * sizeof(double), res * sizeof(double)};
	const bool ok = alloc_all_or_none(ptrs, bytes, 3,
		[](void **p, size_t b){ return hipMalloc(p, b) == hipSuccess; },
		[](void *p){ (void)hipFree(p); });
	if(!ok){
		(void)hipGetLastError();
		set_error("correlator buffers (%zu MB) could not be allocated", 2 * store * 8 >> 20);
		return EPHMC_ERR_ALLOC;
	}
	return EPHMC_OK;
}

// a b - c d with both products rounded: exactly zero where they are equal (lattices of extent 1)
__device__ __forceinline__ double cc_diff(double a, double b, double c, double d)
{
#pragma clang fp contract(off)
	return a * b - c * d;
}

// Thread t takes the sites i = t + BT q, q < S (BT S >= N).  Workgroup b works on item `item` of slice tau, eight
// slices at a time, one to an XCD.
// What bounds it: the 2 nt N^2 values read from memory once (2 GB at 32x32, nt 128); each piece's first and
// last columns and the rows above and below it come a second and third time, from the XCD's L2, to
// which all workgroups of a slice go.  585 us there, 3.6 TB/s; with the gathered entries of all nine
// (a, b) from eight rows in LDS 1975 us.
template <int BT, int S>
__global__ __launch_bounds__(BT) void cc_contract_kernel(const double *__restrict__ Tfin, const double *__restrict__ Rt0,
		const double *__restrict__ R0t, const double *__restrict__ coef, const int *__restrict__ nb, unsigned ns, unsigned nt,
		unsigned l1, unsigned l2, CcShape sh, double *__restrict__ partial)
{
	extern __shared__ double rows[];                 // 2 ns: column j of R_t0, by parity of the step
	__shared__ double red[9][BT / 64];
	// eight slices at a time, one to an XCD (workgroups go to the XCDs in turn)
	const unsigned per = sh.pieces * sh.groups, full = nt / 8 * 8, b = blockIdx.x;
	const unsigned tau = b < full * per ? b / (8 * per) * 8 + b % 8 : full + (b - full * per) / per;
	const unsigned item = b < full * per ? b / 8 % per : (b - full * per) % per;
	const size_t mat = (size_t)ns * ns;
	const double *rt = tau == 0 ? Tfin : Rt0 + (size_t)(nt - tau) * mat;
	const double *r0 = R0t + (size_t)tau * mat;
	const double *ct = coef + (size_t)tau * 6 * ns;
	unsigned site[S];
	int in[S][6];
	double cf[S][6];
#pragma unroll
	for(int q = 0; q < S; q++){
		// a thread past the last site works on it with zero coefficients
		const unsigned i = threadIdx.x + BT * q;
		site[q] = min(i, ns - 1);
#pragma unroll
		for(int d = 0; d < 6; d++){
			in[q][d] = nb[d * ns + site[q]];
			cf[q][d] = i < ns ? coef[d * ns + site[q]] : 0.0;
		}
	}
	double g[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
	const unsigned xa = item % sh.pieces * sh.len, xe = min(xa + sh.len, l1);
	unsigned step = 0;
	for(unsigned y = item / sh.pieces * sh.rows; y < min(item / sh.pieces * sh.rows + sh.rows, l2); y++){
		const double *qc = r0 + (size_t)y * l1 * ns, *qu = r0 + (size_t)((y + 1) % l2) * l1 * ns,
			*qd = r0 + (size_t)((y + l2 - 1) % l2) * l1 * ns, *pc = rt + (size_t)y * l1 * ns;
		auto col = [&](const double *m, unsigned x, int q){ return m[(size_t)x * ns + site[q]]; };
		// Q's rows around j = (x, y): c0, c1 = x - 1, x; c2 = x + 1 (the row above: u0, u1 = x - 1, x; below:
		// d1, d2 = x, x + 1)
		double c0[S], c1[S], c2[S], u0[S], u1[S], d1[S], d2[S], p[S];
#pragma unroll
		for(int q = 0; q < S; q++){
			c0[q] = col(qc, (xa + l1 - 1) % l1, q);
			c1[q] = col(qc, xa, q);
			c2[q] = col(qc, (xa + 1) % l1, q);
			u0[q] = col(qu, (xa + l1 - 1) % l1, q);
			u1[q] = col(qu, xa, q);
			d1[q] = col(qd, xa, q);
			d2[q] = col(qd, (xa + 1) % l1, q);
			p[q] = col(pc, xa, q);
		}
		for(unsigned x = xa; x < xe; x++, step++){
			double *row = rows + (step & 1) * ns;
#pragma unroll
			for(int q = 0; q < S; q++) row[site[q]] = p[q];
			const unsigned j = y * l1 + x, x1 = (x + 1) % l1, x2 = (x + 2) % l1;
			double cj[6];
#pragma unroll
			for(int d = 0; d < 6; d++) cj[d] = ct[d * ns + j];
			__syncthreads();
			// the next j's new values (its row of the other parity was last read before this barrier)
			double nc[S], nu[S], nd[S], np[S];
#pragma unroll
			for(int q = 0; q < S; q++){
				nc[q] = col(qc, x2, q);
				nu[q] = col(qu, x1, q);
				nd[q] = col(qd, x2, q);
				np[q] = col(pc, x1, q);
			}
#pragma unroll
			for(int q = 0; q < S; q++){
				double f[3], h[3];
#pragma unroll
				for(int a = 0; a < 3; a++) f[a] = cc_diff(cf[q][2 * a], row[in[q][2 * a]], cf[q][2 * a + 1], row[in[q][2 * a + 1]]);
				// neighbours of j: right / left, up / down, up-left / down-right
				h[0] = cc_diff(cj[0], c2[q], cj[1], c0[q]);
				h[1] = cc_diff(cj[2], u1[q], cj[3], d1[q]);
				h[2] = cc_diff(cj[4], u0[q], cj[5], d2[q]);
#pragma unroll
				for(int a = 0; a < 3; a++)
#pragma unroll
					for(int bb = 0; bb < 3; bb++) g[a * 3 + bb] = fmac(f[a], h[bb], g[a * 3 + bb]);
				c0[q] = c1[q];
				c1[q] = c2[q];
				c2[q] = nc[q];
				u0[q] = u1[q];
				u1[q] = nu[q];
				d1[q] = d2[q];
				d2[q] = nd[q];
				p[q] = np[q];
			}
		}
	}
	// fixed-order sums: a butterfly within each wave, then the waves in order
	const unsigned lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
	for(int q = 0; q < 9; q++){
		double v = g[q];
#pragma unroll
		for(int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
		if(lane == 0) red[q][wv] = v;
	}
	__syncthreads();
	if(threadIdx.x < 9){
		double t = 0;
		for(int w = 0; w < BT / 64; w++) t += red[threadIdx.x][w];
		partial[((size_t)tau * per + item) * 9 + threadIdx.x] = -t;
	}
}

// out[tau][q] = scale * sum of the block sums of slice tau: workgroup tau, wave q; lane l adds the
// blocks l, l + 64, ... and a butterfly adds the lanes (a fixed order)
__global__ __launch_bounds__(576) void cc_sum_kernel(const double *__restrict__ partial, unsigned nblocks, double scale,
		double *__restrict__ out)
{
	const unsigned tau = blockIdx.x, q = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const double *p = partial + (size_t)tau * nblocks * 9 + q;
	double s = 0;
	for(unsigned b = lane; b < nblocks; b += 64) s += p[(size_t)b * 9];
#pragma unroll
	for(int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
	if(lane == 0) out[tau * 9 + q] = s * scale;
}

// The correlator's kernels with the transfer-matrix stores Rt0, R0t (nt N^2 values each) and the
// block sums `partial` (cc_partials values) given: g_ab(tau) (nt x 9) into out, asynchronous.
static int correlate(ephmc_ctx *c, const double *x, const double *minv, double logdet, double *Rt0, double *R0t,
		double *partial, double *out)
{
	const unsigned ns = c->ns, nt = c->nt;
	EPHMC_TRY(coefficients(c, x, false));
	// ZERO_FILLING / SINGLE_PARTICLE start both propagators from the identity
	// (organic_dense_matrix.c:458-470)
	const bool ident = c->cfg.zero_filling || c->cfg.single_particle;
	// R_t0: slices nt-1 .. 0 applied to M_hat^{-1}, the state stored before every slice: step i
	// (slice nt-1-i) stores slot nt-i, so slot s >= 1 is stored entry nt-s; slot 0 is the result
	EPHMC_TRY(chain_forward(c, EPHMC_FP64, minv, c->d_Tfin, Rt0, 1, 1, ident));
	// R_0t: transposed inverse, then slices 0 .. nt-1 ascending; stored entry tau = state at tau
	if(!ident) EPHMC_TRY(transpose_plus_identity(c, EPHMC_FP64, minv, c->d_gj[0], 0));
	EPHMC_TRY(chain_forward(c, EPHMC_FP64, c->d_gj[0], c->d_gj[1], R0t, 1, 0, ident));
	const CcShape sh = cc_shape(c);
	const unsigned by = sh.pieces * sh.groups;
	const size_t lds = 2 * (size_t)ns * sizeof(double);
#define EPHMC_CC(BT, S)                                                                                    \
	cc_contract_kernel<BT, S><<<by * nt, BT, lds, c->stream>>>(c->d_Tfin, Rt0, R0t, c->d_coef64, c->d_nb, ns, nt, c->l1, \
		c->l2, sh, partial)
	// two sites i per thread, so that a CU holds workgroups enough to cover each other's barriers
	// (32x32: 585 us against 830 with one site on 1024 threads)
	if(ns <= 64) EPHMC_CC(64, 1);
	else if(ns <= 128) EPHMC_CC(64, 2);
	else if(ns <= 256) EPHMC_CC(128, 2);
	else if(ns <= 512) EPHMC_CC(256, 2);
	else if(ns <= 1024) EPHMC_CC(512, 2);
	else if(ns <= 2048) EPHMC_CC(512, 4);
	else { set_error("correlator: %u sites exceed 2048", ns); return EPHMC_ERR_UNSUPPORTED; }
#undef EPHMC_CC
	EPHMC_LAUNCHED();
	cc_sum_kernel<<<nt, 576, 0, c->stream>>>(partial, by, c->cfg.single_particle ? exp(-logdet) : 1.0 / ns,
		out);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// Allocation-free variant (ephmc_cc_correlator_static): its transfer-matrix stores and block sums
// live in this file-scope device array, 64 MiB on every GPU the library runs on, held until the
// process ends.  In host code `scratch` is only a symbol: its device address on each GPU comes from
// hipGetSymbolAddress, taken once per device on the entry point's first call there, and only that
// address is passed to kernels.  Calls that overlap on one GPU share (and race on) the array.
constexpr size_t CC_STATIC_DOUBLES = (size_t)64 << 17;     // 64 MiB of doubles
static __device__ __align__(256) double scratch[CC_STATIC_DOUBLES];

constexpr int CC_MAX_DEVICES = 64;
static double *g_scratch_addr[CC_MAX_DEVICES];
static std::mutex g_scratch_mu;

// device address of `scratch` on the context's GPU (looked up once per device)
static int static_scratch(ephmc_ctx *c, double **out)
{
	if(c->device < 0 || c->device >= CC_MAX_DEVICES){ set_error("device %d out of range", c->device); return EPHMC_ERR_ARG; }
	std::lock_guard<std::mutex> lock(g_scratch_mu);
	if(!g_scratch_addr[c->device]){
		int prev = 0;
		EPHMC_HIP(hipGetDevice(&prev));
		EPHMC_HIP(hipSetDevice(c->device));
		void *p = nullptr;
		const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
		(void)hipSetDevice(prev);
		if(e != hipSuccess || !p){
			(void)hipGetLastError();
			set_error("hipGetSymbolAddress(scratch) failed on device %d: %s", c->device, hipGetErrorString(e));
			return EPHMC_ERR_HIP;
		}
		g_scratch_addr[c->device] = (double *)p;
	}
	*out = g_scratch_addr[c->device];
	return EPHMC_OK;
}

} // namespace ephmc

using namespace ephmc;

extern "C" int ephmc_cc_correlator_static(ephmc_ctx *c, const double *x, const double *minv, double logdet, double *greens_dev)
{
	if(!c || !x || !greens_dev || (!minv && !c->cfg.zero_filling && !c->cfg.single_particle)){
		set_error("null argument");
		return EPHMC_ERR_ARG;
	}
	const size_t store = (size_t)c->nt * c->mat, need = 2 * store + cc_partials(c->ns, c->nt);
	if(need > CC_STATIC_DOUBLES){
		set_error("ephmc_cc_correlator_static: needs %zu doubles (2 nt N^2 + block sums), the static scratch holds %zu "
			"(64 MiB); use ephmc_cc_correlator", need, CC_STATIC_DOUBLES);
		return EPHMC_ERR_ARG;
	}
	double *base = nullptr;
	EPHMC_TRY(static_scratch(c, &base));
	// every value of the stores and block sums is written before it is read: nothing to clear
	return correlate(c, x, minv, logdet, base, base + store, base + 2 * store, greens_dev);
}

extern "C" int ephmc_cc_correlator(ephmc_ctx *c, const double *x, const double *minv, double logdet, double *greens_host)
{
	if(!c || !x || !greens_host || (!minv && !c->cfg.zero_filling && !c->cfg.single_particle)){
		set_error("null argument");
		return EPHMC_ERR_ARG;
	}
	const unsigned ns = c->ns, nt = c->nt;
	const size_t mat = c->mat;
	if(!c->d_Rt0 || !c->d_R0t || !c->d_ccg){
		// all three or none: a failed allocation releases the others, so the next call retries
		// instead of running on a partial set
		const int rc = cc_alloc(c, nt * mat, nt * 9 + cc_partials(ns, nt));
		if(rc != EPHMC_OK) return rc;
	}
	EPHMC_TRY(timer_begin(c, "correlator"));
	EPHMC_TRY(correlate(c, x, minv, logdet, c->d_Rt0, c->d_R0t, c->d_ccg + (size_t)nt * 9, c->d_ccg));
	EPHMC_TRY(timer_end(c, "correlator"));
	EPHMC_HIP(hipMemcpyAsync(greens_host, c->d_ccg, nt * 9 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
	EPHMC_HIP(hipStreamSynchronize(c->stream));
	return EPHMC_OK;
}
