// chain.hip -- slice coefficients and the chained slice product on column blocks.
//
// A slice factor B_tau = p(A_tau) = prod_pairs (1 + a_lin A + a_quad A^2) with
// A_tau = mu + K(x_tau) the symmetric 7-point stencil of the triangular lattice
// (apply_mu_K_to_v, organic_dense_matrix.c:96-120; pair expansion :168-207).  The reference
// applies p(A) as stencils to every column of a dense N x N matrix (:209-216); this file does
// the same on the GPU: one workgroup owns C columns for the whole chain, keeps them in LDS
// (layout [site][column] so a neighbour read fetches C adjacent values) and applies all
// slices in sequence.  Each output site gathers its six bond neighbours:
//   w[i] = mu v[i] + sum_d coef[tau][d][i] v[nb(i,d)],  d = R, L, TR, BL, TL, BR,
// where coef[tau][d][i] = t_k - kappa_k x[tau][link(i,d)] is the coefficient of the bond
// between i and nb(i,d) (k = d/2).  This gather is exactly the reference's scatter over
// forward bonds, including lattices of extent 1 or 2 where bonds alias.
#include "internal.h"
#include "stencil.h"
#include "patch.h"
#include <vector>
#include <cstdlib>
#include <algorithm>
#include <cstring>

namespace ephmc {

__device__ __forceinline__ void coef_body(const double *__restrict__ x, const unsigned *__restrict__ link,
		double t0, double t1, double t2, double k0, double k1, double k2,
		unsigned ns, unsigned nt, double *__restrict__ c64, float *__restrict__ c32, unsigned bx, unsigned gx)
{
	const size_t n = (size_t)nt * 6 * ns;
	for(size_t e = bx * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gx * blockDim.x){
		const size_t tau = e / (6 * ns);
		const unsigned r = (unsigned)(e - tau * 6 * ns);
		const unsigned d = r / ns, s = r - d * ns;
		const unsigned k = d >> 1;
		const double tk = k == 0 ? t0 : (k == 1 ? t1 : t2);
		const double kk = k == 0 ? k0 : (k == 1 ? k1 : k2);
		const double f = tk - kk * x[tau * 3 * ns + link[d * ns + s]];
		if(c64) c64[e] = f;
		if(c32) c32[e] = (float)f;
	}
}

__global__ void coef_kernel(const double *__restrict__ x, const unsigned *__restrict__ link,
		double t0, double t1, double t2, double k0, double k1, double k2,
		unsigned ns, unsigned nt, double *__restrict__ c64, float *__restrict__ c32)
{
	coef_body(x, link, t0, t1, t2, k0, k1, k2, ns, nt, c64, c32, blockIdx.x, gridDim.x);
}

// many chains in one launch (blockIdx.z = chain; each chain's own grid in gx)
struct CoefArgs {
	const double *x;
	const unsigned *link;
	double t[3], k[3];
	unsigned ns, nt, gx;
	double *c64;
	float *c32;
};

__global__ void coef_multi_kernel(const CoefArgs *__restrict__ tab)
{
	const CoefArgs &a = tab[blockIdx.z];
	if(blockIdx.x >= a.gx) return;
	coef_body(a.x, a.link, a.t[0], a.t[1], a.t[2], a.k[0], a.k[1], a.k[2], a.ns, a.nt, a.c64, a.c32, blockIdx.x, a.gx);
}

// the site form's coefficients (blockIdx.x < nt: slice blockIdx.x) and the patch form's
// (blockIdx.x - nt: its slice) of one arithmetic, in one launch.  The slices lie on the grid's first axis,
// the only one that takes more than 65535 workgroups
template <typename R>
__global__ __launch_bounds__(256) void coef_patch_kernel(const double *__restrict__ x, const unsigned *__restrict__ link,
		double t0, double t1, double t2, double k0, double k1, double k2, unsigned ns, unsigned nt, double *__restrict__ c64,
		float *__restrict__ c32, const int *__restrict__ bond, unsigned nbond, R *__restrict__ out)
{
	const bool site = blockIdx.x < nt;
	const size_t tau = site ? blockIdx.x : blockIdx.x - nt;
	const unsigned n = site ? 6 * ns : nbond;
	for(unsigned e = blockIdx.y * 256 + threadIdx.x; e < n; e += gridDim.y * 256){
		const int b = site ? (int)link[e] : bond[e], k = b % 3;
		const double tk = k == 0 ? t0 : (k == 1 ? t1 : t2);
		const double kk = k == 0 ? k0 : (k == 1 ? k1 : k2);
		const double f = tk - kk * x[tau * 3 * ns + b];
		if(site){
			c64[tau * n + e] = f;
			if(c32) c32[tau * n + e] = (float)f;
		}else out[tau * n + e] = (R)f;
	}
}

int coefficients(ephmc_ctx *c, const double *x, bool want32)
{
	const double *t = c->cfg.t, *k = c->cfg.kappa;
	float *c32 = want32 ? c->d_coef32 : nullptr;
	const PatchTab &pt = c->patch[want32 ? 1 : 0];
	c->patch_slot = -1;
	if(patch_on(c, want32 ? EPHMC_MIXED : EPHMC_FP64)){
		c->patch_slot = want32 ? 1 : 0;
		const unsigned m = pt.nk * pt.tp;
		const dim3 g(2 * c->nt, (std::max(m, 6 * c->ns) + 255) / 256);
		if(want32) coef_patch_kernel<float><<<g, 256, 0, c->stream>>>(x, c->d_link, t[0], t[1], t[2], k[0], k[1], k[2], c->ns, c->nt,
			c->d_coef64, c32, pt.bond, m, (float *)pt.coef);
		else coef_patch_kernel<double><<<g, 256, 0, c->stream>>>(x, c->d_link, t[0], t[1], t[2], k[0], k[1], k[2], c->ns, c->nt,
			c->d_coef64, c32, pt.bond, m, (double *)pt.coef);
		EPHMC_LAUNCHED();
		return EPHMC_OK;
	}
	const size_t n = (size_t)c->nt * 6 * c->ns;
	const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
	coef_kernel<<<blocks, 256, 0, c->stream>>>(x, c->d_link, t[0], t[1], t[2], k[0], k[1], k[2], c->ns, c->nt, c->d_coef64, c32);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// ---------------------------------------------------------------------------------------------
template <typename R>
struct ChainArgs {
	const R *coef;          // [nt][6][ns]
	const int *nb;          // [6][ns]
	R mu;
	unsigned ns;
	const R *src;           // start columns (column-major), or null for the identity
	R *dst;                 // result columns
	R *ck;                  // checkpoints: state before every ck_every-th slice, or null
	unsigned ck_every;
	int tau0, dir, ntau;    // slices tau0, tau0+dir, ... (ntau of them)
	int np;
	R a_lin[MAX_PAIRS], a_quad[MAX_PAIRS];
	int cplx[MAX_PAIRS];
};

// out = mu*own + sum_d cf[d] * buf[nb[d]][c]
template <typename R, int C>
__device__ __forceinline__ void stencil_gather(const R *__restrict__ buf, const int (&nbr)[6], const R (&cf)[6],
		R mu, const R (&own)[C], R (&out)[C])
{
#pragma unroll
	for(int c = 0; c < C; c++) out[c] = mu * own[c];
	if constexpr(sizeof(R) == 4){
		// fp32: the six neighbour reads are issued together (fp64 keeps them interleaved with the
		// sums, which holds fewer registers); the sum is taken in the order d = 0..5 either way
		R nv[6][C];
#pragma unroll
		for(int d = 0; d < 6; d++)
#pragma unroll
			for(int c = 0; c < C; c++) nv[d][c] = buf[(size_t)nbr[d] * C + c];
#pragma unroll
		for(int d = 0; d < 6; d++)
#pragma unroll
			for(int c = 0; c < C; c++) out[c] = fmac(cf[d], nv[d][c], out[c]);
	}else{
#pragma unroll
		for(int d = 0; d < 6; d++){
			const R *q = buf + (size_t)nbr[d] * C;
#pragma unroll
			for(int c = 0; c < C; c++) out[c] = fmac(cf[d], q[c], out[c]);
		}
	}
}

// fp32 with one site per thread: every lane loads and gathers (a lane past the last site reads
// site ns-1 or neighbour 0, all in bounds, and stores nothing), so no lane needs zero values of
// its own, and the second LDS buffer sits at the constant offset C * BT, which a read takes as an
// immediate offset
template <typename R, int S>
constexpr bool chain_all_lanes(){ return sizeof(R) == 4 && S == 1; }

template <typename R, int C, int BT, int S>
constexpr size_t chain_lds_bytes(unsigned ns)
{
	return 2 * (chain_all_lanes<R, S>() ? (size_t)C * BT : (size_t)C * ns) * sizeof(R);
}

template <typename R, int C, int BT, int S>
__device__ __forceinline__ void chain_body(const ChainArgs<R> &a, unsigned bx)
{
	extern __shared__ __align__(16) unsigned char smem_raw[];
	constexpr bool ALL_LANES = chain_all_lanes<R, S>();
	const unsigned ns = a.ns;
	R *V = reinterpret_cast<R *>(smem_raw);
	R *W = V + (ALL_LANES ? (size_t)C * BT : (size_t)C * ns);
	const unsigned col0 = bx * C;
	const size_t mat = (size_t)ns * ns;

	unsigned site[S];
	bool act[S];
	int nbr[S][6];
	R v[S][C], w[S][C], cf[S][6];
#pragma unroll
	for(int j = 0; j < S; j++){
		site[j] = threadIdx.x + j * BT;
		act[j] = site[j] < ns;
#pragma unroll
		for(int d = 0; d < 6; d++) nbr[j][d] = act[j] ? a.nb[d * ns + site[j]] : 0;
#pragma unroll
		for(int c = 0; c < C; c++){
			const unsigned col = col0 + c;
			R val = 0;
			if(act[j] && col < ns) val = a.src ? a.src[(size_t)col * ns + site[j]] : (R)(site[j] == col ? 1 : 0);
			v[j][c] = val;
		}
	}

	// coefficients of the next slice are loaded one slice ahead, so their latency overlaps the
	// stencils of the current one
	R cfn[S][6];
	auto load_cf = [&](int i){
		const R *cft = a.coef + (size_t)(a.tau0 + a.dir * i) * 6 * ns;
#pragma unroll
		for(int j = 0; j < S; j++){
			const unsigned sl = ALL_LANES && !act[j] ? ns - 1 : site[j];
#pragma unroll
			for(int d = 0; d < 6; d++) cfn[j][d] = (ALL_LANES || act[j]) ? cft[d * ns + sl] : (R)0;
		}
	};
	if(a.ntau > 0) load_cf(0);
	for(int i = 0; i < a.ntau; i++){
		if(a.ck && (i % a.ck_every) == 0){
			R *ck = a.ck + (size_t)(i / a.ck_every) * mat;
#pragma unroll
			for(int j = 0; j < S; j++)
#pragma unroll
				for(int c = 0; c < C; c++)
					if(act[j] && col0 + c < ns) ck[(size_t)(col0 + c) * ns + site[j]] = v[j][c];
		}
#pragma unroll
		for(int j = 0; j < S; j++)
#pragma unroll
			for(int d = 0; d < 6; d++) cf[j][d] = cfn[j][d];
		if(i + 1 < a.ntau) load_cf(i + 1);

#pragma unroll
		for(int p = 0; p < MAX_PAIRS; p++){
			if(p >= a.np) break;
#pragma unroll
			for(int j = 0; j < S; j++)
				if(act[j])
#pragma unroll
					for(int c = 0; c < C; c++) V[(size_t)site[j] * C + c] = v[j][c];
			__syncthreads();
#pragma unroll
			for(int j = 0; j < S; j++)
				if(ALL_LANES || act[j]) stencil_gather<R, C>(V, nbr[j], cf[j], a.mu, v[j], w[j]);
			if(a.cplx[p]){
				// W is free: its last readers passed the barrier above.  The barrier below also
				// retires every read of V before the next pair overwrites it.
#pragma unroll
				for(int j = 0; j < S; j++)
					if(act[j])
#pragma unroll
						for(int c = 0; c < C; c++) W[(size_t)site[j] * C + c] = w[j][c];
				__syncthreads();
#pragma unroll
				for(int j = 0; j < S; j++){
					if(!ALL_LANES && !act[j]) continue;
					R z[C];
					stencil_gather<R, C>(W, nbr[j], cf[j], a.mu, w[j], z);
#pragma unroll
					for(int c = 0; c < C; c++) v[j][c] = v[j][c] + fmac(a.a_quad[p], z[c], a.a_lin[p] * w[j][c]);
				}
			}else{
				__syncthreads();
#pragma unroll
				for(int j = 0; j < S; j++)
#pragma unroll
					for(int c = 0; c < C; c++) v[j][c] = fmac(a.a_lin[p], w[j][c], v[j][c]);
			}
		}
	}
	if(a.dst){
#pragma unroll
		for(int j = 0; j < S; j++)
#pragma unroll
			for(int c = 0; c < C; c++)
				if(act[j] && col0 + c < ns) a.dst[(size_t)(col0 + c) * ns + site[j]] = v[j][c];
	}
}

template <typename R, int C, int BT, int S>
__global__ __launch_bounds__(BT) void chain_kernel(ChainArgs<R> a)
{
	chain_body<R, C, BT, S>(a, blockIdx.x);
}

// many chains in one launch: blockIdx.z = chain, blockIdx.x = its column block (blocks past the
// chain's own ceil(ns / C) return).  With one site per thread the workgroup may have fewer threads
// than BT (at least ns); the LDS layout stays that of BT.
template <typename R, int C, int BT, int S>
__global__ __launch_bounds__(BT) void chain_multi_kernel(const ChainArgs<R> *__restrict__ tab)
{
	const ChainArgs<R> &a = tab[blockIdx.z];
	if(blockIdx.x >= (a.ns + C - 1) / C) return;
	chain_body<R, C, BT, S>(a, blockIdx.x);
}

// ---------------------------------------------------------------------------------------------
// ---------------------------------------------------------------------------------------------
// Strip form of the same chain (stencil.h): a thread owns M consecutive sites of a lattice row.
// The sum is taken in the same order (d = R, L, TR, BL, TL, BR) as stencil_gather, so both forms
// give identical bits.
template <typename R, int C, int M, int LB>
__global__ __launch_bounds__(LB) void chain_strip_kernel(ChainArgs<R> a)
{
	extern __shared__ __align__(16) unsigned char smem_raw[];
	R *V = reinterpret_cast<R *>(smem_raw);
	R *W = V + (size_t)C * a.ns;
	const unsigned ns = a.ns;
	const unsigned col0 = blockIdx.x * C;
	const size_t mat = (size_t)ns * ns;
	const unsigned s0 = threadIdx.x * M;      // blockDim.x * M == ns
	StripNb<M> sn;
	strip_neighbours<M>(a.nb, ns, s0, sn);
	R v[M][C], w[M][C], cf[M][6];
#pragma unroll
	for(int k = 0; k < M; k++)
#pragma unroll
		for(int c = 0; c < C; c++){
			const unsigned col = col0 + c, site = s0 + k;
			R val = 0;
			if(col < ns) val = a.src ? a.src[(size_t)col * ns + site] : (R)(site == col ? 1 : 0);
			v[k][c] = val;
		}
	for(int i = 0; i < a.ntau; i++){
		const int tau = a.tau0 + a.dir * i;
		if(a.ck && (i % a.ck_every) == 0){
			R *ck = a.ck + (size_t)(i / a.ck_every) * mat;
#pragma unroll
			for(int k = 0; k < M; k++)
#pragma unroll
				for(int c = 0; c < C; c++)
					if(col0 + c < ns) ck[(size_t)(col0 + c) * ns + s0 + k] = v[k][c];
		}
		const R *cft = a.coef + (size_t)tau * 6 * ns;
#pragma unroll
		for(int k = 0; k < M; k++)
#pragma unroll
			for(int d = 0; d < 6; d++) cf[k][d] = cft[d * ns + s0 + k];
		for(int p = 0; p < a.np; p++){
#pragma unroll
			for(int k = 0; k < M; k++)
#pragma unroll
				for(int c = 0; c < C; c++) V[(size_t)(s0 + k) * C + c] = v[k][c];
			__syncthreads();
			strip_gather<R, C, M>(V, sn, cf, a.mu, v, w);
			if(a.cplx[p]){
#pragma unroll
				for(int k = 0; k < M; k++)
#pragma unroll
					for(int c = 0; c < C; c++) W[(size_t)(s0 + k) * C + c] = w[k][c];
				__syncthreads();
				R z[M][C];
				strip_gather<R, C, M>(W, sn, cf, a.mu, w, z);
#pragma unroll
				for(int k = 0; k < M; k++)
#pragma unroll
					for(int c = 0; c < C; c++) v[k][c] = v[k][c] + fmac(a.a_quad[p], z[k][c], a.a_lin[p] * w[k][c]);
			}else{
				__syncthreads();
#pragma unroll
				for(int k = 0; k < M; k++)
#pragma unroll
					for(int c = 0; c < C; c++) v[k][c] = fmac(a.a_lin[p], w[k][c], v[k][c]);
			}
		}
	}
	if(a.dst){
#pragma unroll
		for(int k = 0; k < M; k++)
#pragma unroll
			for(int c = 0; c < C; c++)
				if(col0 + c < ns) a.dst[(size_t)(col0 + c) * ns + s0 + k] = v[k][c];
	}
}

// ---------------------------------------------------------------------------------------------
// Patch form of the same chain (patch.h): a thread owns PX x PY sites of C columns, a workgroup all
// patches of them.  Up to 64 patches are one wave, and its steps need no barrier.  The bonds of the
// next slice are loaded during the current one, except above 512 threads, where the registers for
// them would spill.
//
// What bounds it: LDS reads plus vector issue, which overlap little, as a barrier between any two
// stencils keeps the waves in step.  Against the site form a 2 x 2 patch reads 10 neighbours
// per 4 sites instead of 24, without the bank conflicts of the strip form's consecutive sites, and each
// bond once instead of twice.  us per chain (chain kernel and coefficients), before -> now:
// fp64 6x6 nt 32 38 -> 31, 16x16 nt 64 79 -> 67, 21x19 nt 95 165 -> 141, 27x31 nt 64 325 -> 224,
// 32x32 nt 128 545 -> 433, 64x32 nt 32 1041 -> 548; fp32 21x19 118 -> 111, 24x24 nt 64 178 -> 105,
// 32x32 301 -> 271, 36x36 nt 32 250 -> 156, 45x45 410 -> 354.
template <typename R>
struct PatchArgs {
	const R *coef;          // [nt][bonds][tp]
	const int *halo;        // [halo][tp]: LDS places of the halo sites
	R mu;
	unsigned ns, l1, l2, npx, np, tp;     // patches per row, patches, places per slot
	const R *src;
	R *dst, *ck;
	unsigned ck_every;
	int tau0, dir, ntau, npairs;
	R a_lin[MAX_PAIRS], a_quad[MAX_PAIRS];
};

template <typename R, int C, int PX, int PY, int LB>
__global__ __launch_bounds__(LB) void chain_patch_kernel(PatchArgs<R> a)
{
	extern __shared__ __align__(16) unsigned char smem_raw[];
	constexpr int S = PX * PY, NH = patch_halo(PX, PY), NK = patch_bonds(PX, PY);
	constexpr bool AHEAD = LB <= 512;
	struct alignas(C * sizeof(R) <= 16 ? C * sizeof(R) : 16) Vec { R v[C]; };
	const unsigned tp = a.tp, ns = a.ns, col0 = blockIdx.x * C;
	Vec *V = reinterpret_cast<Vec *>(smem_raw), *W = V + (size_t)S * tp;
	// a thread past the last patch works on it too (the same values, to the same LDS places) and
	// stores nothing
	const bool act = threadIdx.x < a.np;
	const unsigned p = act ? threadIdx.x : a.np - 1;
	const unsigned x0 = p % a.npx * PX, y0 = p / a.npx * PY;
	int halo[NH];
#pragma unroll
	for(int k = 0; k < NH; k++) halo[k] = a.halo[(size_t)k * tp + p];
	R v[S][C], cf[NK], cn[NK];
	// (x, y) of this patch: its column-major place, and whether this patch owns the site
	auto place = [&](int x, int y){ return (y0 + y) % a.l2 * a.l1 + (x0 + x) % a.l1; };
	auto owns = [&](int x, int y){ return act && x0 + x < a.l1 && y0 + y < a.l2; };
#pragma unroll
	for(int s = 0; s < S; s++){
		const unsigned site = place(s % PX, s / PX);
#pragma unroll
		for(int c = 0; c < C; c++){
			const unsigned col = col0 + c;
			v[s][c] = 0;
			if(col < ns) v[s][c] = a.src ? a.src[(size_t)col * ns + site] : (R)(site == col ? 1 : 0);
		}
	}
	auto store = [&](R *m){
#pragma unroll
		for(int c = 0; c < C; c++){
			if(col0 + c >= ns) break;
			R *q = m + (size_t)(col0 + c) * ns;
#pragma unroll
			for(int s = 0; s < S; s++)
				if(owns(s % PX, s / PX)) q[(y0 + s / PX) * a.l1 + x0 + s % PX] = v[s][c];
		}
	};
	auto load_bonds = [&](int i){
		const R *q = a.coef + (size_t)(a.tau0 + a.dir * i) * NK * tp + p;
#pragma unroll
		for(int k = 0; k < NK; k++) cn[k] = q[(size_t)k * tp];
	};
	auto apply = [&](Vec *buf, const R (&in)[S][C], R (&out)[S][C]){
#pragma unroll
		for(int s = 0; s < S; s++){
			Vec t;
#pragma unroll
			for(int c = 0; c < C; c++) t.v[c] = in[s][c];
			buf[s * tp + p] = t;
		}
		__syncthreads();
		R h[NH][C];
#pragma unroll
		for(int k = 0; k < NH; k++){
			const Vec t = buf[halo[k]];
#pragma unroll
			for(int c = 0; c < C; c++) h[k][c] = t.v[c];
		}
		patch_stencil<R, C, PX, PY>(in, h, cf, a.mu, out);
	};
	if(AHEAD && a.ntau > 0) load_bonds(0);
	for(int i = 0; i < a.ntau; i++){
		if(!AHEAD) load_bonds(i);
		if(a.ck && (i % a.ck_every) == 0) store(a.ck + (size_t)(i / a.ck_every) * ns * ns);
#pragma unroll
		for(int k = 0; k < NK; k++) cf[k] = cn[k];
		if(AHEAD && i + 1 < a.ntau) load_bonds(i + 1);
#pragma unroll 1
		for(int q = 0; q < a.npairs; q++){
			// V is free: its last readers passed the barrier of the pair's second stencil, and W's
			// passed the barrier of the next first one
			R w[S][C], z[S][C];
			apply(V, v, w);
			apply(W, w, z);
#pragma unroll
			for(int s = 0; s < S; s++)
#pragma unroll
				for(int c = 0; c < C; c++) v[s][c] = v[s][c] + fmac(a.a_quad[q], z[s][c], a.a_lin[q] * w[s][c]);
		}
	}
	if(a.dst) store(a.dst);
}

template <typename R>
static PatchArgs<R> patch_args(const ephmc_ctx *c, const PatchTab &t)
{
	PatchArgs<R> a{};
	a.coef = (const R *)t.coef;
	a.halo = t.halo;
	a.mu = (R)c->cfg.mu;
	a.ns = c->ns;
	a.l1 = c->l1;
	a.l2 = c->l2;
	a.npx = t.npx;
	a.np = t.np;
	a.tp = t.tp;
	a.npairs = c->poly.np;
	for(int p = 0; p < c->poly.np; p++){
		a.a_lin[p] = (R)c->poly.a_lin[p];
		a.a_quad[p] = (R)c->poly.a_quad[p];
	}
	return a;
}

template <typename R, int C, int PX, int PY>
static int launch_patch_lb(ephmc_ctx *c, const PatchArgs<R> &a)
{
	const size_t lds = 2 * (size_t)C * PX * PY * a.tp * sizeof(R);
	if(lds > 160 * 1024 || a.tp > 1024){ set_error("chain: %zu B of LDS, %u threads", lds, a.tp); return EPHMC_ERR_ARG; }
	const unsigned blocks = (a.ns + C - 1) / C;
#define EPHMC_PATCH_LAUNCH(LB)                                                                          \
	do {                                                                                                \
		(void)hipFuncSetAttribute((const void *)chain_patch_kernel<R, C, PX, PY, LB>,                    \
			hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                                       \
		chain_patch_kernel<R, C, PX, PY, LB><<<blocks, a.tp, lds, c->stream>>>(a);                       \
	} while(0)
	if(a.tp <= 64) EPHMC_PATCH_LAUNCH(64);
	else if(a.tp <= 256) EPHMC_PATCH_LAUNCH(256);
	else if(a.tp <= 512) EPHMC_PATCH_LAUNCH(512);
	else if(a.tp <= 640) EPHMC_PATCH_LAUNCH(640);
	else EPHMC_PATCH_LAUNCH(1024);
#undef EPHMC_PATCH_LAUNCH
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

template <typename R>
static int launch_patch(ephmc_ctx *c, const PatchTab &t, PatchArgs<R> a)
{
#define EPHMC_PATCH(CC, X, Y) if(t.cols == CC && t.px == X && t.py == Y) return launch_patch_lb<R, CC, X, Y>(c, a)
	EPHMC_PATCH(1, 1, 1);
	EPHMC_PATCH(2, 1, 1);
	EPHMC_PATCH(2, 2, 2);
#undef EPHMC_PATCH
	set_error("chain: no patch form for %u columns of %u x %u sites", t.cols, t.px, t.py);
	return EPHMC_ERR_ARG;
}

// Tables of the patch form for one arithmetic, where it is the faster form of the chain (measured
// shapes above): fp64 up to 512 sites one site per thread and one column per workgroup, above 640
// sites 2 x 2 sites and 2 columns (between, the strip form by 3 % where l1 is even); fp32 not up to
// 256 sites (16x16 nt 64: 62 against 55 us for the site form), one site and 2 columns up to 640, 2 x 2
// sites and 2 columns beyond.  Not 2 x 2 where the lattice is one site wide, as half of a patch would be ghosts
// (fp64 1x1024 nt 32 200 us against 120 for the site form, 1500x1 431 against 277 for strips; fp32 1x1024 108
// against 83), nor in fp64 over strips where a quarter would (400x3 273 against 236; 300x5, with a sixth, 292
// against 288; where l1 is odd, patches stay the faster: 3x400 276 against 293).
int patch_reserve(ephmc_ctx *c, int prec)
{
	PatchTab &t = c->patch[prec == EPHMC_FP64 ? 0 : 1];
	const unsigned ns = c->ns;
	if(prec != EPHMC_FP64 && ns <= 256) return EPHMC_OK;
	if(prec == EPHMC_FP64 && ns > 512 && ns <= 640 && c->l1 % 2 == 0) return EPHMC_OK;
	const unsigned X = ns <= 640 ? 1 : 2, Y = X;
	t.cols = prec == EPHMC_FP64 && ns <= 640 ? 1 : 2;
	t.px = X; t.py = Y;
	t.npx = (c->l1 + X - 1) / X;
	t.np = t.npx * ((c->l2 + Y - 1) / Y);
	const bool strips = prec == EPHMC_FP64 && c->l1 % 2 == 0;
	if(X == 2 && (c->l1 == 1 || c->l2 == 1 || (strips && 16 * t.np > 5 * ns))){ t = PatchTab{}; return EPHMC_OK; }
	t.tp = (t.np + 63) / 64 * 64;               // at most 704 (3 x 680 sites)
	t.nk = patch_bonds(X, Y);
	const unsigned nh = patch_halo(X, Y), tp = t.tp;
	std::vector<int> tab((size_t)(nh + t.nk) * tp, 0);
	int *halo = tab.data(), *bond = halo + (size_t)nh * tp;
	for(unsigned p = 0; p < tp; p++){
		const unsigned q = std::min(p, t.np - 1);
		const int x0 = (int)(q % t.npx * X), y0 = (int)(q / t.npx * Y), l1 = (int)c->l1, l2 = (int)c->l2;
		auto wrap = [](int v, int l){ return (v % l + l) % l; };
		auto place = [&](int x, int y){
			const unsigned xs = wrap(x0 + x, l1), ys = wrap(y0 + y, l2);
			return (int)((ys % Y * X + xs % X) * tp + ys / Y * t.npx + xs / X);
		};
		auto link = [&](int x, int y, int k){ return 3 * (wrap(y0 + y, l2) * l1 + wrap(x0 + x, l1)) + k; };
		unsigned h = 0, b = 0;
		auto put = [&](int x, int y){ halo[(size_t)h++ * tp + p] = place(x, y); };
		auto bnd = [&](int x, int y, int k){ bond[(size_t)b++ * tp + p] = link(x, y, k); };
		for(int x = 0; x <= (int)X; x++) put(x - 1, Y);
		for(int x = 0; x <= (int)X; x++) put(x, -1);
		for(int y = 0; y < (int)Y; y++) put(-1, y);
		for(int y = 0; y < (int)Y; y++) put(X, y);
		for(int y = 0; y < (int)Y; y++) for(int x = 0; x < (int)X; x++) for(int k = 0; k < 3; k++) bnd(x, y, k);
		for(int y = 0; y < (int)Y; y++) bnd(-1, y, 0);
		for(int x = 0; x < (int)X; x++) bnd(x, -1, 1);
		for(int x = 0; x < (int)X; x++) bnd(x + 1, -1, 2);
		for(int y = 0; y + 1 < (int)Y; y++) bnd(X, y, 2);
	}
	// one allocation: the coefficients, then both tables
	const size_t csz = (size_t)c->nt * t.nk * tp * (prec == EPHMC_FP64 ? 8 : 4), tsz = tab.size() * sizeof(int);
	if(hipMalloc(&t.coef, csz + tsz) != hipSuccess){
		(void)hipGetLastError();
		t = PatchTab{};
		set_error("patch tables (%zu bytes) could not be allocated", csz + tsz);
		return EPHMC_ERR_ALLOC;
	}
	t.halo = (int *)((char *)t.coef + csz);
	t.bond = t.halo + (size_t)nh * tp;
	EPHMC_HIP(hipMemcpy(t.halo, tab.data(), tsz, hipMemcpyHostToDevice));
	return EPHMC_OK;
}

// Whether the chain of this arithmetic runs in the patch form: not with a shape set by
// ephmc_autotune or by a tuning variable.
bool patch_on(const ephmc_ctx *c, int prec)
{
	const int slot = prec == EPHMC_FP64 ? 0 : 1;
	return c->patch[slot].cols && !c->chain_cols_set[slot] && c->chain_strip_set[slot] < 0 && !getenv("EPHMC_CHAIN_COLS")
		&& !getenv("EPHMC_CHAIN_STRIP") && !getenv("EPHMC_CHAIN_SITES");
}

void patch_release(ephmc_ctx *c)
{
	for(PatchTab &t : c->patch){
		if(t.coef) (void)hipFree(t.coef);
		t = PatchTab{};
	}
}

// Strip width for this lattice and arithmetic (0: site-per-thread form): the width chosen by
// ephmc_autotune, else EPHMC_CHAIN_STRIP=0/2/4, else 2 in fp64 and 0 in fp32.  The strip form
// cuts the LDS reads by a third (M = 2) at a larger register footprint; at 32x32 it is the
// faster fp64 chain (0.53 against 0.76 ms per 128 slices) and the slower fp32 one (0.31 against
// 0.28 ms).
unsigned strip_width(const ephmc_ctx *c, int prec)
{
	const int slot = prec == EPHMC_FP64 ? 0 : 1;
	unsigned m = prec == EPHMC_FP64 ? 2 : 0;
	if(c->chain_strip_set[slot] >= 0) m = (unsigned)c->chain_strip_set[slot];
	else if(const char *e = getenv("EPHMC_CHAIN_STRIP")) m = (unsigned)atoi(e);
	if(m != 2 && m != 4) return 0;
	if(c->l1 % m != 0) m = (m == 4 && c->l1 % 2 == 0) ? 2 : 0;
	if(m == 0 || c->ns / m > 1024) return 0;
	return m;
}

template <typename R, int C, int M>
static int launch_strip(ephmc_ctx *c, const ChainArgs<R> &a)
{
	const unsigned ns = a.ns;
	const size_t lds = 2 * (size_t)C * ns * sizeof(R);
	if(lds > 160 * 1024){ set_error("chain: %zu B of LDS exceeds 160 KiB", lds); return EPHMC_ERR_ARG; }
	const unsigned bt = ns / M, blocks = (ns + C - 1) / C;
#define EPHMC_STRIP_LAUNCH(LB)                                                                          \
	do {                                                                                                \
		(void)hipFuncSetAttribute((const void *)chain_strip_kernel<R, C, M, LB>,                        \
			hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                                       \
		chain_strip_kernel<R, C, M, LB><<<blocks, bt, lds, c->stream>>>(a);                              \
	} while(0)
	if(bt <= 256) EPHMC_STRIP_LAUNCH(256);
	else if(bt <= 512) EPHMC_STRIP_LAUNCH(512);
	else EPHMC_STRIP_LAUNCH(1024);
#undef EPHMC_STRIP_LAUNCH
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// Sites per thread requested by a tuning variable (1 when unset): 2 runs lattices of 513..1024
// sites on 512 threads.
unsigned sites_per_thread(const char *var)
{
	const char *e = getenv(var);
	return (e && atoi(e) == 2) ? 2u : 1u;
}

// Launch shape: threads per workgroup and sites per thread from the lattice size; columns
// per workgroup from the tuning table (ctx->cols) capped by LDS.
template <typename R, int C>
static int launch_chain_c(ephmc_ctx *c, const ChainArgs<R> &a)
{
	const unsigned ns = a.ns;
	const unsigned blocks = (ns + C - 1) / C;
#define EPHMC_CHAIN_LAUNCH(BT, S)                                                                  \
	do {                                                                                           \
		const size_t lds = chain_lds_bytes<R, C, BT, S>(ns);                                       \
		if(lds > 160 * 1024){ set_error("chain: %zu B of LDS exceeds 160 KiB", lds); return EPHMC_ERR_ARG; } \
		(void)hipFuncSetAttribute((const void *)chain_kernel<R, C, BT, S>,                               \
			hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                                 \
		chain_kernel<R, C, BT, S><<<blocks, BT, lds, c->stream>>>(a);                             \
	} while(0)
	if(ns <= 256) EPHMC_CHAIN_LAUNCH(256, 1);
	else if(ns <= 512) EPHMC_CHAIN_LAUNCH(512, 1);
	else if(ns <= 1024 && sites_per_thread("EPHMC_CHAIN_SITES") == 2) EPHMC_CHAIN_LAUNCH(512, 2);
	else if(ns <= 1024) EPHMC_CHAIN_LAUNCH(1024, 1);
	else if(ns <= 2048) EPHMC_CHAIN_LAUNCH(1024, 2);
	else if(ns <= 4096) EPHMC_CHAIN_LAUNCH(1024, 4);
	else { set_error("chain: lattice of %u sites exceeds 4096", ns); return EPHMC_ERR_UNSUPPORTED; }
#undef EPHMC_CHAIN_LAUNCH
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

template <typename R>
static int launch_chain(ephmc_ctx *c, const ChainArgs<R> &a, unsigned cols)
{
	// LDS budget: 2 * C * ns * sizeof(R) <= 160 KiB
	while(cols > 1 && 2 * (size_t)cols * a.ns * sizeof(R) > 160 * 1024) cols >>= 1;
	const unsigned m = strip_width(c, sizeof(R) == 8 ? EPHMC_FP64 : EPHMC_MIXED);
	if(m == 4){
		switch(cols){
			case 1: return launch_strip<R, 1, 4>(c, a);
			case 2: return launch_strip<R, 2, 4>(c, a);
			case 4: return launch_strip<R, 4, 4>(c, a);
			default: return launch_strip<R, 8, 4>(c, a);
		}
	}
	if(m == 2){
		switch(cols){
			case 1: return launch_strip<R, 1, 2>(c, a);
			case 2: return launch_strip<R, 2, 2>(c, a);
			case 4: return launch_strip<R, 4, 2>(c, a);
			default: return launch_strip<R, 8, 2>(c, a);
		}
	}
	switch(cols){
		case 1: return launch_chain_c<R, 1>(c, a);
		case 2: return launch_chain_c<R, 2>(c, a);
		case 4: return launch_chain_c<R, 4>(c, a);
		default: return launch_chain_c<R, 8>(c, a);
	}
}

template <typename R>
static ChainArgs<R> make_args(ephmc_ctx *c, const R *coef)
{
	ChainArgs<R> a{};
	a.coef = coef;
	a.nb = c->d_nb;
	a.mu = (R)c->cfg.mu;
	a.ns = c->ns;
	a.np = c->poly.np;
	for(int p = 0; p < c->poly.np; p++){
		a.a_lin[p] = (R)c->poly.a_lin[p];
		a.a_quad[p] = (R)c->poly.a_quad[p];
		a.cplx[p] = c->poly.cplx[p];
	}
	return a;
}

unsigned chain_cols(const ephmc_ctx *c, int prec)
{
	// columns per workgroup of the forward chain: the widest that gives at least 512 workgroups
	// (two per CU); EPHMC_CHAIN_COLS overrides it for tuning sweeps
	const unsigned ns = c->ns;
	const int slot = prec == EPHMC_FP64 ? 0 : 1;
	if(c->chain_cols_set[slot]) return c->chain_cols_set[slot];
	if(const char *e = getenv("EPHMC_CHAIN_COLS")){
		const unsigned v = (unsigned)atoi(e);
		if(v == 1 || v == 2 || v == 4 || v == 8) return v;
	}
	unsigned cols = 8;
	while(cols > 1 && (ns + cols - 1) / cols < 512) cols >>= 1;
	return cols;
}

// Chain of slices over all columns: dst = B_{tau_last} ... B_{tau_first} src, with the
// slices tau0, tau0+dir, ... (nt of them); src null = identity.  Stores the state before
// every ck_every-th slice into ck.  prec selects fp64 or fp32 storage and arithmetic.
template <typename R>
static ChainArgs<R> forward_args(ephmc_ctx *c, const R *coef, const void *src, void *dst, void *ck, unsigned ck_every,
		int descending, bool from_identity)
{
	ChainArgs<R> a = make_args<R>(c, coef);
	a.src = from_identity ? nullptr : (const R *)src;
	a.dst = (R *)dst;
	a.ck = (R *)ck;
	a.ck_every = ck_every ? ck_every : 1;
	a.tau0 = descending ? (int)c->nt - 1 : 0;
	a.dir = descending ? -1 : 1;
	a.ntau = (int)c->nt;
	return a;
}

// the patch form's coefficients are the current field's (coefficients() wrote them last) and in use
static bool patch_ready(const ephmc_ctx *c, int prec)
{
	return c->patch_slot == (prec == EPHMC_FP64 ? 0 : 1) && patch_on(c, prec);
}

template <typename R>
static int patch_chain(ephmc_ctx *c, const R *src, R *dst, R *ck, unsigned ck_every, int tau0, int dir, int ntau)
{
	const PatchTab &t = c->patch[sizeof(R) == 8 ? 0 : 1];
	PatchArgs<R> a = patch_args<R>(c, t);
	a.src = src;
	a.dst = dst;
	a.ck = ck;
	a.ck_every = ck_every ? ck_every : 1;
	a.tau0 = tau0;
	a.dir = dir;
	a.ntau = ntau;
	return launch_patch<R>(c, t, a);
}

int chain_forward(ephmc_ctx *c, int prec, const void *src, void *dst, void *ck, unsigned ck_every,
		int descending, bool from_identity)
{
	if(patch_ready(c, prec)){
		const int tau0 = descending ? (int)c->nt - 1 : 0, dir = descending ? -1 : 1;
		if(from_identity) src = nullptr;
		if(prec == EPHMC_FP64) return patch_chain<double>(c, (const double *)src, (double *)dst, (double *)ck, ck_every, tau0, dir, (int)c->nt);
		return patch_chain<float>(c, (const float *)src, (float *)dst, (float *)ck, ck_every, tau0, dir, (int)c->nt);
	}
	if(prec == EPHMC_FP64)
		return launch_chain<double>(c, forward_args<double>(c, c->d_coef64, src, dst, ck, ck_every, descending, from_identity),
			chain_cols(c, prec));
	return launch_chain<float>(c, forward_args<float>(c, c->d_coef32, src, dst, ck, ck_every, descending, from_identity),
		chain_cols(c, prec));
}

// dst = B_{tau_last} ... B_{tau0} src over the slices tau0, tau0+dir, ... (ntau of them) in the
// precision prec; src is fp64 (converted for fp32) or null for the identity.
int chain_range(ephmc_ctx *c, int prec, const double *src, void *dst, int tau0, int dir, int ntau)
{
	if(prec == EPHMC_FP64){
		if(patch_ready(c, prec)) return patch_chain<double>(c, src, (double *)dst, nullptr, 1, tau0, dir, ntau);
		ChainArgs<double> a = make_args<double>(c, c->d_coef64);
		a.src = src;
		a.dst = (double *)dst;
		a.ck = nullptr;
		a.ck_every = 1;
		a.tau0 = tau0; a.dir = dir; a.ntau = ntau;
		return launch_chain<double>(c, a, chain_cols(c, prec));
	}
	float *s32 = nullptr;
	if(src){
		s32 = (float *)c->d_seg;        // scratch: the segment buffer holds at least N^2 values
		EPHMC_TRY(convert_f64_to_f32(c, src, s32, c->mat));
	}
	if(patch_ready(c, prec)) return patch_chain<float>(c, s32, (float *)dst, nullptr, 1, tau0, dir, ntau);
	ChainArgs<float> a = make_args<float>(c, c->d_coef32);
	a.src = s32;
	a.dst = (float *)dst;
	a.ck = nullptr;
	a.ck_every = 1;
	a.tau0 = tau0; a.dir = dir; a.ntau = ntau;
	return launch_chain<float>(c, a, chain_cols(c, prec));
}

// fp64 coefficients of the single slice whose 3N couplings are x_tau, into d_coef64 slot 0
int slice_coefficients(ephmc_ctx *c, const double *x_tau)
{
	const unsigned ns = c->ns;
	coef_kernel<<<(6 * ns + 255) / 256, 256, 0, c->stream>>>(x_tau, c->d_link, c->cfg.t[0], c->cfg.t[1], c->cfg.t[2],
		c->cfg.kappa[0], c->cfg.kappa[1], c->cfg.kappa[2], ns, 1, c->d_coef64, nullptr);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// apply_exp_mu_K_to_M with partial pair products (revert/stop, organic_dense_matrix.c:186-194)
// for a single slice whose 3N couplings are x_tau.  Uses d_coef64 slot 0 as scratch.
int apply_exp_partial(ephmc_ctx *c, const double *x_tau, double *M, int revert, int stop)
{
	EPHMC_TRY(slice_coefficients(c, x_tau));
	ChainArgs<double> a = make_args<double>(c, c->d_coef64);
	a.np = 0;
	auto add = [&](int p){
		a.a_lin[a.np] = c->poly.a_lin[p];
		a.a_quad[a.np] = c->poly.a_quad[p];
		a.cplx[a.np] = c->poly.cplx[p];
		a.np++;
	};
	if(revert){ for(int p = c->poly.np - 1; p > stop; p--) add(p); }
	else{ for(int p = 0; p < stop; p++) add(p); }
	if(a.np == 0) return EPHMC_OK;
	a.src = M;
	a.dst = M;       // each workgroup reads its columns before writing them
	a.ck = nullptr;
	a.ck_every = 1;
	a.tau0 = 0; a.dir = 1; a.ntau = 1;
	return launch_chain<double>(c, a, chain_cols(c, EPHMC_FP64));
}

// ---------------------------------------------------------------------------------------------
// M = T^T (+ identity): 32x32 tiles through LDS; T in R, M in fp64.
template <typename R>
__device__ __forceinline__ void transpose_body(const R *__restrict__ T, double *__restrict__ M, unsigned n, int add_identity,
		unsigned bxi, unsigned byi)
{
	__shared__ double tile[32][33];
	const unsigned bx = bxi * 32, by = byi * 32;
	const unsigned tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
	for(unsigned r = ty; r < 32; r += 8){
		const unsigned col = by + r, row = bx + tx;          // T[col][row] (column col of T)
		if(col < n && row < n) tile[r][tx] = (double)T[(size_t)col * n + row];
	}
	__syncthreads();
	for(unsigned r = ty; r < 32; r += 8){
		const unsigned col = bx + r, row = by + tx;          // M column col = row col of T
		if(col < n && row < n) M[(size_t)col * n + row] = tile[tx][r] + ((add_identity && col == row) ? 1.0 : 0.0);
	}
}

template <typename R>
__global__ __launch_bounds__(256) void transpose_kernel(const R *__restrict__ T, double *__restrict__ M,
		unsigned n, int add_identity)
{
	transpose_body<R>(T, M, n, add_identity, blockIdx.x, blockIdx.y);
}

struct TransArgs {
	const void *T;
	double *M;
	unsigned n;
	int add_identity;
};

template <typename R>
__global__ __launch_bounds__(256) void transpose_multi_kernel(const TransArgs *__restrict__ tab)
{
	const TransArgs &a = tab[blockIdx.z];
	const unsigned g = (a.n + 31) / 32;
	if(blockIdx.x >= g || blockIdx.y >= g) return;
	transpose_body<R>((const R *)a.T, a.M, a.n, a.add_identity, blockIdx.x, blockIdx.y);
}

int transpose_plus_identity(ephmc_ctx *c, int prec, const void *T, double *M, int add_identity)
{
	const unsigned n = c->ns;
	dim3 grid((n + 31) / 32, (n + 31) / 32);
	if(prec == EPHMC_FP64) transpose_kernel<double><<<grid, 256, 0, c->stream>>>((const double *)T, M, n, add_identity);
	else transpose_kernel<float><<<grid, 256, 0, c->stream>>>((const float *)T, M, n, add_identity);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

__global__ void add_identity_kernel(double *__restrict__ M, unsigned n)
{
	for(unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) M[(size_t)i * (n + 1)] += 1.0;
}

struct AddIdArgs {
	double *M;
	unsigned n;
};

__global__ void add_identity_multi_kernel(const AddIdArgs *__restrict__ tab)
{
	const AddIdArgs &a = tab[blockIdx.z];
	for(unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += gridDim.x * blockDim.x) a.M[(size_t)i * (a.n + 1)] += 1.0;
}

int add_identity(ephmc_ctx *c, double *M)
{
	add_identity_kernel<<<(c->ns + 255) / 256, 256, 0, c->stream>>>(M, c->ns);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// SINGLE_PARTICLE log det = log tr(B_0 ... B_{nt-1}) (organic_dense_matrix.c:550-551); the force
// factor exp(-logdet) (organic_hmc.c:121) goes to fs_slot when >= 0.
template <typename R>
__global__ __launch_bounds__(256) void log_trace_kernel(const R *__restrict__ M, unsigned n, double *__restrict__ scal,
		int ld_slot, int fs_slot)
{
	__shared__ double red[256];
	double s = 0;
	for(unsigned i = threadIdx.x; i < n; i += 256) s += (double)M[(size_t)i * (n + 1)];
	red[threadIdx.x] = s;
	__syncthreads();
	for(int off = 128; off > 0; off >>= 1){
		if((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
		__syncthreads();
	}
	if(threadIdx.x == 0){
		const double ld = log(red[0]);
		scal[ld_slot] = ld;
		if(fs_slot >= 0) scal[fs_slot] = exp(-ld);
	}
}

int log_trace(ephmc_ctx *c, int prec, const void *M, int ld_slot, int fs_slot)
{
	if(prec == EPHMC_FP64) log_trace_kernel<double><<<1, 256, 0, c->stream>>>((const double *)M, c->ns, c->d_scal, ld_slot, fs_slot);
	else log_trace_kernel<float><<<1, 256, 0, c->stream>>>((const float *)M, c->ns, c->d_scal, ld_slot, fs_slot);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

template <typename R>
__global__ void set_identity_kernel(R *__restrict__ M, unsigned n)
{
	const size_t nn = (size_t)n * n;
	for(size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < nn; e += (size_t)gridDim.x * blockDim.x)
		M[e] = (e % (n + 1) == 0) ? (R)1 : (R)0;
}

int set_identity(ephmc_ctx *c, int prec, void *M)
{
	if(prec == EPHMC_FP64) set_identity_kernel<double><<<1024, 256, 0, c->stream>>>((double *)M, c->ns);
	else set_identity_kernel<float><<<1024, 256, 0, c->stream>>>((float *)M, c->ns);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

__global__ void set_scalar_kernel(double *scal, int slot, double v){ scal[slot] = v; }

int set_scalar(ephmc_ctx *c, int slot, double v)
{
	set_scalar_kernel<<<1, 1, 0, c->stream>>>(c->d_scal, slot, v);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

__global__ void f64_to_f32_kernel(const double *__restrict__ a, float *__restrict__ b, size_t n)
{
	for(size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
		b[e] = (float)a[e];
}

int convert_f64_to_f32(ephmc_ctx *c, const double *a, float *b, size_t n)
{
	const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
	f64_to_f32_kernel<<<blocks, 256, 0, c->stream>>>(a, b, n);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// ---- many chains in one launch (batch.hip).  The chain runs in the site form with 2 columns per
// workgroup on `block` threads (ns <= block <= threads, the LDS layout's workgroup size); every
// column is computed with the arithmetic of every other form and width, so a chain gives the same
// bits in a batch as alone.
int batch_coef(BatchOp &op, ephmc_ctx *c, const double *x, bool want32)
{
	CoefArgs a{};
	a.x = x;
	a.link = c->d_link;
	for(int k = 0; k < 3; k++){ a.t[k] = c->cfg.t[k]; a.k[k] = c->cfg.kappa[k]; }
	a.ns = c->ns;
	a.nt = c->nt;
	const size_t n = (size_t)c->nt * 6 * c->ns;
	a.gx = (unsigned)std::min<size_t>((n + 255) / 256, 4096);     // the grid of coefficients()
	a.c64 = c->d_coef64;
	a.c32 = want32 ? c->d_coef32 : nullptr;
	return op.add((const void *)coef_multi_kernel, 256, 0, a.gx, 1, a);
}

template <typename R, int BT, int C>
static int batch_chain_c(BatchOp &op, unsigned block, const ChainArgs<R> &a)
{
	const size_t lds = chain_lds_bytes<R, C, BT, 1>(a.ns);
	if(lds > 160 * 1024){ set_error("batch chain: %zu B of LDS exceeds 160 KiB", lds); return EPHMC_ERR_ARG; }
	const void *fn = (const void *)chain_multi_kernel<R, C, BT, 1>;
	(void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)std::max(lds, op.lds));
	return op.add(fn, block, lds, (a.ns + C - 1) / C, 1, a);
}

// columns per workgroup: 2, or EPHMC_BATCH_CHAIN_COLS = 1 / 4 for tuning sweeps (any width gives the
// same bits)
template <typename R, int BT>
static int batch_chain_t(BatchOp &op, unsigned block, const ChainArgs<R> &a)
{
	const char *e = getenv("EPHMC_BATCH_CHAIN_COLS");
	const int cols = e ? atoi(e) : 2;
	if(cols == 1) return batch_chain_c<R, BT, 1>(op, block, a);
	if(cols == 4) return batch_chain_c<R, BT, 4>(op, block, a);
	return batch_chain_c<R, BT, 2>(op, block, a);
}

template <typename R>
static int batch_chain_r(BatchOp &op, unsigned threads, unsigned block, const ChainArgs<R> &a)
{
	if(a.ns > block || block > threads || block % 64){
		set_error("batch chain: %u sites on %u of %u threads", a.ns, block, threads);
		return EPHMC_ERR_ARG;
	}
	switch(threads){
		case 256: return batch_chain_t<R, 256>(op, block, a);
		case 512: return batch_chain_t<R, 512>(op, block, a);
		case 1024: return batch_chain_t<R, 1024>(op, block, a);
		default: set_error("batch chain: %u threads per workgroup", threads); return EPHMC_ERR_ARG;
	}
}

int batch_chain(BatchOp &op, ephmc_ctx *c, int prec, unsigned threads, unsigned block, void *dst, void *ck,
		unsigned ck_every, int descending)
{
	if(prec == EPHMC_FP64)
		return batch_chain_r<double>(op, threads, block,
			forward_args<double>(c, c->d_coef64, nullptr, dst, ck, ck_every, descending, true));
	return batch_chain_r<float>(op, threads, block, forward_args<float>(c, c->d_coef32, nullptr, dst, ck, ck_every, descending, true));
}

int batch_transpose(BatchOp &op, ephmc_ctx *c, int prec, const void *T, double *M)
{
	const TransArgs a{T, M, c->ns, 1};
	const unsigned g = (c->ns + 31) / 32;
	const void *fn = prec == EPHMC_FP64 ? (const void *)transpose_multi_kernel<double> : (const void *)transpose_multi_kernel<float>;
	return op.add(fn, 256, 0, g, g, a);
}

int batch_add_identity(BatchOp &op, ephmc_ctx *c, double *M)
{
	const AddIdArgs a{M, c->ns};
	return op.add((const void *)add_identity_multi_kernel, 256, 0, (c->ns + 255) / 256, 1, a);
}

struct CopyArgs {
	const double *src;
	double *dst;
	size_t n;
	const double *gate;
};

// elementwise, so any grid gives the same result
__global__ __launch_bounds__(256) void copy_multi_kernel(const CopyArgs *__restrict__ tab)
{
	const CopyArgs &a = tab[blockIdx.z];
	if(a.gate && a.gate[SCAL_ACC] == 0) return;
	for(size_t e = blockIdx.x * (size_t)256 + threadIdx.x; e < a.n; e += (size_t)gridDim.x * 256) a.dst[e] = a.src[e];
}

int batch_copy(BatchOp &op, const double *src, double *dst, size_t n, const double *gate)
{
	const CopyArgs a{src, dst, n, gate};
	return op.add((const void *)copy_multi_kernel, 256, 0, (unsigned)std::min<size_t>((n + 255) / 256, 1024), 1, a);
}

} // namespace ephmc
