// gj.hip -- log|det| and inverse of M_hat (FP64), replacing LAPACK dgetrf + dgetri in
// logDetM_and_inv_M_hat (organic_dense_matrix.c:547-607).
//
// LAPACK's partial pivoting picks, at elimination step g, the row with the largest |a_rg|
// among rows r >= g (first index on ties).  Elimination without row exchanges makes the same
// choices exactly when every multiplier |l_rg| = |a_rg| / |a_gg| is <= 1; the pivots are then
// the same U_ii, so log|det| = sum log|U_ii| and the sign (organic_dense_matrix.c:582-588)
// agree with LAPACK, and the inverse is the same matrix up to rounding.  For M_hat = 1 + B..B at
// the lattice parameters of the reference (mu at the band bottom) the multipliers are of order
// 1e-2, so:
//
//   fast path: blocked Gauss-Jordan without row exchanges, 32 or 64 columns per block K = [k0, k0+nb),
//     one launch per block over 64 x 64 output tiles.  Every workgroup reads D^{-1} of the diagonal
//     block D = A[K,K], forms the transform rows
//     E[i,:] = -A[i,K] D^{-1} (i not in K) or D^{-1} rows (i in K) of its rows, and writes its
//     tile of A' = [i not in K] A + E A[K,:] (columns inside K: E itself), while one more workgroup
//     forms and inverts the next diagonal block.  The LU multipliers of D and of the rows below K
//     are checked |l| <= 1.  N <= 64 is one block, inverted by one workgroup in one launch
//   check:   any multiplier > 1 sets a device flag; the single-workgroup fallback kernel, always
//            launched, then inverts the untouched input with partial pivoting (in-place
//            Gauss-Jordan with row exchanges and the columns un-permuted at the end); without
//            the flag it returns at once.  No host round trip either way.
#include "internal.h"
#include <cstdlib>

namespace ephmc {

// Columns per block (one launch).  A step costs the longer of its lookahead, a chain that grows with the
// block, and of its tiles, whose traffic (the matrix read and written) does not: 32 columns where the
// lookahead is the longer, 64 where the tiles are: log det and inverse at N = 1024 304 us with 32, 338 with 64,
// 1296 436 and 506, 1440 572 and 558, 1600 666 and 620, 2025 1180 and 1080 (from N = 1409 on the 64 x 64 tiles
// outnumber the 512 places that the wide form has on the chip anyway)
constexpr unsigned GJ_WIDE_ABOVE = 1400;
constexpr int GJ_T = 64, GJ_LE = 72;      // edge of a tile; its row stride in Et and Di

typedef double gj_v4d __attribute__((ext_vector_type(4)));

// LDS: the transform rows and A[K, column block] of a tile; an inversion keeps its pivot columns in the place
// of the one.  The matrix cores take the block's columns k in the order 8 kb + 2 (l / 16),
// 8 kb + 2 (l / 16) + 1 (lane l; any order does, the same in both operands): a lane reads two consecutive
// values of A[K, column], which lies as it does in memory, and rows 72 values apart put the lanes of two
// rows on different banks.  78 KB with 64 columns: two workgroups per CU
template <int NB>
struct GjLds {
	__align__(16) double prow[4][4][16];            // pivot rows of an inversion step, by tile (NB = 32: by step parity and tile)
	union {
		__align__(16) double Et[NB][GJ_LE];         // transform rows, transposed
		__align__(16) double pcs[NB / 4][4 * NB + 2];   // pivot columns of every inversion step, 4 per row (padded:
		                                            // the multiplier pass reads all steps at once)
	};
	union {
		__align__(16) double Yt[GJ_T][NB + 2];      // A[K, column block], by column; with 64 columns the next D, by row
		__align__(16) double Di[NB][GJ_LE];         // D^{-1}, by row
	};
};

// 1/x: hardware reciprocal r (2^-24 or better) refined by one step of third order, r + r (t + t^2), t = 1 - x r
__device__ inline double rcp_nr(double x)
{
	const double r = __builtin_amdgcn_rcp(x), t = fma(-x, r, 1.0);
	return fma(r, fma(t, t, t), r);
}

// lane I of each row of 16 lanes, in all of its lanes
template <int I>
__device__ __forceinline__ double row_lane(double v)
{
	const long long b = __double_as_longlong(v);
	const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b & 0xffffffffLL), 0x150 + I, 0xf, 0xf, true);
	const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + I, 0xf, 0xf, true);
	return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// inverse of the 2 x 2 matrix m by elimination without exchanges
__device__ __forceinline__ void gj_inv2(const double (&m)[2][2], double (&v)[2][2])
{
	const double r0 = rcp_nr(m[0][0]), l = m[1][0] * r0, t = m[0][1] * r0;
	const double r1 = rcp_nr(fmac(-l, m[0][1], m[1][1]));
	v[1][1] = r1;
	v[0][1] = -t * r1;
	v[1][0] = -l * r1;
	v[0][0] = fmac(-t, v[1][0], r0);
}

// y = x P^{-1} for a row x, P = [A B; C D] in 2 x 2 blocks: G = A^{-1} B, S = D - C G,
// y2 = (x2 - x1 G) S^{-1}, y1 = (x1 - y2 C) A^{-1}.  Element i of P by rows is pl of lane i of each row of 16
// lanes; returns -y[k]
__device__ __forceinline__ double gj_solve4(double pl, const double (&x)[4], int k)
{
	const double A[2][2] = {{row_lane<0>(pl), row_lane<1>(pl)}, {row_lane<4>(pl), row_lane<5>(pl)}};
	const double B[2][2] = {{row_lane<2>(pl), row_lane<3>(pl)}, {row_lane<6>(pl), row_lane<7>(pl)}};
	const double C[2][2] = {{row_lane<8>(pl), row_lane<9>(pl)}, {row_lane<12>(pl), row_lane<13>(pl)}};
	const double D[2][2] = {{row_lane<10>(pl), row_lane<11>(pl)}, {row_lane<14>(pl), row_lane<15>(pl)}};
	double Ai[2][2], G[2][2], S[2][2], Si[2][2];
	gj_inv2(A, Ai);
#pragma unroll
	for(int i = 0; i < 2; i++)
#pragma unroll
		for(int j = 0; j < 2; j++) G[i][j] = fmac(Ai[i][1], B[1][j], Ai[i][0] * B[0][j]);
#pragma unroll
	for(int i = 0; i < 2; i++)
#pragma unroll
		for(int j = 0; j < 2; j++) S[i][j] = fmac(-C[i][1], G[1][j], fmac(-C[i][0], G[0][j], D[i][j]));
	gj_inv2(S, Si);
	double z[2], y[4];
#pragma unroll
	for(int j = 0; j < 2; j++) z[j] = fmac(-x[1], G[1][j], fmac(-x[0], G[0][j], x[2 + j]));
#pragma unroll
	for(int j = 0; j < 2; j++) y[2 + j] = fmac(z[1], Si[1][j], z[0] * Si[0][j]);
#pragma unroll
	for(int j = 0; j < 2; j++) z[j] = fmac(-y[3], C[1][j], fmac(-y[2], C[0][j], x[j]));
#pragma unroll
	for(int j = 0; j < 2; j++) y[j] = fmac(z[1], Ai[1][j], z[0] * Ai[0][j]);
	const double lo = (k & 1) ? y[1] : y[0], hi = (k & 1) ? y[3] : y[2];
	return -(k < 2 ? lo : hi);
}

// Inversion of the diagonal block D of nbe <= NB columns (identity past nbe) by in-place Gauss-Jordan
// without exchanges, four pivots g .. g + 3 per step through their 4 x 4 block P, on the FP64 matrix cores:
// with C the pivot columns, R the pivot rows where the pivot columns hold the identity, every element
// becomes
//     [not in a pivot row or column] D - (C P^{-1}) R       with C = -1 in the pivot rows,
// a product of depth four, one instruction per 16 x 16 tile.  Lane l holds a tile's rows 4 e + l / 16 in
// element e and its column l % 16, so that the pivot rows of a step are one element of a tile and the pivot
// columns four lanes each: both pass through LDS, behind one barrier, into the operands' layout, and the
// pivot columns stay there for the multipliers.  A lane solves C P^{-1} for its row; of the step's chain
// (LDS, P, C P^{-1}, the product) the reciprocals in P's elimination are the longest part.  Only four steps
// are unrolled (straight-line code waits for its instructions).
//   NB = 32: wave w holds the tile of rows 16 (w / 2) .. and columns 16 (w % 2) ..
//   NB = 64: wave w holds the rows 16 w .. in four tiles.  The 16 columns at whose pivots the steps are stay
//            in tile 0: the tiles rotate once per four steps.
//
// At the end acc[(cb - rot) & 3] is tile cb of D^{-1}, rot the return value (0 with NB = 32).  The LU
// multipliers L (unit lower triangular) go to lm_out (NB x NB by rows) with LM: row r's of step s are
// C[r] U_P^{-1}, P = L_P U_P; bad is set in the threads that see one above 1.  The pivots go to diag, their
// rows kb.. to piv.  Called by all 256 threads of a workgroup.
template <int NB, bool LM>
__device__ __forceinline__ int gj_invert(GjLds<NB> &sh, unsigned nbe, gj_v4d (&acc)[NB == 64 ? 4 : 1], bool &bad,
		double *__restrict__ lm_out, double *__restrict__ diag, int *__restrict__ piv, unsigned kb)
{
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int m16 = lane & 15, k4 = lane >> 4;
	int rot = 0;
	if constexpr(NB == 32){
		const int wr = wave >> 1, wc = wave & 1, row = 16 * wr + m16;
#pragma clang loop unroll(disable)
		for(int t = 0; t < 2; t++){
#pragma unroll
			for(int e4 = 0; e4 < 4; e4++){
				const int s = 4 * t + e4, b = e4 & 1;
				if(4 * s >= (int)nbe) break;
				const bool pv = (m16 >> 2) == e4, prows = wr == t, pcols = wc == t;
				double *pc = sh.pcs[s];
				if(prows) sh.prow[2 * b + wc][k4][m16] = acc[0][e4];
				if(pcols && pv)
#pragma unroll
					for(int e = 0; e < 4; e++) pc[4 * (16 * wr + 4 * e + k4) + (m16 & 3)] = acc[0][e];
				__syncthreads();
				const double pl = sh.prow[2 * b + t][m16 >> 2][4 * e4 + (m16 & 3)];
				const double2 x01 = *(const double2 *)&pc[4 * row], x23 = *(const double2 *)&pc[4 * row + 2];
				double r = sh.prow[2 * b + wc][k4][m16];
				// the pivot rows: -1 for C, their elements cleared; the pivot columns: R = 1, cleared
				double x[4] = {x01.x, x01.y, x23.x, x23.y};
				if(prows){
#pragma unroll
					for(int j = 0; j < 4; j++) x[j] = pv ? (j == (m16 & 3) ? -1.0 : 0.0) : x[j];
					acc[0][e4] = 0.0;
				}
				if(pcols && pv){
					r = k4 == (m16 & 3) ? 1.0 : 0.0;
					acc[0] = gj_v4d{0.0, 0.0, 0.0, 0.0};
				}
				const double yk = gj_solve4(pl, x, k4);
				acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(yk, r, acc[0], 0, 0, 0);
			}
		}
	} else {
		rot = (int)(nbe + 15) / 16;
		const int row = 16 * wave + m16;
		// the product of a step is done at once for the tile of the next pivots; the other three
		// follow under the next step's chain
		double yk = 0.0, r[4] = {0.0, 0.0, 0.0, 0.0};
		auto product = [&](int c){ acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(yk, r[c], acc[c], 0, 0, 0); };
#pragma clang loop unroll(disable)
		for(int t = 0; t < rot; t++){
			const bool owner = wave == t;
#pragma unroll
			for(int e4 = 0; e4 < 4; e4++){
				const int s = 4 * t + e4;
				if(4 * s >= (int)nbe) break;
				const bool pcol = (m16 >> 2) == e4;             // this lane's column of tile 0 is a pivot column
				double *pc = sh.pcs[s];
				if(owner) sh.prow[0][k4][m16] = acc[0][e4];
				if(pcol)
#pragma unroll
					for(int e = 0; e < 4; e++) pc[4 * (16 * wave + 4 * e + k4) + (m16 & 3)] = acc[0][e];
				__syncthreads();
				const double pl = sh.prow[0][m16 >> 2][4 * e4 + (m16 & 3)];
				const double2 x01 = *(const double2 *)&pc[4 * row], x23 = *(const double2 *)&pc[4 * row + 2];
				const double r0 = sh.prow[0][k4][m16];
#pragma unroll
				for(int c = 1; c < 4; c++) product(c);
				// the pivot rows: -1 for C, their elements cleared once published; the pivot columns: R = 1, cleared
				double x[4] = {x01.x, x01.y, x23.x, x23.y};
				if(owner && pcol){
#pragma unroll
					for(int j = 0; j < 4; j++) x[j] = j == (m16 & 3) ? -1.0 : 0.0;
				}
				yk = gj_solve4(pl, x, k4);
				// three products spread over the chain, which is not to sink below the branch
				asm volatile("" : "+v"(yk));
#pragma unroll
				for(int i = 0; i < 3; i++){
					__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
					__builtin_amdgcn_sched_group_barrier(0x002, 18, 0);
				}
				if(owner){
#pragma unroll
					for(int c = 1; c < 4; c++) sh.prow[c][k4][m16] = acc[c][e4];
#pragma unroll
					for(int c = 0; c < 4; c++) acc[c][e4] = 0.0;
				}
				r[0] = r0;
				if(pcol){
					r[0] = k4 == (m16 & 3) ? 1.0 : 0.0;
					acc[0] = gj_v4d{0.0, 0.0, 0.0, 0.0};
				}
				__syncthreads();
#pragma unroll
				for(int c = 1; c < 4; c++) r[c] = sh.prow[c][k4][m16];
				product(e4 == 3 ? 1 : 0);
			}
			// tile 1 to the front; after a full round it is the one that is done already
			const gj_v4d a0 = acc[0];
			const double q0 = r[0];
#pragma unroll
			for(int c = 0; c < 3; c++){
				acc[c] = acc[c + 1];
				r[c] = r[c + 1];
			}
			acc[3] = a0;
			r[3] = q0;
		}
		// what is left of the last step: all tiles but the one it did at once, which is now 0, or 3 if the last round
		// was not full
		const bool full = 16 * rot - (int)nbe < 4;
		if(full) product(3);
		else product(0);
		product(1);
		product(2);
	}
	// the pivots and the multipliers: thread column j factors the pivot block of its step without exchanges
	// and forms column j & 3 of U_P^{-1}
	const int j = tid % NB, r0 = tid / NB, ii = j & 3;
	const double *pc = sh.pcs[j >> 2];
	double u[4][4], lo[4], rp[4];
	if(j < (int)nbe){
#pragma unroll
		for(int i = 0; i < 4; i++)
#pragma unroll
			for(int q = 0; q < 4; q++) u[i][q] = pc[4 * ((j & ~3) + i) + q];
	} else {
#pragma unroll
		for(int i = 0; i < 4; i++)
#pragma unroll
			for(int q = 0; q < 4; q++) u[i][q] = i == q ? 1.0 : 0.0;
	}
#pragma unroll
	for(int k = 0; k < 4; k++){
		rp[k] = rcp_nr(u[k][k]);
#pragma unroll
		for(int m = k + 1; m < 4; m++){
			const double l = u[m][k] * rp[k];
#pragma unroll
			for(int i = k + 1; i < 4; i++) u[m][i] = fmac(-l, u[k][i], u[m][i]);
		}
	}
	// U lo = unit vector ii
#pragma unroll
	for(int k = 3; k >= 0; k--){
		double x = k == ii ? 1.0 : 0.0;
#pragma unroll
		for(int i = k + 1; i < 4; i++) x = i <= ii ? fmac(-u[k][i], lo[i], x) : x;
		lo[k] = k <= ii ? x * rp[k] : 0.0;
	}
	if(tid < (int)nbe){
		diag[kb + tid] = ii == 0 ? u[0][0] : (ii == 1 ? u[1][1] : (ii == 2 ? u[2][2] : u[3][3]));
		piv[kb + tid] = (int)(kb + tid);
	}
	double l[NB * NB / 256];
#pragma unroll
	for(int q = 0; q < NB * NB / 256; q++){
		const double2 c0 = *(const double2 *)&pc[4 * (256 / NB * q + r0)], c1 = *(const double2 *)&pc[4 * (256 / NB * q + r0) + 2];
		l[q] = fmac(c1.y, lo[3], fmac(c1.x, lo[2], fmac(c0.y, lo[1], c0.x * lo[0])));
	}
#pragma unroll
	for(int q = 0; q < NB * NB / 256; q++){
		const int r = 256 / NB * q + r0;
		asm("" : "+v"(l[q]));                           // (no branch around the reads)
		const bool below = (r > j) & (r < (int)nbe);    // (nbe > r > j: a column that was pivoted on)
		bad |= below & !(fabs(l[q]) <= 1.0);
		if(LM) lm_out[r * NB + j] = below ? l[q] : (r == j ? 1.0 : 0.0);
	}
	return rot;
}

// row and column of element e of tile c of the inversion's layout
template <int NB>
__device__ __forceinline__ unsigned gj_row(int e){ return 16 * (threadIdx.x >> (NB == 64 ? 6 : 7)) + 4 * e + ((threadIdx.x & 63) >> 4); }
template <int NB>
__device__ __forceinline__ unsigned gj_col(int c){ return 16 * (NB == 64 ? c : (threadIdx.x >> 6) & 1) + (threadIdx.x & 15); }

template <int NB>
__device__ __forceinline__ void gj_store(const gj_v4d (&acc)[NB == 64 ? 4 : 1], int rot, double *__restrict__ out)
{
#pragma unroll
	for(int c = 0; c < (NB == 64 ? 4 : 1); c++)
#pragma unroll
		for(int e = 0; e < 4; e++) out[gj_row<NB>(e) * NB + gj_col<NB>((c + rot) & 3)] = acc[c][e];
}

// A[k:k+nbe, k:k+nbe] in the inversion's layout, the identity past nbe
template <int NB>
__device__ __forceinline__ void gj_load(gj_v4d (&acc)[NB == 64 ? 4 : 1], const double *__restrict__ A, unsigned n, unsigned nbe)
{
#pragma unroll
	for(int c = 0; c < (NB == 64 ? 4 : 1); c++)
#pragma unroll
		for(int e = 0; e < 4; e++) acc[c][e] = A[min(gj_col<NB>(c), nbe - 1) * n + min(gj_row<NB>(e), nbe - 1)];
#pragma unroll
	for(int c = 0; c < (NB == 64 ? 4 : 1); c++)
#pragma unroll
		for(int e = 0; e < 4; e++)
			if(gj_row<NB>(e) >= nbe || gj_col<NB>(c) >= nbe) acc[c][e] = gj_row<NB>(e) == gj_col<NB>(c) ? 1.0 : 0.0;
}

__device__ __forceinline__ void gj_clear_flags(double *__restrict__ scal)
{
	if(threadIdx.x == 0){
		scal[SCAL_GJ_FLAG] = 0;     // no multiplier above 1 seen yet
		scal[SCAL_SINGULAR] = 0;
		scal[SCAL_SCHUR_FAIL] = 0;
	}
}

// Inversion of the first diagonal block (one workgroup), N > 64.
template <int NB>
__device__ __forceinline__ void gj_first_body(GjLds<NB> &sh, const double *__restrict__ A, unsigned n,
		double *__restrict__ dinv_out, double *__restrict__ lm_out, double *__restrict__ diag, int *__restrict__ piv,
		double *__restrict__ scal)
{
	gj_v4d acc[NB == 64 ? 4 : 1];
	bool bad = false;
	gj_clear_flags(scal);
	gj_load<NB>(acc, A, n, NB);
	const int rot = gj_invert<NB, true>(sh, NB, acc, bad, lm_out, diag, piv, 0);
	gj_store<NB>(acc, rot, dinv_out);
	const bool any = __syncthreads_or(bad);
	if(any && threadIdx.x == 0) scal[SCAL_GJ_FLAG] = 1;
}

template <int NB>
__global__ __launch_bounds__(256, 2) void gj_first_kernel(const double *__restrict__ A, unsigned n,
		double *__restrict__ dinv_out, double *__restrict__ lm_out, double *__restrict__ diag, int *__restrict__ piv,
		double *__restrict__ scal)
{
	__shared__ GjLds<NB> sh;
	gj_first_body<NB>(sh, A, n, dinv_out, lm_out, diag, piv, scal);
}

// Block step for K = [k0, k0+nbe), grid (row tiles + 1, column tiles) of 64 x 64 tiles, with
// D^{-1} and L of D = A[K,K] read from dinv_cur / lm_cur.
//
// Tile workgroups form the transform rows E[i,:] = -A[i,K] D^{-1} (rows inside K: the rows of D^{-1}) of
// their rows on the FP64 matrix cores (v_mfma_f64_16x16x4) into a transposed LDS panel Et[m][row], and
// update A'[rows, cols] = [rows not in K] A + E A[K, cols] (columns inside K: E itself).  K is a row or two
// of 32 in one row of tiles, so each wave's 16 rows and 32 columns are inside or outside K.  The LU
// multipliers of the rows below K, l = -E L (|l| <= 1), are checked 16 columns of L at a time: tile y takes
// the columns 16 y .., 16 (y + ncb) .. of the block.
//
// Lookahead workgroup (blockIdx = (row tiles, 0)): forms the next diagonal block D' = A'[K', K'],
// K' = [k0+nbe, ...), inverts it and writes D'^{-1}, L' and its pivots for the next step, so that no step
// waits for an inversion of its own.  With 64 columns it runs the tile that D' is.  With 32 it forms
// D' alone, which may differ from the tile that holds it in the last bits: the inversion uses D', the next
// step's panels the tile's values.
//
// A step of 32 columns at N <= 576 takes 8 us, of which 6.6 are the lookahead's: 1 us loads, 1.4 the two products,
// 3.7 the inversion's eight steps (its four-pivot steps on the vector unit, with the pivot columns by
// readlane, took 5.7 and the multipliers 1.4 more, and a step 9.2 to 11.4), 0.5 the multipliers.  At N = 2025 a
// step of 64 takes 34 us for 66 MB of the matrix: 1.9 TB/s, half of what a copy reaches.  Log det and
// inverse before and after: N = 256 84 -> 70 us, 399 124 -> 102, 1024 360 -> 304, 2025 1584 -> 1080
template <int NB>
__device__ __forceinline__ void gj_step_body(GjLds<NB> &sh, const double *__restrict__ A, double *__restrict__ An,
		unsigned n, unsigned k0, unsigned nbe, const double *__restrict__ dinv_cur, const double *__restrict__ lm_cur,
		double *__restrict__ dinv_next, double *__restrict__ lm_next, double *__restrict__ diag, int *__restrict__ piv,
		double *__restrict__ scal, double *__restrict__ out_final, unsigned bx, unsigned by, unsigned ncb)
{
	constexpr int MD = NB * NB / 256, ML = NB * GJ_T / 256, NQ = NB / 4;
	const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
	const int m16 = lane & 15, k4 = lane >> 4;
	const unsigned nrb = (n + GJ_T - 1) / GJ_T, last = (n - 1) * n;
	const unsigned k1 = k0 + nbe;
	const bool look = bx == nrb;
	if(look){
		if(by != 0) return;
		if(k1 >= n){
			// last step: no next block; this workgroup sums log|det| and its sign from the pivots (the
			// flag is final: the last block's multipliers were checked when it was inverted)
			if(scal[SCAL_GJ_FLAG] == 0){
				double *part = &sh.Et[0][0];
				int *negs = reinterpret_cast<int *>(&sh.Yt[0][0]);
				double sl = 0;
				int neg = 0;
				for(unsigned i = tid; i < n; i += 256){
					const double d = diag[i];
					sl += log(fabs(d));
					neg += d < 0;
				}
				part[tid] = sl;
				negs[tid] = neg;
				__syncthreads();
				for(int off = 128; off > 0; off >>= 1){
					if(tid < off){ part[tid] += part[tid + off]; negs[tid] += negs[tid + off]; }
					__syncthreads();
				}
				if(tid == 0){
					scal[SCAL_LOGDET] = part[0];
					scal[SCAL_SIGN] = (negs[0] & 1) ? -1.0 : 1.0;
				}
			}
			return;
		}
	}
	const unsigned nb1 = min((unsigned)NB, n - k1);     // (the lookahead's)
	gj_v4d d[NB == 64 ? 4 : 1];
	if(NB == 32 && look){
		// D' = A[K',K'] + E[K',:] A[K,K'], E[K',:] = -A[K',K] D^{-1}: both products with the rows 16 (w / 2) ..
		// and the columns 16 (w % 2) .. in wave w, E through LDS.  (Every block before the last is full.)
		const int wr = wave >> 1, wc = wave & 1;
		const unsigned row = min(k1 + 16 * wr + m16, n - 1), col = min(k1 + 16 * wc + m16, n - 1);
		double xv[NQ], yv[NQ], dv[NQ];
#pragma unroll
		for(int q = 0; q < NQ; q++){
			const unsigned k = 4 * q + k4;
			xv[q] = A[(k0 + k) * n + row];
			dv[q] = dinv_cur[k * NB + 16 * wc + m16];
			yv[q] = A[col * n + k0 + k];
		}
#pragma unroll
		for(int e = 0; e < 4; e++) d[0][e] = A[col * n + min(k1 + 16 * wr + 4 * e + k4, n - 1)];
		gj_v4d ea[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
		for(int q = 0; q < NQ; q++) ea[q & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(-xv[q], dv[q], ea[q & 1], 0, 0, 0);
#pragma unroll
		for(int e = 0; e < 4; e++) sh.Di[16 * wr + 4 * e + k4][16 * wc + m16] = ea[0][e] + ea[1][e];
		__syncthreads();
#pragma unroll
		for(int q = 0; q < NQ; q++)
			d[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(sh.Di[16 * wr + m16][4 * q + k4], yv[q], d[0], 0, 0, 0);
	} else {
	const unsigned r0 = look ? k1 : bx * GJ_T, c0 = look ? k1 : by * GJ_T;
	// the last step writes the inverse straight to out_final unless the pivoted fallback will run
	// (it inverts the untouched input there)
	double *__restrict__ dst = (out_final && scal[SCAL_GJ_FLAG] == 0) ? out_final : An;
	const int wcb = 2 * (wave >> 1), wrb = 2 * (wave & 1);
	auto in_k = [&](unsigned i){ return i - k0 < (unsigned)NB; };   // of 16 rows or columns: past nbe they are past n
	// ---- every load up front: D^{-1}, A[rows, K] in operand layout (wave w: rows 16 w ..), A[K, columns] and
	// the tile.  Element (row, col) is at col n + row < 2^24: 32-bit offsets, rows and columns past n repeat
	// the last one; past nbe the rows of A[K, columns] and the columns of A[rows, K] count as zero
	double dv[MD], xv[NQ], yv[ML];
#pragma unroll
	for(int q = 0; q < MD; q++) dv[q] = dinv_cur[tid + 256 * q];
	{
		const unsigned xr = min(r0 + 16 * wave + m16, n - 1), x0 = (k0 + 2 * k4) * n + xr;
#pragma unroll
		for(int q = 0; q < NQ; q++) xv[q] = A[min(x0 + (8 * (q >> 1) + (q & 1)) * n, last + xr)];
		const unsigned yr = min(k0 + tid % NB, n - 1), y0 = (c0 + tid / NB) * n + yr;
#pragma unroll
		for(int q = 0; q < ML; q++) yv[q] = A[min(y0 + 256 / NB * q * n, last + yr)];
	}
	// the tile in transposed form, T^T[col][row] += sum_m Y[m][col] E[row][m]: wave w holds the 16 x 16
	// blocks of columns 16 (2 (w >> 1) + cb) and rows 16 (2 (w & 1) + rb); lane l has rows 16 rb' + l % 16
	// (16 lanes read 16 consecutive rows) and columns 16 cb' + 4 e + l / 16 in element e
	gj_v4d acc[2][2];
#pragma unroll
	for(int rb = 0; rb < 2; rb++){
		const unsigned tr = min(r0 + 16 * (wrb + rb) + m16, n - 1), t0 = (c0 + 16 * wcb + k4) * n + tr;
#pragma unroll
		for(int cb = 0; cb < 2; cb++)
#pragma unroll
			for(int e = 0; e < 4; e++) acc[cb][rb][e] = A[min(t0 + (16 * cb + 4 * e) * n, last + tr)];
	}
	// ---- transform rows, transposed: E^T[j][i] = -sum_m D^{-1}[m][j] A[i][k0 + m]; wave w has i = 16 w ..
#pragma unroll
	for(int q = 0; q < MD; q++) sh.Di[tid / NB + 256 / NB * q][tid % NB] = dv[q];
	__syncthreads();
	if(in_k(r0 + 16 * wave)){
		const double *di = sh.Di[r0 + 16 * wave + m16 - k0];
#pragma unroll
		for(int j = 0; j < NQ; j++) sh.Et[4 * j + k4][16 * wave + m16] = di[4 * j + k4];
	} else {
		gj_v4d ea[NB / 16];
#pragma unroll
		for(int jb = 0; jb < NB / 16; jb++) ea[jb] = gj_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
		for(int q = 0; q < NQ; q++){
			const int k = 8 * (q >> 1) + 2 * k4 + (q & 1);
			const double x = k < (int)nbe ? -xv[q] : 0.0;
#pragma unroll
			for(int jb = 0; jb < NB / 16; jb++)
				ea[jb] = __builtin_amdgcn_mfma_f64_16x16x4f64(sh.Di[k][16 * jb + m16], x, ea[jb], 0, 0, 0);
		}
#pragma unroll
		for(int jb = 0; jb < NB / 16; jb++)
#pragma unroll
			for(int e = 0; e < 4; e++) sh.Et[16 * jb + 4 * e + k4][16 * wave + m16] = ea[jb][e];
	}
	__syncthreads();
#pragma unroll
	for(int q = 0; q < ML; q++) sh.Yt[tid / NB + 256 / NB * q][tid % NB] = tid % NB < (int)nbe ? yv[q] : 0.0;
	__syncthreads();
	// ---- LU multipliers of the rows below K: 16 columns of -E L per round, 16 rows per wave
	if(!look && r0 + GJ_T > k1)
		for(unsigned jb = by; jb < (unsigned)NB / 16; jb += ncb){
			gj_v4d ya = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
			for(int kb = 0; kb < NQ; kb++){
				const int k = 4 * kb + k4;
				ya = __builtin_amdgcn_mfma_f64_16x16x4f64(sh.Et[k][16 * wave + m16], lm_cur[k * NB + 16 * jb + m16], ya, 0, 0, 0);
			}
			bool bad = false;
#pragma unroll
			for(int e = 0; e < 4; e++){
				const unsigned i = r0 + 16 * wave + 4 * e + k4;
				bad |= (i >= k1) & (i < n) & (16 * jb + m16 < nbe) & !(fabs(ya[e]) <= 1.0);
			}
			if(bad) scal[SCAL_GJ_FLAG] = 1;
		}
	// ---- tile update: T^T[col][row] += sum_m Y[m][col] E[row][m] (Yt[col][m], Et[m][row])
	if(in_k(c0 + 16 * wcb)){
#pragma unroll
		for(int cb = 0; cb < 2; cb++)
#pragma unroll
			for(int rb = 0; rb < 2; rb++)
#pragma unroll
				for(int e = 0; e < 4; e++)
					acc[cb][rb][e] = sh.Et[c0 + 16 * (wcb + cb) + 4 * e + k4 - k0][16 * (wrb + rb) + m16];
	} else {
		if(in_k(r0 + 16 * wrb))
#pragma unroll
			for(int cb = 0; cb < 2; cb++)
#pragma unroll
				for(int rb = 0; rb < 2; rb++) acc[cb][rb] = gj_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
		for(int kb = 0; kb < NB / 8; kb++){
			const int k = 8 * kb + 2 * k4;
			double2 y[2];
			double ev[2][2];
#pragma unroll
			for(int q = 0; q < 2; q++){
				y[q] = *(const double2 *)&sh.Yt[16 * (wcb + q) + m16][k];
				ev[q][0] = sh.Et[k][16 * (wrb + q) + m16];
				ev[q][1] = sh.Et[k + 1][16 * (wrb + q) + m16];
			}
#pragma unroll
			for(int h = 0; h < 2; h++)
#pragma unroll
				for(int cb = 0; cb < 2; cb++)
#pragma unroll
					for(int rb = 0; rb < 2; rb++)
						acc[cb][rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(h ? y[cb].y : y[cb].x, ev[rb][h], acc[cb][rb], 0, 0, 0);
		}
	}
	if(!look){
#pragma unroll
		for(int cb = 0; cb < 2; cb++)
#pragma unroll
			for(int e = 0; e < 4; e++){
				const unsigned col = c0 + 16 * (wcb + cb) + 4 * e + k4;
#pragma unroll
				for(int rb = 0; rb < 2; rb++){
					const unsigned row = r0 + 16 * (wrb + rb) + m16;
					if(row < n && col < n) dst[col * n + row] = acc[cb][rb][e];
				}
			}
		return;
	}
	if constexpr(NB == 64){
		// D' into the inversion's layout
		__syncthreads();
#pragma unroll
		for(int cb = 0; cb < 2; cb++)
#pragma unroll
			for(int rb = 0; rb < 2; rb++)
#pragma unroll
				for(int e = 0; e < 4; e++) sh.Yt[16 * (wrb + rb) + m16][16 * (wcb + cb) + 4 * e + k4] = acc[cb][rb][e];
		__syncthreads();
#pragma unroll
		for(int c = 0; c < 4; c++)
#pragma unroll
			for(int e = 0; e < 4; e++) d[c][e] = sh.Yt[gj_row<NB>(e)][gj_col<NB>(c)];
	}
	}
	// ---- lookahead: D'^{-1}, the identity past its columns
#pragma unroll
	for(int c = 0; c < (NB == 64 ? 4 : 1); c++)
#pragma unroll
		for(int e = 0; e < 4; e++)
			if(gj_row<NB>(e) >= nb1 || gj_col<NB>(c) >= nb1) d[c][e] = gj_row<NB>(e) == gj_col<NB>(c) ? 1.0 : 0.0;
	bool bad = false;
	const int rot = gj_invert<NB, true>(sh, nb1, d, bad, lm_next, diag, piv, k1);
	gj_store<NB>(d, rot, dinv_next);
	if(bad) scal[SCAL_GJ_FLAG] = 1;
}

template <int NB>
__global__ __launch_bounds__(256, 2) void gj_step_kernel(const double *__restrict__ A, double *__restrict__ An,
		unsigned n, unsigned k0, unsigned nbe, const double *__restrict__ dinv_cur, const double *__restrict__ lm_cur,
		double *__restrict__ dinv_next, double *__restrict__ lm_next, double *__restrict__ diag, int *__restrict__ piv,
		double *__restrict__ scal, double *__restrict__ out_final)
{
	__shared__ GjLds<NB> sh;
	gj_step_body<NB>(sh, A, An, n, k0, nbe, dinv_cur, lm_cur, dinv_next, lm_next, diag, piv, scal, out_final, blockIdx.x, blockIdx.y,
		gridDim.y);
}

// Fallback: in-place Gauss-Jordan with partial pivoting on M (one workgroup).  Runs only when
// the fast path saw a multiplier above 1 (or a non-finite one).  The row interchanges go to
// piv_out (LAPACK's sequential form, 0-based: row g was exchanged with row piv_out[g] at step g).
// A column without a nonzero candidate pivot makes the matrix singular: log|det| = -inf (the
// reference's sum of log|U_ii| with a zero U_ii, organic_dense_matrix.c:582-584), the step is
// recorded in SCAL_SINGULAR, and M is filled with NaN, so that a force or a Metropolis step built
// on it rejects instead of using a partial inverse.
template <unsigned NT>
__device__ __forceinline__ void gj_fallback_body(double *fsh, double *__restrict__ M, unsigned n, double *__restrict__ scal,
		int *__restrict__ piv_out)
{
	double *colg = fsh;                                   // n: multipliers of the step
	double *rowg = fsh + n;                               // n: the scaled pivot row of the step
	int *piv = reinterpret_cast<int *>(fsh + 2 * n);      // n
	__shared__ double rv[NT / 64];
	__shared__ int ri[NT / 64];
	__shared__ double ld_acc;
	__shared__ int neg_acc;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	if(tid == 0){ ld_acc = 0; neg_acc = 0; }
	for(unsigned g = 0; g < n; g++){
		double best = -1;
		int bidx = 0x7fffffff;
		for(unsigned r = g + tid; r < n; r += NT){
			const double a = fabs(M[(size_t)g * n + r]);
			if(a > best){ best = a; bidx = (int)r; }
		}
		for(int off = 32; off >= 1; off >>= 1){
			const double ob = __shfl_xor(best, off, 64);
			const int oi = __shfl_xor(bidx, off, 64);
			if(ob > best || (ob == best && oi < bidx)){ best = ob; bidx = oi; }
		}
		if(lane == 0){ rv[wave] = best; ri[wave] = bidx; }
		__syncthreads();
		best = rv[0]; bidx = ri[0];
		for(int w = 1; w < (int)(NT / 64); w++) if(rv[w] > best || (rv[w] == best && ri[w] < bidx)){ best = rv[w]; bidx = ri[w]; }
		if(best == 0){
			// every candidate in column g is zero (best is the same in every thread): singular
			for(size_t e = tid; e < (size_t)n * n; e += NT) M[e] = __longlong_as_double(0x7ff8000000000000LL);
			if(tid == 0){
				scal[SCAL_LOGDET] = -HUGE_VAL;
				scal[SCAL_SIGN] = 1.0;
				scal[SCAL_SINGULAR] = g + 1;
				scal[SCAL_GJ_FALLBACKS] += 1;
			}
			for(unsigned r = g + tid; r < n; r += NT) piv_out[r] = (int)r;
			return;
		}
		const unsigned p = bidx < (int)n ? (unsigned)bidx : g;
		if(tid == 0){
			piv[g] = (int)p;
			piv_out[g] = (int)p;
		}
		if(p != g)
			for(unsigned cc = tid; cc < n; cc += NT){
				const double t = M[(size_t)cc * n + g];
				M[(size_t)cc * n + g] = M[(size_t)cc * n + p];
				M[(size_t)cc * n + p] = t;
			}
		__syncthreads();
		const double d = M[(size_t)g * n + g];
		for(unsigned r = tid; r < n; r += NT) colg[r] = M[(size_t)g * n + r];
		if(tid == 0){ ld_acc += log(fabs(d)); neg_acc += (d < 0) + (p != g); }
		__syncthreads();
		const double inv = 1.0 / d;
		for(unsigned cc = tid; cc < n; cc += NT){
			double u = 0.0;
			if(cc != g){
				u = M[(size_t)cc * n + g] * inv;
				M[(size_t)cc * n + g] = u;
			}
			rowg[cc] = u;
		}
		__syncthreads();
		// rank-1 update over all threads: thread (r, c0) with r = tid % n, c0 = tid / n takes the columns
		// c0, c0 + cpp, ... (n <= NT); for larger n every thread takes rows tid, tid + NT of all columns
		{
			const bool small = n <= NT;
			const unsigned cpp = small ? NT / n : 1, rstep = small ? n : NT;
			const unsigned r0 = small ? tid % n : tid, c0 = small ? tid / n : 0;
			if(c0 < cpp)
				for(unsigned cc = c0; cc < n; cc += cpp){
					double *mc = M + (size_t)cc * n;
					const double u = rowg[cc];
					for(unsigned r = r0; r < n; r += rstep){
						if(r == g) continue;
						if(cc == g) mc[r] = -colg[r] * inv;
						else mc[r] -= colg[r] * u;
					}
				}
		}
		if(tid == 0) M[(size_t)g * n + g] = inv;         // (no thread writes row g in the update)
		__syncthreads();
	}
	// undo the row exchanges on the columns, in reverse order
	for(int g = (int)n - 1; g >= 0; g--){
		const int p = piv[g];
		if(p != g)
			for(unsigned r = tid; r < n; r += NT){
				const double t = M[(size_t)g * n + r];
				M[(size_t)g * n + r] = M[(size_t)p * n + r];
				M[(size_t)p * n + r] = t;
			}
		__syncthreads();
	}
	if(tid == 0){
		scal[SCAL_LOGDET] = ld_acc;
		scal[SCAL_SIGN] = (neg_acc & 1) ? -1.0 : 1.0;
		scal[SCAL_GJ_FALLBACKS] += 1;
	}
}

__global__ __launch_bounds__(1024) void gj_fallback_kernel(double *__restrict__ M, unsigned n, double *__restrict__ scal,
		int *__restrict__ piv_out)
{
	extern __shared__ double fsh[];
	if(scal[SCAL_GJ_FLAG] != 0) gj_fallback_body<1024>(fsh, M, n, scal, piv_out);
}

// N <= 64: the matrix is one diagonal block, so that one workgroup inverts it in LDS, sums its pivots and,
// where a multiplier exceeds 1, reads the untouched input again and inverts that with partial pivoting
// there.  One launch of 9 us at N = 36 (9 of the 16 four-pivot steps) where first block, two steps and the check
// for the fallback took 28
__device__ __forceinline__ void gj_small_body(GjLds<64> &sh, double *__restrict__ M, unsigned n, double *__restrict__ diag,
		int *__restrict__ piv, double *__restrict__ scal)
{
	const int tid = threadIdx.x;
	gj_v4d acc[4];
	bool bad = false;
	gj_clear_flags(scal);
	gj_load<64>(acc, M, n, n);
	const int rot = gj_invert<64, false>(sh, n, acc, bad, nullptr, diag, piv, 0);
	if(__syncthreads_or(bad)){
		double *m = &sh.Et[0][0];
		static_assert(64 * 64 <= 64 * GJ_LE, "the matrix exceeds the transform rows");
		for(unsigned e = tid; e < n * n; e += 256) m[e] = M[e];
		__syncthreads();
		if(tid == 0) scal[SCAL_GJ_FLAG] = 1;
		gj_fallback_body<256>(&sh.Yt[0][0], m, n, scal, piv);
		__syncthreads();
		for(unsigned e = tid; e < n * n; e += 256) M[e] = m[e];
		return;
	}
#pragma unroll
	for(int c = 0; c < 4; c++)
#pragma unroll
		for(int e = 0; e < 4; e++){
			const unsigned row = gj_row<64>(e), col = gj_col<64>((c + rot) & 3);
			if(row < n && col < n) M[(size_t)col * n + row] = acc[c][e];
		}
	if(tid < 64){
		// this wave's pivots, each written by the thread that reads it
		const double d = tid < (int)n ? diag[tid] : 1.0;
		double sl = log(fabs(d));
		int neg = d < 0;
		for(int off = 32; off > 0; off >>= 1){
			sl += __shfl_xor(sl, off, 64);
			neg += __shfl_xor(neg, off, 64);
		}
		if(tid == 0){
			scal[SCAL_LOGDET] = sl;
			scal[SCAL_SIGN] = (neg & 1) ? -1.0 : 1.0;
		}
	}
}

__global__ __launch_bounds__(256, 2) void gj_small_kernel(double *__restrict__ M, unsigned n, double *__restrict__ diag,
		int *__restrict__ piv, double *__restrict__ scal)
{
	__shared__ GjLds<64> sh;
	gj_small_body(sh, M, n, diag, piv, scal);
}

// M (column-major, N x N, FP64) <- M^{-1}; log|det| and sign into the device scalars.
int gj_logdet_inverse(ephmc_ctx *c, double *M)
{
	const unsigned n = c->ns;
	if(n > 4096){ set_error("gj: N = %u exceeds 4096", n); return EPHMC_ERR_UNSUPPORTED; }
	if(n <= 64){
		gj_small_kernel<<<1, 256, 0, c->stream>>>(M, n, c->d_diag, c->d_piv, c->d_scal);
		EPHMC_LAUNCHED();
		return EPHMC_OK;
	}
	const bool wide = n > GJ_WIDE_ABOVE;
	const unsigned nb = wide ? 64 : 32;
	const double *cur = M;
	double *buf[2] = {c->d_gj[0], c->d_gj[1]};
	int which = 0;
	// D^{-1} and L of the current and the next diagonal block (double-buffered by step parity)
	double *dinv_g[2] = {c->d_dlu, c->d_dlu + 64 * 64}, *lm_g[2] = {c->d_dlu + 2 * 64 * 64, c->d_dlu + 3 * 64 * 64};
	(wide ? gj_first_kernel<64> : gj_first_kernel<32>)<<<1, 256, 0, c->stream>>>(M, n, dinv_g[0], lm_g[0], c->d_diag, c->d_piv, c->d_scal);
	EPHMC_LAUNCHED();
	const dim3 sgrid((n + GJ_T - 1) / GJ_T + 1, (n + GJ_T - 1) / GJ_T);
	int par = 0;
	// from the second step on the input M is no longer read by the steps, so the last step writes
	// the inverse into it and sums the log det itself
	for(unsigned k0 = 0; k0 < n; k0 += nb){
		const unsigned nbe = std::min<unsigned>(nb, n - k0);
		double *next = buf[which];
		double *final_out = k0 + nbe >= n ? M : nullptr;
		(wide ? gj_step_kernel<64> : gj_step_kernel<32>)<<<sgrid, 256, 0, c->stream>>>(cur, next, n, k0, nbe, dinv_g[par], lm_g[par],
			dinv_g[par ^ 1], lm_g[par ^ 1], c->d_diag, c->d_piv, c->d_scal, final_out);
		EPHMC_LAUNCHED();
		cur = next;
		which ^= 1;
		par ^= 1;
	}
	const size_t lds = (size_t)n * (2 * sizeof(double) + sizeof(int));
	(void)hipFuncSetAttribute((const void *)gj_fallback_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
	gj_fallback_kernel<<<1, 1024, lds, c->stream>>>(M, n, c->d_scal, c->d_piv);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

// ---- many chains in one launch (batch.hip): the kernels of gj_logdet_inverse with the arguments
// of chain blockIdx.z read from a table; a chain's blocks past its own grid return.  A chain of
// N <= 64 is done by the first launch and takes no part in the others.
struct GjFirstArgs {
	double *A;
	unsigned n;
	double *dinv_out, *lm_out, *diag;
	int *piv;
	double *scal;
};

__global__ __launch_bounds__(256, 2) void gj_first_multi_kernel(const GjFirstArgs *__restrict__ tab)
{
	const GjFirstArgs &a = tab[blockIdx.z];
	__shared__ union Lds {
		GjLds<64> small;
		GjLds<32> first;
	} sh;
	if(a.n <= 64) gj_small_body(sh.small, a.A, a.n, a.diag, a.piv, a.scal);
	else gj_first_body<32>(sh.first, a.A, a.n, a.dinv_out, a.lm_out, a.diag, a.piv, a.scal);
}

struct GjStepArgs {
	const double *A;
	double *An;
	unsigned n, k0, nbe;
	const double *dinv_cur, *lm_cur;
	double *dinv_next, *lm_next, *diag;
	int *piv;
	double *scal, *out_final;
};

__global__ __launch_bounds__(256, 2) void gj_step_multi_kernel(const GjStepArgs *__restrict__ tab)
{
	const GjStepArgs &a = tab[blockIdx.z];
	const unsigned nrb = (a.n + GJ_T - 1) / GJ_T, ncb = nrb;
	if(blockIdx.x > nrb || blockIdx.y >= ncb) return;
	__shared__ GjLds<32> sh;
	gj_step_body<32>(sh, a.A, a.An, a.n, a.k0, a.nbe, a.dinv_cur, a.lm_cur, a.dinv_next, a.lm_next, a.diag, a.piv, a.scal, a.out_final,
		blockIdx.x, blockIdx.y, ncb);
}

struct GjFallbackArgs {
	double *M;
	unsigned n;
	double *scal;
	int *piv_out;
};

__global__ __launch_bounds__(1024) void gj_fallback_multi_kernel(const GjFallbackArgs *__restrict__ tab)
{
	const GjFallbackArgs &a = tab[blockIdx.z];
	extern __shared__ double fsh[];
	if(a.scal[SCAL_GJ_FLAG] != 0) gj_fallback_body<1024>(fsh, a.M, a.n, a.scal, a.piv_out);
}

int batch_gj(BatchOp &first, std::vector<BatchOp> &steps, BatchOp &fallback, ephmc_ctx *c, double *M)
{
	const unsigned n = c->ns;
	if(n <= 32 || n > GJ_WIDE_ABOVE){ set_error("batch gj: N = %u (the batch inverts 33 <= N <= %u)", n, GJ_WIDE_ABOVE); return EPHMC_ERR_UNSUPPORTED; }
	double *dinv_g[2] = {c->d_dlu, c->d_dlu + 64 * 64}, *lm_g[2] = {c->d_dlu + 2 * 64 * 64, c->d_dlu + 3 * 64 * 64};
	const GjFirstArgs fa{M, n, dinv_g[0], lm_g[0], c->d_diag, c->d_piv, c->d_scal};
	EPHMC_TRY(first.add((const void *)gj_first_multi_kernel, 256, 0, 1, 1, fa));
	if(n <= 64) return EPHMC_OK;
	const unsigned nrb = (n + GJ_T - 1) / GJ_T, ncb = nrb, nb = 32;
	const unsigned nsteps = (n + nb - 1) / nb;
	if(steps.size() < nsteps) steps.resize(nsteps);
	const double *cur = M;
	double *buf[2] = {c->d_gj[0], c->d_gj[1]};
	int which = 0, par = 0;
	for(unsigned i = 0; i < nsteps; i++){
		const unsigned k0 = i * nb, nbe = std::min(nb, n - k0);
		double *next = buf[which];
		GjStepArgs a{cur, next, n, k0, nbe, dinv_g[par], lm_g[par], dinv_g[par ^ 1], lm_g[par ^ 1], c->d_diag, c->d_piv,
			c->d_scal, k0 + nbe >= n ? M : nullptr};
		EPHMC_TRY(steps[i].add((const void *)gj_step_multi_kernel, 256, 0, nrb + 1, ncb, a));
		cur = next;
		which ^= 1;
		par ^= 1;
	}
	const size_t lds = (size_t)n * (2 * sizeof(double) + sizeof(int));
	(void)hipFuncSetAttribute((const void *)gj_fallback_multi_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
		(int)std::max(lds, fallback.lds));
	const GjFallbackArgs fb{M, n, c->d_scal, c->d_piv};
	return fallback.add((const void *)gj_fallback_multi_kernel, 1024, lds, 1, 1, fb);
}

} // namespace ephmc
