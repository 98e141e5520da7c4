// binary_step.hip -- the whole binary-fluid time step in one launch.
//
// The reference performs, per step (ludwig.c:528-860): the thermodynamic
// force from phi_t, the Cahn-Hilliard update phi_t -> phi_t+1 with the
// velocity of the previous collision, the collision of f_t with that force
// (giving rho_t, u_t), and the propagation.  Here one block owns a tile of
// (y, z) columns and marches along x through a chunk of planes
// (step_tile.h): for each site it forms F and the new phi from the LDS
// tiles, then collides the site's 19 pulled distributions with that F.  The
// force never goes to memory.
//
// Traffic per site (FP64): f 19 read + 19 write, phi read + write, u of the
// previous step read, u and rho written: 376 B (against 448 B for three
// separate passes).  Buffers: phi and u are double-buffered so that no block
// reads a value another block has already replaced.  Arithmetic is that of
// fe_ch.hip and lb_collide.hip, so FP64 results are bit-identical to the
// reference.

#include <hip/hip_runtime.h>

#include "kernels.h"
#include "step_tile.h"

namespace ldw {

namespace {

using namespace tile;

template <typename T, class S, int ORDER, int METHOD, bool GZ, bool CONS, bool GMU>
__global__ void __launch_bounds__(S::NT)
binary_step_kernel(Geom g, FeParams fe, LbParams prm, int nbz, int nby, int nbx, int remap,
		   const T * __restrict__ phi, T * __restrict__ phi_out,
		   const T * __restrict__ u_prev, T * __restrict__ u_next,
		   T * __restrict__ rho, const T * __restrict__ g_in,
		   T * __restrict__ g_out, T fz0, T fz1, T fz2, T * __restrict__ csum) {

  __shared__ Smem<T, S> s;

  int bzi, byi, bxi;
  if (!tile_of_block(nbz, nby, nbx, remap, bzi, byi, bxi)) return;
  // nbx chunks of planes, even to within one plane
  const int xq = g.nx/nbx, xr = g.nx - xq*nbx;
  const int xb = bxi*xq + min(bxi, xr);
  const int xe = xb + xq + (bxi < xr ? 1 : 0);
  step_tile<T, S, ORDER, METHOD, GZ, CONS, GMU>(s, g, fe, prm, byi*S::TY, bzi*S::TZ, xb, xe, phi, phi_out,
					   u_prev, u_next, rho, g_in, g_out, fz0, fz1, fz2, csum);
}

// The kernel for these parameters.  Advection order 4 is built for the 64 x 8
// tile only (launch() picks it).
template <typename T, class S, bool CONS, bool GMU>
auto step_kernel(const FeParams & fe, const LbParams & prm) {
  const bool gz = (prm.relax == 0);
#define K_G(O, M) (gz ? &binary_step_kernel<T, S, O, M, true, CONS, GMU> \
		   : &binary_step_kernel<T, S, O, M, false, CONS, GMU>)
#define K_M(O) (fe.force_method == 0 ? K_G(O, 0) : K_G(O, 1))
  if constexpr (S::TZ == 64) {
    if (fe.order == 4) return K_M(4);
  }
  return fe.order == 1 ? K_M(1) : (fe.order == 2 ? K_M(2) : K_M(3));
#undef K_M
#undef K_G
}

// Blocks of that kernel that the whole GPU holds at once (resident blocks per
// CU times the CUs); cached.  The kernels differ: FP32 with 32 x 8 tiles, 3 per
// CU, but 2 with advection order 3 (48x20x100: 11.0 us per step; 19.6 with the
// blocks of order 1 counted, which makes two rounds).
template <typename T, class S, bool CONS, bool GMU>
int resident_slots(const FeParams & fe, const LbParams & prm) {
  static int cache[5][2][2];
  int & slots = cache[(fe.order >= 1 && fe.order <= 4) ? fe.order : 0][fe.force_method == 0][prm.relax == 0];
  if (slots == 0) {
    int per_cu = 0, dev = 0;
    hipDeviceProp_t prop;
    const void * kernel = reinterpret_cast<const void *>(step_kernel<T, S, CONS, GMU>(fe, prm));
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess
	|| hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, S::NT, 0) != hipSuccess || per_cu < 1) {
      (void) hipGetLastError();
      return 256;
    }
    slots = per_cu*prop.multiProcessorCount;
  }
  return slots;
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1)/b; }

// Chunks of x planes for 64 x 8 tiles of a lattice that takes many rounds of
// blocks.  A block that marches over xc planes first loads 4 phi planes and
// forms 2 Q planes (about 3 planes of work), so a launch costs about
// ceil(blocks/slots)*(xc + 3) plane-times; the chunk that minimises it
// balances the prologue against the last, partly filled round (on MI355X
// 3.6 % faster than a fixed 2048-block grid at 256^3 FP64, 3.4 % at 128^3
// FP32).
//
// remap: the XCD-contiguous tile order, unless a chunk has more column tiles
// than an XCD holds blocks and the XCDs would share chunks (192^3 FP64, 7
// chunks of 72 columns: 534 us in linear order, 545 contiguous; 122x46x214, 10
// chunks of 24: 138 and 122).
struct StepPlan { int tz, nchunk, remap; };

inline StepPlan rounds_plan(const Geom & g, int slots) {
  const int nx = g.nx;
  const int64_t ncol = ceil_div(g.nz, 64)*ceil_div(g.ny, 8);
  int best = 1;
  int64_t best_cost = -1;
  for (int xc = nx; ; xc = (xc + 1)/2) {
    const int n = (int) ceil_div(nx, xc);
    const int64_t cost = ceil_div(ncol*n, slots)*(xc + 3);
    if (best_cost < 0 || cost <= best_cost) { best = n; best_cost = cost; }
    if (xc <= 1) break;
  }
  return {64, best, (8*ncol <= slots || best % 8 == 0) ? 1 : 0};
}

// The tile (its z extent; 8 rows in y) and the number of x chunks.
//
// A small lattice is bound by the length of one block: prologue and planes in
// a row.  It takes one round of blocks with as few planes each as fill the
// resident slots (2 blocks of 32 x 8 or 4 of 16 x 8 threads fit where one of
// 64 x 8 does), of the tile whose padding in y and z leaves the fewest planes
// per block.  A large one is bound by memory: 64-wide rows where z pads little,
// with long chunks; else 32-wide ones with chunks of 3 planes, so that
// neighbouring tiles of an XCD run close together and share their edge lines
// in its L2.  Measured over 60 lattices of 16^3 to 256^3, cubic and ragged (us
// per step, with one 64 x 8 tile of at least 4 planes before): FP64 32^3 28.9 ->
// 9.7, 64^3 33 -> 22, 80^3 65 -> 42, 91x88x66 92 -> 46, 102x221x150 375 -> 333,
// 128^3 174 -> 171, 256^3 unchanged; FP32 64^3 22 -> 15, 96^3 52 -> 34,
// 144^3 223 -> 153.  The best of all tiles and chunks is 3 % (FP64) and 6 %
// (FP32) faster on average.  The lines between the two: at 0.8 M sites (FP64;
// 1.0 M: 87x78x169 137 us in one round of 16 x 8 tiles, 109 in 64 x 8 chunks)
// and 1.25 M (FP32), and at 1.2 of padding (FP64 87x58x212, 1.21: 104 us with 64
// x 8, 108 with 32 x 8; 82x173x150, 1.28: 237 and 209).
template <typename T>
StepPlan step_plan(const Geom & g, const FeParams & fe, const LbParams & prm) {
  static const int tzs[3] = {16, 32, 64};
  const int slots[3] = {resident_slots<T, Shape<16, 8>, false, false>(fe, prm),
			resident_slots<T, Shape<32, 8>, false, false>(fe, prm),
			resident_slots<T, Shape<64, 8>, false, false>(fe, prm)};
  // a plane of the narrower tiles costs slightly more or less than its share
  static const double weight64[3] = {1.00, 1.02, 1.10}, weight32[3] = {1.05, 1.00, 1.10};
  const double * weight = (sizeof(T) == 8) ? weight64 : weight32;
  const int64_t small = (sizeof(T) == 8) ? 800000 : 1250000;
  const int forced = tune_step_tile();
  if (g.nsite <= small) {
    StepPlan best = {0, 0, 1};
    double best_cost = 0.0;
    for (int k = 0; k < 3; k++) {
      if (forced && tzs[k] != forced) continue;
      const int64_t ncol = ceil_div(g.nz, tzs[k])*ceil_div(g.ny, 8);
      if (slots[k] < ncol) continue;
      const int64_t xc = ceil_div(g.nx, slots[k]/ncol);
      const double cost = (double) (xc + 2)*weight[k];
      if (best.tz == 0 || cost < best_cost) { best = {tzs[k], (int) ceil_div(g.nx, xc), 1}; best_cost = cost; }
    }
    if (best.tz) return best;
  }
  if (forced == 64 || (!forced && ceil_div(g.nz, 64)*64*5 <= (int64_t) g.nz*6))
    return rounds_plan(g, slots[2]);
  return {forced ? forced : 32, (int) ceil_div(g.nx, 3), 1};
}

template <typename T, class S, bool CONS, bool GMU>
void launch_shape(const Geom & g, const FeParams & fe, const LbParams & prm, const T * phi,
		  T * phi_out, const T * u_prev, T * u_next, T * rho, const T * g_in,
		  T * g_out, const double fzero[3], T * csum, const StepPlan & plan, hipStream_t st) {
  const int bz = (g.nz + S::TZ - 1)/S::TZ;
  const int by = (g.ny + S::TY - 1)/S::TY;
  int bx = plan.nchunk;
  if (getenv("LDW_MIN_BLOCKS")) {
    // the fixed rule: halve the chunk until the grid has that many blocks
    int xchunk = g.nx;
    const int want = tune_min_blocks();
    while (xchunk > 8 && (int64_t) bz*by*((g.nx + xchunk - 1)/xchunk) < want) xchunk = (xchunk + 1)/2;
    bx = (g.nx + xchunk - 1)/xchunk;
  }
  const int ntile = bz*by*bx;
  dim3 grid(((ntile + NXCD - 1)/NXCD)*NXCD), block(S::TZ, S::TY, 1);
  const T f0 = T(fzero[0]), f1 = T(fzero[1]), f2 = T(fzero[2]);
  hipLaunchKernelGGL((step_kernel<T, S, CONS, GMU>(fe, prm)), grid, block, 0, st, g, fe, prm, bz, by, bx,
		     tune_remap_step(plan.remap), phi, phi_out, u_prev, u_next, rho, g_in, g_out, f0, f1, f2, csum);
}

// The tile changes only which block computes a site, not the arithmetic.
// With a compensation array (conserve 1), advection order 4 or an external
// chemical potential gradient the 64 x 8 tile is used, so those kernels are
// built for one tile only.  The kernels without the external gradient leave
// its code out, which keeps the FP32 kernels at 3 waves per SIMD.
template <typename T>
void launch(const Geom & g, const FeParams & fe, const LbParams & prm, const T * phi,
	    T * phi_out, const T * u_prev, T * u_next, T * rho, const T * g_in,
	    T * g_out, const double fzero[3], T * csum, hipStream_t st) {
  using S64 = Shape<64, 8>;
#define S64_(CONS, GMU) launch_shape<T, S64, CONS, GMU>(g, fe, prm, phi, phi_out, u_prev, u_next, rho, g_in, g_out, fzero, \
						       csum, rounds_plan(g, resident_slots<T, S64, CONS, GMU>(fe, prm)), st)
  if (fe.gmu_on || csum || fe.order == 4) {
    if (fe.gmu_on && csum) S64_(true, true);
    else if (fe.gmu_on) S64_(false, true);
    else if (csum) S64_(true, false);
    else S64_(false, false);
    return;
  }
#undef S64_
  const StepPlan p = step_plan<T>(g, fe, prm);
#define TILE_(TZ) launch_shape<T, Shape<TZ, 8>, false, false>(g, fe, prm, phi, phi_out, u_prev, u_next, rho, g_in, g_out, \
						       fzero, nullptr, p, st)
  if (p.tz == 16) TILE_(16);
  else if (p.tz == 32) TILE_(32);
  else TILE_(64);
#undef TILE_
}

}  // namespace

void launch_binary_step_f64(const Geom & g, const FeParams & fe, const LbParams & prm,
			    const double * phi, double * phi_out, const double * u_prev,
			    double * u_next, double * rho, const double * g_in,
			    double * g_out, const double fzero[3], double * csum, hipStream_t s) {
  launch<double>(g, fe, prm, phi, phi_out, u_prev, u_next, rho, g_in, g_out, fzero, csum, s);
}

void launch_binary_step_f32(const Geom & g, const FeParams & fe, const LbParams & prm,
			    const float * phi, float * phi_out, const float * u_prev,
			    float * u_next, float * rho, const float * g_in,
			    float * g_out, const double fzero[3], float * csum, hipStream_t s) {
  launch<float>(g, fe, prm, phi, phi_out, u_prev, u_next, rho, g_in, g_out, fzero, csum, s);
}

}  // namespace ldw
