// conv3d.hip -- 3 x 3 x 3 convolutions on periodic lattices as implicit
// GEMMs on the MFMA units (BF16 operands, FP32 accumulation), for the
// learned surrogate's network.
//
// Layout: activations are channels-last, x[p][c] with p = ((b*nx + x)*ny + y)*nz + z
// over the batch, so the 27 taps of a position are 27 contiguous channel
// rows.  Padding is periodic (the lattice is periodic), so no halo exists
// and the adjoint of a convolution is again a convolution.  Channel
// counts are multiples of 16.
//
// Forward, y = b + sum_t W_t x(p + o_t):  GEMM with M = Cout, N = positions,
//   K = 27 Cin; tiles of x with their halo are staged in LDS 16 channels at a
//   time, each read for up to 3 taps.
// Backward data, dx = sum_t W_{26-t}^T dy(p + o_t): the same kernel with the
//   weights flipped and transposed (conv3_weights_prep).
// Backward weight, dW_t = sum_p dy(p) x(p + o_t)^T:  GEMM with M = Cout,
//   N = Cin, K = positions; tiles of dy and x are staged through LDS, read as
//   transposed fragments, and the blocks' sums are added in a fixed order
//   (deterministic).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "conv_plan.h"
#include "kernels.h"
#include "silu.h"

namespace ldw {

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int wrapi(int i, int n) {
  return (i < 0) ? i + n : (i >= n ? i - n : i);
}

typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4a __attribute__((ext_vector_type(4), aligned(8)));   // 16 bytes, 8-byte aligned
typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t h4a __attribute__((ext_vector_type(4), aligned(2)));

// ---------------------------------------------------------------------------
// Forward pass (and, on the flipped weights, the backward-data pass).
//
// A block works through CT_X x TY x ZT tiles (CT_X = 4*16/ZT) for 16*NT output
// channels.  Wave w owns TY rows of 16 positions: z0 .. z0+15 at x0 + w
// (ZT = 16), or 8 z at two neighbouring x (ZT = 8, for lattices up to 8 deep).
// Input channels go 16 at a time; such a slice of the tile with its halo lies
// in LDS, 32 bytes per position.
//
// A unit is up to two (dx, dz) columns of the stencil, whose 16 channels each
// fill the K = 32 of v_mfma_f32_16x16x32_bf16: lanes q = 0, 1 hold the first
// column, q = 2, 3 the second.  Five units make a slice: dz = 0 and 1 for each
// dx, dz = 2 for dx = 0 and 1, and the ninth column alone (K = 16, which
// occupies the unit as long: 10 MFMAs do the work of 9).  A unit's weights, three
// dy taps, are held in registers while the wave walks the TY + 2 halo rows,
// so one LDS read of a row serves up to 3 taps x NT MFMAs (a read per tap
// makes LDS the bound: 6 reads per 8 MFMAs at NT = 2).
//
// Everything is staged by loads straight to LDS, two buffers each, so no
// registers hold data in flight: the next unit's weights are requested at a
// unit's start and waited for at its end; the next slice's halo (of the next
// tile after the last slice) is requested over the first units of a slice and
// waited for at its end, the other waits let that unit's halo loads go on.
//
// The weights are the first MFMA operand and the positions the second, so
// lane (r, q) ends with channels 4q .. 4q+3 of position r: 16-byte stores.
//
// Bound by the halo loads beside the MFMAs (which are busy 42 % of the time):
// without them 80 -> 32 channels on 8 x 64^3 would take 264 us.  It takes 342 us
// (847 TFLOP/s), 373 with the SiLU, and the network's 12 layers on 8 x 64^3 1.01
// ms, against 500 us and 1.62 ms for a tile per block, staged through registers
// with two barriers per three taps and a read per tap.

constexpr int NUNIT = 5;
constexpr int NXCD = 8;

template <int TY, int ZT>
struct ConvTile {
  static constexpr int XW = 16/ZT;            // x planes of a wave
  static constexpr int X = 4*XW, HX = X + 2, HY = TY + 2, HZ = ZT + 2;
  static constexpr int HP = HY*HZ, N = HX*HP; // halo positions of a plane, of the tile
  static constexpr int HL = (2*N + 63)/64;    // loads of a wave (64 vectors of 16 bytes) in all
  static constexpr int HW = (HL + 3)/4;       // per wave
  static constexpr int HU = (HW + NUNIT - 2)/(NUNIT - 1);   // per unit, none in a slice's last
  static constexpr int in_unit(int u) { return (HW > (u + 1)*HU) ? HU : (HW > u*HU ? HW - u*HU : 0); }
};

// Weight rows are 4 x 16 bytes, halo rows 2 x 16.  The 16 lanes of a fragment
// read consecutive rows at one 16-byte part; XOR-swizzling the part with bits
// of the consecutive index (output channel, z) spreads them over all banks and
// leaves the other indices plain offsets.
__device__ __forceinline__ int w_part(int i, int part) { return part ^ ((i >> 1) & 3); }
__device__ __forceinline__ int h_part(int z, int part) { return part ^ ((z >> 3) & 1); }

// the lattice coordinate of halo offset i: periodic wrap; what lies further
// out belongs to positions outside the lattice, whose results are dropped
__device__ __forceinline__ int halo_at(int i, int n) {
  i = wrapi(i, n);
  return (i < n) ? i : 0;
}

// 16 bytes per lane from global memory to LDS at byte offset `to` + 16 lane.
// The compiler does not know that the load is in flight: wait_barrier waits.
// The offset goes through M0, which the compiler sets.
__device__ __forceinline__ void load_to_lds(const void * from, uint32_t to) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(from), "{m0}"(to) : "memory");
}

// all but this wave's last N memory operations and all its LDS reads done,
// then the block barrier
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

// DMA: x and w are 16-byte aligned, as the loads to LDS need it.  Otherwise the
// same loads go through registers: requested at the same places, written to
// LDS at the unit's end (weights) and the next unit's (halo).
template <int NT, int TY, int ZT, bool DMA>
__global__ void __launch_bounds__(256, 2)
conv3_fwd_kernel(const uint16_t * __restrict__ x, const uint16_t * __restrict__ w,
		 const float * __restrict__ bias, float * __restrict__ y, uint16_t * __restrict__ act,
		 int nx, int ny, int nz, int cin, int cout, int accumulate, int ntx, int nty, int ntz, int ntile) {
  using C = ConvTile<TY, ZT>;
  constexpr int NW = 3*16*NT*4;               // weight vectors of a unit
  constexpr int WL = NW/64, WW = (WL + 3)/4;  // loads of a wave: in all, per wave
  __shared__ u4 lds[2*NW + 2*64*C::HL];       // weights, then halo slices
  const uint32_t base = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) &lds[0];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4, hi = q >> 1;
  const int64_t nsite = (int64_t) nx*ny*nz;
  const int n0 = blockIdx.y*16*NT;

  // This lane's halo vectors: load i of the wave covers vectors 64 j .. + 63,
  // j = wave + 4 i, two per position.  Loads and positions past the end repeat
  // the last ones, so that every wave issues as many.
  int hc[C::HW];                              // halo coordinates and part
  uint32_t hs[C::HW];                         // site in the tile being fetched
#pragma unroll
  for (int i = 0; i < C::HW; i++) {
    const int v = 64*min(wave + 4*i, C::HL - 1) + lane;
    const int p = min(v >> 1, C::N - 1);
    const int hz = p % C::HZ, hy = (p/C::HZ) % C::HY, hx = p/C::HP;
    hc[i] = hx | (hy << 8) | (hz << 16) | (h_part(hz, v & 1) << 24);
  }
  int x0, y0, z0;
  int64_t p0;                                 // first position of the sample
  auto locate = [&](int t, int & tx, int & ty, int & tz, int64_t & tp) {
    tz = (t % ntz)*ZT; t /= ntz;
    ty = (t % nty)*TY; t /= nty;
    tx = (t % ntx)*C::X;
    tp = (int64_t) (t/ntx)*nsite;
  };
  auto sites = [&](int tx, int ty, int tz) {
#pragma unroll
    for (int i = 0; i < C::HW; i++) {
      const int cx = halo_at(tx + (hc[i] & 255) - 1, nx), cy = halo_at(ty + ((hc[i] >> 8) & 255) - 1, ny);
      hs[i] = ((uint32_t) cx*ny + cy)*nz + halo_at(tz + ((hc[i] >> 16) & 255) - 1, nz);
    }
  };
  // loads [i0, i1) of slice c0 of the sample at tp into halo buffer hb
  u4 rh[C::HW], rw[WW];                       // (not DMA) in flight
  auto halo_row = [&](int i, int hb) { return 2*NW + 64*(hb*C::HL + min(wave + 4*i, C::HL - 1)); };
  auto fetch_halo = [&](int i0, int i1, int64_t tp, int c0, int hb) {
#pragma unroll
    for (int i = 0; i < C::HW; i++) {
      if (i < i0 || i >= i1) continue;
      const uint16_t * from = x + (tp + hs[i])*cin + (c0 + 8*(hc[i] >> 24));
      if constexpr (DMA) load_to_lds(from, base + 16*halo_row(i, hb));
      else rh[i] = *reinterpret_cast<const u4a *>(from);
    }
  };
  auto put_halo = [&](int i0, int i1, int hb) {
#pragma unroll
    for (int i = 0; i < C::HW; i++)
      if (i >= i0 && i < i1) lds[halo_row(i, hb) + lane] = rh[i];
  };

  // This lane's weight vectors: row dy*16*NT + n, part; parts 2, 3 belong to
  // the unit's second column.  Rows past the last output channel repeat it.
  int wo[WW];
  const int tap = cout*cin;
#pragma unroll
  for (int k = 0; k < WW; k++) {
    const int i = 64*min(wave + 4*k, WL - 1) + lane;
    const int row = i >> 2, part = w_part(row, i & 3);
    const int n = min(n0 + row % (16*NT), cout - 1);
    wo[k] = ((3*(row/(16*NT))*cout + n)*cin + 8*(part & 1))*2 + (part >> 1);
  }
  auto w_row = [&](int k, int buf) { return buf*NW + 64*min(wave + 4*k, WL - 1); };
  auto fetch_w = [&](int u, int c0, int buf) {
    // second column: dz + 1 (units 0-2), dx + 1 (unit 3), none (unit 4)
    const int col = (u < 3) ? 9*u : (u == 3 ? 2 : 20), step = (u < 3) ? 1 : (u == 3 ? 9 : 0);
#pragma unroll
    for (int k = 0; k < WW; k++) {
      const uint16_t * from = w + ((int64_t) col*tap + c0) + ((wo[k] >> 1) + (wo[k] & 1)*(step*tap));
      if constexpr (DMA) load_to_lds(from, base + 16*w_row(k, buf));
      else rw[k] = *reinterpret_cast<const u4a *>(from);
    }
  };
  auto put_w = [&](int buf) {
#pragma unroll
    for (int k = 0; k < WW; k++) lds[w_row(k, buf) + lane] = rw[k];
  };

  f4 acc[TY][NT];
#pragma unroll
  for (int j = 0; j < TY; j++)
#pragma unroll
    for (int n = 0; n < NT; n++) acc[j][n] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // halo row of lane r in this wave's row Y = 0, column (dx, dz) = (0, 0)
  const int rz = (ZT == 16) ? r : (r & 7), rx = C::XW*wave + (ZT == 16 ? 0 : r >> 3);
  const int hrow = rx*C::HP + rz;
  auto unit32 = [&](int buf, int hb, int dx, int dz) {
    const u4 * pw = &lds[buf*NW + 4*r + w_part(r, q)];
    const u4 * pa = &lds[2*NW + 64*C::HL*hb + 2*(hrow + dx*C::HP + dz) + h_part(rz + dz, q & 1)];
    b8 bw[3][NT];
#pragma unroll
    for (int dy = 0; dy < 3; dy++)
#pragma unroll
      for (int n = 0; n < NT; n++) bw[dy][n] = __builtin_bit_cast(b8, pw[64*(dy*NT + n)]);
#pragma unroll
    for (int Y = 0; Y < TY + 2; Y++) {
      const b8 a = __builtin_bit_cast(b8, pa[2*Y*C::HZ]);
#pragma unroll
      for (int dy = 0; dy < 3; dy++) {
	const int j = Y - dy;
	if (j < 0 || j >= TY) continue;
#pragma unroll
	for (int n = 0; n < NT; n++)
	  acc[j][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[dy][n], a, acc[j][n], 0, 0, 0);
      }
    }
  };
  // the ninth column: lane (r, q) holds channels 4q .. 4q+3, the (q & 1) half
  // of part q >> 1
  auto unit16 = [&](int buf, int hb) {
    auto half = [&](const u4 * v) {
      return *reinterpret_cast<const s4 *>(reinterpret_cast<const char *>(v) + 8*(q & 1));
    };
    const u4 * pw = &lds[buf*NW + 4*r + w_part(r, hi)];
    const u4 * pa = &lds[2*NW + 64*C::HL*hb + 2*(hrow + 2*C::HP + 2) + h_part(rz + 2, hi)];
    s4 bw[3][NT];
#pragma unroll
    for (int dy = 0; dy < 3; dy++)
#pragma unroll
      for (int n = 0; n < NT; n++) bw[dy][n] = half(pw + 64*(dy*NT + n));
#pragma unroll
    for (int Y = 0; Y < TY + 2; Y++) {
      const s4 a = half(pa + 2*Y*C::HZ);
#pragma unroll
      for (int dy = 0; dy < 3; dy++) {
	const int j = Y - dy;
	if (j < 0 || j >= TY) continue;
#pragma unroll
	for (int n = 0; n < NT; n++)
	  acc[j][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bw[dy][n], a, acc[j][n], 0, 0, 0);
      }
    }
  };

  // results of the tile: lane (r, q) has channels 4q .. 4q+3 of position r of
  // each row
  auto store_tile = [&]() {
    const int gx = x0 + rx, gz = z0 + rz;
    if (gx >= nx || gz >= nz) return;
    const int64_t o0 = (p0 + ((int64_t) gx*ny + y0)*nz + gz)*cout + n0 + 4*q;
#pragma unroll
    for (int n = 0; n < NT; n++) {
      if (n0 + 16*n >= cout) continue;
      f4 bv = f4{0.0f, 0.0f, 0.0f, 0.0f};
      if (bias) bv = *reinterpret_cast<const f4a *>(bias + n0 + 16*n + 4*q);
#pragma unroll
      for (int j = 0; j < TY; j++) {
	if (y0 + j >= ny) continue;
	const int64_t o = o0 + (int64_t) j*nz*cout + 16*n;
	f4 v = acc[j][n] + bv;
	if (y) {
	  f4a * yo = reinterpret_cast<f4a *>(y + o);
	  if (accumulate) v += f4(*yo);
	  *yo = v;
	}
	if (act) {
	  const float z[4] = {v[0], v[1], v[2], v[3]};
	  uint16_t a[4];
	  silu_bf16(z, a);
	  *reinterpret_cast<h4a *>(act + o) = h4a{a[0], a[1], a[2], a[3]};
	}
      }
    }
  };

  // Blocks are dispatched round-robin over the 8 XCDs.  Where the grid allows,
  // XCD g takes the tiles [g per, (g + 1) per) in order, all its blocks side by
  // side, so that neighbouring tiles share their halos and the 128-byte lines
  // of their slices in its L2.
  const bool xcd = (gridDim.x % NXCD == 0);
  const int per = xcd ? (ntile + NXCD - 1)/NXCD : ntile;
  const int step = xcd ? (int) gridDim.x/NXCD : (int) gridDim.x;
  const int first = xcd ? (int) (blockIdx.x % NXCD)*per : 0;
  const int end = min(first + per, ntile);
  int tile = first + (xcd ? (int) blockIdx.x/NXCD : (int) blockIdx.x);
  if (tile >= end) return;
  locate(tile, x0, y0, z0, p0);
  sites(x0, y0, z0);
  fetch_w(0, 0, 0);
  fetch_halo(0, C::HW, p0, 0, 0);
  if constexpr (!DMA) { put_w(0); put_halo(0, C::HW, 0); }
  wait_barrier<0>();
  int buf = 0, hb = 0, c0 = 0;
#pragma unroll 1
  for (;;) {
    // the slice that follows; after the block's last one, that one again (not
    // used, but every unit then waits for the same number of loads)
    const bool last = (c0 + 16 >= cin);
    const bool done = last && (tile + step >= end);
    const int cn = done ? c0 : (last ? 0 : c0 + 16);
    const int tn = (last && !done) ? tile + step : tile;
    int xn = x0, yn = y0, zn = z0;
    int64_t pn = p0;
    if (last) {
      locate(tn, xn, yn, zn, pn);
      sites(xn, yn, zn);
    }
#pragma unroll
    for (int u = 0; u < NUNIT; u++) {
      if (u + 1 < NUNIT) fetch_w(u + 1, c0, buf ^ 1);
      else fetch_w(0, cn, buf ^ 1);
      if (u + 1 < NUNIT) fetch_halo(u*C::HU, (u + 1)*C::HU, pn, cn, hb ^ 1);
      if (u < 3) unit32(buf, hb, u, hi);
      else if (u == 3) unit32(buf, hb, hi, 2);
      else unit16(buf, hb);
      if constexpr (!DMA) {
	put_w(buf ^ 1);
	if (u > 0) put_halo((u - 1)*C::HU, u*C::HU, hb ^ 1);
      }
      // wait for the weights; this unit's halo loads may go on
      if (u == 0) wait_barrier<C::in_unit(0)>();
      else if (u == 1) wait_barrier<C::in_unit(1)>();
      else if (u == 2) wait_barrier<C::in_unit(2)>();
      else if (u == 3) wait_barrier<C::in_unit(3)>();
      else wait_barrier<0>();
      buf ^= 1;
    }
    if (last) {
      store_tile();
      if (done) break;
#pragma unroll
      for (int j = 0; j < TY; j++)
#pragma unroll
	for (int n = 0; n < NT; n++) acc[j][n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    hb ^= 1;
    tile = tn;
    c0 = cn;
    x0 = xn; y0 = yn; z0 = zn; p0 = pn;
  }
}

// ---------------------------------------------------------------------------
// Weight gradient, dW_t[co][ci] = sum_p dy(p)[co] x(p + o_t)[ci].
//
// One of the two arrays is read in place ("fixed", the one with more
// channels), the other at the 27 shifted positions; shifting dy instead of x
// only turns tap t into tap 26 - t.  A block owns 16 channels of the shifted
// array and 16*NF of the fixed one, and marches along x over a WT_Y x WT_Z
// (y, z) tile: LDS holds four planes of the shifted tile with its halo and
// two of the fixed tile, so each plane is fetched once for the 27 taps and
// the next plane's loads are in flight while the current one is used.  Wave w
// accumulates taps 7w .. 7w+6 over all positions of the tile.
//
// K of the GEMM is the position, which is the strided index of the
// channels-last arrays.  ds_read_b64_tr_b16 transposes on the way out of LDS:
// 16 lanes read 4 positions x 16 channels and lane r receives channel r of
// the 4 positions, so two reads make the 8-position fragment of
// v_mfma_f32_16x16x32_bf16.  Both operands use the same order of positions.
// LDS rows are 16 channels (32 bytes), one block of rows per 16 channels: the
// 16 rows of a read are then 512 contiguous bytes, without bank conflicts.
//
// A block's sums stay in registers over all its columns and are written
// once; wgrad_reduce_kernel adds the blocks' sums in a fixed order.
//
// Bound by LDS reads and MFMAs alike: (7 + NF) fragments are read per 7 NF
// MFMAs, so the array with more channels is the fixed one; NF is at most 5,
// which is what 256 registers hold.  On 4 x 64^3, 80 -> 32 channels takes
// 133 us (1.09 PFLOP/s), and the 12 layers of the network 0.52 ms with the
// reductions, against 14.6 ms when every block staged its positions again
// for each tap and transposed the fragments with 2-byte LDS reads.

constexpr int WT_Y = 8, WT_Z = 16;
constexpr int WT_N = WT_Y*WT_Z;                       // positions of a tile plane
constexpr int WH_Z = WT_Z + 2, WH_N = (WT_Y + 2)*WH_Z; // with the halo
constexpr int WT_TAPS = 7;                            // taps per wave
constexpr int WG_BLOCKS = 512;                        // blocks of a launch: two per CU
constexpr int WG_NF_MAX = 5;

struct WgradPlan {
  int shift_x;                   // x is the shifted array (else dy)
  int nf, nfg, ns;               // fixed 16-channel blocks per block, groups of them; shifted blocks
  int ty, tz, xlen, xc;          // tiles in y and z, planes per item, items along x
  int items, nchunk;             // (sample, column, x range) items; blocks that share them
};

WgradPlan wgrad_plan(int batch, int nx, int ny, int nz, int cin, int cout) {
  WgradPlan w;
  const int bi = cin/16, bo = cout/16;
  w.shift_x = (cin <= cout);
  w.ns = w.shift_x ? bi : bo;
  const int f = w.shift_x ? bo : bi;
  w.nfg = (f + WG_NF_MAX - 1)/WG_NF_MAX;
  w.nf = (f + w.nfg - 1)/w.nfg;
  w.ty = (ny + WT_Y - 1)/WT_Y;
  w.tz = (nz + WT_Z - 1)/WT_Z;
  const int cols = batch*w.ty*w.tz;
  int want = WG_BLOCKS/(w.ns*w.nfg);
  if (want < 1) want = 1;
  // x ranges of at least 2 planes (each reads 2 halo planes more) until the
  // items make the wanted number of blocks; single planes where even those
  // leave most of the GPU idle (16 -> 16 on 8^3: 7.9 -> 7.2 us)
  int xc = (want + cols - 1)/cols;
  const int most = (cols*nx <= want/8) ? nx : (nx + 1)/2;
  if (xc > most) xc = most;
  w.xlen = (nx + xc - 1)/xc;
  w.xc = (nx + w.xlen - 1)/w.xlen;
  w.items = cols*w.xc;
  w.nchunk = (w.items < want) ? w.items : want;
  return w;
}

__device__ __forceinline__ s4 read_tr(const uint16_t * p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
    (__attribute__((address_space(3))) s4 *) const_cast<uint16_t *>(p));
}

__device__ __forceinline__ b8 join8(s4 lo, s4 hi) {
  const s8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(b8, v);
}

// fx, sx: the fixed and the shifted array, cf and cs channels.  EDGE: some
// tiles reach past the lattice.
template <int NF, bool SHIFT_X, bool EDGE>
__global__ void __launch_bounds__(256, 2)
conv3_wgrad_kernel(const uint16_t * __restrict__ fx, const uint16_t * __restrict__ sx,
		   float * __restrict__ part, int nx, int ny, int nz, int cf, int cs,
		   int ty, int tz, int xlen, int xc, int items) {
  __shared__ __attribute__((aligned(16))) uint16_t ls[4][WH_N*16];
  __shared__ __attribute__((aligned(16))) uint16_t lf[2][NF][WT_N*16];
  __shared__ __attribute__((aligned(16))) uint16_t lz[(WH_Z + 1)*16];   // zeros
  const int tid = threadIdx.x;
  if (EDGE && tid < (WH_Z + 1)*2) *reinterpret_cast<u4 *>(&lz[8*tid]) = u4{0u, 0u, 0u, 0u};
  const int lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int s0 = 16*(blockIdx.y % (cs/16));              // first shifted channel
  const int f0 = 16*NF*(blockIdx.y / (cs/16));           // first fixed channel

  f4 acc[WT_TAPS][NF];
#pragma unroll
  for (int j = 0; j < WT_TAPS; j++)
#pragma unroll
    for (int k = 0; k < NF; k++) acc[j][k] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // this lane's part of a transposing read: position 4q + (r >> 2) of a row
  // of 16, channels 4 (r & 3) .. + 3
  const int lpos = 4*q + (r >> 2), lch = 4*(r & 3);
  const int half = 8*(tid & 1);                          // staging: 8 channels per thread

  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    int c = item;
    const int xi = c % xc; c /= xc;
    const int z0 = (c % tz)*WT_Z; c /= tz;
    const int y0 = (c % ty)*WT_Y;
    const int b = c / ty;
    const int xb = xi*xlen;
    const int n = min(xlen, nx - xb);                    // planes of this item
    const int64_t plane = (int64_t) ny*nz;
    const uint16_t * fb = fx + (int64_t) b*nx*plane*cf + f0 + half;
    const uint16_t * sb = sx + (int64_t) b*nx*plane*cs + s0 + half;

    // staging positions within a plane; -1: outside the lattice, staged as
    // zeros (in the shifted tile everything past the wrapped halo)
    const int fr = tid >> 1;
    const int fy = y0 + fr/WT_Z, fz = z0 + fr%WT_Z;
    const int64_t fo = (fy < ny && fz < nz) ? ((int64_t) fy*nz + fz)*cf : -1;
    int64_t so[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int row = (tid + 256*k) >> 1;
      const int y = y0 + row/WH_Z - 1, z = z0 + row%WH_Z - 1;
      so[k] = (row < WH_N && y <= ny && z <= nz) ? ((int64_t) wrapi(y, ny)*nz + wrapi(z, nz))*cs : -1;
    }
    // Outside the lattice the fixed tile is zero, but a shifted position may
    // wrap into it, and zero times infinity must not enter the sums: there the
    // shifted operand is read from zeros.  (1 to 5 % on ragged lattices; 32 ->
    // 16 on 4 x 33x47x65: 33.6 us before, 34.3 so, 43.7 with masked fragments.)
    const bool zin = !EDGE || (z0 + lpos < nz);
    const int pair = zin ? 2*WH_Z*16 : 0;                // from one pair of rows to the next
    const int nks = EDGE ? min(WT_Y/2, (ny - y0 + 1)/2) : WT_Y/2;
    u4 rf[NF], rs[2];
    auto fetch_f = [&](int x) {
#pragma unroll
      for (int k = 0; k < NF; k++) {
	rf[k] = u4{0u, 0u, 0u, 0u};
	if (fo >= 0 && f0 + 16*k < cf) rf[k] = *reinterpret_cast<const u4a *>(fb + x*plane*cf + fo + 16*k);
      }
    };
    auto fetch_s = [&](int x) {
      const int xw = wrapi(x, nx);
#pragma unroll
      for (int k = 0; k < 2; k++) {
	rs[k] = u4{0u, 0u, 0u, 0u};
	if (so[k] >= 0) rs[k] = *reinterpret_cast<const u4a *>(sb + xw*plane*cs + so[k]);
      }
    };
    auto store_f = [&](int i) {
#pragma unroll
      for (int k = 0; k < NF; k++) *reinterpret_cast<u4 *>(&lf[i & 1][k][8*tid]) = rf[k];
    };
    auto store_s = [&](int i) {
#pragma unroll
      for (int k = 0; k < 2; k++)
	if (tid + 256*k < 2*WH_N) *reinterpret_cast<u4 *>(&ls[i & 3][8*(tid + 256*k)]) = rs[k];
    };

    // shifted plane xb - 1 + i sits in slot i & 3, fixed plane xb + i in i & 1
    fetch_s(xb - 1); store_s(0);
    fetch_s(xb); store_s(1);
    fetch_s(xb + 1); store_s(2);
    fetch_f(xb); store_f(0);
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < n; i++) {
      const bool more = (i + 1 < n);
      if (more) { fetch_s(xb + i + 2); fetch_f(xb + i + 1); }
      const uint16_t * pf = &lf[i & 1][0][lpos*16 + lch];
      const uint16_t * ps[WT_TAPS];
#pragma unroll
      for (int j = 0; j < WT_TAPS; j++) {
	const int t = min(WT_TAPS*wave + j, 26);
	const int dx = t/9, dy = (t/3)%3, dz = t%3;
	ps[j] = zin ? &ls[(i + dx) & 3][(dy*WH_Z + dz + lpos)*16 + lch] : &lz[lch];
      }
#pragma unroll 1
      for (int ks = 0; ks < nks; ks++) {
	b8 ff[NF];
#pragma unroll
	for (int k = 0; k < NF; k++)
	  ff[k] = join8(read_tr(pf + (k*WT_N + 2*ks*WT_Z)*16), read_tr(pf + (k*WT_N + (2*ks + 1)*WT_Z)*16));
	const bool second = !EDGE || (y0 + 2*ks + 1 < ny);
#pragma unroll
	for (int j = 0; j < WT_TAPS; j++) {
	  const uint16_t * p0 = ps[j] + ks*pair, * p1 = second ? p0 + WH_Z*16 : &lz[lch];
	  const b8 sf = join8(read_tr(p0), read_tr(p1));
#pragma unroll
	  for (int k = 0; k < NF; k++)
	    acc[j][k] = SHIFT_X ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(ff[k], sf, acc[j][k], 0, 0, 0)
				: __builtin_amdgcn_mfma_f32_16x16x32_bf16(sf, ff[k], acc[j][k], 0, 0, 0);
	}
      }
      // the slots written here were last read one plane ago
      if (more) { store_s(i + 3); store_f(i + 1); }
      __syncthreads();
    }
  }

  // part[block][t][co][ci]; D: lane holds rows (co) 4q + i of column (ci) r
  const int cin = SHIFT_X ? cs : cf, cout = SHIFT_X ? cf : cs;
#pragma unroll
  for (int j = 0; j < WT_TAPS; j++) {
    const int st = WT_TAPS*wave + j;
    if (st >= 27) continue;
    const int t = SHIFT_X ? st : 26 - st;
#pragma unroll
    for (int k = 0; k < NF; k++) {
      if (f0 + 16*k >= cf) continue;
      const int co = (SHIFT_X ? f0 + 16*k : s0) + 4*q, ci = (SHIFT_X ? s0 : f0 + 16*k) + r;
#pragma unroll
      for (int i = 0; i < 4; i++)
	part[(((int64_t) blockIdx.x*27 + t)*cout + co + i)*cin + ci] = acc[j][k][i];
    }
  }
}

// dw[i] (+)= sum over the blocks of part[block][i]: 64 values per block, the
// four waves take every fourth partial and their sums are added in order
__global__ void __launch_bounds__(256)
wgrad_reduce_kernel(const float * __restrict__ part, float * __restrict__ dw, int nchunk, int64_t n,
		    int accumulate) {
  __shared__ float sh[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i = (int64_t) blockIdx.x*64 + lane;
  float s = 0.0f;
  if (i < n) {
#pragma unroll 8
    for (int c = wave; c < nchunk; c += 4) s += part[(int64_t) c*n + i];
  }
  sh[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && i < n) {
    const float v = (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]);
    dw[i] = accumulate ? dw[i] + v : v;
  }
}

__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t) ((u >> 16) | 0x40u);   // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);                                              // nearest even
  return (uint16_t) (u >> 16);
}

// wf[t][co][ci] = bf16(w[t][co][ci]); wd[t][ci][co] = bf16(w[26 - t][co][ci])
__global__ void weights_prep_kernel(const float * __restrict__ w, uint16_t * __restrict__ wf,
				    uint16_t * __restrict__ wd, int cin, int cout) {
  const int64_t n = (int64_t) 27*cout*cin;
  for (int64_t i = blockIdx.x*(int64_t) blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x*blockDim.x) {
    const int ci = (int) (i % cin);
    const int co = (int) ((i / cin) % cout);
    const int t = (int) (i / ((int64_t) cin*cout));
    const uint16_t v = to_bf16(w[i]);
    if (wf) wf[i] = v;
    if (wd) wd[((int64_t) (26 - t)*cin + ci)*cout + co] = v;
  }
}

__global__ void to_bf16_kernel(const float * __restrict__ a, uint16_t * __restrict__ b, int64_t n) {
  for (int64_t i = blockIdx.x*(int64_t) blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x*blockDim.x)
    b[i] = to_bf16(a[i]);
}

int grid_for(int64_t n) {
  int64_t g = (n + 255)/256;
  return (int) (g < 8192 ? (g > 0 ? g : 1) : 8192);
}

template <int NT, int TY, int ZT, bool DMA>
void launch_conv(const uint16_t * x, const uint16_t * w, const float * bias, float * y, uint16_t * act,
		 int batch, int nx, int ny, int nz, int cin, int cout, int accumulate, hipStream_t s) {
  constexpr int X = ConvTile<TY, ZT>::X;
  const int ntx = (nx + X - 1)/X, nty = (ny + TY - 1)/TY, ntz = (nz + ZT - 1)/ZT;
  const int ntile = batch*ntx*nty*ntz, nb = (cout/16 + NT - 1)/NT;
  int nblk = CONV_BLOCKS/nb;
  if (nblk < 1) nblk = 1;
  if (nblk >= NXCD) nblk -= nblk % NXCD;
  if (nblk > ntile) nblk = ntile;
  hipLaunchKernelGGL((conv3_fwd_kernel<NT, TY, ZT, DMA>), dim3(nblk, nb), dim3(256), 0, s, x, w, bias, y, act, nx, ny, nz,
		     cin, cout, accumulate, ntx, nty, ntz, ntile);
}

}  // namespace

hipError_t launch_conv3_fwd(const uint16_t * x, const uint16_t * w, const float * bias, float * y,
			    uint16_t * act, int batch, int nx, int ny, int nz, int cin, int cout,
			    int accumulate, hipStream_t s) {
  const int nb16 = cout/16;
  const bool dma = (((uintptr_t) x | (uintptr_t) w) % 16 == 0);
  const ConvShape c = conv_shape(batch, nx, ny, nz, nb16, dma);
#define CONV_(NT, TY, ZT, DMA) \
  launch_conv<NT, TY, ZT, DMA>(x, w, bias, y, act, batch, nx, ny, nz, cin, cout, accumulate, s)
#define CONV_Z(NT, TY, DMA) do { if (c.zt == 16) CONV_(NT, TY, 16, DMA); else CONV_(NT, TY, 8, DMA); } while (0)
#define CONV_4(NT) do { if (dma) CONV_Z(NT, 4, true); else CONV_Z(NT, 4, false); } while (0)
  if (c.ty == 8) {
    if (c.nt == 2) CONV_Z(2, 8, true);
    else CONV_Z(1, 8, true);
  }
  else {
    switch (c.nt) {
    case 6: CONV_4(6); break;
    case 4: CONV_4(4); break;
    case 3: CONV_4(3); break;
    case 2: CONV_4(2); break;
    default: CONV_4(1); break;
    }
  }
#undef CONV_4
#undef CONV_Z
#undef CONV_
  return hipGetLastError();
}

int64_t conv3_wgrad_workspace(int batch, int nx, int ny, int nz, int cin, int cout) {
  return (int64_t) wgrad_plan(batch, nx, ny, nz, cin, cout).nchunk*27*cout*cin;
}

hipError_t launch_conv3_wgrad(const uint16_t * x, const uint16_t * dy, float * dw, float * work,
			      int batch, int nx, int ny, int nz, int cin, int cout, int accumulate,
			      hipStream_t s) {
  const WgradPlan w = wgrad_plan(batch, nx, ny, nz, cin, cout);
  const dim3 grid(w.nchunk, w.ns*w.nfg), block(256);
  const bool edge = (ny % WT_Y || nz % WT_Z);
#define WG_E(NF, EDGE) do { \
    if (w.shift_x) hipLaunchKernelGGL((conv3_wgrad_kernel<NF, true, EDGE>), grid, block, 0, s, dy, x, work, nx, ny, nz, \
				      cout, cin, w.ty, w.tz, w.xlen, w.xc, w.items); \
    else hipLaunchKernelGGL((conv3_wgrad_kernel<NF, false, EDGE>), grid, block, 0, s, x, dy, work, nx, ny, nz, \
			    cin, cout, w.ty, w.tz, w.xlen, w.xc, w.items); \
  } while (0)
#define WG_(NF) do { if (edge) WG_E(NF, true); else WG_E(NF, false); } while (0)
  switch (w.nf) {
  case 1: WG_(1); break;
  case 2: WG_(2); break;
  case 3: WG_(3); break;
  case 4: WG_(4); break;
  default: WG_(5); break;
  }
#undef WG_
#undef WG_E
  const int64_t n = (int64_t) 27*cout*cin;
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned) ((n + 63)/64)), dim3(256), 0, s, work, dw, w.nchunk, n,
		     accumulate);
  return hipGetLastError();
}

hipError_t launch_conv3_weights_prep(const float * w, uint16_t * wf, uint16_t * wd, int cin, int cout,
				     hipStream_t s) {
  const int64_t n = (int64_t) 27*cout*cin;
  hipLaunchKernelGGL(weights_prep_kernel, dim3(grid_for(n)), dim3(256), 0, s, w, wf, wd, cin, cout);
  return hipGetLastError();
}

hipError_t launch_to_bf16(const float * a, uint16_t * b, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_for(n)), dim3(256), 0, s, a, b, n);
  return hipGetLastError();
}

}  // namespace ldw
