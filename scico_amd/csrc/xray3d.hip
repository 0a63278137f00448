// Parallel-beam 3D X-ray projector (scico.linop.xray.XRayTransform3D) for
// gfx950.
//
// Model (scico/linop/xray/_xray3d.py:206-266): voxel (i, j, k) has centre
// x = (i + 1/2, j + 1/2, k + 1/2); for view v with float32 matrix m (2 x 4)
//   Px_r = ((m[r][0] x0 + m[r][1] x1) + m[r][2] x2) + m[r][3]
//   left = Px - 1/4,  t = min(ceil(left) - left, 1/2),  ul = floor(left)
// and the voxel splats onto the 2 x 2 detector pixels at ul with weights
// (t0 t1) 4, ((1/2 - t0) t1) 4, (t0 (1/2 - t1)) 4, ((1/2 - t0)(1/2 - t1)) 4,
// each zeroed when its pixel is off the detector.
//
// Slice mode.  When one detector axis d depends only on one volume axis s
// (the rotation axis) through the same coefficient and offset for every
// view, and that axis maps slice n exactly onto detector column n + delta
// with t_d = 1/2, the other two weights of every voxel are exactly zero and
// the transform splits into independent 2D slices that share one in-plane
// weight table.  The kernels then run with the SLICE index across the
// lanes: a wave owns 64 lanes x 4 consecutive slices, computes each
// (pixel, view) weight once in one lane, broadcasts it with readlane and
// applies it to 256 slices with float4 loads of contiguous slice rows.
// Volume and projections are used in a canonical layout with the slice
// index fastest: vol_c[p][q][s] and proj_c[v][u][s] (p < q the in-plane
// volume axes, u the in-plane detector axis); a tiled transpose converts
// to and from the caller's layout when it differs.
//
// General mode (any other geometry): the forward splats blocks of voxels
// into detector windows held in LDS and adds the windows up in a fixed
// order; the adjoint gathers per voxel from windows staged in LDS.  Both are
// deterministic.  Geometries whose windows do not fit take gathers from
// global memory.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.h"

namespace scxr {
namespace xr3d {

enum { MODE_GENERAL = 0, MODE_SLICE = 1 };

constexpr int FB = 8;   // forward: detector bins per wave
constexpr int FBL = 7;  // the same of fwd_slice16_kernel: 8 bin groups of 2 slots fill a lane row
constexpr int AR = 8;   // adjoint: pixels per wave (2 x 4 block)

struct Plan {
  int X = 0, Y = 0, Z = 0, V = 0, D0 = 0, D1 = 0;
  int mode = MODE_GENERAL;
  int sax = -1, dax = -1, delta = 0, pax = -1, qax = -1;
  int P = 0, Q = 0, S = 0, SQ = 0, U = 0;  // SQ = slice quads (slices padded to 4)
  int cpr = 32;                            // forward candidates per row
  int spg = 2;                             // forward slots per bin group
  bool slot16 = false;                     // forward by fwd_slice16_kernel
  bool vol_direct = false, proj_direct = false;
  bool adj_staged = false;                 // adjoint rows staged in LDS (adj_slice_staged_kernel)
  void* tables = nullptr;  // general mode: one block of the tables below (mats included)
  float* mats = nullptr;   // (V, 2, 4) float32
  float4* geom = nullptr;  // slice mode: (a, b, t, 0) in-plane row per view
  float* volc = nullptr;   // canonical volume workspace (P Q rows of 4 SQ floats)
  float* proja = nullptr;  // canonical projection workspace (V U 4 SQ)
  struct GenView* gview = nullptr;  // general mode: per-view gather set-up
  // general mode, windows in LDS (gen_splat_kernel, gen_adj_tile_kernel)
  bool splat = false, adj_tiled = false;
  struct SplatView* sview = nullptr;
  struct SplatItem* sitem = nullptr;
  float* zterm = nullptr;             // adjoint: m[r][2] (k + 1/2), 8 voxels at a time
  int slot = 0;                       // window floats of a splat item
  bool need_t = false;                // some view marches along z: volume copy [z][x][y]
  std::vector<int> ifirst;            // first item of every view (V + 1 entries)
  std::vector<int> chunk;             // first view of every pass over the items (and V)
  long long ws_floats = 0;            // forward workspace
};

// General-mode splat set-up of one view.  The view marches along volume axis
// a (the one whose complementary 2 x 2 minor is largest); b < c are the other
// two.  At plane t the whole lattice of voxel blocks is shifted by
// (rint(bb (t - tc)), rint(bc (t - tc))) voxels along (b, c), which keeps a
// block's projection in place, so one window of detector pixels holds all of
// the block's planes.
struct SplatView {
  int a, sb, sc, pitch, rows, first, last, pad;  // items [first, last)
  float bb, bc, tc, pad2;
  float m[8];
};
// One block of 8 sb x 8 sc voxels per plane (b from p8 + shift, c from q8 +
// shift) over planes [t0, t1), with the window at detector pixel (lo0, lo1).
struct SplatItem {
  int view, p8, q8, lo0, lo1, t0, t1, pad;
};

// General-mode forward set-up of one view.  The detector pixel (d0, d1)
// receives from the voxels whose projected centre P satisfies
// floor(P_r - 1/4) in {d_r - 1, d_r}, i.e. P_r in [d_r - 3/4, d_r + 5/4).
// The kernel marches along volume axis a (the one whose complementary
// 2 x 2 minor of the matrix is largest) and, per plane, solves for the
// other two coordinates (b, c) of the box centre with the inverse minor;
// the candidates are the nb x nc integer points of the box's bounding
// rectangle (half-extents hb, hc plus a rounding margin).
struct GenView {
  int a, nb, nc, pad;
  float i00, i01, i10, i11, hb, hc, pad2, pad3;
};

// ------------------------------------------------------------ weights --

struct Tap {
  int ul;
  float wl, wr;
};

// In-plane weights of pixel (p, q) for a slice-mode view with in-plane row
// (a, b, t): P = (a (p + 1/2) + b (q + 1/2)) + t, the two taps at ul and
// ul + 1 carry (t 1/2) 4 and ((1/2 - t) 1/2) 4 (the slice axis has
// t_d = 1/2), zeroed off the detector.
__device__ __forceinline__ Tap slice_tap(float a, float b, float t, int p, int q, int U) {
  const float xp = __fadd_rn(static_cast<float>(p), 0.5f);
  const float xq = __fadd_rn(static_cast<float>(q), 0.5f);
  const float P = __fadd_rn(__fadd_rn(__fmul_rn(a, xp), __fmul_rn(b, xq)), t);
  const float left = __fsub_rn(P, 0.25f);
  const float tt = fminf(__fsub_rn(ceilf(left), left), 0.5f);
  Tap r;
  r.ul = static_cast<int>(floorf(left));
  r.wl = __fmul_rn(__fmul_rn(tt, 0.5f), 4.0f);
  r.wr = __fmul_rn(__fmul_rn(__fsub_rn(0.5f, tt), 0.5f), 4.0f);
  if (!(r.ul >= 0 && r.ul < U)) r.wl = 0.0f;
  if (!(r.ul + 1 >= 0 && r.ul + 1 < U)) r.wr = 0.0f;
  return r;
}

// Full reference weights of voxel (i, j, k) for matrix m (general mode).
__device__ __forceinline__ void gen_weights(const float* __restrict__ m, int i, int j, int k,
                                            int D0, int D1, int ul[2], float w[4]) {
  const float x0 = __fadd_rn(static_cast<float>(i), 0.5f);
  const float x1 = __fadd_rn(static_cast<float>(j), 0.5f);
  const float x2 = __fadd_rn(static_cast<float>(k), 0.5f);
  float t[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const float* mr = m + 4 * r;
    const float P = __fadd_rn(
        __fadd_rn(__fadd_rn(__fmul_rn(mr[0], x0), __fmul_rn(mr[1], x1)), __fmul_rn(mr[2], x2)),
        mr[3]);
    const float left = __fsub_rn(P, 0.25f);
    t[r] = fminf(__fsub_rn(ceilf(left), left), 0.5f);
    ul[r] = static_cast<int>(floorf(left));
  }
  const float s0 = __fsub_rn(0.5f, t[0]), s1 = __fsub_rn(0.5f, t[1]);
  w[0] = __fmul_rn(__fmul_rn(t[0], t[1]), 4.0f);
  w[1] = __fmul_rn(__fmul_rn(s0, t[1]), 4.0f);
  w[2] = __fmul_rn(__fmul_rn(t[0], s1), 4.0f);
  w[3] = __fmul_rn(__fmul_rn(s0, s1), 4.0f);
  const bool a0 = ul[0] >= 0 && ul[0] < D0, b0 = ul[0] + 1 >= 0 && ul[0] + 1 < D0;
  const bool a1 = ul[1] >= 0 && ul[1] < D1, b1 = ul[1] + 1 >= 0 && ul[1] + 1 < D1;
  if (!(a0 && a1)) w[0] = 0.0f;
  if (!(b0 && a1)) w[1] = 0.0f;
  if (!(a0 && b1)) w[2] = 0.0f;
  if (!(b0 && b1)) w[3] = 0.0f;
}

__device__ __forceinline__ float4 fma4(float w, float4 x, float4 acc) {
  return make_float4(__builtin_fmaf(w, x.x, acc.x), __builtin_fmaf(w, x.y, acc.y),
                     __builtin_fmaf(w, x.z, acc.z), __builtin_fmaf(w, x.w, acc.w));
}

__device__ __forceinline__ int rl(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }


__device__ __forceinline__ float rlf(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// ------------------------------------------------------ slice kernels --

// Bin group and view group of a workgroup of the slice forward.
template <bool UP>
__device__ __forceinline__ void slice_block(int& bg, int& vg) {
  // Workgroup order: consecutive workgroups go to the 8 XCDs in turn; each
  // XCD is given a contiguous run of an order that takes the view groups
  // in blocks of about an eighth of them, every bin group of a block with
  // its views adjacent.  Each XCD then works on its own range of views
  // (neighbouring views' strips share most of their pixel rows, so they
  // share its L2) across all bin groups (whose strips differ in length,
  // so every XCD gets a similar share of work).  A bijection of the grid.
  // (UP: an eighth rounded up: rounded down, a run ends in the long strips of
  // one block more; fwd_slice16_kernel at 256^3 with 360 and 180 views 1256, 741
  // -> 1196, 698 us, two slots at a spacing of 0.57 with 180 and 45 views 812,
  // 447 -> 750, 418.  Three slots a bin group are 3 to 8 % slower with it at a
  // spacing of 0.35, 0 to 7 % faster or slower at 0.4 to 0.5, and keep the
  // eighth rounded down.)
  const int GX = gridDim.x, GY = gridDim.y, G = GX * GY, G8 = (G / 8) * 8;
  int L = blockIdx.y * GX + blockIdx.x;
  if (L < G8) L = (L % 8) * (G8 / 8) + L / 8;
  const int VB = UP ? (GY + 7) / 8 : max(GY / 8, 1);  // view groups per block
  const int blk = L / (GX * VB);
  const int nb = min(VB, GY - blk * VB);  // the last block may be short
  const int within = L - blk * GX * VB;
  bg = within / nb;
  vg = blk * VB + (within - bg * nb);
}

// Forward: each wave owns FB consecutive bins of one view for 256 slices
// and gathers the strip of pixels that touch them, row by row along the
// slow in-plane axis.  Lane kk of a row pass holds candidate kk of the
// row, ordered so that its bin is non-decreasing; ballots give the first
// candidate of every bin group g (ul = u0 + g, g = -1 .. FB - 1).  Each
// group has SPG static slots (a group holds at most SPG pixels: pixel
// centres are at least |f| apart along the fast axis), so the whole row is
// straight-line code apart from wave-uniform branches: every occupied
// slot's row of slices is loaded independently and accumulated into
// static registers.  For spacings below 0.67 (32 or 64 candidates a row); the
// others take fwd_slice16_kernel.
template <int CPR, int SPG>
__global__ __launch_bounds__(256) void fwd_slice_kernel(const float4* __restrict__ vol,
                                                        float4* __restrict__ proj,
                                                        const float4* __restrict__ geom, int P,
                                                        int Q, int SQ, int U, int V,
                                                        const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  constexpr int RPP = 64 / CPR;
  constexpr int BIG = INT_MAX / 2;
  const int lane = threadIdx.x & 63;
  int bg, vg;
  slice_block<(SPG < 3)>(bg, vg);
  const int v = vg * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (v >= V) return;
  const int u0 = bg * FB;
  const unsigned quad = blockIdx.z * 64 + lane;
  const bool qok = quad < static_cast<unsigned>(SQ);
  const unsigned qoff = (qok ? quad : 0u) * 16u;
  // vol holds P Q rows of SQ slice quads
  const int rowb = SQ * 16;
  const __amdgpu_buffer_rsrc_t vr = make_rsrc(vol, P * Q * rowb);
  const float4 g = geom[v];
  const float a = g.x, b = g.y, t = g.z;
  const bool qfast = fabsf(b) >= fabsf(a);
  const float f = qfast ? b : a, sc = qfast ? a : b;
  const int nslow = qfast ? P : Q, nfast = qfast ? Q : P;
  // pixel index step along the fast axis, in candidate order
  const int kstep = (f > 0.0f ? 1 : -1) * (qfast ? 1 : Q);
  const float plo = static_cast<float>(u0) - 0.75f;
  const float phi = static_cast<float>(u0 + FB) + 0.25f;
  const float rf = 1.0f / f;
  const int kk = lane % CPR;

  float4 acc[FB];
#pragma unroll
  for (int j = 0; j < FB; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);

  for (int r0 = 0; r0 < nslow; r0 += RPP) {
    const int row = r0 + lane / CPR;
    // Approximate fast-index interval of the strip in this row, widened by
    // one pixel each side; the exact bin of each candidate decides.
    const float c = sc * (static_cast<float>(row) + 0.5f) + t;
    const float ka = (plo - c) * rf - 0.5f, kb = (phi - c) * rf - 0.5f;
    const int klo = max(0, static_cast<int>(floorf(fminf(ka, kb))) - 1);
    const int khi = min(nfast - 1, static_cast<int>(ceilf(fmaxf(ka, kb))) + 1);
    const int k0 = (f > 0.0f) ? klo : khi;  // fast index of candidate 0
    const int pix0 = qfast ? row * Q + k0 : k0 * Q + row;
    int gi = BIG;
    float wl = 0.0f, wr = 0.0f;
    if (row < nslow && kk <= khi - klo) {
      const int k = (f > 0.0f) ? klo + kk : khi - kk;
      const int p = qfast ? row : k, q = qfast ? k : row;
      const Tap tp = slice_tap(a, b, t, p, q, U);
      gi = tp.ul - u0;
      wl = tp.wl;
      wr = tp.wr;
    }
#pragma unroll
    for (int rr = 0; rr < RPP; ++rr) {
      if (r0 + rr >= nslow) break;
      const int base = rr * CPR;
      const int rpix = rl(pix0, base);
      int first[FB + 2];
#pragma unroll
      for (int gg = -1; gg <= FB; ++gg) {
        const unsigned long long bal = __ballot(gi < gg);
        const int cnt =
            CPR == 64 ? __popcll(bal) : __popc(static_cast<unsigned>(bal >> (rr * CPR)));
        first[gg + 1] = base + cnt;
      }
      // Groups in chunks of GC: the loads of a chunk's occupied slots are
      // issued first, then those slots are accumulated.  Emptiness is
      // wave-uniform, so empty slots are skipped by scalar branches: they
      // issue no load (an out-of-range load would still take its cycles
      // in the texture addresser, which bounds this kernel).
      constexpr int NG = FB + 1, GC = 5;
      // byte offset of slot L: (rpix + (L - base) kstep) rowb, formed once
      // per group and stepped by kstep rowb from slot to slot
      const int rbyte = rpix * rowb, kbyte = kstep * rowb;
#pragma unroll
      for (int g0 = 0; g0 < NG; g0 += GC) {
        float4 xs[GC][SPG];
#pragma unroll
        for (int c = 0; c < GC; ++c) {
          const int gg = g0 + c - 1;
          if (gg < FB) {
            const int gbyte = rbyte + (first[gg + 1] - base) * kbyte;
#pragma unroll
            for (int k = 0; k < SPG; ++k) {
              const int L = first[gg + 1] + k;
              // an empty slot's register is never read
              if (L < first[gg + 2]) xs[c][k] = bload4(vr, qoff, gbyte + k * kbyte);
            }
          }
        }
#pragma unroll
        for (int c = 0; c < GC; ++c) {
          const int gg = g0 + c - 1;
          if (gg < FB) {
#pragma unroll
            for (int k = 0; k < SPG; ++k) {
              const int L = first[gg + 1] + k;
              if (L < first[gg + 2]) {
                const float cl = rlf(wl, L), cr = rlf(wr, L);
                if (gg >= 0) acc[gg] = fma4(cl, xs[c][k], acc[gg]);
                if (gg + 1 < FB) acc[gg + 1] = fma4(cr, xs[c][k], acc[gg + 1]);
              }
            }
          }
        }
      }
    }
  }
  if (!qok) return;
#pragma unroll
  for (int j = 0; j < FB; ++j)
    if (u0 + j < U) proj[(static_cast<size_t>(v) * U + u0 + j) * SQ + quad] = acc[j];
}

// Value of lane N of every 16-lane row, for the whole row (N a constant).
template <int N>
__device__ __forceinline__ int row_bcast(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 | N, 0xf, 0xf, true);
}
template <int N>
__device__ __forceinline__ float4 fma4_bcast(float w, float4 x, float4 acc) {
  const float wn = __int_as_float(row_bcast<N>(__float_as_int(w)));
  return fma4(wn, x, acc);
}

// Forward for in-plane spacings near 1 (at most 16 candidates in a row, two
// per bin group): the strip gather of fwd_slice_kernel with most of its scalar
// work per pixel taken out; the same sums in the same order.  A pass
// evaluates the taps of four image rows (16 candidates each) and files them
// by slot, two for each of the 8 bin groups, in an LDS table of the wave.  A
// row's 16 entries are read back into every 16-lane row, where a slot's
// weights are a row broadcast of a constant lane and one ballot tells which
// slots are taken.  Bound by the vector loads (a 16-byte load of 64 lanes for
// each pixel, view and bin group: 23 TB/s from the CUs' caches at 256^3 with
// 360 views) and their latency.  Against fwd_slice_kernel: 256^3 with 360, 180
// and 45 views 1372, 844, 405 -> 1196, 698, 323 us, 128^3 with 90 views 194 ->
// 151 us.  (Eight loads at a time, before slice_block rounded up: 1212, 787,
// 376, 171 against 1256, 741, 330, 153 us.)
// (Sharing the pixel rows of four views through LDS takes two thirds off the
// loads, but with a barrier per image row too little is in flight: 1602 us.)
__global__ __launch_bounds__(256) void fwd_slice16_kernel(
    const float4* __restrict__ vol, float4* __restrict__ proj, const float4* __restrict__ geom,
    int P, int Q, int SQ, int U, int V, const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  constexpr int BIG = INT_MAX / 2;
  __shared__ int4 table[4][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bg, vg;
  slice_block<true>(bg, vg);
  const int v = vg * 4 + w;
  if (v >= V) return;
  const int u0 = bg * FBL;
  const unsigned quad = blockIdx.z * 64 + lane;
  const bool qok = quad < static_cast<unsigned>(SQ);
  const unsigned qoff = (qok ? quad : 0u) * 16u;
  const int rowb = SQ * 16;
  const __amdgpu_buffer_rsrc_t vr = make_rsrc(vol, P * Q * rowb);
  const float4 g = geom[v];
  const float a = g.x, b = g.y, t = g.z;
  const bool qfast = fabsf(b) >= fabsf(a);
  const float f = qfast ? b : a, sc = qfast ? a : b, rf = 1.0f / f;
  const int nslow = qfast ? P : Q, nfast = qfast ? Q : P;
  const float plo = static_cast<float>(u0) - 0.75f;
  const float phi = static_cast<float>(u0 + FBL) + 0.25f;
  const int kk = lane & 15, lr = lane >> 4;
  int4* ent = table[w];

  float4 acc[FBL];
#pragma unroll
  for (int j = 0; j < FBL; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);

  for (int r0 = 0; r0 < nslow; r0 += 4) {
    // taps of rows r0 .. r0 + 3, filed by slot; the interval of the strip in
    // a row is widened by one pixel each side, the exact bin decides
    {
      const int row = r0 + lr;
      const float c = sc * (static_cast<float>(row) + 0.5f) + t;
      const float ka = (plo - c) * rf - 0.5f, kb = (phi - c) * rf - 0.5f;
      const int klo = max(0, static_cast<int>(floorf(fminf(ka, kb))) - 1);
      const int khi = min(nfast - 1, static_cast<int>(ceilf(fmaxf(ka, kb))) + 1);
      int gi = BIG, off = 0;
      float wl = 0.0f, wr = 0.0f;
      if (row < nslow && kk <= khi - klo) {
        const int k = f > 0.0f ? klo + kk : khi - kk;  // bins do not decrease with kk
        const int p = qfast ? row : k, q = qfast ? k : row;
        const Tap tp = slice_tap(a, b, t, p, q, U);
        gi = tp.ul - u0;
        wl = tp.wl;
        wr = tp.wr;
        off = (p * Q + q) * rowb;
      }
      // the second pixel of its bin group? (lane before, within the row)
      const int prev = __builtin_amdgcn_update_dpp(-BIG, gi, 0x111, 0xf, 0xf, false);
      // Lanes clear, file and read one another's entries: LDS executes a
      // wave's accesses in order, the fences keep the compiler to it.
      ent[lane] = make_int4(0, 0, 0, 0);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_wave_barrier();
      if (gi >= -1 && gi < FBL)
        ent[lr * 16 + 2 * (gi + 1) + (gi == prev)] =
            make_int4(off, __float_as_int(wl), __float_as_int(wr), 1);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
#pragma unroll 1
    for (int rr = 0; rr < min(4, nslow - r0); ++rr) {
      const int4 e = ent[rr * 16 + kk];
      const unsigned occ = static_cast<unsigned>(__builtin_amdgcn_ballot_w64(e.w != 0)) & 0xffffu;
      if (occ == 0) continue;
      const float wl = __int_as_float(e.y), wr = __int_as_float(e.z);
      // taken slots only (wave-uniform), all loads before the first sum
      float4 x[16];
      auto load = [&](auto N) {
        constexpr int n = decltype(N)::value;
        if (occ & (1u << n)) x[n % 16] = bload4(vr, qoff, rl(e.x, n));
      };
      auto use = [&](auto N) {
        constexpr int n = decltype(N)::value, gg = n / 2 - 1;
        if (occ & (1u << n)) {
          if constexpr (gg >= 0) acc[gg] = fma4_bcast<n>(wl, x[n % 16], acc[gg]);
          if constexpr (gg + 1 < FBL) acc[gg + 1] = fma4_bcast<n>(wr, x[n % 16], acc[gg + 1]);
        }
      };
#define SCXR_X3_SLOT(N) std::integral_constant<int, N>{}
      load(SCXR_X3_SLOT(0)); load(SCXR_X3_SLOT(1)); load(SCXR_X3_SLOT(2)); load(SCXR_X3_SLOT(3));
      load(SCXR_X3_SLOT(4)); load(SCXR_X3_SLOT(5)); load(SCXR_X3_SLOT(6)); load(SCXR_X3_SLOT(7));
      load(SCXR_X3_SLOT(8)); load(SCXR_X3_SLOT(9)); load(SCXR_X3_SLOT(10)); load(SCXR_X3_SLOT(11));
      load(SCXR_X3_SLOT(12)); load(SCXR_X3_SLOT(13)); load(SCXR_X3_SLOT(14)); load(SCXR_X3_SLOT(15));
      use(SCXR_X3_SLOT(0)); use(SCXR_X3_SLOT(1)); use(SCXR_X3_SLOT(2)); use(SCXR_X3_SLOT(3));
      use(SCXR_X3_SLOT(4)); use(SCXR_X3_SLOT(5)); use(SCXR_X3_SLOT(6)); use(SCXR_X3_SLOT(7));
      use(SCXR_X3_SLOT(8)); use(SCXR_X3_SLOT(9)); use(SCXR_X3_SLOT(10)); use(SCXR_X3_SLOT(11));
      use(SCXR_X3_SLOT(12)); use(SCXR_X3_SLOT(13)); use(SCXR_X3_SLOT(14)); use(SCXR_X3_SLOT(15));
#undef SCXR_X3_SLOT
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
  }
  if (!qok) return;
#pragma unroll
  for (int j = 0; j < FBL; ++j)
    if (u0 + j < U) proj[(static_cast<size_t>(v) * U + u0 + j) * SQ + quad] = acc[j];
}

// Adjoint: each wave owns a 2 x 4 block of pixels for 256 slices and walks
// the views in order, 8 at a time: lane (view j, pixel r) computes that
// pair's taps, then every (view, pixel) pair is broadcast and applied as
// acc += wl * proj_c[v][ul] + wr * proj_c[v][ul + 1] (float4 per lane).
__global__ __launch_bounds__(256) void adj_slice_kernel(const float4* __restrict__ proj,
                                                        float4* __restrict__ vol,
                                                        const float4* __restrict__ geom, int P,
                                                        int Q, int SQ, int U, int V,
                                                        const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int p0 = blockIdx.y * 4 + 2 * (w >> 1), q0 = blockIdx.x * 8 + 4 * (w & 1);
  const int quad = blockIdx.z * 64 + lane;
  const bool qok = quad < SQ;
  const unsigned qoff = (qok ? quad : 0) * 16u;
  const int rowb = SQ * 16;
  const __amdgpu_buffer_rsrc_t yr = make_rsrc(proj, V * U * rowb);
  const int r = lane & (AR - 1), jv = lane / AR;
  const int pp = p0 + (r >> 2), qq = q0 + (r & 3);
  const bool pok = pp < P && qq < Q;

  float4 acc[AR];
#pragma unroll
  for (int i = 0; i < AR; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);

  for (int v0 = 0; v0 < V; v0 += 64 / AR) {
    const int vv = v0 + jv;
    int ul = 0;
    float wl = 0.0f, wr = 0.0f;
    if (vv < V && pok) {
      const float4 g = geom[vv];
      const Tap tp = slice_tap(g.x, g.y, g.z, pp, qq, U);
      ul = tp.ul;
      wl = tp.wl;
      wr = tp.wr;
    }
    const int nv = min(64 / AR, V - v0);
    for (int j = 0; j < nv; ++j) {
      const int vb = (v0 + j) * U;
      // The bin pair (u, u + 1) is uniform across the wave; consecutive
      // pixels of a row move it by at most one bin, so rows already loaded
      // for the previous pixel are reused (scalar branches).
      auto row = [&](int u) { return bload4(yr, qoff, (vb + min(max(u, 0), U - 1)) * rowb); };
      int ucur = INT_MIN / 2;
      float4 ya = make_float4(0.f, 0.f, 0.f, 0.f), yb = ya;
#pragma unroll
      for (int i = 0; i < AR; ++i) {
        const int L = j * AR + i;
        const int u = rl(ul, L);
        const float cl = rlf(wl, L), cr = rlf(wr, L);
        if (u == ucur + 1) {
          ya = yb;
          yb = row(u + 1);
        } else if (u == ucur - 1) {
          yb = ya;
          ya = row(u);
        } else if (u != ucur) {
          ya = row(u);
          yb = row(u + 1);
        }
        ucur = u;
        acc[i] = fma4(cr, yb, fma4(cl, ya, acc[i]));
      }
    }
  }
  if (!qok) return;
#pragma unroll
  for (int i = 0; i < AR; ++i) {
    const int p = p0 + (i >> 2), q = q0 + (i & 3);
    if (p < P && q < Q) vol[(static_cast<size_t>(p) * Q + q) * SQ + quad] = acc[i];
  }
}

// Copy one 64-quad row of slices (1 KiB per wave) from global memory into
// LDS at dst without passing through registers (lane i writes dst + 16 i).
__device__ __forceinline__ void lds_row_load(__amdgpu_buffer_rsrc_t r, float4* dst, unsigned voff,
                                             int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16,
                                           voff, soff, 0, 0);
}
// Adjoint with the detector rows staged in LDS.  The workgroup's four
// waves cover a 4 x 8 pixel tile; for each view the tile's bins lie
// between those of its corner pixels (the projected centre is monotone in
// p and q, in float32 too), a range of at most ceil(3 |a| + 7 |b|) + 2
// rows.  That range is copied into LDS once per view (buffer loads that
// write LDS directly, one view ahead), and each wave reads its pixels'
// rows from there with the same reuse and accumulation order as
// adj_slice_kernel, so the results are bitwise the same; the texture data
// path then moves each row once per workgroup instead of once per wave.
// The host takes this kernel when every view's range fits ADJ_NW rows.
constexpr int ADJ_NW = 12;  // staged detector rows per view

__global__ __launch_bounds__(256) void adj_slice_staged_kernel(
    const float4* __restrict__ proj, float4* __restrict__ vol, const float4* __restrict__ geom,
    int P, int Q, int SQ, int U, int V, const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  __shared__ float4 stage[2][ADJ_NW][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pt = blockIdx.y * 4, qt = blockIdx.x * 8;  // tile origin
  const int p0 = pt + 2 * (w >> 1), q0 = qt + 4 * (w & 1);
  const int quad = blockIdx.z * 64 + lane;
  const bool qok = quad < SQ;
  const unsigned qoff = (qok ? quad : 0) * 16u;
  const int rowb = SQ * 16;
  const __amdgpu_buffer_rsrc_t yr = make_rsrc(proj, V * U * rowb);
  const int r = lane & (AR - 1), jv = lane / AR;
  const int pp = p0 + (r >> 2), qq = q0 + (r & 3);
  const bool pok = pp < P && qq < Q;

  // Staged range (first row, row count) of views c0 .. c0 + 15: lane
  // 4 k + corner computes corner `corner` of view c0 + k; a quad reduction
  // leaves the range in lane 4 k.
  auto ranges = [&](int c0, int& lo, int& n) {
    const int vv = min(c0 + (lane >> 2), V - 1), c = lane & 3;
    const float4 g = geom[vv];
    const int ul = slice_tap(g.x, g.y, g.z, pt + 3 * (c >> 1), qt + 7 * (c & 1), U).ul;
    int mn = ul, mx = ul;
    mn = min(mn, __builtin_amdgcn_mov_dpp(mn, 0xB1, 0xF, 0xF, true));  // quad_perm 1 0 3 2
    mx = max(mx, __builtin_amdgcn_mov_dpp(mx, 0xB1, 0xF, 0xF, true));
    mn = min(mn, __builtin_amdgcn_mov_dpp(mn, 0x4E, 0xF, 0xF, true));  // quad_perm 2 3 0 1
    mx = max(mx, __builtin_amdgcn_mov_dpp(mx, 0x4E, 0xF, 0xF, true));
    lo = mn;
    n = mx - mn + 2;
  };
  int lo_c, n_c, lo_n = 0, n_n = 0;  // ranges of the current and the next 16 views
  ranges(0, lo_c, n_c);
  if (V > 16) ranges(16, lo_n, n_n);
  // stage view v's rows into buffer b
  auto stage_view = [&](int v, int lo, int n, int b) {
    for (int k = w; k < n; k += 4)
      lds_row_load(yr, &stage[b][k][0], qoff, (v * U + min(max(lo + k, 0), U - 1)) * rowb);
  };

  float4 acc[AR];
#pragma unroll
  for (int i = 0; i < AR; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);

  stage_view(0, rl(lo_c, 0), rl(n_c, 0), 0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int ul = 0;  // the pixel's first detector row
  float wl = 0.0f, wr = 0.0f;
#pragma unroll 1
  for (int v = 0; v < V; ++v) {
    const int j = v & 7;
    if (j == 0) {  // taps of the wave's 8 pixels for views v .. v + 7
      const int vv = v + jv;
      ul = 0;
      wl = wr = 0.0f;
      if (vv < V) {
        const float4 g = geom[vv];
        const Tap tp = slice_tap(g.x, g.y, g.z, pp, qq, U);
        ul = tp.ul;
        wl = pok ? tp.wl : 0.0f;
        wr = pok ? tp.wr : 0.0f;
      }
    }
    // this view's range, then the next view's, from the 16-view range sets
    const int lo = rl(lo_c, 4 * (v & 15));
    if (v + 1 < V) {
      const int vn = v + 1, kn = 4 * (vn & 15);
      const bool nxt_set = (vn & 15) == 0;
      const int lon = nxt_set ? rl(lo_n, kn) : rl(lo_c, kn);
      const int nn = nxt_set ? rl(n_n, kn) : rl(n_c, kn);
      stage_view(vn, lon, nn, vn & 1);
    }
    // both rows of four pixels first (no reuse branches: LDS reads
    // are cheap), then the accumulation in adj_slice_kernel's order
    const char* sb = reinterpret_cast<const char*>(&stage[v & 1][0][0] + lane);
    // byte offset of the first staged row (64 float4 = 1 KiB apart): every
    // pixel's rows lie in [lo, lo + n), n <= ADJ_NW (the range is taken over
    // the tile's corner bins)
    const int ra = (ul - lo) * 1024;
#pragma unroll
    for (int i0 = 0; i0 < AR; i0 += 4) {
      float4 ya[4], yb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4* y = reinterpret_cast<const float4*>(sb + rl(ra, j * AR + i0 + i));
        ya[i] = y[0];
        yb[i] = y[64];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int L = j * AR + i0 + i;
        const float cl = rlf(wl, L), cr = rlf(wr, L);
        acc[i0 + i] = fma4(cr, yb[i], fma4(cl, ya[i], acc[i0 + i]));
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if ((v & 15) == 15) {  // the next 16 views become current
      lo_c = lo_n;
      n_c = n_n;
      if (v + 17 < V) ranges(v + 17, lo_n, n_n);
    }
  }
  if (!qok) return;
#pragma unroll
  for (int i = 0; i < AR; ++i) {
    const int p = p0 + (i >> 2), q = q0 + (i & 3);
    if (p < P && q < Q) vol[(static_cast<size_t>(p) * Q + q) * SQ + quad] = acc[i];
  }
}

// ----------------------------------------------------- layout kernels --

// Batched 2D transpose with offsets and zero fill:
//   out[b ob + c oc + r] = in[b ib + (r + roff) ir + (c + coff)]
// when 0 <= r + roff < Rin and 0 <= c + coff < Cin, else 0, for
// r < Rout, c < Cout.  32 x 32 tiles through LDS.
__global__ __launch_bounds__(256) void transpose_kernel(const float* __restrict__ in,
                                                        float* __restrict__ out, int Rout,
                                                        int Cout, int Rin, int Cin, int roff,
                                                        int coff, long long ib, long long ir,
                                                        long long ob, long long oc,
                                                        const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  __shared__ float tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const long long b = blockIdx.z;
  for (int rr = ty; rr < 32; rr += 8) {
    const int ri = r0 + rr + roff, ci = c0 + tx + coff;
    float val = 0.0f;
    if (ri >= 0 && ri < Rin && ci >= 0 && ci < Cin) val = in[b * ib + ri * ir + ci];
    tile[rr][tx] = val;
  }
  __syncthreads();
  for (int cc = ty; cc < 32; cc += 8) {
    const int c = c0 + cc, r = r0 + tx;
    if (c < Cout && r < Rout) out[b * ob + c * oc + r] = tile[tx][cc];
  }
}

// Row copy with a column shift and zero fill:
//   out[row os + s] = in[row is + s + off] if 0 <= s + off < Cin else 0.
__global__ __launch_bounds__(256) void shift_rows_kernel(const float* __restrict__ in,
                                                         float* __restrict__ out, long long rows,
                                                         int Cout, int Cin, int off, long long is,
                                                         long long os,
                                                         const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  const long long n = rows * Cout;
  for (long long e = blockIdx.x * 256LL + threadIdx.x; e < n; e += 256LL * gridDim.x) {
    const long long row = e / Cout;
    const int s = static_cast<int>(e - row * Cout);
    const int c = s + off;
    out[row * os + s] = (c >= 0 && c < Cin) ? in[row * is + c] : 0.0f;
  }
}

// ------------------------------------------------- general-mode kernels --

// One detector axis of a voxel: its lower pixel and the share min(ceil(left)
// - left, 1/2) that falls there (the reference's operations; P carries its
// rounding order).
__device__ __forceinline__ float axis_share(float P, int& ul) {
  const float left = __fsub_rn(P, 0.25f);
  ul = cvt_flr_i32(left);
  return fminf(__fsub_rn(ceilf(left), left), 0.5f);
}

// LDS address row * u0 + 4 * u1 + base of a window pixel in two instructions
// (row bytes in a vector register, the window's base in a scalar one); left
// to itself the compiler takes a 32-bit multiply at quarter rate.
__device__ __forceinline__ int win_offset(int u0, int row, int u1, int base) {
  int r;
  asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(u0), "v"(row), "s"(base));
  return r + (u1 << 2);
}

// Forward, general mode.  Each wave takes one item: a block of voxels that
// it splats, plane by plane, into its own window of detector pixels in LDS.
// No atomics: in one instruction the 64 lanes take an 8 x 8 lattice of
// voxels sb and sc apart, whose 2 x 2 footprints are disjoint (the host
// picks the strides so that any two of them are 2.0625 pixels apart along a
// detector axis), so a plain LDS read-modify-write is race free, and LDS
// executes a wave's accesses in order.  Every voxel's weights are evaluated
// once (a gather per detector pixel evaluates each about four times, and
// tests as many candidates again).
//
// Bound by the LDS (a read and a write of four words per voxel and view, with
// the bank conflicts of a rotated lattice: the host takes the window pitch
// that a bank model rates cheapest for the view) and by VALU issue together:
// 129 x 130 x 131 with 60 views 1872 -> 212 us (window sums 22 us of it), the
// LDS busy 90 % of the kernel, VALU issue 93 %.
template <int A, int SB_, int SC_>
__device__ __forceinline__ void splat_item(__amdgpu_buffer_rsrc_t vr, const SplatView& g,
                                           const SplatItem& it, int wbase, int nb, int nc,
                                           int sta, int stb) {
  constexpr int B = A == 0 ? 1 : 0, C = A == 2 ? 1 : 2;
  constexpr bool FIX = SB_ > 0;
  const int SB = FIX ? SB_ : g.sb, SC = FIX ? SC_ : g.sc;
  const int lane = threadIdx.x & 63;
  const int ob = SB * (lane >> 3), oc = SC * (lane & 7);
  const float ma0 = g.m[A], ma1 = g.m[4 + A], mb0 = g.m[B], mb1 = g.m[4 + B], mc0 = g.m[C],
              mc1 = g.m[4 + C], mt0 = g.m[3], mt1 = g.m[7];
  int row = 4 * g.pitch;  // bytes of a window row
  const int base = wbase - (it.lo0 * row + 4 * it.lo1);
  asm("" : "+v"(row));
  auto shift = [&](float beta, int t) {
    return __builtin_amdgcn_readfirstlane(
        static_cast<int>(rintf(__fmul_rn(beta, __fsub_rn(static_cast<float>(t), g.tc)))));
  };
  // byte offset of voxel (t, b, c): an index off the volume moves it past
  // the buffer's end (at most 2^30 bytes), where loads return zero
  auto row_off = [&](int t, int b) {
    return static_cast<unsigned>(b) < static_cast<unsigned>(nb)
               ? static_cast<unsigned>(t * sta + b * stb) * 4u
               : 0x80000000u;
  };
  auto col_off = [&](int c) {
    return static_cast<unsigned>(c) < static_cast<unsigned>(nc) ? static_cast<unsigned>(c) * 4u
                                                                : 0x40000000u;
  };
  // P_r = ((m_r0 x0 + m_r1 x1) + m_r2 x2) + m_r3 in the reference's order:
  // pab holds the terms of the march axis and b where both come before c
  // (A < 2), else b's term alone, and pa is added last
  auto voxel = [&](float x, float pab0, float pab1, float pc0, float pc1, float pa0, float pa1) {
    float P0 = __fadd_rn(pab0, pc0), P1 = __fadd_rn(pab1, pc1);
    if (A == 2) {
      P0 = __fadd_rn(P0, pa0);
      P1 = __fadd_rn(P1, pa1);
    }
    int u0, u1;
    const float w0 = axis_share(__fadd_rn(P0, mt0), u0), w1 = axis_share(__fadd_rn(P1, mt1), u1);
    // the factor 4 of the weights (an exact scaling) is applied to the sums
    const float v0 = __fsub_rn(0.5f, w0);
    const float xl = __fmul_rn(w1, x), xr = __fmul_rn(__fsub_rn(0.5f, w1), x);
    const int at = win_offset(u0, row, u1, base);
    LdsFloat* q = lds_at(at);
    LdsFloat* r = lds_at(at + row);
    const float a00 = q[0], a01 = q[1], a10 = r[0], a11 = r[1];
    q[0] = fmaf(w0, xl, a00);
    q[1] = fmaf(w0, xr, a01);
    r[0] = fmaf(v0, xl, a10);
    r[1] = fmaf(v0, xr, a11);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
  };
  if constexpr (FIX) {
    float nxt[SB_][SC_];
    const unsigned lane_off = static_cast<unsigned>(ob * stb + oc) * 4u;
    auto load = [&](int t, int sb, int sc) {
      const int bu = it.p8 + sb, cu = it.q8 + sc;
      if (bu >= 0 && bu + 8 * SB_ <= nb && cu >= 0 && cu + 8 * SC_ <= nc) {
        // inside the volume: a scalar offset per row, the lane's own offset
#pragma unroll
        for (int rb = 0; rb < SB_; ++rb)
#pragma unroll
          for (int rc = 0; rc < SC_; ++rc)
            nxt[rb][rc] =
                bload1(vr, lane_off + 4u * rc, (t * sta + (bu + rb) * stb + cu) * 4);
        return;
      }
      const int b0 = bu + ob, c0 = cu + oc;
      unsigned co[SC_];
#pragma unroll
      for (int rc = 0; rc < SC_; ++rc) co[rc] = col_off(c0 + rc);
#pragma unroll
      for (int rb = 0; rb < SB_; ++rb) {
        const unsigned ro = row_off(t, b0 + rb);
#pragma unroll
        for (int rc = 0; rc < SC_; ++rc) nxt[rb][rc] = bload1(vr, ro + co[rc], 0);
      }
    };
    int sb = shift(g.bb, it.t0), sc = shift(g.bc, it.t0);
    load(it.t0, sb, sc);
#pragma unroll 1
    for (int t = it.t0; t < it.t1; ++t) {
      float cur[SB_][SC_];
#pragma unroll
      for (int rb = 0; rb < SB_; ++rb)
#pragma unroll
        for (int rc = 0; rc < SC_; ++rc) cur[rb][rc] = nxt[rb][rc];
      const float xb0 = static_cast<float>(it.p8 + sb + ob);
      const float xc0 = static_cast<float>(it.q8 + sc + oc);
      if (t + 1 < it.t1) {
        sb = shift(g.bb, t + 1);
        sc = shift(g.bc, t + 1);
        load(t + 1, sb, sc);
      }
      const float xa = __fadd_rn(static_cast<float>(t), 0.5f);
      const float pa0 = __fmul_rn(ma0, xa), pa1 = __fmul_rn(ma1, xa);
      float pc0[SC_], pc1[SC_];
#pragma unroll
      for (int rc = 0; rc < SC_; ++rc) {
        const float xc = __fadd_rn(xc0, static_cast<float>(rc) + 0.5f);
        pc0[rc] = __fmul_rn(mc0, xc);
        pc1[rc] = __fmul_rn(mc1, xc);
      }
#pragma unroll
      for (int rb = 0; rb < SB_; ++rb) {
        const float xb = __fadd_rn(xb0, static_cast<float>(rb) + 0.5f);
        float pb0 = __fmul_rn(mb0, xb), pb1 = __fmul_rn(mb1, xb);
        if (A < 2) {
          pb0 = __fadd_rn(pa0, pb0);
          pb1 = __fadd_rn(pa1, pb1);
        }
#pragma unroll
        for (int rc = 0; rc < SC_; ++rc)
          voxel(cur[rb][rc], pb0, pb1, pc0[rc], pc1[rc], pa0, pa1);
      }
    }
  } else {
    for (int t = it.t0; t < it.t1; ++t) {
      const int b0 = it.p8 + shift(g.bb, t) + ob, c0 = it.q8 + shift(g.bc, t) + oc;
      const float xa = __fadd_rn(static_cast<float>(t), 0.5f);
      const float pa0 = __fmul_rn(ma0, xa), pa1 = __fmul_rn(ma1, xa);
      for (int rb = 0; rb < SB; ++rb) {
        const float xb = __fadd_rn(static_cast<float>(b0 + rb), 0.5f);
        const unsigned ro = row_off(t, b0 + rb);
        float pb0 = __fmul_rn(mb0, xb), pb1 = __fmul_rn(mb1, xb);
        if (A < 2) {
          pb0 = __fadd_rn(pa0, pb0);
          pb1 = __fadd_rn(pa1, pb1);
        }
        for (int rc = 0; rc < SC; ++rc) {
          const float x = bload1(vr, ro + col_off(c0 + rc), 0);
          const float xc = __fadd_rn(static_cast<float>(c0 + rc), 0.5f);
          voxel(x, pb0, pb1, __fmul_rn(mc0, xc), __fmul_rn(mc1, xc), pa0, pa1);
        }
      }
    }
  }
}

// Strides 3 x 3 (a minor near a rotation, the usual case) are compiled;
// other strides take run-time loops.
__global__ __launch_bounds__(256) void gen_splat_kernel(const float* __restrict__ vol,
                                                        const float* __restrict__ volt,
                                                        float* __restrict__ parts,
                                                        const SplatView* __restrict__ views,
                                                        const SplatItem* __restrict__ items,
                                                        int item0, int item1, int slot, int X,
                                                        int Y, int Z,
                                                        const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  extern __shared__ float splat_win[];  // [4 waves][slot]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = item0 + blockIdx.x * 4 + wave;
  if (i >= item1) return;  // waves are independent: no workgroup barrier below
  const SplatItem it = items[i];
  const SplatView g = views[it.view];
  float* win = splat_win + wave * slot;
  const int n = g.rows * g.pitch;
  for (int e = lane; e < n; e += 64) win[e] = 0.0f;
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_wave_barrier();
  const __amdgpu_buffer_rsrc_t vr = make_rsrc(g.a == 2 ? volt : vol, X * Y * Z * 4);
  const bool fix = g.sb == 3 && g.sc == 3;
  const int wbase = lds_address(splat_win) + wave * slot * 4;
  if (g.a == 0) {
    if (fix)
      splat_item<0, 3, 3>(vr, g, it, wbase, Y, Z, Y * Z, Z);
    else
      splat_item<0, 0, 0>(vr, g, it, wbase, Y, Z, Y * Z, Z);
  } else if (g.a == 1) {
    if (fix)
      splat_item<1, 3, 3>(vr, g, it, wbase, X, Z, Z, Y * Z);
    else
      splat_item<1, 0, 0>(vr, g, it, wbase, X, Z, Z, Y * Z);
  } else {
    if (fix)
      splat_item<2, 3, 3>(vr, g, it, wbase, X, Y, X * Y, Y);
    else
      splat_item<2, 0, 0>(vr, g, it, wbase, X, Y, X * Y, Y);
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_wave_barrier();
  float* dst = parts + static_cast<size_t>(i - item0) * slot;
  for (int e = lane; e < n; e += 64) dst[e] = __fmul_rn(4.0f, win[e]);
}

// Detector pixel = sum of the windows that cover it, in item order.  One
// workgroup per 16 x 16 pixels of a view; each wave finds the items that
// reach its 16 x 4 pixels by ballots over the view's items.
__global__ __launch_bounds__(256) void gen_splat_sum_kernel(const float* __restrict__ parts,
                                                            float* __restrict__ proj,
                                                            const SplatView* __restrict__ views,
                                                            const SplatItem* __restrict__ items,
                                                            int view0, int item0, int slot, int D0,
                                                            int D1,
                                                            const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  const int v = view0 + blockIdx.z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = blockIdx.y * 16 + wave * 4, c0 = blockIdx.x * 16;
  const int d0 = r0 + (lane >> 4), d1 = c0 + (lane & 15);
  const int rows = views[v].rows, pitch = views[v].pitch;
  const int first = views[v].first, last = views[v].last;
  float sum = 0.0f;
  for (int i0 = first; i0 < last; i0 += 64) {
    const int i = i0 + lane;
    int lo0 = 0, lo1 = 0;
    bool hit = false;
    if (i < last) {
      lo0 = items[i].lo0;
      lo1 = items[i].lo1;
      hit = lo0 < r0 + 4 && lo0 + rows > r0 && lo1 < c0 + 16 && lo1 + pitch > c0;
    }
    unsigned long long todo = __ballot(hit);
    while (todo) {  // four windows at a time: their loads are in flight together
      float x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        x[q] = 0.0f;
        if (todo) {
          const int k = __builtin_ctzll(todo);
          todo &= todo - 1;
          const int r = d0 - rl(lo0, k), c = d1 - rl(lo1, k);
          if (static_cast<unsigned>(r) < static_cast<unsigned>(rows) &&
              static_cast<unsigned>(c) < static_cast<unsigned>(pitch))
            x[q] = parts[static_cast<size_t>(i0 + k - item0) * slot + r * pitch + c];
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) sum = __fadd_rn(sum, x[q]);
    }
  }
  if (d0 < D0 && d1 < D1) proj[(static_cast<size_t>(v) * D0 + d0) * D1 + d1] = sum;
}

// Adjoint, general mode.  Each wave takes an 8 x 8 x 8 block of voxels (lane
// (i, j), eight k per lane) and walks its share of the views: the 16 x 16
// detector pixels that the block can reach are copied into the wave's LDS
// window (zero off the detector, so the taps need no range tests; the next
// view's pixels are in flight meanwhile), and every voxel reads its four
// taps there.  The terms m[r][2] (k + 1/2) are uniform over the wave and
// come from a table by scalar loads; (m[r][0] x0 + m[r][1] x1) serves a
// lane's eight voxels: about 31 vector instructions per voxel and view with
// the staging, the bound (97 % of the issue rate), against 130 for taps
// clamped and read from global memory per voxel: 129 x 130 x 131 with 60
// views 457 -> 84 us.
constexpr int GA = 8, GWIN = 16, GPITCH = 17;

__global__ __launch_bounds__(256) void gen_adj_tile_kernel(
    const float* __restrict__ proj, float* __restrict__ vol, const float* __restrict__ mats,
    const float* __restrict__ zterm, int X, int Y, int Z, int V, int D0, int D1, int vs,
    const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  __shared__ float wins[4][GWIN * GPITCH];
  __shared__ float share[3][GA][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nti = (X + GA - 1) / GA, ntj = (Y + GA - 1) / GA, ntk = (Z + GA - 1) / GA;
  const int tile = blockIdx.x * (4 / vs) + wave / vs, vg = wave % vs;
  const bool live = tile < nti * ntj * ntk;
  const int tk = live ? tile % ntk : 0, tj = live ? (tile / ntk) % ntj : 0,
            ti = live ? tile / (ntk * ntj) : 0;
  const int i = ti * GA + (lane >> 3), j = tj * GA + (lane & 7), k0 = tk * GA;
  const float x0 = __fadd_rn(static_cast<float>(i), 0.5f);
  const float x1 = __fadd_rn(static_cast<float>(j), 0.5f);
  float* win = wins[wave];
  const int wbase = lds_address(&wins[0][0]) + wave * GWIN * GPITCH * 4;
  int row = 4 * GPITCH;
  asm("" : "+v"(row));
  const int chunk = (V + vs - 1) / vs;
  const int vb = live ? min(V, vg * chunk) : 0, ve = live ? min(V, vb + chunk) : 0;
  float acc[GA];
#pragma unroll
  for (int k = 0; k < GA; ++k) acc[k] = 0.0f;
  // window origins of views [c0, c0 + 64), one per lane: the lower bound of
  // both detector indices over the block (its lowest corner), with a margin
  // far above the float32 rounding of the projected centres
  int olo0 = 0, olo1 = 0;
  auto origins = [&](int c0) {
    const float* m = mats + 8 * min(c0 + lane, V - 1);
    int o[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const float* mr = m + 4 * r;
      const float c = static_cast<float>(GA - 1);
      const float xa = static_cast<float>(ti * GA) + (mr[0] < 0.0f ? c : 0.0f) + 0.5f;
      const float xb = static_cast<float>(tj * GA) + (mr[1] < 0.0f ? c : 0.0f) + 0.5f;
      const float xc = static_cast<float>(tk * GA) + (mr[2] < 0.0f ? c : 0.0f) + 0.5f;
      const float lo = mr[0] * xa + mr[1] * xb + mr[2] * xc + mr[3] - 0.26f;
      o[r] = static_cast<int>(floorf(lo));
    }
    olo0 = o[0];
    olo1 = o[1];
  };
  float nxt[4];
  auto fetch = [&](int v, int lo0, int lo1) {
    const __amdgpu_buffer_rsrc_t yr =
        make_rsrc(proj + static_cast<size_t>(v) * D0 * D1, D0 * D1 * 4);
    // rows off the detector fall outside the view's buffer; columns off it
    // are moved there (rows and columns are below 2^14)
    const int row = lo0 + (lane >> 4), col = lo1 + (lane & 15);
    const unsigned off = static_cast<unsigned>(col) < static_cast<unsigned>(D1)
                             ? static_cast<unsigned>(row * D1 + col) * 4u
                             : 0x80000000u;
#pragma unroll
    for (int q = 0; q < 4; ++q) nxt[q] = bload1(yr, off + static_cast<unsigned>(q * 16 * D1), 0);
  };
  if (vb < ve) {
    origins(vb);
    fetch(vb, rl(olo0, 0), rl(olo1, 0));
  }
#pragma unroll 1
  for (int v = vb; v < ve; ++v) {
    const int q6 = (v - vb) & 63;
    const int lo0 = rl(olo0, q6), lo1 = rl(olo1, q6);
#pragma unroll
    for (int q = 0; q < 4; ++q) win[((lane >> 4) + 4 * q) * GPITCH + (lane & 15)] = nxt[q];
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
    if (v + 1 < ve) {
      if (q6 == 63) origins(v + 1);
      const int n6 = (v + 1 - vb) & 63;
      fetch(v + 1, rl(olo0, n6), rl(olo1, n6));
    }
    const float* m = mats + 8 * v;
    const float* zt = zterm + (static_cast<size_t>(v) * ntk + tk) * (2 * GA);
    const float a0 = __fadd_rn(__fmul_rn(m[0], x0), __fmul_rn(m[1], x1));
    const float a1 = __fadd_rn(__fmul_rn(m[4], x0), __fmul_rn(m[5], x1));
    const float t0 = m[3], t1 = m[7];
    const int base = wbase - (lo0 * GPITCH + lo1) * 4;
#pragma unroll
    for (int k = 0; k < GA; ++k) {
      int u0, u1;
      const float w0 = axis_share(__fadd_rn(__fadd_rn(a0, zt[k]), t0), u0);
      const float w1 = axis_share(__fadd_rn(__fadd_rn(a1, zt[GA + k]), t1), u1);
      const LdsFloat* y = lds_at(win_offset(u0, row, u1, base));
      // the factor 4 of the weights (an exact scaling) is applied to the sums
      const float v0 = __fsub_rn(0.5f, w0), v1 = __fsub_rn(0.5f, w1);
      const float left = fmaf(v0, y[GPITCH], __fmul_rn(w0, y[0]));
      const float right = fmaf(v0, y[GPITCH + 1], __fmul_rn(w0, y[1]));
      acc[k] = fmaf(v1, right, fmaf(w1, left, acc[k]));
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
  }
  if (vs > 1) {  // add the other waves' shares of the views, in order
    const int slot0 = (wave / vs) * (vs - 1);
    if (vg > 0)
#pragma unroll
      for (int k = 0; k < GA; ++k) share[slot0 + vg - 1][k][lane] = acc[k];
    __syncthreads();
    if (vg > 0) return;
    for (int g = 1; g < vs; ++g)
#pragma unroll
      for (int k = 0; k < GA; ++k) acc[k] = __fadd_rn(acc[k], share[slot0 + g - 1][k][lane]);
  }
  if (!live || i >= X || j >= Y) return;
#pragma unroll
  for (int k = 0; k < GA; ++k) acc[k] = __fmul_rn(4.0f, acc[k]);
  float* out = vol + (static_cast<size_t>(i) * Y + j) * Z + k0;
  if (Z % 4 == 0 && k0 + GA <= Z && (reinterpret_cast<uintptr_t>(vol) & 15) == 0) {
    reinterpret_cast<float4*>(out)[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    reinterpret_cast<float4*>(out)[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
  } else {
#pragma unroll
    for (int k = 0; k < GA; ++k)
      if (k0 + k < Z) out[k] = acc[k];
  }
}

// The gathers below read global memory; they take what the windows cannot
// hold (projected voxels far apart on the detector, or nearly on one line).

__global__ __launch_bounds__(256) void gen_adj_kernel(const float* __restrict__ proj,
                                                      float* __restrict__ vol,
                                                      const float* __restrict__ mats, int X,
                                                      int Y, int Z, int V, int D0, int D1,
                                                      const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  const long long n = static_cast<long long>(X) * Y * Z;
  const long long e = blockIdx.x * 256LL + threadIdx.x;
  if (e >= n) return;
  const int k = static_cast<int>(e % Z), j = static_cast<int>((e / Z) % Y),
            i = static_cast<int>(e / (static_cast<long long>(Y) * Z));
  float acc = 0.0f;
  for (int v = 0; v < V; ++v) {
    int ul[2];
    float w[4];
    gen_weights(mats + 8 * v, i, j, k, D0, D1, ul, w);
    const float* y = proj + static_cast<size_t>(v) * D0 * D1;
    const int a0 = min(max(ul[0], 0), D0 - 1), b0 = min(max(ul[0] + 1, 0), D0 - 1);
    const int a1 = min(max(ul[1], 0), D1 - 1), b1 = min(max(ul[1] + 1, 0), D1 - 1);
    // _xray3d.py:200-203, in order
    acc = __fadd_rn(acc, __fmul_rn(y[a0 * D1 + a1], w[0]));
    acc = __fadd_rn(acc, __fmul_rn(y[b0 * D1 + a1], w[1]));
    acc = __fadd_rn(acc, __fmul_rn(y[a0 * D1 + b1], w[2]));
    acc = __fadd_rn(acc, __fmul_rn(y[b0 * D1 + b1], w[3]));
  }
  vol[e] = acc;
}

// General-mode forward as a gather: one thread per (view, detector pixel)
// sums w * vol over the voxels whose reference taps land on the pixel, the
// weights evaluated per voxel exactly as gen_weights does.  Deterministic,
// no atomics.
template <int A>
__device__ __forceinline__ float gen_gather(const float* __restrict__ vol,
                                            const float* __restrict__ m, const GenView& g,
                                            int X, int Y, int Z, int d0, int d1, int t0,
                                            int t1) {
  constexpr int B = A == 0 ? 1 : 0, C = A == 2 ? 1 : 2;
  const int dims[3] = {X, Y, Z};
  const float r0 = __fsub_rn(__fadd_rn(static_cast<float>(d0), 0.25f), m[3]);
  const float r1 = __fsub_rn(__fadd_rn(static_cast<float>(d1), 0.25f), m[7]);
  float acc = 0.0f;
  for (int t = t0; t < t1; ++t) {
    const float xa = static_cast<float>(t) + 0.5f;
    const float q0 = r0 - m[A] * xa, q1 = r1 - m[4 + A] * xa;
    const float cb = g.i00 * q0 + g.i01 * q1, cc = g.i10 * q0 + g.i11 * q1;
    const int lob = static_cast<int>(ceilf(cb - g.hb - 0.5f));
    const int loc = static_cast<int>(ceilf(cc - g.hc - 0.5f));
    for (int kb = 0; kb < g.nb; ++kb) {
      const int ib = lob + kb;
      if (ib < 0 || ib >= dims[B]) continue;
      // Within the row the contributing voxels satisfy, for both detector
      // axes r, P_r - (d_r + 1/4) = m_r[B] xb + m_r[C] xc - q_r in [-1, 1):
      // an interval of xc per axis.  Their intersection, widened by 0.01 in
      // P (far above this estimate's float32 error), bounds the
      // candidates; the exact taps below still decide.
      const float xb = static_cast<float>(ib) + 0.5f;
      int c0 = max(loc, 0), c1 = min(loc + g.nc - 1, dims[C] - 1);
      {
        const float s0 = m[B] * xb - q0, s1 = m[4 + B] * xb - q1;
        const float e0 = m[C], e1 = m[4 + C];
        const float cmax = static_cast<float>(dims[C]);
        if (fabsf(e0) > 1e-6f) {
          const float u = (-1.01f - s0) / e0, w = (1.01f - s0) / e0;
          // clamped to the volume before the conversions (|u|, |w| can be huge)
          c0 = max(c0, static_cast<int>(ceilf(fmaxf(fminf(u, w) - 0.5f, -1.0f))));
          c1 = min(c1, static_cast<int>(floorf(fminf(fmaxf(u, w) - 0.5f, cmax))));
        } else if (!(fabsf(s0) <= 1.01f)) {
          continue;
        }
        if (fabsf(e1) > 1e-6f) {
          const float u = (-1.01f - s1) / e1, w = (1.01f - s1) / e1;
          // clamped to the volume before the conversions (|u|, |w| can be huge)
          c0 = max(c0, static_cast<int>(ceilf(fmaxf(fminf(u, w) - 0.5f, -1.0f))));
          c1 = min(c1, static_cast<int>(floorf(fminf(fmaxf(u, w) - 0.5f, cmax))));
        } else if (!(fabsf(s1) <= 1.01f)) {
          continue;
        }
      }
      for (int ic = c0; ic <= c1; ++ic) {
        const int i = A == 0 ? t : (B == 0 ? ib : ic);
        const int j = A == 1 ? t : (B == 1 ? ib : ic);
        const int k = A == 2 ? t : (C == 2 ? ic : ib);
        const float x0 = __fadd_rn(static_cast<float>(i), 0.5f);
        const float x1 = __fadd_rn(static_cast<float>(j), 0.5f);
        const float x2 = __fadd_rn(static_cast<float>(k), 0.5f);
        float tr[2];
        int ul[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float* mr = m + 4 * r;
          const float P = __fadd_rn(__fadd_rn(__fadd_rn(__fmul_rn(mr[0], x0),
                                                        __fmul_rn(mr[1], x1)),
                                              __fmul_rn(mr[2], x2)),
                                    mr[3]);
          const float left = __fsub_rn(P, 0.25f);
          tr[r] = fminf(__fsub_rn(ceilf(left), left), 0.5f);
          ul[r] = static_cast<int>(floorf(left));
        }
        const bool h0 = ul[0] == d0, l0 = ul[0] == d0 - 1;
        const bool h1 = ul[1] == d1, l1 = ul[1] == d1 - 1;
        if ((h0 || l0) && (h1 || l1)) {
          const float f0 = h0 ? tr[0] : __fsub_rn(0.5f, tr[0]);
          const float f1 = h1 ? tr[1] : __fsub_rn(0.5f, tr[1]);
          const float w = __fmul_rn(__fmul_rn(f0, f1), 4.0f);
          acc = __builtin_fmaf(w, vol[(static_cast<size_t>(i) * Y + j) * Z + k], acc);
        }
      }
    }
  }
  return acc;
}

// One workgroup per (view, 64 consecutive pixels): wave w of GEN_W takes
// planes [w n / GEN_W, (w + 1) n / GEN_W) of the march axis and the
// partial sums are added in wave order.  Few views give few pixel groups,
// so the planes are split over 16 waves to fill the chip (4 waves: 148 us,
// 16: 120 us on the three-view 129 x 130 x 131 comparison geometry).
constexpr int GEN_W = 16;
__global__ __launch_bounds__(64 * GEN_W) void gen_fwd_kernel(const float* __restrict__ vol,
                                                          float* __restrict__ proj,
                                                          const float* __restrict__ mats,
                                                          const GenView* __restrict__ gv,
                                                          int X, int Y, int Z, int D0, int D1,
                                                          const int32_t* __restrict__ pred) {
  if (pred_off(pred)) return;
  __shared__ float part[GEN_W][64];
  const int v = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long e = blockIdx.x * 64LL + lane;
  const bool ok = e < static_cast<long long>(D0) * D1;
  const int d0 = ok ? static_cast<int>(e / D1) : 0, d1 = ok ? static_cast<int>(e % D1) : 0;
  const float* m = mats + 8 * v;
  const GenView g = gv[v];
  const int n = g.a == 0 ? X : (g.a == 1 ? Y : Z);
  const int t0 = (wave * n) / GEN_W, t1 = ((wave + 1) * n) / GEN_W;
  float acc = 0.0f;
  if (ok) {
    if (g.a == 0)
      acc = gen_gather<0>(vol, m, g, X, Y, Z, d0, d1, t0, t1);
    else if (g.a == 1)
      acc = gen_gather<1>(vol, m, g, X, Y, Z, d0, d1, t0, t1);
    else
      acc = gen_gather<2>(vol, m, g, X, Y, Z, d0, d1, t0, t1);
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && ok) {
    float sum = part[0][lane];
    for (int w = 1; w < GEN_W; ++w) sum = __fadd_rn(sum, part[w][lane]);
    proj[static_cast<size_t>(v) * D0 * D1 + e] = sum;
  }
}

// Reference weight arrays of one view: ul (2, X, Y, Z) int32 and
// w (4, X, Y, Z) float32 (_xray3d.py:206-266), computed by the same device
// functions that the projection kernels use.
__global__ __launch_bounds__(256) void weights_kernel(Plan p, int view, int32_t* __restrict__ ul,
                                                      float* __restrict__ w) {
  const long long n = static_cast<long long>(p.X) * p.Y * p.Z;
  const long long e = blockIdx.x * 256LL + threadIdx.x;
  if (e >= n) return;
  const int idx[3] = {static_cast<int>(e / (static_cast<long long>(p.Y) * p.Z)),
                      static_cast<int>((e / p.Z) % p.Y), static_cast<int>(e % p.Z)};
  int u[2];
  float ww[4];
  if (p.mode == MODE_SLICE) {
    const float4 g = p.geom[view];
    const Tap tp = slice_tap(g.x, g.y, g.z, idx[p.pax], idx[p.qax], p.U);
    const int col = idx[p.sax] + p.delta;
    const int Dd = p.dax == 0 ? p.D0 : p.D1;
    const bool cok = col >= 0 && col < Dd;
    u[p.dax] = col;
    u[1 - p.dax] = tp.ul;
    // taps (ul0, ul1), (ul0 + 1, ul1), (ul0, ul1 + 1), (ul0 + 1, ul1 + 1)
    ww[0] = cok ? tp.wl : 0.0f;
    ww[3] = 0.0f;
    if (p.dax == 1) {
      ww[1] = cok ? tp.wr : 0.0f;
      ww[2] = 0.0f;
    } else {
      ww[1] = 0.0f;
      ww[2] = cok ? tp.wr : 0.0f;
    }
  } else {
    gen_weights(p.mats + 8 * view, idx[0], idx[1], idx[2], p.D0, p.D1, u, ww);
  }
  ul[e] = u[0];
  ul[n + e] = u[1];
  for (int t = 0; t < 4; ++t) w[t * n + e] = ww[t];
}

// ------------------------------------------------------------- host --

static float mat(const std::vector<float>& m, int v, int r, int c) { return m[8 * v + 4 * r + c]; }

// Slice decomposition test for slice axis sax and detector axis dax, all in
// the reference's float32 arithmetic.
static bool try_slice(Plan& p, const std::vector<float>& m, int sax, int dax) {
  const int e = 1 - dax;
  const int shape[3] = {p.X, p.Y, p.Z};
  const int S = shape[sax];
  int delta = 0;
  for (int v = 0; v < p.V; ++v) {
    for (int a = 0; a < 3; ++a)
      if (a != sax && mat(m, v, dax, a) != 0.0f) return false;
    if (mat(m, v, e, sax) != 0.0f) return false;
    // Every view must map slice s to column s + delta with t_d = 1/2,
    // evaluated as the reference does: ((0 + m x) + 0) + t up to exact zeros.
    const float ms = mat(m, v, dax, sax), td = mat(m, v, dax, 3);
    if (!(ms != 0.0f)) return false;
    for (int s = 0; s < S; ++s) {
      const float x = static_cast<float>(s) + 0.5f;
      const float prod = ms * x;
      const float P = prod + td;
      const float left = P - 0.25f;
      const float ce = std::ceil(left);
      const float tt = std::fmin(ce - left, 0.5f);
      if (tt != 0.5f) return false;
      const int d = static_cast<int>(std::floor(left)) - s;
      if (v == 0 && s == 0)
        delta = d;
      else if (d != delta)
        return false;
    }
  }
  int pax = -1, qax = -1;
  for (int a = 0; a < 3; ++a)
    if (a != sax) (pax < 0 ? pax : qax) = a;
  float fmin = INFINITY;
  for (int v = 0; v < p.V; ++v) {
    const float a = mat(m, v, e, pax), b = mat(m, v, e, qax), t = mat(m, v, e, 3);
    if (!std::isfinite(a) || !std::isfinite(b) || !std::isfinite(t)) return false;
    fmin = std::fmin(fmin, std::fmax(std::fabs(a), std::fabs(b)));
  }
  if (!(fmin > 0.0f)) return false;
  const double need = std::ceil((FB + 1) / static_cast<double>(fmin)) + 6.0;
  if (need > 64.0) return false;
  p.cpr = need <= 32.0 ? 32 : 64;
  // pixels of one bin group (left in [g, g + 1)) along the fast axis
  const double spg = std::ceil(1.0 / static_cast<double>(fmin) + 0.01);
  if (spg > 3.0) return false;
  p.spg = spg <= 2.0 ? 2 : 3;
  // 16 candidates hold a strip of FBL + 1 bins, rounded outwards and widened
  // by a pixel each side
  p.slot16 = (FBL + 1) / static_cast<double>(fmin) < 11.99;
  if (p.slot16) p.cpr = 16;
  p.mode = MODE_SLICE;
  p.sax = sax;
  p.dax = dax;
  p.delta = delta;
  p.pax = pax;
  p.qax = qax;
  p.P = shape[pax];
  p.Q = shape[qax];
  p.S = S;
  p.SQ = (S + 3) / 4;
  p.U = e == 0 ? p.D0 : p.D1;
  // The forward reads the canonical (slice-fastest) volume through one
  // buffer resource; buffer offsets are 32-bit.
  p.vol_direct = false;
  const double rowb = 16.0 * ((S + 3) / 4);
  if (static_cast<double>(p.P) * p.Q * rowb >= 2147483647.0) return false;
  const int Ue = e == 0 ? p.D0 : p.D1;
  if (static_cast<double>(p.V) * Ue * rowb >= 2147483647.0) return false;
  p.proj_direct = dax == 1 && delta == 0 && p.D1 == S && S % 4 == 0;
  return true;
}

void destroy(Plan& p) {
  if (p.mats && !p.tables) (void)hipFree(p.mats);
  if (p.tables) (void)hipFree(p.tables);
  p.tables = nullptr;
  if (p.geom) (void)hipFree(p.geom);
  if (p.volc) (void)hipFree(p.volc);
  if (p.proja) (void)hipFree(p.proja);
  p.gview = nullptr;
  p.sview = nullptr;
  p.sitem = nullptr;
  p.zterm = nullptr;
  p.mats = nullptr;
  p.geom = nullptr;
  p.volc = p.proja = nullptr;
}

static int dev_alloc(void** ptr, size_t bytes) {
  if (hipMalloc(ptr, bytes) != hipSuccess) {
    (void)hipGetLastError();
    *ptr = nullptr;
    return fail(SCXR_ERR_NOMEM, "hipMalloc of %zu bytes failed", bytes);
  }
  return SCXR_OK;
}

// Where the windows in LDS are the faster path: both sides' times in us,
// fitted to graph replays over volumes of 8^3 to 256^3 and thin ones, few and
// many views, detectors smaller and larger than the volume (most within a
// fifth).  A flag forces either.
//
// The gather of the forward pays for every detector pixel, for the candidate
// voxels of the pixels that the volume covers, and for the march of a pixel
// along its planes; the windows take two or three launches and a workspace,
// and at these sizes little else.  (Windows against gather: 16^3 with 10 views
// 18 against 12, with 60 views 22 against 22, 64^3 with one view 25 against 25,
// 40^3 with 6 23 against 28; on a detector of 500^2 pixels 32^3 with 3 views 19
// against 81; 512 x 512 x 1 with one view 36 against 531.)
static bool splat_pays(const Plan& p, const std::vector<float>& m, const std::vector<GenView>& gv) {
  const int dims[3] = {p.X, p.Y, p.Z};
  double pixels = 0.0, candidates = 0.0;
  int planes = 0;
  bool copy = false;
  for (int v = 0; v < p.V; ++v) {
    const int na = dims[gv[v].a];
    double e[2];
    for (int r = 0; r < 2; ++r)
      e[r] = std::fabs(mat(m, v, r, 0)) * p.X + std::fabs(mat(m, v, r, 1)) * p.Y +
             std::fabs(mat(m, v, r, 2)) * p.Z + 2.0;
    pixels += 1e-6 * p.D0 * p.D1 * (45.0 + na);
    candidates += 1e-6 * std::min<double>(p.D0, e[0]) * std::min<double>(p.D1, e[1]) * na *
                  gv[v].nb * gv[v].nc;
    planes = std::max(planes, na);
    copy = copy || gv[v].a == 2;
  }
  const double gather = 6.0 + pixels + std::max(0.2 * planes, candidates + 0.1 * planes);
  return gather >= 16.0 + 0.07 * planes + (copy ? 3.5 : 0.0);
}

// The adjoint's waves walk their share of the views one after the other (half
// of them below 32 views, a quarter from there on), and a block that the
// volume fills in part costs as much as a whole one; the gather's threads walk
// all views, at a rate that depends on how many of a wave's voxels lie along
// the fast axis.  (Tiles against gather: 16^3 with 30 views 16.0 against 10.4,
// with 32 9.9 against 10.9; 64^3 with 2 views 5.6 against 4.5, with 5 7.2 against
// 8.1; 256^3 with one view 88 against 68, with two 91 against 149; 512 x 512 x 1
// with 40 views 52 against 24, 512 x 512 x 4 51 against 74.)
static bool adj_tiles_pay(const Plan& p) {
  const double n = static_cast<double>(p.X) * p.Y * p.Z, V = p.V;
  const double blocks = std::ceil(p.X / 8.0) * std::ceil(p.Y / 8.0) * std::ceil(p.Z / 8.0);
  const double rate = p.Z < 8 ? 1.85 : p.Z < 32 ? 2.5 : std::min(p.X, p.Y) < 8 ? 5.5 : 4.3;
  const double tiles = std::max(2.6 + (V >= 32 ? 0.217 : 0.445) * V,
                                3.5 + 1e-3 * blocks * (2.0 + 0.26 * V));
  return tiles <= std::max(1.9 + 0.28 * V, 2.0 + 1e-6 * rate * n * V);
}

// Detector coordinates of every voxel centre stay below this (float32
// rounding of P far below the window margins, window offsets within int32).
constexpr double GEN_PMAX = 8192.0;
constexpr double GEN_MARGIN = 0.01;

static bool gen_in_range(const Plan& p, const std::vector<float>& m) {
  if (p.D0 > 16384 || p.D1 > 16384 || static_cast<double>(p.D0) * p.D1 > 2.6e8) return false;
  for (int v = 0; v < p.V; ++v)
    for (int r = 0; r < 2; ++r)
      if (std::fabs(mat(m, v, r, 0)) * p.X + std::fabs(mat(m, v, r, 1)) * p.Y +
              std::fabs(mat(m, v, r, 2)) * p.Z + std::fabs(mat(m, v, r, 3)) >
          GEN_PMAX)
        return false;
  return true;
}

// Tables of the tiled adjoint; false if some view's 8 x 8 x 8 blocks reach
// over more than GWIN detector pixels.
static bool build_adj_tiles(const Plan& p, const std::vector<float>& m, std::vector<float>& zt) {
  for (int v = 0; v < p.V; ++v)
    for (int r = 0; r < 2; ++r) {
      const double ext = (GA - 1.0) * (std::fabs(mat(m, v, r, 0)) + std::fabs(mat(m, v, r, 1)) +
                                       std::fabs(mat(m, v, r, 2)));
      if (std::floor(ext + 2 * GEN_MARGIN) + 3 > GWIN) return false;
    }
  const int ntk = (p.Z + GA - 1) / GA;
  zt.resize(static_cast<size_t>(p.V) * ntk * 2 * GA);
  for (int v = 0; v < p.V; ++v)
    for (int t = 0; t < ntk; ++t)
      for (int r = 0; r < 2; ++r)
        for (int k = 0; k < GA; ++k)
          zt[((static_cast<size_t>(v) * ntk + t) * 2 + r) * GA + k] =
              mat(m, v, r, 2) * (static_cast<float>(t * GA + k) + 0.5f);
  return true;
}

// Lane strides (sb, sc) of the splat: the smallest product for which any two
// voxels of the 8 x 8 lane lattice project at least 2.0625 pixels apart along
// one detector axis (their 2 x 2 footprints are then disjoint, with a margin
// far above the rounding of the projected centres).
static bool splat_strides(const double mb[2], const double mc[2], int& sb, int& sc) {
  auto disjoint = [&](int SB, int SC) {
    for (int a = 0; a < 8; ++a)
      for (int b = -7; b < 8; ++b) {
        if (a == 0 && b <= 0) continue;
        const double d0 = std::fabs(a * SB * mb[0] + b * SC * mc[0]);
        const double d1 = std::fabs(a * SB * mb[1] + b * SC * mc[1]);
        if (std::max(d0, d1) < 2.0625) return false;
      }
    return true;
  };
  int best = 65;
  for (int SB = 1; SB <= 8; ++SB)
    for (int SC = 1; SC <= 8; ++SC)
      if (SB * SC < best && disjoint(SB, SC)) {
        best = SB * SC;
        sb = SB;
        sc = SC;
      }
  return best < 65;
}

// Window pitch for lane strides (sb, sc): of the width and the 16 values above
// it, the one for which the bank model rates the lattice cheapest (the LDS
// serves 32 lanes at a time over 32 banks, so a half-wave costs the largest
// number of its lanes on one bank).  Over the angles of a 74 degree tilt the
// model averages 2.1 cycles per access against 2.9 for a fixed odd pitch (and
// the counters of that one showed 2.9).
static int splat_pitch(const double mb[2], const double mc[2], int sb, int sc, int width) {
  int d0[64], at[64];
  for (int l = 0; l < 64; ++l) {
    const double b = sb * (l >> 3), c = sc * (l & 7);
    d0[l] = static_cast<int>(std::floor(512.31 + b * mb[0] + c * mc[0]));
    at[l] = d0[l] * width + static_cast<int>(std::floor(512.83 + b * mb[1] + c * mc[1]));
  }
  int best = width, low = INT_MAX;
  for (int pitch = width; pitch <= width + 16; ++pitch) {
    int cost = 0;
    for (int h = 0; h < 2; ++h) {
      unsigned char cnt[32] = {0};
      unsigned char mx = 0;
      for (int l = 32 * h; l < 32 * h + 32; ++l) {
        const unsigned char n = ++cnt[at[l] & 31];
        mx = n > mx ? n : mx;
        at[l] += d0[l];
      }
      cost += mx;
    }
    if (cost < low) {
      low = cost;
      best = pitch;
    }
  }
  return best;
}

// Splat tables: march axes, lane strides, blocks and their windows.  False
// where a view has no strides up to 8 x 8 or its windows do not fit
// 4 x 16 KiB of LDS.
static bool build_splat(Plan& p, const std::vector<float>& m, const std::vector<GenView>& gv,
                        std::vector<SplatView>& views, std::vector<SplatItem>& items) {
  const long long vox = static_cast<long long>(p.X) * p.Y * p.Z;
  if (vox * 4 > (1LL << 30)) return false;
  const int dims[3] = {p.X, p.Y, p.Z};
  struct Block {
    int p, q, lo0, lo1, t0, t1;
  };
  views.resize(p.V);
  std::vector<Block> blocks;  // of all views in turn; view v's end at bend[v]
  std::vector<size_t> bend(p.V);
  long long planes = 0;
  int slot = 0;
  bool need_t = false;
  for (int v = 0; v < p.V; ++v) {
    SplatView g{};
    g.a = gv[v].a;
    const int b = g.a == 0 ? 1 : 0, c = g.a == 2 ? 1 : 2;
    const int na = dims[g.a], nb = dims[b], nc = dims[c];
    const double ma[2] = {mat(m, v, 0, g.a), mat(m, v, 1, g.a)};
    const double mb[2] = {mat(m, v, 0, b), mat(m, v, 1, b)};
    const double mc[2] = {mat(m, v, 0, c), mat(m, v, 1, c)};
    if (!splat_strides(mb, mc, g.sb, g.sc)) return false;
    const double det = mb[0] * mc[1] - mc[0] * mb[1];
    const double bb = -(mc[1] * ma[0] - mc[0] * ma[1]) / det;
    const double bc = -(-mb[1] * ma[0] + mb[0] * ma[1]) / det;
    const double tc = na / 2;
    g.bb = static_cast<float>(bb);
    g.bc = static_cast<float>(bc);
    g.tc = static_cast<float>(tc);
    for (int k = 0; k < 8; ++k) g.m[k] = m[8 * v + k];
    const int wb = 8 * g.sb, wc = 8 * g.sc;
    int size[2];
    double low[2];  // lowest corner of a block relative to its origin voxel
    for (int r = 0; r < 2; ++r) {
      // the shift is within half a voxel (and its rounding) of the exact one
      low[r] = std::min(mb[r] * -0.501, mb[r] * (wb - 0.499)) +
               std::min(mc[r] * -0.501, mc[r] * (wc - 0.499));
      const double ext = std::fabs(mb[r]) * (wb + 0.002) + std::fabs(mc[r]) * (wc + 0.002);
      size[r] = static_cast<int>(std::floor(ext + 2 * GEN_MARGIN)) + 3;
    }
    g.rows = size[0];
    g.pitch = size[1];
    if (g.rows * (g.pitch + 16) > 4096) return false;
    g.pitch = splat_pitch(mb, mc, g.sb, g.sc, size[1]);
    slot = std::max(slot, g.rows * g.pitch);
    need_t = need_t || g.a == 2;
    const double smb = std::fabs(bb) * (na / 2 + 1) + 1, smc = std::fabs(bc) * (na / 2 + 1) + 1;
    const int p0 = static_cast<int>(std::floor(-smb / wb)),
              p1 = static_cast<int>(std::floor((nb + smb) / wb));
    const int q0 = static_cast<int>(std::floor(-smc / wc)),
              q1 = static_cast<int>(std::floor((nc + smc) / wc));
    for (int bp = p0; bp <= p1; ++bp)
      for (int bq = q0; bq <= q1; ++bq) {
        // planes where the block meets the volume: 0 <= origin + width and
        // origin < n along both axes, half a voxel to spare for the rounding
        double lo = 0.0, hi = na - 1.0;
        auto meet = [&](double o, double beta, int w, int n) {
          // -w < o + beta (t - tc) + [-0.51, 0.51] < n
          const double l = -w - 0.51 - o, h = n + 0.51 - o;
          if (std::fabs(beta) < 1e-12) {
            if (!(l < 0.0 && 0.0 < h)) hi = -1.0;
            return;
          }
          const double ta = tc + l / beta, tb = tc + h / beta;
          lo = std::max(lo, std::floor(std::min(ta, tb)));
          hi = std::min(hi, std::ceil(std::max(ta, tb)));
        };
        meet(static_cast<double>(bp) * wb, bb, wb, nb);
        meet(static_cast<double>(bq) * wc, bc, wc, nc);
        if (hi < lo) continue;
        Block k;
        k.p = bp * wb;
        k.q = bq * wc;
        k.t0 = static_cast<int>(lo);
        k.t1 = static_cast<int>(hi) + 1;
        int origin[2];
        for (int r = 0; r < 2; ++r)
          origin[r] = static_cast<int>(std::floor(ma[r] * (tc + 0.5) + mb[r] * (k.p + 0.5) +
                                                  mc[r] * (k.q + 0.5) + mat(m, v, r, 3) + low[r] -
                                                  0.25 - GEN_MARGIN));
        k.lo0 = origin[0];
        k.lo1 = origin[1];
        // off the detector: its window would add nothing
        if (k.lo0 >= p.D0 || k.lo0 + g.rows <= 0 || k.lo1 >= p.D1 || k.lo1 + g.pitch <= 0) continue;
        planes += k.t1 - k.t0;
        blocks.push_back(k);
      }
    views[v] = g;
    bend[v] = blocks.size();
  }
  // Planes per item: about 16384 items (16 waves a SIMD) of at least 16
  // planes, a shorter item being mostly the clearing and writing of its
  // window; 8 planes where 16 would leave most of the chip idle.  Measured
  // with a 74 degree tilt, items of 8192, 16384 at least 16, 16384 at least 8
  // planes: 144^3 with 90 views 407, 380, 383 us, with 20 views 107, 108, 115
  // us; 64^3 with 3 views (about 500 items of 16) 26.5, 26.5, 20.4 us.
  const int most = std::max(p.X, std::max(p.Y, p.Z));
  const long long least = planes / 16 < 1024 ? 8 : 16;
  const int len = static_cast<int>(
      std::min<long long>(most, std::max<long long>(least, (planes + 16383) / 16384)));
  p.ifirst.assign(p.V + 1, 0);
  for (int v = 0; v < p.V; ++v) {
    views[v].first = static_cast<int>(items.size());
    for (size_t e = v ? bend[v - 1] : 0; e < bend[v]; ++e) {
      const Block& k = blocks[e];
      const int n = k.t1 - k.t0, parts = (n + len - 1) / len;
      for (int s = 0; s < parts; ++s)
        items.push_back(SplatItem{v, k.p, k.q, k.lo0, k.lo1, k.t0 + n * s / parts,
                                  k.t0 + n * (s + 1) / parts, 0});
    }
    views[v].last = static_cast<int>(items.size());
    p.ifirst[v + 1] = views[v].last;
  }
  // Passes of whole views whose windows fit 128 MiB (the last-level cache
  // holds 256 MiB), at most 65535 views (the grid's z extent).
  const long long room = (32LL << 20) / std::max(slot, 1);
  long long most_items = 1;
  p.chunk.assign(1, 0);
  for (int v = 0; v < p.V; ++v) {
    const int c0 = p.chunk.back();
    if (v > c0 && (p.ifirst[v + 1] - p.ifirst[c0] > room || v - c0 >= 65535)) p.chunk.push_back(v);
    most_items = std::max<long long>(most_items, p.ifirst[v + 1] - p.ifirst[p.chunk.back()]);
  }
  p.chunk.push_back(p.V);
  p.slot = slot;
  p.need_t = need_t;
  p.ws_floats = most_items * slot + (need_t ? vox : 0);
  return true;
}

// General mode: one device block for every table (one allocation and one
// copy, which set the time of making a plan).
static int upload_tables(Plan& p, const std::vector<float>& m, const std::vector<GenView>& gv,
                         const std::vector<SplatView>& views, const std::vector<SplatItem>& items,
                         const std::vector<float>& zt) {
  std::vector<char> host;
  auto add = [&](const void* src, size_t bytes) {
    const size_t at = (host.size() + 255) & ~static_cast<size_t>(255);
    host.resize(at + bytes);
    if (bytes) std::memcpy(host.data() + at, src, bytes);
    return at;
  };
  const size_t am = add(m.data(), m.size() * sizeof(float));
  const size_t ag = add(gv.data(), gv.size() * sizeof(GenView));
  const size_t av = add(views.data(), views.size() * sizeof(SplatView));
  const size_t ai = add(items.data(), items.size() * sizeof(SplatItem));
  const size_t az = add(zt.data(), zt.size() * sizeof(float));
  const int rc = dev_alloc(&p.tables, host.size());
  if (rc) return rc;
  SCXR_HIP(hipMemcpy(p.tables, host.data(), host.size(), hipMemcpyHostToDevice));
  char* base = static_cast<char*>(p.tables);
  p.mats = reinterpret_cast<float*>(base + am);
  p.gview = reinterpret_cast<GenView*>(base + ag);
  p.sview = reinterpret_cast<SplatView*>(base + av);
  p.sitem = reinterpret_cast<SplatItem*>(base + ai);
  p.zterm = reinterpret_cast<float*>(base + az);
  return SCXR_OK;
}

int create(Plan& p, int X, int Y, int Z, int V, const float* mats, int D0, int D1,
           int allow_slice) {
  p.X = X;
  p.Y = Y;
  p.Z = Z;
  p.V = V;
  p.D0 = D0;
  p.D1 = D1;
  std::vector<float> m(mats, mats + 8 * static_cast<size_t>(V));
  for (float f : m)
    SCXR_REQUIRE(std::isfinite(f), SCXR_ERR_GEOM, "non-finite projection matrix entry");
  if (allow_slice & 1) {
    for (int dax = 1; dax >= 0 && p.mode != MODE_SLICE; --dax)
      for (int sax = 0; sax < 3 && p.mode != MODE_SLICE; ++sax) try_slice(p, m, sax, dax);
  }
  int rc;
  if (p.mode == MODE_GENERAL) {
    std::vector<GenView> gv(V);
    for (int v = 0; v < V; ++v) {
      double best = 0.0;
      int ba = -1;
      for (int a = 0; a < 3; ++a) {
        const int b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
        const double det = static_cast<double>(mat(m, v, 0, b)) * mat(m, v, 1, c) -
                           static_cast<double>(mat(m, v, 0, c)) * mat(m, v, 1, b);
        if (std::fabs(det) > std::fabs(best)) {
          best = det;
          ba = a;
        }
      }
      SCXR_REQUIRE(ba >= 0 && std::fabs(best) > 1e-6, SCXR_ERR_GEOM,
                   "projection matrix of view %d has rank < 2", v);
      const int b = ba == 0 ? 1 : 0, c = ba == 2 ? 1 : 2;
      GenView g{};
      g.a = ba;
      const double i00 = mat(m, v, 1, c) / best, i01 = -mat(m, v, 0, c) / best;
      const double i10 = -mat(m, v, 1, b) / best, i11 = mat(m, v, 0, b) / best;
      // box half-width 1 in P; margin for the float32 solve
      const double hb = std::fabs(i00) + std::fabs(i01) + 1e-2;
      const double hc = std::fabs(i10) + std::fabs(i11) + 1e-2;
      g.i00 = static_cast<float>(i00);
      g.i01 = static_cast<float>(i01);
      g.i10 = static_cast<float>(i10);
      g.i11 = static_cast<float>(i11);
      g.hb = static_cast<float>(hb);
      g.hc = static_cast<float>(hc);
      g.nb = static_cast<int>(std::floor(2.0 * hb)) + 2;
      g.nc = static_cast<int>(std::floor(2.0 * hc)) + 2;
      gv[v] = g;
    }
    std::vector<SplatView> views;
    std::vector<SplatItem> items;
    std::vector<float> zt;
    if (!(allow_slice & 4) && gen_in_range(p, m)) {
      const bool always = allow_slice & 8;
      p.splat = (always || splat_pays(p, m, gv)) && build_splat(p, m, gv, views, items);
      p.adj_tiled = (always || adj_tiles_pay(p)) && build_adj_tiles(p, m, zt);
    }
    return upload_tables(p, m, gv, views, items, zt);
  }
  rc = dev_alloc(reinterpret_cast<void**>(&p.mats), m.size() * sizeof(float));
  if (rc) return rc;
  SCXR_HIP(hipMemcpy(p.mats, m.data(), m.size() * sizeof(float), hipMemcpyHostToDevice));
  if (p.mode == MODE_SLICE) {
    const int e = 1 - p.dax;
    std::vector<float4> g(V);
    for (int v = 0; v < V; ++v)
      g[v] = make_float4(mat(m, v, e, p.pax), mat(m, v, e, p.qax), mat(m, v, e, 3), 0.0f);
    // Staged adjoint: a 4 x 8 tile's rows per view, at most
    // ceil(3 |a| + 7 |b| + rounding) + 2 (the corner bins' spread plus the
    // right-hand tap), must fit ADJ_NW.  The rounding margin covers the
    // float32 evaluation of the corner centres (a few ulps of |P|); beyond
    // 65536 detector rows, where those reach a tap, rows are read from global
    // memory.
    p.adj_staged = !(allow_slice & 2) && p.U < 65536;
    for (int v = 0; v < V && p.adj_staged; ++v) {
      const double a = std::fabs(static_cast<double>(g[v].x)),
                   b = std::fabs(static_cast<double>(g[v].y));
      const double pmax = a * (p.P + 1) + b * (p.Q + 1) + std::fabs(static_cast<double>(g[v].z));
      const double spread = 3.0 * a + 7.0 * b + 1e-3 + 1e-6 * (pmax + 2.0);
      if (std::ceil(spread) + 2.0 > ADJ_NW) p.adj_staged = false;
    }
    rc = dev_alloc(reinterpret_cast<void**>(&p.geom), V * sizeof(float4));
    if (rc) return rc;
    SCXR_HIP(hipMemcpy(p.geom, g.data(), V * sizeof(float4), hipMemcpyHostToDevice));
    const size_t s4 = 4 * static_cast<size_t>(p.SQ);
    {
      const size_t rows = static_cast<size_t>(p.P) * p.Q;
      rc = dev_alloc(reinterpret_cast<void**>(&p.volc), rows * s4 * sizeof(float));
      if (rc) return rc;
    }
    if (!p.proj_direct) {
      rc = dev_alloc(reinterpret_cast<void**>(&p.proja),
                     static_cast<size_t>(V) * p.U * s4 * sizeof(float));
      if (rc) return rc;
    }
  }
  return SCXR_OK;
}

static int transpose(const float* in, float* out, int B, int Rout, int Cout, int Rin, int Cin,
                     int roff, int coff, long long ib, long long ir, long long ob, long long oc,
                     const int32_t* pred, hipStream_t s) {
  dim3 grid(ceil_div(Cout, 32), ceil_div(Rout, 32), B);
  hipLaunchKernelGGL(transpose_kernel, grid, dim3(256), 0, s, in, out, Rout, Cout, Rin, Cin, roff,
                     coff, ib, ir, ob, oc, pred);
  SCXR_LAUNCHED("xr3d transpose");
  return SCXR_OK;
}

static int shift_rows(const float* in, float* out, long long rows, int Cout, int Cin, int off,
                      long long is, long long os, const int32_t* pred, hipStream_t s) {
  const long long n = rows * Cout;
  const unsigned blocks = static_cast<unsigned>(std::min<long long>((n + 255) / 256, 65536));
  hipLaunchKernelGGL(shift_rows_kernel, dim3(blocks), dim3(256), 0, s, in, out, rows, Cout, Cin,
                     off, is, os, pred);
  SCXR_LAUNCHED("xr3d shift_rows");
  return SCXR_OK;
}

// vol (X, Y, Z) -> vol_c[p][q][s] (slices padded to 4 SQ with zeros)
static int vol_to_canon(const Plan& p, const float* vol, float* vc, const int32_t* pred,
                        hipStream_t s) {
  const int S4 = 4 * p.SQ;
  switch (p.sax) {
    case 2:
      return shift_rows(vol, vc, static_cast<long long>(p.X) * p.Y, S4, p.S, 0, p.S, S4, pred,
                        s);
    case 1:  // vol[p][s][q] -> vc[p][q][s]
      return transpose(vol, vc, p.X, S4, p.Z, p.S, p.Z, 0, 0,
                       static_cast<long long>(p.Y) * p.Z, p.Z,
                       static_cast<long long>(p.Z) * S4, S4, pred, s);
    default: {  // vol[s][pq] -> vc[pq][s]
      const int PQ = p.Y * p.Z;
      return transpose(vol, vc, 1, S4, PQ, p.S, PQ, 0, 0, 0, PQ, 0, S4, pred, s);
    }
  }
}

static int canon_to_vol(const Plan& p, const float* vc, float* vol, const int32_t* pred,
                        hipStream_t s) {
  const int S4 = 4 * p.SQ;
  switch (p.sax) {
    case 2:
      return shift_rows(vc, vol, static_cast<long long>(p.X) * p.Y, p.S, S4, 0, S4, p.S, pred,
                        s);
    case 1:  // vol[p][s][q] = vc[p][q][s]
      return transpose(vc, vol, p.X, p.Z, p.S, p.Z, S4, 0, 0,
                       static_cast<long long>(p.Z) * S4, S4,
                       static_cast<long long>(p.Y) * p.Z, p.Z, pred, s);
    default: {  // vol[s][pq] = vc[pq][s]
      const int PQ = p.Y * p.Z;
      return transpose(vc, vol, 1, PQ, p.S, PQ, S4, 0, 0, 0, S4, 0, PQ, pred, s);
    }
  }
}

// proj (V, D0, D1) -> proj_c[v][u][s]
static int proj_to_canon(const Plan& p, const float* y, float* yc, const int32_t* pred,
                         hipStream_t s) {
  const int S4 = 4 * p.SQ;
  if (p.dax == 1)  // proj[v][u][s + delta]
    return shift_rows(y, yc, static_cast<long long>(p.V) * p.D0, S4, p.D1, p.delta, p.D1, S4,
                      pred, s);
  // proj[v][s + delta][u] -> yc[v][u][s]
  return transpose(y, yc, p.V, S4, p.U, p.D0, p.D1, p.delta, 0,
                   static_cast<long long>(p.D0) * p.D1, p.D1,
                   static_cast<long long>(p.U) * S4, S4, pred, s);
}

static int canon_to_proj(const Plan& p, const float* yc, float* y, const int32_t* pred,
                         hipStream_t s) {
  const int S4 = 4 * p.SQ;
  if (p.dax == 1)  // proj[v][u][c] = yc[v][u][c - delta] for c - delta in [0, S)
    return shift_rows(yc, y, static_cast<long long>(p.V) * p.D0, p.D1, p.S, -p.delta, S4, p.D1,
                      pred, s);
  // proj[v][c][u] = yc[v][u][c - delta]
  return transpose(yc, y, p.V, p.U, p.D0, p.U, p.S, 0, -p.delta,
                   static_cast<long long>(p.U) * S4, S4,
                   static_cast<long long>(p.D0) * p.D1, p.D1, pred, s);
}

// Splat forward: ws holds the transposed volume (if a view marches along z),
// then the windows of one pass over the items.
static int forward_splat(const Plan& p, const float* vol, float* proj, float* ws,
                         const int32_t* pred, hipStream_t s) {
  const float* volt = vol;
  float* parts = ws;
  if (p.need_t) {
    const int XY = p.X * p.Y;  // vol[xy][z] -> volt[z][xy]
    const int rc = transpose(vol, ws, 1, XY, p.Z, XY, p.Z, 0, 0, 0, p.Z, 0, XY, pred, s);
    if (rc) return rc;
    volt = ws;
    parts = ws + static_cast<size_t>(XY) * p.Z;
  }
  for (size_t c = 0; c + 1 < p.chunk.size(); ++c) {
    const int v0 = p.chunk[c], v1 = p.chunk[c + 1];
    const int i0 = p.ifirst[v0], i1 = p.ifirst[v1];
    if (i1 > i0) {
      hipLaunchKernelGGL(gen_splat_kernel, dim3(ceil_div(i1 - i0, 4)), dim3(256),
                         4 * p.slot * sizeof(float), s, vol, volt, parts, p.sview, p.sitem, i0, i1,
                         p.slot, p.X, p.Y, p.Z, pred);
      SCXR_LAUNCHED("xr3d general forward");
    }
    hipLaunchKernelGGL(gen_splat_sum_kernel, dim3(ceil_div(p.D1, 16), ceil_div(p.D0, 16), v1 - v0),
                       dim3(256), 0, s, parts, proj, p.sview, p.sitem, v0, i0, p.slot, p.D0, p.D1,
                       pred);
    SCXR_LAUNCHED("xr3d general forward window sums");
  }
  return SCXR_OK;
}

int forward(const Plan& p, const float* vol, float* proj, float* ws, const int32_t* pred,
            hipStream_t s) {
  if (p.mode == MODE_GENERAL) {
    if (p.splat && ws) return forward_splat(p, vol, proj, ws, pred, s);
    const long long npix = static_cast<long long>(p.D0) * p.D1;
    hipLaunchKernelGGL(gen_fwd_kernel, dim3(ceil_div(npix, 64), p.V), dim3(64 * GEN_W), 0, s, vol,
                       proj, p.mats, p.gview, p.X, p.Y, p.Z, p.D0, p.D1, pred);
    SCXR_LAUNCHED("xr3d general forward");
    return SCXR_OK;
  }
  const float* vc = vol;
  if (!p.vol_direct) {
    int rc = vol_to_canon(p, vol, p.volc, pred, s);
    if (rc) return rc;
    vc = p.volc;
  }
  float* yc = p.proj_direct ? proj : p.proja;
  const float4* v4 = reinterpret_cast<const float4*>(vc);
  float4* y4 = reinterpret_cast<float4*>(yc);
  if (p.slot16) {
    const dim3 g16(ceil_div(p.U, FBL), ceil_div(p.V, 4), ceil_div(p.SQ, 64));
    hipLaunchKernelGGL(fwd_slice16_kernel, g16, dim3(256), 0, s, v4, y4, p.geom, p.P, p.Q, p.SQ,
                       p.U, p.V, pred);
    SCXR_LAUNCHED("xr3d slice forward (16 slots)");
    if (!p.proj_direct) return canon_to_proj(p, yc, proj, pred, s);
    return SCXR_OK;
  }
  const dim3 grid(ceil_div(p.U, FB), ceil_div(p.V, 4), ceil_div(p.SQ, 64));
#define SCXR_FWD3(C, G)                                                                       \
  hipLaunchKernelGGL((fwd_slice_kernel<C, G>), grid, dim3(256), 0, s, v4, y4, p.geom, p.P, p.Q, \
                     p.SQ, p.U, p.V, pred)
  // (two slots: spacings of 0.5 to 0.67, at most 24 candidates)
  if (p.spg == 2)
    SCXR_FWD3(32, 2);
  else if (p.cpr == 32)
    SCXR_FWD3(32, 3);
  else
    SCXR_FWD3(64, 3);
#undef SCXR_FWD3
  SCXR_LAUNCHED("xr3d slice forward");
  if (!p.proj_direct) return canon_to_proj(p, yc, proj, pred, s);
  return SCXR_OK;
}

int adjoint(const Plan& p, const float* proj, float* vol, const int32_t* pred, hipStream_t s) {
  if (p.mode == MODE_GENERAL) {
    const long long n = static_cast<long long>(p.X) * p.Y * p.Z;
    if (p.adj_tiled) {
      // The four waves of a workgroup take four shares of one block's views,
      // or two of two blocks' where a share would be under 8 views: more and
      // shorter waves, also where there are blocks enough to fill the chip.
      // 1, 2, 4 shares: 48^3 with 90 views 81, 42, 23.5 us, 130^3 with 90
      // views 144, 128, 123 us; 64^3 with 20 views 20.7, 12.0, 15.1 us, 144^3
      // with 3 views 13.0, 13.0, 15.8 us.
      const int tiles = ceil_div(p.X, GA) * ceil_div(p.Y, GA) * ceil_div(p.Z, GA);
      const int vs = p.V >= 32 ? 4 : 2;
      hipLaunchKernelGGL(gen_adj_tile_kernel, dim3(ceil_div(tiles, 4 / vs)), dim3(256), 0, s, proj,
                         vol, p.mats, p.zterm, p.X, p.Y, p.Z, p.V, p.D0, p.D1, vs, pred);
      SCXR_LAUNCHED("xr3d general adjoint (tiled)");
      return SCXR_OK;
    }
    hipLaunchKernelGGL(gen_adj_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, proj, vol, p.mats,
                       p.X, p.Y, p.Z, p.V, p.D0, p.D1, pred);
    SCXR_LAUNCHED("xr3d general adjoint");
    return SCXR_OK;
  }
  const float* yc = proj;
  if (!p.proj_direct) {
    int rc = proj_to_canon(p, proj, p.proja, pred, s);
    if (rc) return rc;
    yc = p.proja;
  }
  float* vc = p.vol_direct ? vol : p.volc;
  dim3 grid(ceil_div(p.Q, 8), ceil_div(p.P, 4), ceil_div(p.SQ, 64));
  hipLaunchKernelGGL(p.adj_staged ? adj_slice_staged_kernel : adj_slice_kernel, grid, dim3(256), 0,
                     s, reinterpret_cast<const float4*>(yc), reinterpret_cast<float4*>(vc),
                     p.geom, p.P, p.Q, p.SQ, p.U, p.V, pred);
  SCXR_LAUNCHED("xr3d slice adjoint");
  if (!p.vol_direct) return canon_to_vol(p, vc, vol, pred, s);
  return SCXR_OK;
}

}  // namespace xr3d
}  // namespace scxr

struct scxr_xr3d_plan {
  scxr::xr3d::Plan p;
};

using namespace scxr;

extern "C" {

int scxr_xr3d_plan_create(int32_t X, int32_t Y, int32_t Z, int32_t V, const float* matrices,
                          int32_t D0, int32_t D1, int32_t allow_slice, scxr_xr3d_plan** out) {
  SCXR_REQUIRE(out && matrices, SCXR_ERR_ARG, "null argument to xr3d_plan_create");
  SCXR_REQUIRE(X > 0 && Y > 0 && Z > 0 && V > 0 && D0 > 0 && D1 > 0, SCXR_ERR_SHAPE,
               "non-positive size (X=%d Y=%d Z=%d V=%d D0=%d D1=%d)", X, Y, Z, V, D0, D1);
  SCXR_REQUIRE(static_cast<long long>(X) * Y * Z < (1LL << 31) &&
                   static_cast<long long>(D0) * D1 < (1LL << 31),
               SCXR_ERR_SHAPE, "volume or detector too large");
  auto* plan = new scxr_xr3d_plan();
  int rc = xr3d::create(plan->p, X, Y, Z, V, matrices, D0, D1, allow_slice);
  if (rc != SCXR_OK) {
    xr3d::destroy(plan->p);
    delete plan;
    return rc;
  }
  *out = plan;
  return SCXR_OK;
}

int scxr_xr3d_plan_destroy(scxr_xr3d_plan* plan) {
  if (!plan) return SCXR_OK;
  xr3d::destroy(plan->p);
  delete plan;
  return SCXR_OK;
}

int scxr_xr3d_info(const scxr_xr3d_plan* plan, int32_t* out) {
  SCXR_REQUIRE(plan && out, SCXR_ERR_ARG, "null argument to xr3d_info");
  const auto& p = plan->p;
  out[0] = p.mode;
  out[1] = p.sax;
  out[2] = p.dax;
  out[3] = p.delta;
  out[4] = p.cpr;
  out[5] = p.vol_direct;
  out[6] = p.proj_direct;
  out[7] = p.U;
  out[8] = p.adj_staged;
  return SCXR_OK;
}

int scxr_xr3d_forward(const scxr_xr3d_plan* plan, const float* vol, float* proj,
                      const int32_t* pred, void* stream) {
  SCXR_REQUIRE(plan && vol && proj, SCXR_ERR_ARG, "null argument to xr3d_forward");
  return xr3d::forward(plan->p, vol, proj, nullptr, pred, as_stream(stream));
}

int64_t scxr_xr3d_forward_ws(const scxr_xr3d_plan* plan) {
  return plan && plan->p.splat ? static_cast<int64_t>(plan->p.ws_floats) : 0;
}

int scxr_xr3d_forward_with(const scxr_xr3d_plan* plan, const float* vol, float* proj, float* ws,
                           const int32_t* pred, void* stream) {
  SCXR_REQUIRE(plan && vol && proj, SCXR_ERR_ARG, "null argument to xr3d_forward_with");
  SCXR_REQUIRE(ws || !plan->p.splat, SCXR_ERR_ARG, "xr3d_forward_with needs its workspace");
  return xr3d::forward(plan->p, vol, proj, ws, pred, as_stream(stream));
}

int scxr_xr3d_adjoint(const scxr_xr3d_plan* plan, const float* proj, float* vol,
                      const int32_t* pred, void* stream) {
  SCXR_REQUIRE(plan && vol && proj, SCXR_ERR_ARG, "null argument to xr3d_adjoint");
  return xr3d::adjoint(plan->p, proj, vol, pred, as_stream(stream));
}

int scxr_xr3d_weights(const scxr_xr3d_plan* plan, int32_t view, int32_t* ul, float* w,
                      void* stream) {
  SCXR_REQUIRE(plan && ul && w, SCXR_ERR_ARG, "null argument to xr3d_weights");
  const auto& p = plan->p;
  SCXR_REQUIRE(view >= 0 && view < p.V, SCXR_ERR_ARG, "view %d out of range", view);
  const long long n = static_cast<long long>(p.X) * p.Y * p.Z;
  hipLaunchKernelGGL(xr3d::weights_kernel, dim3(ceil_div(n, 256)), dim3(256), 0,
                     as_stream(stream), p, view, ul, w);
  SCXR_LAUNCHED("xr3d weights");
  return SCXR_OK;
}

}  // extern "C"
