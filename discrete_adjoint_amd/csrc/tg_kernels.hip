// FP64 kernels of the forward step and the per-step discrete adjoint on
// uniform blocks of cells.  Tiles of 256 cells (tile table), of one member
// each, so an ensemble of uneven blocks runs in one launch.
//
// Forward step s (replaces step.C:38-232, order 1):
//   k_coef   : forward slopes -> kact (getcoef.f) + per-instance CFL min /
//              hmax reduction (get_coef_and_eigen.C:29-180)
//   k_update : dt = 0.5*min(0.5*min(dx/ev), 0.9*sqrt(hmax eps Gs/9.8)) and
//              incrtime; slopes, HLL edge fluxes with outflow copies,
//              update_states
// Reverse step s (replaces calc_jacobian + calc_adjoint, dual_solver.C:200-206):
//   k_adjoint: gathers lambda^s_c = g_c - sum_j J_j[slot->c]^T lambda^{s+1}_j,
//              recomputing every Jacobian block from U^s in registers.
// Small meshes launch a workgroup per tile of each (..._tile); on large ones
// the first pass of a step lists the tiles that have work for the second.
#include "tg_kernels.h"
#include "tg_math.h"

namespace tg {

namespace {

__device__ __forceinline__ unsigned long long dbits(double v) {
  return (unsigned long long)__double_as_longlong(v);
}

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    double w = __shfl_xor(v, o, 64);
    v = (w < v) ? w : v;
  }
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    double w = __shfl_xor(v, o, 64);
    v = (w > v) ? w : v;
  }
  return v;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

struct Cell {
  int i, j;
  long long c;
  bool act;
  bool hasE, hasW, hasN, hasS;
};

template <int TX>
__device__ __forceinline__ Cell cell_of(const TileDev& t, const InstDev& I) {
  Cell q;
  q.i = t.x0 + (int)(threadIdx.x % TX);
  q.j = t.y0 + (int)(threadIdx.x / TX);
  q.act = q.i < I.nx && q.j < I.ny;
  q.c = I.off + (long long)q.j * I.nx + q.i;
  q.hasE = q.i + 1 < I.nx;
  q.hasW = q.i > 0;
  q.hasN = q.j + 1 < I.ny;
  q.hasS = q.j > 0;
  return q;
}

template <int TX>
__device__ __forceinline__ Cell cell_of(const TileRef& t) {
  Cell q;
  q.i = t.x0 + (int)(threadIdx.x % TX);
  q.j = t.y0 + (int)(threadIdx.x / TX);
  q.act = q.i < t.nx && q.j < t.ny;
  q.c = t.off + (long long)q.j * t.nx + q.i;
  q.hasE = q.i + 1 < t.nx;
  q.hasW = q.i > 0;
  q.hasN = q.j + 1 < t.ny;
  q.hasS = q.j > 0;
  return q;
}

// ------------------------------------------------------------- zero marks --

__device__ __forceinline__ bool bitzero3(double a, double b, double c) {
  return (dbits(a) | dbits(b) | dbits(c)) == 0ull;
}
// Records in the output marks whether the tile holds +0.0 only (all: the
// workgroup's reduction of "this cell is +0.0 in all three fields or
// outside the member").  Thread 0 stores the tile's byte.
template <int TX, class T>
__device__ __forceinline__ void mark_store(uint32_t* mk, const T& t, bool all) {
  if (threadIdx.x == 0) ((unsigned char*)(mk + t.mw))[mark_byte<TX>(t)] = all ? 1 : 0;
}

// Skips decided from the marks alone, for a whole mark block.
// Update: the block and the four side blocks of U are +0.0 -- every cell
// and side neighbour has h < tiny, so the fluxes are zero and there are no
// sources, and U^{s+1} = U^s - dtdx*(0 - 0) - dtdy*(0 - 0) = +0.0 for a
// finite dt -- so nothing is to do where the output already holds +0.0.
template <class Blk>
__device__ __forceinline__ bool update_skip(const uint32_t* in, const Blk& B) {
  return in[B.mw] == MARK_FULL &&
         (B.mwW < 0 || in[B.mwW] == MARK_FULL) && (B.mwE < 0 || in[B.mwE] == MARK_FULL) &&
         (B.mwS < 0 || in[B.mwS] == MARK_FULL) && (B.mwN < 0 || in[B.mwN] == MARK_FULL);
}
// Adjoint: the block of U^s is +0.0 (void cells: lambda^s = +0.0), that of
// lambda^{s+1} too when the gradient is wanted (no bed-friction terms): nothing
// is to do where lambda^s already holds +0.0.
__device__ __forceinline__ bool adjoint_skip(const uint32_t* mu, const uint32_t* ml, int mw) {
  return mu[mw] == MARK_FULL && (!ml || ml[mw] == MARK_FULL);
}
// the byte of block word mw that tile byte b owns
__device__ __forceinline__ void mark_byte_store(uint32_t* mk, int mw, int b, bool zero) {
  ((unsigned char*)(mk + mw))[b] = zero ? 1 : 0;
}
// the list entry of tile byte b of a block
template <int TX>
__device__ __forceinline__ TileRef tile_ref(const BlockDev& B, int b) {
  constexpr int TY = BLOCK / TX, PER_ROW = MARK_W / TX;
  return TileRef{B.inst, B.tile[b], B.x0 + (b % PER_ROW) * TX, B.y0 + (b / PER_ROW) * TY,
                 B.mw, B.nx, B.ny, 0, B.off};
}
// The cells of a block's four tiles this thread handles (one per tile).
template <int TX>
__device__ __forceinline__ void block_cells(const BlockDev& B, Cell q[4]) {
  constexpr int TY = BLOCK / TX, PER_ROW = MARK_W / TX;
  InstDev I;  // the fields cell_of reads, carried by the block record
  I.nx = B.nx; I.ny = B.ny; I.off = B.off;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    q[b].act = false;
    if (B.tile[b] < 0) continue;
    // tile byte b (mark_byte) from the block origin: no tile record to load
    TileDev t{};
    t.inst = B.inst;
    t.x0 = B.x0 + (b % PER_ROW) * TX;
    t.y0 = B.y0 + (b / PER_ROW) * TY;
    q[b] = cell_of<TX>(t, I);
  }
}

// ---------------------------------------------------------------- forward --

// Limited slope from its two one-sided differences dp = (u+ - u)/dx and
// dm = (u - u-)/dx (Element::get_slopes, element2.C:886-897; same operands
// as slope_fwd); inv_s = 1 / (dx + dx).
__device__ __forceinline__ double slope_from(double dp, double dm, double dx, double inv_s,
                                             double gamma, double tiny) {
  const double dc = div_r(dp * dx + dm * dx, dx + dx, inv_s);
  return .5 * (c_sgn(dp, tiny) + c_sgn(dm, tiny)) *
         dmin3(gamma * dabs(dp), gamma * dabs(dm), dabs(dc));
}
__device__ __forceinline__ double slope3(double up, double uc, double um, double dx, double inv,
                                         double inv_s, double gamma, double tiny) {
  return slope_from(div_r(up - uc, dx, inv), div_r(uc - um, dx, inv), dx, inv_s, gamma, tiny);
}

// Coefficients of one cell above tiny: kact from its forward slopes
// (getcoef.f), written, and its terms of the CFL reduction
// (get_coef_and_eigen.C:29-180).  Every load is issued before the first use.
__device__ __forceinline__ void coef_cell(const StepArgs& a, const InstDev& I, int i, int j,
                                          double h, int reduce, double& minev, double& hmax) {
  const long long c = I.off + (long long)j * I.nx + i;
  // cells on the domain boundary have zero slopes: with themselves as
  // neighbours every difference is 0
  const bool inner = i + 1 < I.nx && i > 0 && j + 1 < I.ny && j > 0;
  const long long ox = inner ? 1 : 0, oy = inner ? I.nx : 0;
  const double hu = a.U.hu[c], hv = a.U.hv[c], g3 = a.S.gz[c];
  const double hE = a.U.h[c + ox], hW = a.U.h[c - ox], hN = a.U.h[c + oy], hS = a.U.h[c - oy];
  const double uE = a.U.hu[c + ox], uW = a.U.hu[c - ox];
  const double vN = a.U.hv[c + oy], vS = a.U.hv[c - oy];
  const double kroot = mat_of(I, a.mat, a.mtab, c).kroot;
  const double hx = slope3(hE, h, hW, I.dx, I.inv_dx, I.inv_sx, a.gamma, a.tiny);
  const double hux = slope3(uE, hu, uW, I.dx, I.inv_dx, I.inv_sx, a.gamma, a.tiny);
  const double hy = slope3(hN, h, hS, I.dy, I.inv_dy, I.inv_sy, a.gamma, a.tiny);
  const double hvy = slope3(vN, hv, vS, I.dy, I.inv_dy, I.inv_sy, a.gamma, a.tiny);
  // getcoef and eigen (tg_math.h) for h > tiny
  const double inv = 1. / h, hh = h * h, ihh = 1. / hh;
  const double vx = div_r(hu, h, inv), vy = div_r(hv, h, inv);
  const double vel = div_r(hux, h, inv) - div_r(hu * hx, hh, ihh) + div_r(hvy, h, inv) -
                     div_r(hv * hy, hh, ihh);
  double k = I.kc1 * (1. - f_sgn(vel, a.tiny) * kroot) - 1.;
  if (fabs(vx) < a.tiny && fabs(vy) < a.tiny) k = 1.;
  if (k < 0.) k = 0.;
  k = k * I.eps;
  a.kact[c] = k;
  if (reduce) {
    const double w = sqrt(k * g3 * h);
    const double ex = fabs(vx) + w, ey = fabs(vy) + w;
    const double ev = (ex > ey) ? ex : ey;
    if (ev > 1000000000.) atomicOr(a.err, 2);
    const double mdx = (I.dx > I.dy) ? I.dy : I.dx;
    const double m = mdx / ev;
    minev = (m < minev) ? m : minev;
    hmax = (h > hmax) ? h : hmax;
  }
}

// The workgroup's CFL terms into the member's reduction cells (every thread
// calls it; any: some thread has one).
__device__ __forceinline__ void coef_reduce(const StepArgs& a, int b, double minev, double hmax,
                                            bool any) {
  if (!__syncthreads_or(any)) return;
  __shared__ double smin[BLOCK / 64], smax[BLOCK / 64];
  minev = wave_min(minev);
  hmax = wave_max(hmax);
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  if (l == 0) { smin[w] = minev; smax[w] = hmax; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < BLOCK / 64; k++) {
      minev = (smin[k] < minev) ? smin[k] : minev;
      hmax = (smax[k] > hmax) ? smax[k] : hmax;
    }
    red_add(a, b, minev, hmax);
  }
}

// First pass on large meshes, one workgroup per mark block.
//
// Coefficients: forward slopes -> kact (getcoef.f) and the per-instance CFL
// min / hmax reduction (get_coef_and_eigen.C:29-180).  The block's wet cells
// are listed in LDS and worked off 256 at a time, so a block that a front
// crosses takes as many rounds as it has wet cells, not one for each of its
// four tiles.
//
// Tiles for the update: a tile whose cells and side neighbours all hold h <
// tiny has every face flux zero (the physical flux is zero below tiny and
// riemannflux of two such sides is zero) and no source terms (update_states
// adds them only above tiny); it goes on the dry list, unless the marks show
// that input and output hold +0.0 already.  Every other tile goes on the full
// list.  (No dt is needed for that: see k_update for one that is not finite.)
// Both jobs read h of the same blocks; in two passes they took 12.4 + 12.4 us
// of a 2048 x 2048 step and 15.5 + 20 us on 64 members of 5.8 M cells, in one
// 18 and 24 us.
template <int TX>
__global__ __launch_bounds__(BLOCK) void k_coef(StepArgs a, int reduce) {
  constexpr int TY = BLOCK / TX;
  // (the block table is indexed by mark word)
  const BlockDev B = a.blocks[blockIdx.x];
  if (a.mk_in && a.mk_out[B.mw] == MARK_FULL && update_skip(a.mk_in, B)) return;
  __shared__ int s_n;
  __shared__ unsigned s_wet;
  __shared__ unsigned short s_cell[4 * BLOCK];
  __shared__ double s_h[4 * BLOCK];
  if (threadIdx.x == 0) { s_n = 0; s_wet = 0u; }
  Cell q[4];
  block_cells<TX>(B, q);
  // tiles of the block holding +0.0 in the input / output state (mark bytes):
  // their h is not read
  const uint32_t zin = (a.mk_in && a.zbytes) ? a.mk_in[B.mw] : 0u;
  const uint32_t zout = (a.mk_out && a.zbytes) ? a.mk_out[B.mw] : 0u;
  const long long nx = B.nx;
  const int tx = (int)(threadIdx.x % TX), ty = (int)(threadIdx.x / TX);
  double h[4];
  unsigned flows = 0u;  // tiles with a cell or side neighbour not below tiny
#pragma unroll
  for (int b = 0; b < 4; b++)
    h[b] = q[b].act && !((zin >> (8 * b)) & 1u) ? a.U.h[q[b].c] : 0.;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    if (!q[b].act) continue;
    const long long c = q[b].c;
    bool w = !(h[b] < a.tiny);
    if (tx == 0 && q[b].hasW) w = w || !(a.U.h[c - 1] < a.tiny);
    if (tx == TX - 1 && q[b].hasE) w = w || !(a.U.h[c + 1] < a.tiny);
    if (ty == 0 && q[b].hasS) w = w || !(a.U.h[c - nx] < a.tiny);
    if (ty == TY - 1 && q[b].hasN) w = w || !(a.U.h[c + nx] < a.tiny);
    if (w) flows |= 1u << b;
  }
  const InstDev I = a.inst[B.inst];
  __syncthreads();  // s_n, s_wet set
  if (flows) atomicOr(&s_wet, flows);
  int nwet = 0, nshort = 0;
  const int lane = threadIdx.x % 64;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const bool wet = q[b].act && h[b] > a.tiny;
    const unsigned long long m = __ballot(wet);
    if (m) {
      int base = 0;
      if (lane == 0) base = atomicAdd(&s_n, __popcll(m));
      base = __shfl(base, 0, 64);
      if (wet) {
        const int k = base + __popcll(m & ((1ull << lane) - 1ull));
        s_cell[k] = (unsigned short)((q[b].j - B.y0) * MARK_W + q[b].i - B.x0);
        s_h[k] = h[b];
      }
    }
    if (!q[b].act || ((zin >> (8 * b)) & 1u)) continue;
    if (wet) {
      nwet++;
    } else {
      nshort++;
      // kact is read only where h >= tiny (the physical flux is zero below
      // tiny, update_states uses kact only above it): at or below tiny the
      // value is epsilon, and below tiny it is not written
      if (!(h[b] < a.tiny)) a.kact[q[b].c] = I.eps;
    }
  }
  if (a.active) {
    const int cnt = (int)wave_sum((double)nwet);
    if (threadIdx.x % 64 == 0 && cnt) atomicAdd(a.active, (unsigned long long)cnt);
  }
  if (a.short_cells) {
    const int cnt = (int)wave_sum((double)nshort);
    if (threadIdx.x % 64 == 0 && cnt) atomicAdd(a.short_cells, (unsigned long long)cnt);
  }
  __syncthreads();  // the wet cells and tiles are complete
  if (a.copy_dry) {
    // dry_cell for a dt known to be zero or positive: the state, h clamped
#pragma unroll
    for (int b = 0; b < 4; b++) {
      if (!q[b].act || ((s_wet >> b) & 1u)) continue;
      const long long c = q[b].c;
      const double hu = a.U.hu[c], hv = a.U.hv[c];
      if (!isfinite(h[b]) || !isfinite(hu) || !isfinite(hv)) atomicOr(a.err, 1);
      a.h_out[c] = (h[b] < 0.) ? 0. : h[b];
      a.hu_out[c] = hu;
      a.hv_out[c] = hv;
    }
  }
  if (threadIdx.x == 0) {
    unsigned full = s_wet, dry = 0u;
#pragma unroll
    for (int b = 0; b < 4 && !a.copy_dry; b++)
      if (B.tile[b] >= 0 && !((full >> b) & 1u) && !(((zin & zout) >> (8 * b)) & 1u)) dry |= 1u << b;
    int kf = full ? atomicAdd(a.tile_count, __popc(full)) : 0;
    int kd = dry ? atomicAdd(a.tile_count + 1, __popc(dry)) : 0;
    // the full list grows from the front of the array, the dry one from its
    // end: a tile is on at most one of them
#pragma unroll
    for (int b = 0; b < 4; b++) {
      if ((full >> b) & 1u) a.tile_list[kf++] = tile_ref<TX>(B, b);
      if ((dry >> b) & 1u) a.tile_list[a.ntiles - 1 - kd++] = tile_ref<TX>(B, b);
    }
  }
  const int n = s_n;
  double minev = HUGE_VAL, hmax = 0.;
  for (int k = (int)threadIdx.x; k < n; k += BLOCK)
    coef_cell(a, I, B.x0 + s_cell[k] % MARK_W, B.y0 + s_cell[k] / MARK_W, s_h[k], reduce, minev,
              hmax);
  if (reduce) coef_reduce(a, B.inst, minev, hmax, (int)threadIdx.x < n);
}

// the tile of a workgroup of the passes over every tile
template <class A>
__device__ __forceinline__ int tile_of(const A& a) {
  const int p = (int)blockIdx.x;
  return a.by_tile == 2 ? unbanded(p, a.ntiles) : p;
}

// Coefficient pass on small meshes, one workgroup per tile (128 x 128 cells:
// 5 us; a workgroup per mark block, four tiles in turn, 12 us).
template <int TX>
__global__ __launch_bounds__(BLOCK) void k_coef_tile(StepArgs a, int reduce) {
  const TileDev t = a.tiles[tile_of(a)];
  const uint32_t z = a.mk_in ? a.mk_in[t.mw] : 0u;
  if (z == MARK_FULL || (a.zbytes && ((z >> (8 * mark_byte<TX>(t))) & 1u))) return;
  const InstDev I = a.inst[t.inst];
  const int i = t.x0 + (int)(threadIdx.x % TX), j = t.y0 + (int)(threadIdx.x / TX);
  const bool act = i < t.nx && j < t.ny;
  const long long c = t.off + (long long)j * t.nx + i;
  const double h = act ? a.U.h[c] : 0.;
  const bool wet = act && h > a.tiny;
  double minev = HUGE_VAL, hmax = 0.;
  if (wet) coef_cell(a, I, i, j, h, reduce, minev, hmax);
  else if (act && !(h < a.tiny)) a.kact[c] = I.eps;  // (as in k_coef)
  if (a.active) {
    const int cnt = __syncthreads_count(wet);
    if (threadIdx.x == 0 && cnt) atomicAdd(a.active, (unsigned long long)cnt);
  }
  if (a.short_cells) {
    const int cnt = __syncthreads_count(act && !wet);
    if (threadIdx.x == 0 && cnt) atomicAdd(a.short_cells, (unsigned long long)cnt);
  }
  if (reduce) coef_reduce(a, t.inst, minev, hmax, wet);
}

// Both sets of reduction cells, and each member's clock slot of the step about
// to be taken.
__global__ void k_reset_red(RedDev* red, int ninst, const double* time, double* clock,
                            long long stride) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < ninst) {
    for (int k = 0; k < NRED; k++) {
      red_clear(red, b, k);
      red_clear(red, ninst + b, k);
    }
    if (clock) clock[b * stride] = time[b];
  }
}

// Plain fill / copy kernels: used instead of memset / memcpy nodes so a
// captured sweep holds kernel nodes only.
__global__ void k_zero_u32(uint32_t* p, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = 0u;
}
__global__ void k_copy_u32(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                           long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// MaxH box record (check_maxh, calc_adjoint.C:443-465): each workgroup
// takes one chunk of a member's box cells and raises rec[member][step] to
// the largest h > 0 among them.  The running value starts at +0.0 and only
// grows by a strict '>' (NaN never wins), so it is a non-negative double
// whose bit pattern orders like the integer: an integer atomicMax is exact.
template <class S>
__global__ void __launch_bounds__(256) k_box_max(const BoxChunk* __restrict__ ch,
                                                 const long long* __restrict__ cells,
                                                 const S* __restrict__ h,
                                                 unsigned long long* rec, int max_steps,
                                                 int step) {
  __shared__ double wm[4];
  const BoxChunk c = ch[blockIdx.x];
  double m = 0.;
  for (int i = c.begin + (int)threadIdx.x; i < c.end; i += 256) {
    const double v = (double)h[cells[i]];
    m = (v > m) ? v : m;
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; w++) m = (wm[w] > m) ? wm[w] : m;
    if (m > 0.) atomicMax(rec + (long long)c.inst * max_steps + step, dbits(m));
  }
}

// The three field ranges [off, off + count) of one member (words of `es`
// bytes in buffers of `field_bytes` per field): copied from src, or zeroed
// when src is null; the member's zero-mark words [mw0, mw0 + nmw) of dst are
// cleared (nothing known) after a copy.
__global__ void k_member_fill(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                              long long field_words, long long off_words, long long nwords,
                              uint32_t* mk, long long mw0, long long nmw) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long t0 = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  for (int f = 0; f < 3; f++) {
    const long long base = f * field_words + off_words;
    for (long long i = t0; i < nwords; i += stride)
      dst[base + i] = src ? src[base + i] : 0u;
  }
  if (src && mk)
    for (long long i = t0; i < nmw; i += stride) mk[mw0 + i] = 0u;
}

// Face records of one tile: every face flux and every one-sided difference
// the tile's cells use is computed once (a face is shared by two cells) and
// staged in LDS.  x-face fi of row fj lies between tile columns fi-1 and fi.
template <int TX>
struct FaceLds {
  static constexpr int TY = BLOCK / TX, RX = TX + 2, RXY = (TX + 2) * (TY + 2);
  double fx[3][TY][TX + 1], fy[3][TY + 1][TX];
  double dxh[TY][TX + 1], dxhv[TY][TX + 1];  // (U_right - U_left) / dx of h, hv
  double dyh[TY + 1][TX], dyhu[TY + 1][TX];  // (U_top - U_bottom) / dy of h, hu
  // records of the tile and its side strips: the state and, for h >= tiny,
  // hu/h, hv/h and sqrt(kact h g2) -- hfv_fwd's values, evaluated once per
  // cell instead of once per face
  double h[RXY], hu[RXY], hv[RXY], vx[RXY], vy[RXY], sq[RXY];
};
// threads of the update: one for every face of a tile, or one for every record
// (the faces then take two rounds)
template <int TX>
constexpr int face_threads() {
  return ((TX + 1) * (BLOCK / TX) + TX * (BLOCK / TX + 1) + 63) / 64 * 64;
}
template <int TX>
constexpr int record_threads() {
  return BLOCK + (2 * TX + 2 * (BLOCK / TX) + 63) / 64 * 64;
}

// riemannflux (tg_math.h) of the face between records l and r along dir
// (0 x, 1 y) and their one-sided differences: the three quotients share the
// reciprocal of their denominator
template <int TX>
__device__ __forceinline__ void face_flux(const FaceLds<TX>& L, int dir, int l, int r,
                                          double tiny, double flux[3]) {
  const double lh = L.h[l] < tiny ? 0. : L.h[l], rh = L.h[r] < tiny ? 0. : L.h[r];
  flux[0] = flux[1] = flux[2] = 0.;
  if (lh == 0. && rh == 0.) return;
  const double* V = dir ? L.vy : L.vx;
  const bool lz = L.h[l] < tiny, rz = L.h[r] < tiny;
  const double lu[3] = {lh, lz ? 0. : L.hu[l], lz ? 0. : L.hv[l]};
  const double ru[3] = {rh, rz ? 0. : L.hu[r], rz ? 0. : L.hv[r]};
  const double lv = V[l], rv = V[r], la = L.sq[l], ra = L.sq[r];  // 0 below tiny
  double lf[3], rf[3];
  lf[0] = dir ? lu[2] : lu[1];
  rf[0] = dir ? ru[2] : ru[1];
  const double lp = 0.5 * la * la * lh, rp = 0.5 * ra * ra * rh;
  lf[1] = lu[1] * lv; lf[2] = lu[2] * lv;
  rf[1] = ru[1] * rv; rf[2] = ru[2] * rv;
  if (dir) { lf[2] += lp; rf[2] += rp; }
  else { lf[1] += lp; rf[1] += rp; }
  const double lw0 = lv - la, lw2 = lv + la, rw0 = rv - ra, rw2 = rv + ra;
  double sl, sr;
  if (lh == 0.) {
    sl = umin(0, 2.0 * rw0 - rv);
    sr = umax(0, 2.0 * rw2 - rv);
  } else if (rh == 0.) {
    sl = umin(0, 2.0 * lw0 - lv);
    sr = umax(0, 2.0 * lw2 - lv);
  } else {
    sl = umin(0, umin(lw0, rw0));
    sr = umax(0, umax(lw2, rw2));
  }
  if (sl >= 0.0) {
#pragma unroll
    for (int v = 0; v < 3; v++) flux[v] = lf[v];
  } else if (sr <= 0.0) {
#pragma unroll
    for (int v = 0; v < 3; v++) flux[v] = rf[v];
  } else {
    const double d = sr - sl, g = 1. / d, ss = sl * sr;
#pragma unroll
    for (int v = 0; v < 3; v++)
      flux[v] = div_r(sr * lf[v] - sl * rf[v] + ss * (ru[v] - lu[v]), d, g);
  }
}

// The dry tile's cells: update_states' own arithmetic with zero fluxes, bit for
// bit (U - dtdx (0 - 0) - dtdy (0 - 0), h clamped at 0; inf and NaN included).
// Returns whether the new state is +0.0.
__device__ __forceinline__ bool dry_cell(const StepArgs& a, const InstDev& I, double dt,
                                         double h, double hu, double hv, double out[3]) {
  const double dtdx = dt / I.dx, dtdy = dt / I.dy, zero = 0.;
  out[0] = h; out[1] = hu; out[2] = hv;
#pragma unroll
  for (int v = 0; v < 3; v++) out[v] = out[v] - dtdx * (zero - zero) - dtdy * (zero - zero);
  if (out[0] < 0.) out[0] = 0;
  if (!isfinite(out[0]) || !isfinite(out[1]) || !isfinite(out[2])) atomicOr(a.err, 1);
  return bitzero3(out[0], out[1], out[2]);
}

// What the corrector reads of a tile's own cell besides the faces.
struct CellIn {
  double h, hu, hv, k, gx, gy, gz, dgx, dgy, kx, ky;
};

// update_tile's per-cell part: slopes from the staged differences, the four
// face fluxes with outflow copies, update_states; z: the new state is +0.0.
template <int TX>
__device__ __forceinline__ void update_cell(const StepArgs& a, const TileRef& t,
                                            const InstDev& I, const Cell& q, const CellIn& u,
                                            double dt, const FaceLds<TX>& L, bool& z) {
  const int tx = (int)(threadIdx.x % TX), ty = (int)(threadIdx.x / TX);
  const long long c = q.c;
  const double prev[3] = {u.h, u.hu, u.hv};
  // Element::get_slopes, element2.C:830-939 (only the components the
  // corrector reads: hx, hvx, hy, huy); boundary cells keep zero slopes
  double hx = 0., hvx = 0., hy = 0., huy = 0.;
  if (q.hasE && q.hasW && q.hasN && q.hasS) {
    hx = slope_from(L.dxh[ty][tx + 1], L.dxh[ty][tx], I.dx, I.inv_sx, a.gamma, a.tiny);
    hvx = slope_from(L.dxhv[ty][tx + 1], L.dxhv[ty][tx], I.dx, I.inv_sx, a.gamma, a.tiny);
    hy = slope_from(L.dyh[ty + 1][tx], L.dyh[ty][tx], I.dy, I.inv_sy, a.gamma, a.tiny);
    huy = slope_from(L.dyhu[ty + 1][tx], L.dyhu[ty][tx], I.dy, I.inv_sy, a.gamma, a.tiny);
  }
  // a face on the domain boundary takes the flux of the opposite face
  // (boundary_flux, element2.C:3374-3411)
  double fE[3], fW[3], fN[3], fS[3];
  for (int v = 0; v < 3; v++) {
    fE[v] = q.hasE ? L.fx[v][ty][tx + 1] : (q.hasW ? L.fx[v][ty][tx] : 0.);
    fW[v] = q.hasW ? L.fx[v][ty][tx] : fE[v];
    fN[v] = q.hasN ? L.fy[v][ty + 1][tx] : (q.hasS ? L.fy[v][ty][tx] : 0.);
    fS[v] = q.hasS ? L.fy[v][ty][tx] : fN[v];
  }
  // correct() -> update_states (corrector.C:36-140, residual.C:162-275)
  const double kc = (prev[0] > a.tiny) ? u.k : I.eps;
  double out[3];
  SrcInfo si;
  update_states(prev, out, fE, fN, fW, fS, div_r(dt, I.dx, I.inv_dx), div_r(dt, I.dy, I.inv_dy),
                dt, hx, hvx, hy, huy, u.kx, u.ky, I.sin_int,
                mat_of(I, a.mat, a.mtab, c).tan_bed, u.gx, u.gy, u.gz, u.dgx, u.dgy, kc, a.ft,
                a.tiny, &si);
  if (!isfinite(out[0]) || !isfinite(out[1]) || !isfinite(out[2])) atomicOr(a.err, 1);
  a.h_out[c] = out[0];
  a.hu_out[c] = out[1];
  a.hv_out[c] = out[2];
  z = bitzero3(out[0], out[1], out[2]);
}

// Update of one tile: records of the tile and its side strips (the first 256
// threads the tile's own cells, whose corrector inputs stay in registers),
// every face once, update_states per cell.  MAYBE_DRY: the tile is not known
// to be wet; a dry one is written here as the classifying pass would.
// What bounds it is the chain of one tile: one round trip to memory, then
// records, faces and cells; so each phase has a thread per item where a tile
// is all a CU has (576 to 640 threads, 9 to 7 us for 128 x 128 cells, the
// list walk's 256 threads 9.5 us), and a thread per record, two rounds of
// faces, where several tiles share a CU (64 members, 5.8 M cells: 20 us;
// one thread per face 40 us, 256 threads on 64 x 4 tiles 27.5 us).
template <int TX, int NT, bool MAYBE_DRY>
__device__ __forceinline__ void update_tile(const StepArgs& a, const TileRef& t, double dt,
                                            FaceLds<TX>& L) {
  constexpr int TY = BLOCK / TX, RX = FaceLds<TX>::RX, RY = TY + 2, NHALO = 2 * TX + 2 * TY;
  constexpr int NFX = (TX + 1) * TY, NFY = TX * (TY + 1);
  static_assert(BLOCK + NHALO <= NT, "one thread per record");
  const InstDev I = a.inst[t.inst];
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));  // indexes rebuilt per tile, not held over the tile loop
  Cell q = cell_of<TX>(t);
  q.act = q.act && tid < BLOCK;
  CellIn u = {};
  bool wet = false;
  if (tid < BLOCK + NHALO) {
    int rx, ry;
    const int h0 = tid - BLOCK;
    if (h0 < 0) { rx = tid % TX + 1; ry = tid / TX + 1; }
    else if (h0 < TX) { rx = h0 + 1; ry = 0; }
    else if (h0 < 2 * TX) { rx = h0 - TX + 1; ry = RY - 1; }
    else if (h0 < 2 * TX + TY) { rx = 0; ry = h0 - 2 * TX + 1; }
    else { rx = RX - 1; ry = h0 - 2 * TX - TY + 1; }
    const int gi = t.x0 - 1 + rx, gj = t.y0 - 1 + ry;
    if (gi >= 0 && gi < t.nx && gj >= 0 && gj < t.ny) {
      const long long c = t.off + (long long)gj * t.nx + gi;
      double h = a.U.h[c], hu = a.U.hu[c], hv = a.U.hv[c], k = a.kact[c], gz = a.S.gz[c];
      if (h0 < 0) {
        u.gx = a.S.gx[c]; u.gy = a.S.gy[c]; u.dgx = a.S.dgx[c]; u.dgy = a.S.dgy[c];
        u.kx = a.S.kx[c]; u.ky = a.S.ky[c];
      }
      // all of them in flight together, not each where it is used
      asm volatile("" : "+v"(hu), "+v"(hv), "+v"(k), "+v"(gz), "+v"(u.gx), "+v"(u.gy),
                        "+v"(u.dgx), "+v"(u.dgy), "+v"(u.kx), "+v"(u.ky));
      u.h = h; u.hu = hu; u.hv = hv; u.k = k; u.gz = gz;
      wet = !(h < a.tiny);
      const int r = ry * RX + rx;
      L.h[r] = h; L.hu[r] = hu; L.hv[r] = hv;
      double vx = 0., vy = 0., sq = 0.;
      if (wet) {
        const double inv = 1. / h;
        vx = div_r(hu, h, inv);
        vy = div_r(hv, h, inv);
        sq = sqrt(k * h * gz);
      }
      L.vx[r] = vx; L.vy[r] = vy; L.sq[r] = sq;
    }
  }
  if (MAYBE_DRY) {
    if (!__syncthreads_or(wet)) {
      // every face flux is zero and there are no sources: update_states'
      // own arithmetic with zero fluxes
      const bool zin = a.mk_in && a.zbytes && (a.mk_in[t.mw] >> (8 * mark_byte<TX>(t))) & 1u;
      const bool keep = zin && a.mk_out && isfinite(dt) &&
                        (a.mk_out[t.mw] >> (8 * mark_byte<TX>(t))) & 1u;
      bool z = true;
      if (q.act) {
        double out[3];
        z = dry_cell(a, I, dt, u.h, u.hu, u.hv, out);
        if (!keep) {
          a.h_out[q.c] = out[0];
          a.hu_out[q.c] = out[1];
          a.hv_out[q.c] = out[2];
        }
      }
      if (a.short_cells) {
        const int cnt = __syncthreads_count(q.act);
        if (tid == 0) atomicAdd(a.short_cells, (unsigned long long)cnt);
      }
      if (a.mk_out) mark_store<TX>(a.mk_out, t, __syncthreads_and(z));
      return;
    }
  } else {
    __syncthreads();
  }
  if (a.active) {
    const int cnt = __syncthreads_count(q.act);
    if (tid == 0) atomicAdd(a.active, (unsigned long long)cnt);
  }
  // faces with a cell of the member on both sides (calc_edge_states,
  // element2.C:2744-3072)
#pragma unroll 1
  for (int k = tid; k < NFX + NFY; k += NT) {
    const bool isx = k < NFX;
    const int f = isx ? k : k - NFX, W = isx ? TX + 1 : TX;
    const int fi = f % W, fj = f / W;
    const int gi = t.x0 + fi, gj = t.y0 + fj;
    if (gi < t.nx && gj < t.ny && (isx ? gi > 0 : gj > 0)) {
      const int r = (fj + 1) * RX + fi + 1, l = isx ? r - 1 : r - RX;  // upper cell, lower cell
      double fl[3];
      if (isx) {
        face_flux<TX>(L, 0, l, r, a.tiny, fl);
        for (int v = 0; v < 3; v++) L.fx[v][fj][fi] = fl[v];
        L.dxh[fj][fi] = div_r(L.h[r] - L.h[l], I.dx, I.inv_dx);
        L.dxhv[fj][fi] = div_r(L.hv[r] - L.hv[l], I.dx, I.inv_dx);
      } else {
        face_flux<TX>(L, 1, l, r, a.tiny, fl);
        for (int v = 0; v < 3; v++) L.fy[v][fj][fi] = fl[v];
        L.dyh[fj][fi] = div_r(L.h[r] - L.h[l], I.dy, I.inv_dy);
        L.dyhu[fj][fi] = div_r(L.hu[r] - L.hu[l], I.dy, I.inv_dy);
      }
    }
  }
  __syncthreads();
  bool z = true;
  if (q.act) update_cell<TX>(a, t, I, q, u, dt, L, z);
  if (a.mk_out) mark_store<TX>(a.mk_out, t, __syncthreads_and(z));
}

// A listed dry tile.
template <int TX, int NT>
__device__ __forceinline__ void update_dry_tile(const StepArgs& a, const TileRef& t, double dt) {
  const InstDev I = a.inst[t.inst];
  const Cell q = cell_of<TX>(t);
  const bool act = q.act && threadIdx.x < BLOCK;
  bool z = true;
  if (act) {
    double out[3];
    z = dry_cell(a, I, dt, a.U.h[q.c], a.U.hu[q.c], a.U.hv[q.c], out);
    a.h_out[q.c] = out[0];
    a.hu_out[q.c] = out[1];
    a.hv_out[q.c] = out[2];
  }
  if (a.short_cells) {
    const int cnt = __syncthreads_count(act);
    if (threadIdx.x == 0) atomicAdd(a.short_cells, (unsigned long long)cnt);
  }
  if (a.mk_out) mark_store<TX>(a.mk_out, t, __syncthreads_and(z));
}

// Second pass on large meshes: a fixed grid walks the full list, then the dry
// one.  The first workgroups also keep the members' records (step_dt); a dt
// that is not finite makes every cell so, the unlisted ones too, so it is
// reported here as the state it would give is (see k_spoil_members).
template <int TX>
__global__ __launch_bounds__(record_threads<TX>(), 5) void k_update(StepArgs a) {
  __shared__ FaceLds<TX> L;
  const int n = a.tile_count[0], nd = a.tile_count[1];
  if (blockIdx.x == 0 && threadIdx.x < 2) a.count_next[threadIdx.x] = 0;
  for (int b = (int)blockIdx.x; b < a.ninst; b += (int)gridDim.x)
    if (!isfinite(step_dt(a, b, true)) && threadIdx.x == 0) atomicOr(a.err, 1);
  for (int i = (int)blockIdx.x; i < n; i += (int)gridDim.x) {
    const TileRef t = a.tile_list[list_band(i, n)];
    update_tile<TX, record_threads<TX>(), false>(a, t, step_dt(a, t.inst, false), L);
    __syncthreads();  // LDS reused by the next tile
  }
  // (from the grid's end: its last workgroups have the fewest full tiles)
  for (int i = (int)(gridDim.x - 1 - blockIdx.x); i < nd; i += (int)gridDim.x) {
    const TileRef t = a.tile_list[a.ntiles - 1 - i];
    update_dry_tile<TX, record_threads<TX>()>(a, t, step_dt(a, t.inst, false));
  }
}

__device__ __forceinline__ TileRef ref_of(const TileDev& t, int tile) {
  return TileRef{t.inst, tile, t.x0, t.y0, t.mw, t.nx, t.ny, 0, t.off};
}

// Update on small meshes, one workgroup per tile, nothing listed.
template <int TX>
__global__ __launch_bounds__(face_threads<TX>()) void k_update_tile(StepArgs a) {
  __shared__ FaceLds<TX> L;
  const int tile = tile_of(a);
  const TileDev t = a.tiles[tile];
  const bool own = t.x0 == 0 && t.y0 == 0;  // keeps the member's records
  // (looked at before dt is made, which the workgroups of empty tiles then never
  // do; a dt that is not finite: see k_spoil_members)
  const bool skip = a.mk_in && update_skip(a.mk_in, t) && out_marked_zero<TX>(a.mk_out, t);
  if (skip && !own) return;
  const double dt = step_dt(a, t.inst, own);
  if (own && threadIdx.x == 0 && !isfinite(dt)) atomicOr(a.err, 1);
  if (skip && isfinite(dt)) return;
  update_tile<TX, face_threads<TX>(), true>(a, ref_of(t, tile), dt, L);
}

__global__ __launch_bounds__(BLOCK) void k_stats(const InstDev* inst, const TileDev* tiles,
                                                 Fields U, const uint32_t* mk,
                                                 double* part_mass, double* part_hmax,
                                                 double tiny) {
  const TileDev t = tiles[blockIdx.x];
  if (mk && mk[t.mw] == MARK_FULL) {  // the block holds +0.0: no mass, no depth
    if (threadIdx.x == 0) { part_mass[blockIdx.x] = 0.; part_hmax[blockIdx.x] = 0.; }
    return;
  }
  const InstDev I = inst[t.inst];
  const Cell q = cell_of<64>(t, I);
  double m = 0., hm = 0.;
  if (q.act) {
    double h = U.h[q.c];
    m = I.dx * I.dy * h;
    if (h > tiny) hm = h;
  }
  __shared__ double sm[BLOCK / 64], sh[BLOCK / 64];
  m = wave_sum(m);
  hm = wave_max(hm);
  if (threadIdx.x % 64 == 0) { sm[threadIdx.x / 64] = m; sh[threadIdx.x / 64] = hm; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < BLOCK / 64; k++) { m += sm[k]; hm = (sh[k] > hm) ? sh[k] : hm; }
    part_mass[blockIdx.x] = m;
    part_hmax[blockIdx.x] = hm;
  }
}

// Copies a state buffer's three fields (raw bits, W the element's width)
// one mark block per workgroup and gives the source and the copy the zero
// marks of what it read: byte b of the block's word is 1 when tile b
// (block_cells' order, TX the update's tile width) holds +0.0 in all three
// fields.  A source whose marks were cleared (a state set from the host)
// and its checkpoint copy then let the next steps skip what is empty.  With
// dst and mk_dst null, only the source's marks are written.  A block of the
// copy marked whole +0.0 (MARK_FULL, meaningful in every tile shape) whose
// source block is +0.0 is not rewritten.
template <int TX, class W>
__global__ __launch_bounds__(BLOCK) void k_copy_marking(const BlockDev* blocks, const W* s0,
                                                        const W* s1, const W* s2, W* dst,
                                                        long long ncell, uint32_t* mk_src,
                                                        uint32_t* mk_dst) {
  const BlockDev B = blocks[blockIdx.x];
  __shared__ unsigned s_nz;
  if (threadIdx.x == 0) s_nz = 0u;
  // a copy whose block already holds +0.0 (word MARK_FULL) is not rewritten
  // where the source block is +0.0 too
  const bool dst_zero = mk_dst && mk_dst[B.mw] == MARK_FULL;
  Cell q[4];
  block_cells<TX>(B, q);
  W v[4][3];
  unsigned nz = 0u;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    v[b][0] = v[b][1] = v[b][2] = (W)0;
    if (!q[b].act) continue;
    const long long c = q[b].c;
    v[b][0] = s0[c]; v[b][1] = s1[c]; v[b][2] = s2[c];
    if ((v[b][0] | v[b][1] | v[b][2]) != (W)0) nz |= 1u << b;
  }
  __syncthreads();  // s_nz cleared
  if (nz) atomicOr(&s_nz, nz);
  __syncthreads();
  if (dst && !(dst_zero && s_nz == 0u)) {
#pragma unroll
    for (int b = 0; b < 4; b++) {
      if (!q[b].act) continue;
      const long long c = q[b].c;
      dst[c] = v[b][0];
      dst[ncell + c] = v[b][1];
      dst[2 * ncell + c] = v[b][2];
    }
  }
  if (threadIdx.x == 0) {
    uint32_t w = 0u;
#pragma unroll
    for (int b = 0; b < 4; b++)
      if (B.tile[b] >= 0 && !((s_nz >> b) & 1u)) w |= 1u << (8 * b);
    mk_src[B.mw] = w;
    if (mk_dst) mk_dst[B.mw] = w;
  }
}

// One workgroup per member b: out[b] = sum of sum_part over member b's
// tiles idx[off[b] .. off[b+1]) (each lane adds its strided share in list
// order, the lanes combine by a fixed tree, so the result does not depend on
// the launch), out[n + b] = the max of max_part over them (when given),
// out[2n + b] = time[b] and out[3n + b] = dt_rec[b * stride + col] (when
// given), out[4n] = *err.  out is pinned host memory, so that one wait for the
// stream hands a step's results to the host; two copies to it, of the error
// word and of the results, each with a wait of its own, and the parameters'
// upload before it took longer than the step's kernels (128 x 128 cells, a
// host's own loop: 61 us a step against 37).
__global__ __launch_bounds__(BLOCK) void k_member_reduce(const double* sum_part,
                                                         const double* max_part,
                                                         const int* off, const int* idx, int n,
                                                         const double* time,
                                                         const double* dt_rec, long long stride,
                                                         int col, const int* err, double* out) {
  const int b = blockIdx.x;
  double s = 0., m = 0.;
  for (int j = off[b] + (int)threadIdx.x; j < off[b + 1]; j += BLOCK) {
    const int t = idx[j];
    s += sum_part[t];
    if (max_part) m = (max_part[t] > m) ? max_part[t] : m;
  }
  __shared__ double ss[BLOCK / 64], sm[BLOCK / 64];
  s = wave_sum(s);
  m = wave_max(m);
  if (threadIdx.x % 64 == 0) { ss[threadIdx.x / 64] = s; sm[threadIdx.x / 64] = m; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < BLOCK / 64; k++) { s += ss[k]; m = (sm[k] > m) ? sm[k] : m; }
    out[b] = s;
    if (max_part) out[n + b] = m;
    if (time) out[2 * n + b] = time[b];
    if (dt_rec) out[3 * n + b] = dt_rec[(long long)b * stride + col];
    if (b == 0) out[4 * n] = (double)*err;
  }
}

__global__ void k_set_time(double* time, int n, double t, int* err) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < n) time[b] = t;
  if (b == 0 && err) *err = 0;
}

// After a step whose dt was not finite (one of `steps` recorded ones): every
// cell of the member is NaN, as inf - inf makes it.  The passes that leave tiles
// of +0.0 alone do so without a look at dt; looking there costs every step (2 %
// of 64 members' steps by its registers alone), this only the failing call.
constexpr int SPOIL_GRID = 64;  // workgroups a member
template <class S>
__global__ __launch_bounds__(BLOCK) void k_spoil_members(const InstDev* inst, const double* dt_rec,
                                                         long long stride, int steps, S* h, S* hu,
                                                         S* hv, uint32_t* mk) {
  const int b = (int)blockIdx.x / SPOIL_GRID;
  bool bad = false;
  for (int s = (int)threadIdx.x; s < steps; s += BLOCK) bad = bad || !isfinite(dt_rec[b * stride + s]);
  if (!__syncthreads_or(bad)) return;
  const InstDev I = inst[b];
  const long long n = (long long)I.nx * I.ny, m = (long long)I.nsx * I.nsy;
  const long long first = (long long)(blockIdx.x % SPOIL_GRID) * BLOCK + threadIdx.x;
  for (long long i = first; i < n; i += SPOIL_GRID * BLOCK)
    h[I.off + i] = hu[I.off + i] = hv[I.off + i] = (S)NAN;
  for (long long i = first; mk && i < m; i += SPOIL_GRID * BLOCK) mk[I.soff + i] = 0u;
}

// (one launch for a copy and two fills; with the three fields of lambda in one
// copy each way and the gradient read with lambda's wait, a reverse step from
// and to the host takes 200 us against 263 at 301 x 257 cells)
__global__ void k_reverse_setup(double* dt_rec, long long stride, int n, double dt, uint32_t* z0,
                                long long n0, uint32_t* z1, long long n1) {
  const long long t0 = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  const long long all = (long long)gridDim.x * blockDim.x;
  for (long long i = t0; i < n; i += all) dt_rec[i * stride] = dt;
  for (long long i = t0; i < n0; i += all) z0[i] = 0u;
  for (long long i = t0; i < n1; i += all) z1[i] = 0u;
}

// ---------------------------------------------------------------- adjoint --

// A double from the other thread of a pair (two 32-bit DPP moves, no LDS).
__device__ __forceinline__ double swap_pair(double v) {
  constexpr int ctrl = 1 | (0 << 2) | (3 << 4) | (2 << 6);
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Reverse step, one tile of 256 cells by 512 threads.
//
// Phase 1, one thread per record (the tile's cells and the four side
// strips of its halo): the dual slopes, kact, source switches and what the
// faces and blocks read of a cell, staged in LDS with its lambda^{s+1}.  Every
// load of a record is issued before any of it is looked at.
// Phase 2, two threads per cell, one its y faces and one its x faces: the
// faces' Jacobians with respect to the cell (dual_riemannflux,
// dualmesh.C:1628-1843) in the face's own frame -- 0 depth, n normal and t
// tangential momentum -- where seven of the nine entries can differ from
// zero (rows 0 and n have no t column), then the gather lambda^s = g -
// sum_j J_j^T lambda_j, whose running sum the pair hands back and forth in the
// reference's order self, S, E, N, W (neighbor[0..3] with positive_x_side =
// 1).  The products left out are exact zeros where lambda^{s+1} is finite, and
// adding a zero to a running sum that starts at +0.0 changes nothing, so the
// result is the reference's bit for bit.  The bed-friction gradient's face
// fluxes come out of the same evaluation.
//
// What bounds it: FP64 instruction issue (52 % of the issue slots at 128
// VGPRs, four waves per SIMD) and, per tile, three round trips to memory (list
// entry, records, results).  A 64-member ensemble of 5.8 M cells: 60 us per
// step against 81 us for one thread per cell with every face's forward and
// dual flux evaluated apart; one tile alone (128 x 128 cells): 12 against 27
// us.  One thread per cell needs 168 VGPRs (81 us), four per cell repeat the
// self block (75 us).
template <int TX, bool DPHI>
struct DualLds {
  static constexpr int RX = TX + 2, RN = (TX + 2) * (BLOCK / TX + 2);
  // records: the state, +0.0 where h < tiny (the flux functions' void side),
  // 1/h and sqrt(kact h g2)
  double h[RN], hu[RN], hv[RN], inv[RN], sq[RN];
  // the source term that the cell's block as x- / x+ / y- / y+ neighbour's
  // neighbour subtracts (compute_jacobian_elem.C:44-51)
  double src[4][RN];
  double lam[3][RN];  // lambda^{s+1}
  // bed-friction gradient: hu/h and hv/h, and d kact / d phi_bed times d F_n /
  // d kact and d sqrt(kact h g2) / d kact
  double vx[DPHI ? RN : 1], vy[DPHI ? RN : 1], dF[DPHI ? RN : 1], dw[DPHI ? RN : 1];
  // the tile's cells: what the self block subtracts from its entries 10, 10,
  // 11, 20, 20, 22 (compute_jacobian_elem.C:55-110), the sources' phi_bed
  // derivatives, and whether h != 0
  double self[6][BLOCK];
  double dsrc[2][DPHI ? BLOCK : 1];
  double sp[BLOCK / 64];
  unsigned char nz[BLOCK];
};
constexpr int ADJ_THREADS = 2 * BLOCK;

// .5 * c_sgn and f_sgn (tg_math.h) by the sign bit
__device__ __forceinline__ double half_sgn(double z, double tiny) {
  return fabs(z) > tiny ? copysign(.5, z) : 0.;
}
// slope_dual (tg_math.h); hs: its sensitivities for the cell itself and its
// minus and plus neighbour
__device__ __forceinline__ double dslope(double up, double uc, double um, double dx, double inv,
                                         double inv_s, double gamma, double tiny,
                                         double* hs = nullptr) {
  const double dp = (up - uc) * inv, dm = (uc - um) * inv;
  const double dc = (dp * dx + dm * dx) * inv_s;
  const double gp = gamma * fabs(dp), gm = gamma * fabs(dm);
  const double mn = fmin(fmin(gp, gm), fabs(dc));
  const double sg = half_sgn(dp, tiny) + half_sgn(dm, tiny);
  if (hs) {
    const bool on = sg != 0., P = mn == gp, M = !P && mn == gm, C = !P && !M;
    const double cen = inv * (dx * inv_s), one = on ? inv : 0.;
    hs[0] = P ? -one : M ? one : 0.;
    hs[1] = M ? -one : (on && C) ? -cen : 0.;
    hs[2] = P ? one : (on && C) ? cen : 0.;
  }
  return sg * mn;
}

// The record of cell (i, j) in slot r; own >= 0: also the self terms of the
// tile's cell `own` (DualElem after update_dual_grid, dual_grid_routines.C:
// 68-84, and update_states in calc_jacobian).  Returns whether the cell is not
// void (h != 0, or with the gradient lambda^{s+1} != 0).
template <int TX, bool DPHI>
__device__ __forceinline__ bool dual_record(const AdjArgs& a, const TileRef& t, const InstDev& I,
                                            int i, int j, double dt, DualLds<TX, DPHI>& L, int r,
                                            int own) {
  const long long c = t.off + (long long)j * t.nx + i;
  // cells on the domain boundary have zero slopes: with themselves as
  // neighbours every difference is 0, and so are slope and sensitivities
  const bool inner = i + 1 < t.nx && i > 0 && j + 1 < t.ny && j > 0;
  const long long ox = inner ? 1 : 0, oy = inner ? t.nx : 0;
  double h = a.U.h[c], hu = a.U.hu[c], hv = a.U.hv[c];
  double hE = a.U.h[c + ox], hW = a.U.h[c - ox], hN = a.U.h[c + oy], hS = a.U.h[c - oy];
  double uE = a.U.hu[c + ox], uW = a.U.hu[c - ox], uN = a.U.hu[c + oy], uS = a.U.hu[c - oy];
  double vE = a.U.hv[c + ox], vW = a.U.hv[c - ox], vN = a.U.hv[c + oy], vS = a.U.hv[c - oy];
  double g2 = a.S.gz[c], k0 = a.S.kx[c], k1 = a.S.ky[c];
  double l0 = a.lam_next.h[c], l1 = a.lam_next.hu[c], l2 = a.lam_next.hv[c];
  double g0 = 0., g1 = 0., dg0 = 0., dg1 = 0.;
  if (own >= 0) { g0 = a.S.gx[c]; g1 = a.S.gy[c]; dg0 = a.S.dgx[c]; dg1 = a.S.dgy[c]; }
  // all of them in flight together (used only below a test of h, they
  // would be loaded after it)
  asm volatile("" : "+v"(hE), "+v"(hW), "+v"(hN), "+v"(hS), "+v"(uE), "+v"(uW), "+v"(uN),
                    "+v"(uS), "+v"(vE), "+v"(vW), "+v"(vN), "+v"(vS));
  asm volatile("" : "+v"(g2), "+v"(k0), "+v"(k1), "+v"(g0), "+v"(g1), "+v"(dg0), "+v"(dg1),
                    "+v"(l0), "+v"(l1), "+v"(l2));
  L.lam[0][r] = l0; L.lam[1][r] = l1; L.lam[2][r] = l2;
  const bool busy = h != 0. || (DPHI && !(l0 == 0. && l1 == 0. && l2 == 0.));
  if (own >= 0) L.nz[own] = h != 0.;
  if (!(h > a.tiny)) {
    // void side of every flux, or (h = tiny, or not a number) a dry cell:
    // kact = epsilon, no slopes and no sources
    const bool flows = !(h < a.tiny);
    L.h[r] = flows ? h : 0.;
    L.hu[r] = flows ? hu : 0.;
    L.hv[r] = flows ? hv : 0.;
    L.inv[r] = flows ? 1. / h : 0.;
    L.sq[r] = flows ? sqrt(1. * I.eps * h * g2) : 0.;
#pragma unroll
    for (int k = 0; k < 4; k++) L.src[k][r] = 0.;
    if (DPHI) {
      L.vx[r] = flows ? hu / h : 0.;
      L.vy[r] = flows ? hv / h : 0.;
      L.dF[r] = L.dw[r] = 0.;
    }
    if (own >= 0) {
#pragma unroll
      for (int k = 0; k < 6; k++) L.self[k][own] = 0.;
      if (DPHI) L.dsrc[0][own] = L.dsrc[1][own] = 0.;
    }
    return busy;
  }
  const MatDev M = mat_of(I, a.mat, a.mtab, c);
  const double ix = I.inv_dx, isx = I.inv_sx, iy = I.inv_dy, isy = I.inv_sy;
  double sx[3], sy[3];
  const double hx = dslope(hE, h, hW, I.dx, ix, isx, a.gamma, a.tiny, sx);
  const double hy = dslope(hN, h, hS, I.dy, iy, isy, a.gamma, a.tiny, sy);
  const double hux = dslope(uE, hu, uW, I.dx, ix, isx, a.gamma, a.tiny);
  const double hvx = dslope(vE, hv, vW, I.dx, ix, isx, a.gamma, a.tiny);
  const double huy = dslope(uN, hu, uS, I.dy, iy, isy, a.gamma, a.tiny);
  const double hvy = dslope(vN, hv, vS, I.dy, iy, isy, a.gamma, a.tiny);
  const double inv = 1. / h;
  const double vx = div_r(hu, h, inv), vy = div_r(hv, h, inv);
  L.h[r] = h; L.hu[r] = hu; L.hv[r] = hv; L.inv[r] = inv;
  // getcoef (tg_math.h) and its phi_bed derivative
  const double hh = h * h, ihh = 1. / hh;
  const double vel = div_r(hux, h, inv) - div_r(hu * hx, hh, ihh) + div_r(hvy, h, inv) -
                     div_r(hv * hy, hh, ihh);
  const double sg = fabs(vel) < a.tiny ? 0. : copysign(1., vel);
  const bool still = fabs(vx) < a.tiny && fabs(vy) < a.tiny;
  const double kf = I.kc1 * (1. - sg * M.kroot) - 1.;
  const double k = (still ? 1. : (kf < 0. ? 0. : kf)) * I.eps;
  const double sq = sqrt(k * h * g2);
  L.sq[r] = sq;
  // src_switches (tg_math.h)
  const double tb = M.tan_bed;
  const double sgn0 = tiny_sgn(inv * (huy - vx * hy), a.ft), sgn2 = tiny_sgn(vx, a.ft);
  const double sgn1 = tiny_sgn(inv * (hvx - vy * hx), a.ft), sgn3 = tiny_sgn(vy, a.ft);
  const double fx = umax(g2 * h + vx * hu * k0, 0.0), fy = umax(g2 * h + vy * hv * k1, 0.0);
  const bool stop0 = sgn2 * fx * tb == 0. && sgn2 != 0.;
  const bool stop1 = sgn3 * fy * tb == 0. && sgn3 != 0.;
  const double alpha = I.sin_int * sgn0 * k, betta = I.sin_int * sgn1 * k;
  const double bx = stop1 ? 0. : -dt * h * betta * g2, by = stop0 ? 0. : -dt * h * alpha * g2;
  L.src[0][r] = bx * sx[1]; L.src[1][r] = bx * sx[2];
  L.src[2][r] = by * sy[1]; L.src[3][r] = by * sy[2];
  double dk = 0.;
  if (DPHI) {
    dk = (still || kf < 0.) ? 0. : -I.kc1 * sg * M.dkroot * I.eps;
    L.dw[r] = (sq > 0.) ? dk * ((h * g2) / (2. * sq)) : 0.;
    L.dF[r] = dk * (0.5 * h * g2 * h);
    L.vx[r] = vx;
    L.vy[r] = vy;
  }
  if (own >= 0) {
    L.self[0][own] = dt * (g0 - alpha * h * (2 * dg1 + g2 * sy[0]) - alpha * g2 * hy);
    L.self[3][own] = dt * (g1 - betta * h * (2 * dg0 + g2 * sx[0]) - betta * g2 * hx);
    const double f0 = (sgn2 != 0. && !stop0) ? -dt * sgn2 * tb : 0.;
    const double f1 = (sgn3 != 0. && !stop1) ? -dt * sgn3 * tb : 0.;
    L.self[1][own] = f0 * (g2 - vx * vx * k0);
    L.self[2][own] = f0 * (2 * vx * k0);
    L.self[4][own] = f1 * (g2 - vy * vy * k1);
    L.self[5][own] = f1 * (2 * vy * k1);
    if (DPHI) {
      const double sec2 = 1. + tb * tb;
      L.dsrc[0][own] = dt * (-(sgn0 * h * dk * (g2 * hy + dg1 * h) * I.sin_int) - sgn2 * fx * sec2);
      L.dsrc[1][own] = dt * (-(sgn1 * h * dk * (g2 * hx + dg0 * h) * I.sin_int) - sgn3 * fy * sec2);
    }
  }
  return busy;
}

// One face's Jacobian with respect to the cell, in the face's frame: the
// entries 00, 0n, n0, nn, t0, tn, tt.
struct FaceJac {
  double a00, a0n, an0, ann, at0, atn, att;
};
// The derivative of the face's momentum fluxes along d kact / d phi_bed on both
// sides.
struct FaceDk {
  double dn, dt;
};

// dual_riemann_side (tg_math.h) of the face between the cell's record rc and
// its neighbour's rn, along x (isx) or y, towards plus or minus.  The normal
// axis points from the cell to the neighbour, so the cell is the left side
// of every face: where the axis is reversed (plus false) normal momenta and
// velocities, the mass and the tangential flux change sign and sl, sr become
// -sr, -sl.  All of it rounds the same, so the caller takes the signs back
// (of a00, ann, at0, att; flux0, d0, dt).  Only the choice between equal
// sides depends on the direction.
template <int TX, bool DPHI>
__device__ __forceinline__ FaceJac face_jac(const DualLds<TX, DPHI>& L, bool isx, bool plus,
                                            int rc, int rn, FaceDk& D) {
  const double* Q = isx ? L.hu : L.hv;  // normal and tangential momentum
  const double* T = isx ? L.hv : L.hu;
  const double ch = L.h[rc], ct = T[rc], ci = L.inv[rc], ca = L.sq[rc];
  const double nh = L.h[rn], nt = T[rn], ni = L.inv[rn], na = L.sq[rn];
  double cq = Q[rc], nq = Q[rn];
  if (!plus) { cq = -cq; nq = -nq; }
  const bool cvoid = ch == 0., nvoid = nh == 0.;
  const double cv = cq * ci, nv = nq * ni;
  // wave speeds; next to a void side 2 w - vel of the other one (a void
  // side's own are 0, so it drops out of the minimum and maximum with 0)
  const double cw0 = cv - ca, cw2 = cv + ca, nw0 = nv - na, nw2 = nv + na;
  const double c0 = nvoid ? 2. * cw0 - cv : cw0, c2 = nvoid ? 2. * cw2 - cv : cw2;
  const double n0 = cvoid ? 2. * nw0 - nv : nw0, n2 = cvoid ? 2. * nw2 - nv : nw2;
  const double sl = fmin(0., fmin(c0, n0)), sr = fmax(0., fmax(c2, n2));
  // the cell's flux Jacobian
  const double cvi = cv * ci, fn0 = ca * ca - cv * cv, ft0 = -cv * ct * ci, ftn = ct * ci;
  double dwc = 0., dwn = 0., dFc = 0., dFn = 0., dsl = 0., dsr = 0.;
  if (DPHI) {
    dwc = L.dw[rc]; dwn = L.dw[rn]; dFc = L.dF[rc]; dFn = L.dF[rn];
    const double dv = 2. * (cvoid ? dwn : dwc);
    const bool one = cvoid || nvoid;
    if (sl < 0.) dsl = -(one ? dv : (c0 > n0 ? dwn : dwc));
    if (sr > 0.) dsr = one ? dv : (c2 > n2 ? dwc : dwn);
  }
  FaceJac J;
  if (sl >= 0. || sr <= 0.) {  // upwind: one side's flux
    const bool own = plus ? sl >= 0. : !(sr <= 0.);
    J.a00 = 0.;
    J.a0n = (own && !cvoid) ? 1. : 0.;
    J.an0 = own ? fn0 : 0.; J.ann = own ? 2 * cv : 0.;
    J.at0 = own ? ft0 : 0.; J.atn = own ? ftn : 0.; J.att = own ? cv : 0.;
    if (DPHI) {
      D.dt = 0.;
      D.dn = own ? dFc : dFn;
    }
    return J;
  }
  // d sl, d sr by the cell (0, n entries; 2 ci - ci = ci)
  const double hai = .5 * ca * ci;
  const double e0 = -hai - cvi, e2 = hai - cvi;
  const bool usel = sl != 0. && (plus ? sl == c0 : sl != n0);
  const bool user = sr != 0. && (plus ? sr == c2 : sr != n2);
  const double dsl0 = usel ? (nvoid ? 2 * e0 - -cvi : e0) : 0., dsln = usel ? ci : 0.;
  const double dsr0 = user ? (nvoid ? 2 * e2 - -cvi : e2) : 0., dsrn = user ? ci : 0.;
  const double g = 1. / (sr - sl), ss = sl * sr;
  const double slg = -sl * g, srg = sr * g, jv = -sr * sl * g;
  {
    const double vd = nh - ch;
    const double fx = (sr * cq - sl * nq + ss * vd) * g;
    const double p = (cq + sl * vd - fx) * g, m = (-nq + sr * vd + fx) * g;
    J.a00 = p * dsr0 + m * dsl0 + jv;
    J.a0n = p * dsrn + m * dsln + (cvoid ? 0. : srg);
  }
  {
    const double cf = cq * cv + 0.5 * ca * ca * ch, nf = nq * nv + 0.5 * na * na * nh;
    const double vd = nq - cq;
    const double fx = (sr * cf - sl * nf + ss * vd) * g;
    const double p = (cf + sl * vd - fx) * g, m = (-nf + sr * vd + fx) * g;
    J.an0 = p * dsr0 + m * dsl0 + srg * fn0;
    J.ann = p * dsrn + m * dsln + srg * (2 * cv) + jv;
    if (DPHI) D.dn = p * dsr + m * dsl + srg * dFc + slg * dFn;
  }
  {
    const double cf = ct * cv, nf = nt * nv, vd = nt - ct;
    const double fx = (sr * cf - sl * nf + ss * vd) * g;
    const double p = (cf + sl * vd - fx) * g, m = (-nf + sr * vd + fx) * g;
    J.at0 = p * dsr0 + m * dsl0 + srg * ft0;
    J.atn = p * dsrn + m * dsln + srg * ftn;
    J.att = srg * cv + jv;
    if (DPHI) D.dt = p * dsr + m * dsl;
  }
  return J;
}

// Adjoint pass 1 (one workgroup per mark block, one cell of each of its four
// tiles per thread): a tile of void cells (h == 0) gets lambda^s = 0 --
// every block that multiplies a void cell's state is zero
// (calc_jacobain.C:117-122), as in the per-cell path of pass 2 -- and, with
// lambda^{s+1} == 0 on the tile, zero bed-friction terms; it is written
// here.  Every other tile is appended to the list pass 2 walks.
template <int TX>
__global__ __launch_bounds__(BLOCK) void k_adjoint_classify(AdjArgs a) {
  // the block record is read alongside the mark words (a skipped block
  // wastes its 64 bytes; a listed one saves a round trip)
  const BlockDev B = a.blocks[blockIdx.x];
  if (a.mk_out && a.mk_out[blockIdx.x] == MARK_FULL &&
      adjoint_skip(a.mk_U, a.dphi_part ? a.mk_lnext : nullptr, (int)blockIdx.x))
    return;
  __shared__ unsigned s_busy;
  if (threadIdx.x == 0) s_busy = 0u;
  // tiles the marks show to be void (U +0.0 and, with the gradient,
  // lambda^{s+1} +0.0): nothing to read; output tiles already +0.0: nothing
  // to write for a void tile
  uint32_t zvoid = 0u, zout = 0u;
  if (a.mk_out && a.l_bytes) {
    if (a.u_bytes) zvoid = a.mk_U[B.mw];
    if (a.dphi_part) zvoid &= a.mk_lnext[B.mw];
    zout = a.mk_out[B.mw];
  }
  Cell q[4];
  block_cells<TX>(B, q);
  // every load in flight at once (a test between them would make each wait for
  // the one before)
  double u[4], l[4][3];
#pragma unroll
  for (int b = 0; b < 4; b++) {
    u[b] = l[b][0] = l[b][1] = l[b][2] = 0.;
    if (!q[b].act || ((zvoid >> (8 * b)) & 1u)) continue;
    const long long c = q[b].c;
    u[b] = a.U.h[c];
    if (a.dphi_part) {
      l[b][0] = a.lam_next.h[c]; l[b][1] = a.lam_next.hu[c]; l[b][2] = a.lam_next.hv[c];
    }
  }
  unsigned busy = 0u;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    // (bitwise on purpose: no branch between the operands)
    const bool nz = (u[b] != 0.) | !((l[b][0] == 0.) & (l[b][1] == 0.) & (l[b][2] == 0.));
    if (nz) busy |= 1u << b;
  }
  __syncthreads();  // s_busy set
  if (busy) atomicOr(&s_busy, busy);
  __syncthreads();
  const unsigned W = s_busy;
  if (threadIdx.x == 0 && W) {
    int k = atomicAdd(a.tile_count, __popc(W));
#pragma unroll
    for (int b = 0; b < 4; b++)
      if ((W >> b) & 1u) a.tile_list[k++] = tile_ref<TX>(B, b);
  }
  int nshort = 0;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    if (!q[b].act || ((W >> b) & 1u)) continue;
    nshort++;
    if ((zout >> (8 * b)) & 1u) continue;  // already +0.0
    a.lam_h[q[b].c] = 0.;
    a.lam_hu[q[b].c] = 0.;
    a.lam_hv[q[b].c] = 0.;
  }
  if (a.short_cells) {
    const int cnt = (int)wave_sum((double)nshort);
    if (threadIdx.x % 64 == 0 && cnt) atomicAdd(a.short_cells, (unsigned long long)cnt);
  }
  if (a.mk_out && threadIdx.x == 0) {
#pragma unroll
    for (int b = 0; b < 4; b++)
      if (B.tile[b] >= 0 && !((W >> b) & 1u)) mark_byte_store(a.mk_out, B.mw, b, true);
  }
}


// The face's mass flux and its derivative along d kact / d phi_bed on both
// sides (riemann and driemann, tg_math.h, component 0), mirrored as in
// face_jac.  It has the forward flux's own velocities hu/h, not the dual
// flux's hu (1/h): where the functional is the whole mass the terms of all
// faces cancel, and what is left is the rounding of exactly these values.
template <int TX>
__device__ __forceinline__ void face_mass_dk(const DualLds<TX, true>& L, bool isx, bool plus,
                                             int rc, int rn, double& flux, double& d0) {
  const double* Q = isx ? L.hu : L.hv;
  const double* V = isx ? L.vx : L.vy;
  const double ch = L.h[rc], ca = L.sq[rc], nh = L.h[rn], na = L.sq[rn];
  double cq = Q[rc], nq = Q[rn], cv = V[rc], nv = V[rn];
  if (!plus) { cq = -cq; nq = -nq; cv = -cv; nv = -nv; }
  const bool cvoid = ch == 0., nvoid = nh == 0.;
  const double cw0 = cv - ca, cw2 = cv + ca, nw0 = nv - na, nw2 = nv + na;
  const double c0 = nvoid ? 2. * cw0 - cv : cw0, c2 = nvoid ? 2. * cw2 - cv : cw2;
  const double n0 = cvoid ? 2. * nw0 - nv : nw0, n2 = cvoid ? 2. * nw2 - nv : nw2;
  const double sl = fmin(0., fmin(c0, n0)), sr = fmax(0., fmax(c2, n2));
  if (sl >= 0. || sr <= 0.) {
    flux = (plus ? sl >= 0. : !(sr <= 0.)) ? cq : nq;
    d0 = 0.;
    return;
  }
  const double dwc = L.dw[rc], dwn = L.dw[rn], dv = 2. * (cvoid ? dwn : dwc);
  const bool one = cvoid || nvoid;
  const double dsl = -(one ? dv : (c0 > n0 ? dwn : dwc)), dsr = one ? dv : (c2 > n2 ? dwc : dwn);
  const double g = 1. / (sr - sl), vd = nh - ch;
  flux = (sr * cq - sl * nq + sl * sr * vd) * g;
  d0 = (cq + sl * vd - flux) * g * dsr + (-nq + sr * vd + flux) * g * dsl;
}

// Adjoint pass 2, one tile.  MAYBE_VOID: the tile is not known to hold
// anything; a void one is written here as the classifying pass would.
template <int TX, bool DPHI, bool MAYBE_VOID>
__device__ __forceinline__ void adjoint_tile(const AdjArgs& a, const TileRef& t,
                                             DualLds<TX, DPHI>& L) {
  const InstDev I = a.inst[t.inst];
  constexpr int TY = BLOCK / TX, RX = TX + 2, RY = TY + 2, NHALO = 2 * TX + 2 * TY;
  static_assert(BLOCK + NHALO <= ADJ_THREADS, "one thread per record");
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));  // indexes rebuilt per tile, not held over the tile loop
  const double dt = a.dt_rec[(long long)t.inst * a.max_steps + a.step];
  // phase 1: the halo is the four side strips (the stencil reads no corner)
  bool busy = false;
  if (tid < BLOCK + NHALO) {
    int rx, ry, own = -1;
    const int h = tid - BLOCK;
    if (h < 0) { rx = tid % TX + 1; ry = tid / TX + 1; own = tid; }
    else if (h < TX) { rx = h + 1; ry = 0; }
    else if (h < 2 * TX) { rx = h - TX + 1; ry = RY - 1; }
    else if (h < 2 * TX + TY) { rx = 0; ry = h - 2 * TX + 1; }
    else { rx = RX - 1; ry = h - 2 * TX - TY + 1; }
    const int i = t.x0 - 1 + rx, j = t.y0 - 1 + ry;
    if (i >= 0 && i < t.nx && j >= 0 && j < t.ny)
      busy = dual_record<TX, DPHI>(a, t, I, i, j, dt, L, ry * RX + rx, own) && own >= 0;
  }
  const int p = tid & 1, q = tid >> 1;
  const bool isx = p;
  const int gi = t.x0 + q % TX, gj = t.y0 + q / TX;
  const bool act = gi < t.nx && gj < t.ny;
  const long long c = t.off + (long long)gj * t.nx + gi;
  if (MAYBE_VOID) {
    if (!__syncthreads_or(busy)) {
      const bool keep = a.mk_out && a.l_bytes && (a.mk_out[t.mw] >> (8 * mark_byte<TX>(t))) & 1u;
      if (act && isx && !keep) { a.lam_h[c] = 0.; a.lam_hu[c] = 0.; a.lam_hv[c] = 0.; }
      if (a.short_cells) {
        const int cnt = __syncthreads_count(act && isx);
        if (tid == 0) atomicAdd(a.short_cells, (unsigned long long)cnt);
      }
      if (a.mk_out) {
        __syncthreads();  // every thread has read the byte
        mark_store<TX>(a.mk_out, t, true);
      }
      return;
    }
  } else {
    __syncthreads();
  }
  double dphi = 0.;
  bool zero_out = true;
  if (act) {
    const bool full = L.nz[q];  // a void cell receives nothing (calc_jacobain.C:117-122)
    const int rc = (q / TX + 1) * RX + q % TX + 1;
    const double* LN = isx ? L.lam[1] : L.lam[2];  // normal and tangential adjoint
    const double* LT = isx ? L.lam[2] : L.lam[1];
    const double lc0 = L.lam[0][rc], lcn = LN[rc], lct = LT[rc];
    const double hraw = L.h[rc];
    double out[3] = {0., 0., 0.};
    // a cell with lambda^{s+1} = 0 adds lambda . dU/dphi = 0 to the gradient
    if (full || (DPHI && !(lc0 == 0. && lcn == 0. && lct == 0.))) {
      const double dtd = isx ? dt / I.dx : dt / I.dy, dts = isx ? dtd : -dtd;
      // faces in visiting order: A is S (y) or E (x), B is N or W; the
      // neighbours beyond them up to the member's edge
      const int pos = isx ? gi : gj, last = (isx ? t.nx : t.ny) - 1;
      const int aheadA = isx ? last - pos : pos, aheadB = last - aheadA;
      const bool hasA = aheadA > 0, hasB = aheadB > 0;
      const int stepA = isx ? 1 : -RX;
      // (a missing neighbour: any face, its entries are replaced below)
      const int rA = hasA ? rc + stepA : rc, rB = hasB ? rc - stepA : rc;
      FaceDk DA, DB;
      FaceJac A = face_jac<TX, DPHI>(L, isx, isx, rc, rA, DA);
      FaceJac B = face_jac<TX, DPHI>(L, isx, !isx, rc, rB, DB);
      if constexpr (DPHI) {
        // lambda^{s+1}_c . d U^{s+1}_c / d phi_bed at frozen dt (no reference
        // counterpart): the flux differences of this thread's direction, plus
        // face minus minus face (mass and tangential: mirrored, so their sum);
        // an outflow face copies the opposite face, so the pair's difference
        // vanishes; h clamped at 0 does not vary
        double fA, fB, dA, dB;
        face_mass_dk<TX>(L, isx, isx, rc, rA, fA, dA);
        face_mass_dk<TX>(L, isx, !isx, rc, rB, fB, dB);
        const bool pair = hasA && hasB;
        const double f0 = dtd * (pair ? fA + fB : 0.);
        const double m0 = dtd * (pair ? dA + dB : 0.), mt = dtd * (pair ? DA.dt + DB.dt : 0.);
        const double mn = dts * (pair ? DA.dn - DB.dn : 0.);
        // out = -x - y: the x thread adds them up (its n = 1, t = 2)
        const double y0 = swap_pair(m0), y2 = swap_pair(mn), y1 = swap_pair(mt);
        const double fy = swap_pair(f0);
        double o0 = -m0 - y0, o1 = -mn - y1, o2 = -mt - y2;
        if (hraw - f0 - fy < 0.) o0 = 0.;
        o1 += L.dsrc[0][q];
        o2 += L.dsrc[1][q];
        dphi = lc0 * o0 + lcn * o1 + lct * o2;
      }
      if (full) {
        // an outflow face copies the opposite face (boundary_flux): its
        // mirrored entries are the opposite's with the signs taken back
        if (!hasA || !hasB) {
          auto flip = [](const FaceJac& J) {
            return FaceJac{-J.a00, J.a0n, J.an0, -J.ann, -J.at0, J.atn, -J.att};
          };
          const FaceJac Z = {0., 0., 0., 0., 0., 0., 0.};
          if (!hasA) A = hasB ? flip(B) : Z;
          if (!hasB) B = hasA ? flip(A) : Z;
        }
        // the neighbours' blocks (calc_jacobian_elem): -dtd J of a plus face
        // (it is the neighbour's minus face), +dtd J of a minus face; zero
        // where the neighbour's other side is a domain boundary (both its
        // sides then carry this face); with the source term on the
        // tangential row, times the neighbour's lambda
        const double sA = aheadA > 1 ? -dtd : 0., pA = isx ? sA : -sA;
        const double sB = aheadB > 1 ? -dtd : 0., pB = isx ? -sB : sB;
        const double a0 = hasA ? L.lam[0][rA] : 0., an = hasA ? LN[rA] : 0.,
                     at = hasA ? LT[rA] : 0.;
        const double b0 = hasB ? L.lam[0][rB] : 0., bn = hasB ? LN[rB] : 0.,
                     bt = hasB ? LT[rB] : 0.;
        const double At0 = sA * A.at0 - L.src[isx ? 0 : 3][rA];
        const double Bt0 = sB * B.at0 - L.src[isx ? 1 : 2][rB];
        // rows 1 and 2 in order: x faces n, t; y faces t, n
        const double An0 = an * (pA * A.an0), Ann = an * (sA * A.ann);
        const double Bn0 = bn * (pB * B.an0), Bnn = bn * (sB * B.ann);
        const double At0l = at * At0, Atn = at * (pA * A.atn);
        const double Bt0l = bt * Bt0, Btn = bt * (pB * B.atn);
        // self block: dtd * (plus face - minus face) of both directions - 1,
        // minus the sources; the y thread (n = 2, t = 1) forms it
        auto other = [](double v) { return swap_pair(v); };
        const double D00 = dtd * (A.a00 + B.a00), D0n = dts * (A.a0n - B.a0n);
        const double Dn0 = dts * (A.an0 - B.an0), Dnn = dtd * (A.ann + B.ann);
        const double Dt0 = dtd * (A.at0 + B.at0), Dtn = dts * (A.atn - B.atn);
        const double Dtt = dtd * (A.att + B.att);
        double r0 = 0. + lc0 * ((D00 + other(D00)) - 1.);
        double rt = 0. + lc0 * other(D0n), rn = 0. + lc0 * D0n;
        r0 += lct * ((other(Dn0) + Dt0) - L.self[0][q] - L.self[1][q]);
        rt += lct * ((other(Dnn) + Dtt) - 1. - L.self[2][q]);
        rn += lct * Dtn;
        r0 += lcn * ((other(Dt0) + Dn0) - L.self[3][q] - L.self[4][q]);
        rt += lcn * other(Dtn);
        rn += lcn * ((other(Dtt) + Dnn) - 1. - L.self[5][q]);
        // the pair hands the sum back and forth: n and t change roles
        auto pass = [&]() {
          r0 = swap_pair(r0);
          const double x = swap_pair(rt);
          rt = swap_pair(rn);
          rn = x;
        };
        const double A1 = isx ? An0 : At0l, A2 = isx ? At0l : An0;
        const double A1n = isx ? Ann : Atn, A2n = isx ? Atn : Ann;
        const double A0 = a0 * (sA * A.a00), A0n = a0 * (pA * A.a0n);
        const double B0 = b0 * (sB * B.a00), B0n = b0 * (pB * B.a0n);
        double Att = at * (sA * A.att), Btt = bt * (sB * B.att);
        if (!isfinite(a0 + an + b0 + bn)) {  // 0 * inf: the products left out count
          Att += 0. * a0 + 0. * an;
          Btt += 0. * b0 + 0. * bn;
        }
        auto addA = [&]() {
          r0 += A0; rn += A0n; rt += Att;
          r0 += A1; rn += A1n;
          r0 += A2; rn += A2n;
        };
        const double B1 = isx ? Bn0 : Bt0l, B2 = isx ? Bt0l : Bn0;
        const double B1n = isx ? Bnn : Btn, B2n = isx ? Btn : Bnn;
        auto addB = [&]() {
          r0 += B0; rn += B0n; rt += Btt;
          r0 += B1; rn += B1n;
          r0 += B2; rn += B2n;
        };
        addA(); pass(); addA(); pass();  // S, E
        addB(); pass(); addB();          // N, W
        // the x thread holds the sum (n = 1, t = 2)
        out[0] = 0. - r0; out[1] = 0. - rn; out[2] = 0. - rt;
#pragma unroll
        for (int k = 0; k < 3; k++)
          if (fabs(out[k]) < 1e-16) out[k] = 0.;  // calc_adjoint.C:150-152
      }
    }
    if (isx) {
      a.lam_h[c] = out[0];
      a.lam_hu[c] = out[1];
      a.lam_hv[c] = out[2];
      zero_out = bitzero3(out[0], out[1], out[2]);
    }
  }
  if (a.active) {
    const int cnt = __syncthreads_count(act && isx);
    if (tid == 0) atomicAdd(a.active, (unsigned long long)cnt);
  }
  // the cell's term where its self terms were (only this pair reads them)
  if (DPHI && isx) L.self[0][q] = dphi;
  const bool all = a.mk_out || DPHI ? __syncthreads_and(zero_out) : false;
  if (DPHI) {  // the tile's sum: 64 cells to a wave, then the waves in order
    if (tid < BLOCK) {
      dphi = wave_sum(L.self[0][tid]);
      if (tid % 64 == 0) L.sp[tid / 64] = dphi;
    }
    __syncthreads();
    if (tid == 0) {
      for (int k = 1; k < BLOCK / 64; k++) dphi += L.sp[k];
      unsafeAtomicAdd(a.dphi_part + t.tile, dphi);  // its only writer: nothing waits for it
    }
  }
  if (a.mk_out) mark_store<TX>(a.mk_out, t, all);
}

template <int TX, bool DPHI>
__global__ __launch_bounds__(ADJ_THREADS, 4) void k_adjoint(AdjArgs a) {
  __shared__ DualLds<TX, DPHI> L;
  const int n = *a.tile_count;
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.count_next = 0;
  for (int i = (int)blockIdx.x; i < n; i += (int)gridDim.x) {
    adjoint_tile<TX, DPHI, false>(a, a.tile_list[list_band(i, n)], L);
    __syncthreads();  // LDS reused by the next tile
  }
}

// Reverse step on small meshes, one workgroup per tile, nothing listed.
template <int TX, bool DPHI>
__global__ __launch_bounds__(ADJ_THREADS, 4) void k_adjoint_tile(AdjArgs a) {
  __shared__ DualLds<TX, DPHI> L;
  const int tile = tile_of(a);
  const TileDev t = a.tiles[tile];
  if (a.mk_out && adjoint_skip(a.mk_U, DPHI ? a.mk_lnext : nullptr, t.mw) &&
      out_marked_zero<TX>(a.mk_out, t))
    return;
  adjoint_tile<TX, DPHI, true>(a, ref_of(t, tile), L);
}

}  // namespace

// one instantiation per built tile width; a.shape selects it
#define TG_LAUNCH_TX(shape, KERNEL, GRID, ...)                                      \
  do {                                                                             \
    switch (SHAPE_TX[shape]) {                                                     \
      case 64: hipLaunchKernelGGL(KERNEL<64>, GRID, dim3(BLOCK), 0, __VA_ARGS__); break; \
      case 32: hipLaunchKernelGGL(KERNEL<32>, GRID, dim3(BLOCK), 0, __VA_ARGS__); break; \
      default: hipLaunchKernelGGL(KERNEL<16>, GRID, dim3(BLOCK), 0, __VA_ARGS__); break; \
    }                                                                              \
  } while (0)

void launch_coef(const StepArgs& a, bool reduce, hipStream_t s) {
  if (a.by_tile) TG_LAUNCH_TX(a.shape, k_coef_tile, dim3(a.ntiles), s, a, reduce ? 1 : 0);
  else TG_LAUNCH_TX(a.shape, k_coef, dim3(a.nblocks), s, a, reduce ? 1 : 0);
}
void launch_update(const StepArgs& a, hipStream_t s) {
  const int g = a.by_tile || a.ntiles < LIST_GRID ? a.ntiles : LIST_GRID;
#define TG_UPD(TX)                                                                             \
  if (a.by_tile)                                                                               \
    hipLaunchKernelGGL(k_update_tile<TX>, dim3(g), dim3(face_threads<TX>()), 0, s, a);         \
  else                                                                                         \
    hipLaunchKernelGGL(k_update<TX>, dim3(g), dim3(record_threads<TX>()), 0, s, a)
  switch (SHAPE_TX[a.shape]) {
    case 64: TG_UPD(64); break;
    case 32: TG_UPD(32); break;
    default: TG_UPD(16); break;
  }
#undef TG_UPD
}
void launch_adjoint(const AdjArgs& a, hipStream_t s) {
  if (!a.by_tile) TG_LAUNCH_TX(a.shape, k_adjoint_classify, dim3(a.nblocks), s, a);
  const dim3 g(a.by_tile || a.ntiles < ADJ_GRID ? a.ntiles : ADJ_GRID), b(ADJ_THREADS);
#define TG_ADJ(TX, DPHI)                                                            \
  if (a.by_tile) hipLaunchKernelGGL((k_adjoint_tile<TX, DPHI>), g, b, 0, s, a);     \
  else hipLaunchKernelGGL((k_adjoint<TX, DPHI>), g, b, 0, s, a)
  const int tx = SHAPE_TX[a.shape];
  if (a.dphi_part) {
    if (tx == 64) { TG_ADJ(64, true); }
    else if (tx == 32) { TG_ADJ(32, true); }
    else { TG_ADJ(16, true); }
  } else {
    if (tx == 64) { TG_ADJ(64, false); }
    else if (tx == 32) { TG_ADJ(32, false); }
    else { TG_ADJ(16, false); }
  }
#undef TG_ADJ
}
static unsigned grid_for(long long n) {
  const long long b = (n + 255) / 256;
  return (unsigned)(b < 4096 ? (b < 1 ? 1 : b) : 4096);
}
void launch_zero(void* p, size_t bytes, hipStream_t s) {
  const long long n = (long long)(bytes / 4);
  hipLaunchKernelGGL(k_zero_u32, dim3(grid_for(n)), dim3(256), 0, s, (uint32_t*)p, n);
}
void launch_copy(const void* src, void* dst, size_t bytes, hipStream_t s) {
  const long long n = (long long)(bytes / 4);
  hipLaunchKernelGGL(k_copy_u32, dim3(grid_for(n)), dim3(256), 0, s, (const uint32_t*)src,
                     (uint32_t*)dst, n);
}
template <class S>
void launch_box_max(const BoxChunk* ch, int nchunks, const long long* cells, const S* h,
                    double* rec, int max_steps, int step, hipStream_t s) {
  if (nchunks <= 0) return;
  hipLaunchKernelGGL(k_box_max<S>, dim3(nchunks), dim3(256), 0, s, ch, cells, h,
                     (unsigned long long*)rec, max_steps, step);
}
template void launch_box_max<double>(const BoxChunk*, int, const long long*, const double*,
                                     double*, int, int, hipStream_t);
template void launch_box_max<float>(const BoxChunk*, int, const long long*, const float*,
                                    double*, int, int, hipStream_t);
void launch_member_fill(const void* src, void* dst, int es, long long ncell, long long off,
                        long long count, uint32_t* mk, long long mw0, long long nmw,
                        hipStream_t s) {
  const long long w = es / 4;  // 32-bit words per value
  const long long n = count * w > nmw ? count * w : nmw;
  hipLaunchKernelGGL(k_member_fill, dim3(grid_for(n)), dim3(256), 0, s, (const uint32_t*)src,
                     (uint32_t*)dst, ncell * w, off * w, count * w, mk, mw0, nmw);
}
void launch_reset_red(RedDev* red, int ninst, const double* time, double* clock, long long stride,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_reset_red, dim3((ninst + 63) / 64), dim3(64), 0, s, red, ninst, time,
                     clock, stride);
}
void launch_stats(const InstDev* inst, const TileDev* tiles, int ntiles, Fields U,
                  const uint32_t* mk, double* part_mass, double* part_hmax, double tiny,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_stats, dim3(ntiles), dim3(BLOCK), 0, s, inst, tiles, U, mk, part_mass,
                     part_hmax, tiny);
}

void launch_copy_marking(const BlockDev* blocks, int nblocks, int shape, int es,
                         const void* const src[3], void* dst, long long ncell, uint32_t* mk_src,
                         uint32_t* mk_dst, hipStream_t s) {
  if (nblocks <= 0) return;
  if (es == 8) {
    const uint64_t* f[3] = {(const uint64_t*)src[0], (const uint64_t*)src[1],
                            (const uint64_t*)src[2]};
    switch (SHAPE_TX[shape]) {
      case 64: hipLaunchKernelGGL((k_copy_marking<64, uint64_t>), dim3(nblocks), dim3(BLOCK), 0,
                                  s, blocks, f[0], f[1], f[2], (uint64_t*)dst, ncell, mk_src,
                                  mk_dst); break;
      case 32: hipLaunchKernelGGL((k_copy_marking<32, uint64_t>), dim3(nblocks), dim3(BLOCK), 0,
                                  s, blocks, f[0], f[1], f[2], (uint64_t*)dst, ncell, mk_src,
                                  mk_dst); break;
      default: hipLaunchKernelGGL((k_copy_marking<16, uint64_t>), dim3(nblocks), dim3(BLOCK), 0,
                                  s, blocks, f[0], f[1], f[2], (uint64_t*)dst, ncell, mk_src,
                                  mk_dst); break;
    }
  } else {
    const uint32_t* f[3] = {(const uint32_t*)src[0], (const uint32_t*)src[1],
                            (const uint32_t*)src[2]};
    switch (SHAPE_TX[shape]) {
      case 64: hipLaunchKernelGGL((k_copy_marking<64, uint32_t>), dim3(nblocks), dim3(BLOCK), 0,
                                  s, blocks, f[0], f[1], f[2], (uint32_t*)dst, ncell, mk_src,
                                  mk_dst); break;
      case 32: hipLaunchKernelGGL((k_copy_marking<32, uint32_t>), dim3(nblocks), dim3(BLOCK), 0,
                                  s, blocks, f[0], f[1], f[2], (uint32_t*)dst, ncell, mk_src,
                                  mk_dst); break;
      default: hipLaunchKernelGGL((k_copy_marking<16, uint32_t>), dim3(nblocks), dim3(BLOCK), 0,
                                  s, blocks, f[0], f[1], f[2], (uint32_t*)dst, ncell, mk_src,
                                  mk_dst); break;
    }
  }
}

void launch_member_reduce(const double* sum_part, const double* max_part, const int* off,
                          const int* idx, int n, const double* time, const double* dt_rec,
                          long long stride, int col, const int* err, double* out,
                          hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_member_reduce, dim3(n), dim3(BLOCK), 0, s, sum_part, max_part, off, idx,
                     n, time, dt_rec, stride, col, err, out);
}
void launch_set_time(double* time, int n, double t, int* err, hipStream_t s) {
  hipLaunchKernelGGL(k_set_time, dim3((n + 63) / 64), dim3(64), 0, s, time, n, t, err);
}
template <class S>
void launch_spoil_members(const InstDev* inst, int n, const double* dt_rec, long long stride,
                          int steps, S* h, S* hu, S* hv, uint32_t* mk, hipStream_t s) {
  hipLaunchKernelGGL(k_spoil_members<S>, dim3(n * SPOIL_GRID), dim3(BLOCK), 0, s, inst, dt_rec,
                     stride, steps, h, hu, hv, mk);
}
template void launch_spoil_members<double>(const InstDev*, int, const double*, long long, int,
                                           double*, double*, double*, uint32_t*, hipStream_t);
template void launch_spoil_members<float>(const InstDev*, int, const double*, long long, int,
                                          float*, float*, float*, uint32_t*, hipStream_t);
void launch_reverse_setup(double* dt_rec, long long stride, int n, double dt, uint32_t* z0,
                          long long n0, uint32_t* z1, long long n1, hipStream_t s) {
  long long m = n0 > n1 ? n0 : n1;
  if (n > m) m = n;
  hipLaunchKernelGGL(k_reverse_setup, dim3(grid_for(m)), dim3(256), 0, s, dt_rec, stride, n, dt,
                     z0, n0, z1, n1);
}

}  // namespace tg
