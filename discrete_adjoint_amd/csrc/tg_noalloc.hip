// tg_step_noalloc: one order-1 forward step of a uniform block with every
// intermediate kept in a fixed device array of this file (no device memory
// is allocated or freed by the call).  It runs the kernels of
// tg_forward_step -- coefficient / CFL pass and update -- on caller-owned
// device arrays, so its results are those of tg_forward_step on the same
// state, bit for bit.
//
// Scratch: the member record, the tile and mark-block tables of the 64x4
// row-major tile variant, the CFL reduction cells, the dt / time / error
// words, the update's tile list and kact of every cell.  The array is
// per device and per process; calls on one device share it, so calls that
// overlap on one device race (the call is synchronous, and a process-wide
// mutex serialises the host side).
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/tg.h"
#include "tg_kernels.h"

using namespace tg;

namespace {

constexpr long long NA_MAX_CELLS = TG_NOALLOC_MAX_CELLS;
constexpr int NA_MAX_TILES = TG_NOALLOC_MAX_CELLS / 256 * 2;  // 64x4 tiles, partial edges
// 64x16 mark blocks: a block of at most four rows has one for each of its tiles
constexpr int NA_MAX_BLOCKS = NA_MAX_TILES;
constexpr int NA_MAX_DEVICES = 64;

constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// byte offsets into the scratch array
constexpr size_t OFF_INST = 0;
constexpr size_t OFF_RED = OFF_INST + align256(sizeof(InstDev));
constexpr size_t OFF_MISC = OFF_RED + align256(2 * NRED * sizeof(RedDev));  // dt, time, err, count
constexpr size_t OFF_TILES = OFF_MISC + 256;
constexpr size_t OFF_BLOCKS = OFF_TILES + align256(sizeof(TileDev) * NA_MAX_TILES);
constexpr size_t OFF_LIST = OFF_BLOCKS + align256(sizeof(BlockDev) * NA_MAX_BLOCKS);
constexpr size_t OFF_KACT = OFF_LIST + align256(sizeof(TileRef) * NA_MAX_TILES);
constexpr size_t NA_BYTES = OFF_KACT + align256(sizeof(double) * NA_MAX_CELLS);

__device__ __align__(256) unsigned char scratch[NA_BYTES];

std::mutex g_mu;
unsigned char* g_ptr[NA_MAX_DEVICES] = {};  // scratch's address on each device

struct Misc {
  double dt_rec, time, clock[2];
  int err, tile_count[2], count_next[2];
};

int device_scratch(int device, unsigned char** out) {
  if (device < 0 || device >= NA_MAX_DEVICES) return TG_ERR_ARG;
  if (!g_ptr[device]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return TG_ERR_HIP;
    g_ptr[device] = (unsigned char*)p;
  }
  *out = g_ptr[device];
  return TG_OK;
}

// The member's record, the step's words, the reduction cells and the tile and
// block tables of the 64x4 row-major variant for one nx x ny member (as
// tg_set_mesh builds them for variant 0), written by one launch whose arguments
// carry what the host knows: the call copies nothing to the device (four copies
// and a host loop over the tables took 40 us of a 64 x 64 call's 76 us).
__global__ __launch_bounds__(256) void k_noalloc_setup(InstDev I, Misc m, InstDev* inst,
                                                       Misc* misc, RedDev* red, TileDev* tiles,
                                                       BlockDev* blocks, int ntx, int ntiles,
                                                       int nblocks) {
  constexpr int TX = SHAPE_TX[0], TY = BLOCK / TX, ROWS = MARK_H / TY;
  static_assert(TX == MARK_W, "a mark block is a column of tiles");
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i == 0) {
    *inst = I;
    *misc = m;
  }
  if (i < NRED) red_clear(red, 0, i);
  const int nsx = I.nsx;
  if (i < ntiles) {
    const int bx = i % ntx, ty = i / ntx, by = ty / ROWS, mw = by * nsx + bx;
    tiles[i] = TileDev{0, bx * TX, ty * TY, mw, bx > 0 ? mw - 1 : -1, bx + 1 < nsx ? mw + 1 : -1,
                       by > 0 ? mw - nsx : -1, by + 1 < I.nsy ? mw + nsx : -1, I.nx, I.ny, 0};
  }
  if (i < nblocks) {
    const int bx = i % nsx, by = i / nsx;
    BlockDev B{0, i, bx > 0 ? i - 1 : -1, bx + 1 < nsx ? i + 1 : -1, by > 0 ? i - nsx : -1,
               by + 1 < I.nsy ? i + nsx : -1, {-1, -1, -1, -1}, bx * MARK_W, by * MARK_H, I.nx,
               I.ny, 0};
    for (int k = 0; k < ROWS; k++)
      if ((by * ROWS + k) * TY < I.ny) B.tile[k] = (by * ROWS + k) * ntx + bx;
    blocks[i] = B;
  }
}

int step_on_device(const tg_config* cfg, const tg_noalloc_block* blk, const tg_params* prm,
                   int step, double time, const double* d_h, const double* d_hu,
                   const double* d_hv, double* d_h_out, double* d_hu_out, double* d_hv_out,
                   hipStream_t s, double* dt_out);

#define NA_CHK(call)                                  \
  do {                                                \
    if ((call) != hipSuccess) return TG_ERR_HIP;      \
  } while (0)

}  // namespace

extern "C" int tg_step_noalloc(const tg_config* cfg, const tg_noalloc_block* blk,
                               const tg_params* prm, int step, double time,
                               const double* d_h, const double* d_hu, const double* d_hv,
                               double* d_h_out, double* d_hu_out, double* d_hv_out,
                               void* stream, double* dt_out) {
  if (!cfg || !blk || !prm || !d_h || !d_hu || !d_hv || !d_h_out || !d_hu_out || !d_hv_out ||
      !blk->statics || step < 0)
    return TG_ERR_ARG;
  if (blk->nx < 1 || blk->ny < 1 || !(blk->dx > 0) || !(blk->dy > 0)) return TG_ERR_ARG;
  const long long n = (long long)blk->nx * blk->ny;
  const long long ntiles_need = (long long)((blk->nx + 63) / 64) * ((blk->ny + 3) / 4);
  if (n > NA_MAX_CELLS || ntiles_need > NA_MAX_TILES) return TG_ERR_TOO_LARGE;
  std::lock_guard<std::mutex> lock(g_mu);
  int dev = -1;
  NA_CHK(hipGetDevice(&dev));
  if (cfg->device != dev) NA_CHK(hipSetDevice(cfg->device));
  const int rc = step_on_device(cfg, blk, prm, step, time, d_h, d_hu, d_hv, d_h_out, d_hu_out,
                                d_hv_out, (hipStream_t)stream, dt_out);
  if (cfg->device != dev) (void)hipSetDevice(dev);  // the caller's device again
  return rc;
}

extern "C" long long tg_noalloc_scratch_bytes(void) { return (long long)NA_BYTES; }

namespace {

int step_on_device(const tg_config* cfg, const tg_noalloc_block* blk, const tg_params* prm,
                   int step, double time, const double* d_h, const double* d_hu,
                   const double* d_hv, double* d_h_out, double* d_hu_out, double* d_hv_out,
                   hipStream_t s, double* dt_out) {
  const long long n = (long long)blk->nx * blk->ny;
  unsigned char* base = nullptr;
  int rc = device_scratch(cfg->device, &base);
  if (rc) return rc;

  constexpr int TX = SHAPE_TX[0], TY = BLOCK / TX;
  InstDev I{};
  I.nx = blk->nx; I.ny = blk->ny; I.off = 0;
  I.nsx = (blk->nx + MARK_W - 1) / MARK_W;
  I.nsy = (blk->ny + MARK_H - 1) / MARK_H;
  I.soff = 0;
  I.dx = blk->dx; I.dy = blk->dy;
  I.inv_dx = 1 / blk->dx; I.inv_sx = 1 / (blk->dx + blk->dx);
  I.inv_dy = 1 / blk->dy; I.inv_sy = 1 / (blk->dy + blk->dy);
  I.sin_int = prm->sin_int; I.tan_bed = prm->tan_bed;
  I.kc1 = prm->kact_c1; I.kroot = prm->kact_root; I.dkroot = prm->dkroot_dphi;
  I.eps = prm->epsilon; I.gscale = prm->gravity_scale;
  I.maxtime = prm->maxtime; I.nextoutput = prm->nextoutput;
  I.nextsave = prm->nextsave;
  const Misc misc{0.0, time, {time, 0.0}, 0, {0, 0}, {0, 0}};
  const int ntx = (blk->nx + TX - 1) / TX, ntiles = ntx * ((blk->ny + TY - 1) / TY);
  const int nblocks = I.nsx * I.nsy;
  Misc* md = (Misc*)(base + OFF_MISC);
  hipLaunchKernelGGL(k_noalloc_setup, dim3((ntiles + 255) / 256), dim3(256), 0, s, I, misc,
                     (InstDev*)(base + OFF_INST), md, (RedDev*)(base + OFF_RED),
                     (TileDev*)(base + OFF_TILES), (BlockDev*)(base + OFF_BLOCKS), ntx, ntiles,
                     nblocks);

  StepArgs a{};
  a.inst = (const InstDev*)(base + OFF_INST);
  a.tiles = (const TileDev*)(base + OFF_TILES);
  a.ntiles = ntiles;
  a.shape = 0;
  a.blocks = (const BlockDev*)(base + OFF_BLOCKS);
  a.nblocks = nblocks;
  a.U = Fields{d_h, d_hu, d_hv};
  const double* st = blk->statics;
  a.S = Statics{st, st + n, st + 2 * n, st + 3 * n, st + 4 * n, st + 5 * n, st + 6 * n};
  a.kact = (double*)(base + OFF_KACT);
  a.red = (RedDev*)(base + OFF_RED);
  a.dt_rec = &md->dt_rec;
  a.red_next = a.red + NRED;
  a.nred = reduction_cells(ntiles, 1);
  a.time = &md->time;
  a.clock = md->clock;
  a.fold = 1;
  a.by_tile = ntiles <= TILE_LAUNCH_MAX ? 1 : 0;
  a.copy_dry = time <= prm->maxtime && time <= prm->nextoutput && time <= prm->nextsave;
  a.max_steps = 1;
  a.step = 0;
  a.ft = (step < cfg->frict_tiny_switch) ? cfg->frict_tiny_early : cfg->frict_tiny_late;
  a.tiny = cfg->tiny; a.gamma = cfg->gamma;
  a.cfl_inner = cfg->cfl_inner; a.cfl_outer = cfg->cfl_outer;
  a.h_out = d_h_out; a.hu_out = d_hu_out; a.hv_out = d_hv_out;
  a.err = &md->err;
  a.active = nullptr;
  a.tile_list = (TileRef*)(base + OFF_LIST);
  a.tile_count = md->tile_count;
  a.count_next = md->count_next;
  a.ninst = 1;
  a.mk_in = nullptr;   // no zero marks: every tile is classified from its cells
  a.mk_out = nullptr;
  a.short_cells = nullptr;

  launch_coef(a, true, s);
  launch_update(a, s);
  NA_CHK(hipGetLastError());
  Misc back{};
  NA_CHK(hipMemcpyAsync(&back, md, sizeof(Misc), hipMemcpyDeviceToHost, s));
  NA_CHK(hipStreamSynchronize(s));
  if (back.err & 1) {
    if (!a.by_tile) {  // the dry tiles were written before dt was known
      launch_spoil_members(a.inst, 1, a.dt_rec, 1, 1, d_h_out, d_hu_out, d_hv_out, nullptr, s);
      NA_CHK(hipStreamSynchronize(s));
    }
    return TG_ERR_NONFINITE;
  }
  if (back.err & 2) return TG_ERR_EIGEN;
  if (dt_out) *dt_out = back.dt_rec;
  return TG_OK;
}

}  // namespace
