// fp32 NHWC convolution on the bf16 matrix cores, without losing fp32 accuracy: the forward pass
// and, read with the flipped, channel-transposed filter, the dx of a stride-1 convolution.
//
// Arithmetic.  Each operand is scaled by 2^23 and split into three bf16 numbers, x = x0 + x1 + x2
// (round to nearest even at each step: 8 + 8 + 8 significant bits hold all 24 of an fp32 value, and
// the scale keeps the pieces of the smallest ones normal).  A product is the six terms x2 w0, x0 w2, x1 w1, x0 w1, x1 w0, x0 w0; the dropped
// ones are together at most 2^-24 of it (both operands 1 + 2^-8 - 2^-17, all terms one sign: a relative
// error of 5.9e-8, which v_mfma_f32_16x16x4f32 has there too), 2^-27 rms for normal operands.  The terms of 32 reduction values sum from zero in that order, and
// the sum is added to the fp32 accumulator.  Error against 64 bits, K = 576 / 4608 normal
// inputs: 0.9e-7 / 2.3e-7 relative, where a chain of v_mfma_f32_16x16x4f32 gives 4.4e-7 / 1.2e-6
// (one rounding of the running sum per 32 products, not per 4).  Six
// v_mfma_f32_16x16x32_bf16 issue in 0.38 of the time of the eight v_mfma_f32_16x16x4f32 they
// replace; a loop of them alone sustains 1680 TFLOP/s on this card, 280 of them the convolution's.
// The matrix core's sums lean towards minus infinity by a part of their last bit (a mean error of 0.3
// of its rms at K = 576), so half of the K-blocks compute on negated operands and are subtracted:
// the second of a stage (stages of 8 octets), every second chunk (of 4: the running sums change sign
// with it) or stage (blocked dx).  A layer of one chunk keeps its lean in the 4-wave tiles: a sign that
// turns every few stages cost those 4-7%.
// What the split does not carry is found at the end of a tile, as a result that is infinite or NaN,
// and the whole tile is computed again with v_mfma_f32_16x16x4f32: an infinite or NaN input, an
// input of about 2^105 or more, a scaled sum past the fp32 range (a result of 2^82 or more).
//
// Work.  A workgroup computes a tile of ti images x th x tw output positions (at most
// 16 NSEG WM) and 32 WN channels of one group; wave (wm, wn) computes 16 NSEG of the positions
// x 32 channels.  The reduction runs over chunks of `co` octets (8 channels) and, within a
// chunk, over the R S co (tap, octet) pairs, 4 to a K-block (one pair per lane group):
//   - A: the tile's input halo of the chunk is read once from memory, split once, and kept in LDS
//     as [octet][halo position][3 pieces] of 16 bytes; every tap reads it at its own offset.  The
//     implicit GEMM gathers (and would split) each value once per tap.
//   - B: the filter values of SO octets a stage, [octet][channel][3 pieces], double-buffered.
// The next stage's filter values and the next chunk's halo are in flight in registers while a
// stage's MFMAs run.
//
// Measured (us, back to back; before: the fp32 implicit GEMM of conv_f32.hip): 32 x 56 x 56, 64 -> 64
// 3x3 59 (106), its dx 59 (118); 32 x 28 x 28, 128 -> 256 100 (198), dx 95 (218), 2 x 4 filter blocks
// 102 (199); 16 x 64 x 64 dilated 34 (59); four groups of 32 70 (115); one 56 x 56 image 12.8 (30.8).
// Few tiles are bound by the stages' latency: 8 waves on 16 positions each (NSEG 1) halve the
// stages of 4 waves on 32 (one image 15.4 -> 13.1, 4 x 16 x 16, 256 -> 64 42 -> 38).
// Bound by the matrix instructions and the power they draw: with everything but the MFMAs and
// their LDS reads taken out the 28 x 28 dx still took 67 us; the filter's split and stores cost 8,
// its loads 8 and the halo 4.  The 56 x 56 layer loses a further 9 us per workgroup at its start
// and end (halo load and split, stores), which a second workgroup per CU hides only in part.

#include "f32_split.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace miq {
namespace {

constexpr int kSplitMaxReach = 64;         // filter blocks that the halo of a tile touches (blocked dx)
// floor(65536 / n) + 1: t / n = t * kInv16[n] >> 16 for t < 256
__constant__ unsigned kInv16[17] = {0, 65537, 32769, 21846, 16385, 13108, 10923, 9363, 8193,
                                    7282, 6554, 5958, 5462, 5042, 4682, 4370, 4097};
constexpr int kSplitUnits = 4;             // halo (position, octet) pairs per thread
constexpr int kSplitMaxOct = 1024;         // (tap, octet) pairs of a chunk

struct SplitArgs {
  const float* x;
  const float* w;
  const float* bias;
  float* y;
  Geom g;
  int kdim;        // R * S * Cg
  int tn;          // channel tiles per group
  int tiles;       // pixel tiles * tn per region
  int nty, ntx;    // tile rows and columns per region
  int ti, th, tw;  // images, rows and columns of a tile
  int hh, hw;      // halo rows and columns per image
  int twp;         // tile columns a row of positions takes (tw, or tw rounded up to 16)
  int hp;          // halo positions, ti * hh * hw
  int hps;         // slots per octet plane (a multiple of 16, >= hp)
  int co;          // octets per chunk
  int ash;         // extra slots before every second octet plane
  int lgh;         // log2(co / 2) for 2, 4 or 8 octets, else -1
  int nchunk;
  int noct;        // R * S * co
  int nst;         // stages per chunk
  int ow_taps, ow_cg;  // transposed filter: R * S and channels per group of the original
  int rx, nreg, rh, rw;  // output regions of rh x rw positions, rx per row (forward: the filter blocks)
  int By, Bx, bias_mode;
  int bho, bwo;  // positions of a filter block (blocked dx: of dy)
  int nfast;     // tile positions in (row, column, image) order instead of (image, row, column)
  FastDivM fd_tn, fd_tiles, fd_reg, fd_rx, fd_ntx, fd_nty, fd_co, fd_s, fd_hw, fd_hhw, fd_twp, fd_thw, fd_ti;
};

__device__ __forceinline__ int f32s_slot(int row, int g) { return 4 * row + (g ^ (((row >> 3) & 1) << 1)); }

// MODE kSplitFwd: the forward convolution, a region's positions use its block's filter.  kSplitTrans:
// the filter read as the dx filter of a stride-1 convolution (ow_* extents).  kSplitTransBlocked:
// the same with a blocked filter, whose blocks partition this kernel's input (dy): a chunk's halo
// is staged once and the reduction runs once per block that the tile's taps reach, over the taps
// that reach it, each lane reading zeros for the positions of other blocks and each pair of
// segments skipping the taps that none of its lanes uses.  With the image the fastest index of a
// tile (16 images: a segment is one position) nearly every tap of a segment falls in one block.
// Measured (us; before: the fp32 implicit GEMM's blocked form): 32 x 28 x 28, 128 -> 256 in 2 x 4
// blocks 215 (368); 32 x 56 x 56, 64 -> 64 in 2 x 2 125 (127), in 4 x 4 119 (158); one image in
// 4 x 4 44 (80). The stages of a neighbour's few taps bound it: a stage's filter values cost the
// same whatever its MFMAs, so fetching them two stages ahead and keeping the reach in LDS (five
// divisions a block otherwise) took the first from 404 to 226.
enum SplitMode : int { kSplitFwd = 0, kSplitTrans = 1, kSplitTransBlocked = 2 };

template <int MODE, int NSEG, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN, 2) f32_split_kernel(SplitArgs a) {
  constexpr bool TRANS = MODE != kSplitFwd;
  constexpr bool MULTI = MODE == kSplitTransBlocked;
  constexpr int NT = 64 * WM * WN;
  constexpr int BM = 16 * NSEG * WM;
  constexpr int BN = 32 * WN;
  constexpr int SO = 2 * WM < 4 ? 4 : 2 * WM;  // filter octets per stage
  constexpr int BU = SO * BN / NT;             // filter (channel, octet) pairs per thread
  constexpr int BSH = 16 / SO;                 // extra slots before every second filter octet
  constexpr int BSZ = 3 * (SO * BN + BSH * SO / 2);  // 16-byte slots of a filter buffer
  static_assert(BU == 1 && NT == SO * BN && (SO == 4 || SO == 8), "whole filter stages, one pair per thread");
  extern __shared__ v4u lds[];
  const Geom& g = a.g;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wn = wave % WN;
  const int wm = wave / WN;

  v4u* const sA = lds;                                  // 3 * co * hps slots
  v4u* const sB = lds + 3 * (a.co * a.hps + 8);         // two filter buffers
  int* const tab = reinterpret_cast<int*>(sB + 2 * BSZ);  // nst * SO entries, then the flag

  const int lin = xcd_tile(blockIdx.x, gridDim.x);
  const int gr = fdiv(lin, a.fd_tiles);  // group * regions + region
  const int rem = lin - gr * a.tiles;
  const int grp = fdiv(gr, a.fd_reg);
  const int reg = gr - grp * a.nreg;
  const int rgy = fdiv(reg, a.fd_rx);
  const int rgx = reg - rgy * a.rx;
  const int tmi = fdiv(rem, a.fd_tn);
  const int n0 = (rem - tmi * a.tn) * BN;  // first channel of the group
  const int tq = fdiv(tmi, a.fd_ntx);
  const int tx0 = (tmi - tq * a.ntx) * a.tw;
  const int tim = fdiv(tq, a.fd_nty);
  const int ty0 = (tq - tim * a.nty) * a.th;
  const int img0 = tim * a.ti;
  const int row0 = rgy * a.rh, col0 = rgx * a.rw;
  const int h0 = (row0 + ty0) * g.sh - g.ph;  // input position of the halo's origin
  const int w0 = (col0 + tx0) * g.sw - g.pw;

  // a tile position m: image, row and column in the tile, and whether it is an output
  auto decode = [&](int m, int& im, int& lr, int& lc) -> bool {
    int p;
    if (MULTI && a.nfast) {
      p = fdiv(m, a.fd_ti);
      im = m - p * a.ti;
      if (p >= a.th * a.twp) return false;
    } else {
      im = fdiv(m, a.fd_thw);
      p = m - im * (a.th * a.twp);
    }
    lr = fdiv(p, a.fd_twp);
    lc = p - lr * a.twp;
    return im < a.ti && img0 + im < g.N && lc < a.tw && ty0 + lr < a.rh && tx0 + lc < a.rw &&
           (!MULTI || (row0 + ty0 + lr < g.Ho && col0 + tx0 + lc < g.Wo));  // the last regions are clipped
  };

  // LDS slot (in units of 48 bytes) of octet oc's plane.  ds_read_b128 serves lane quads of both
  // 16-lane groups of a half-wave in one cycle, so the planes of an even and the next odd octet
  // lie a multiple of 16 apart; ds_write_b128 serves 8 consecutive lanes, which stage octets of
  // one parity: those planes are `ash` further on each.
  auto plane = [&](int oc) { return oc * a.hps + (oc >> 1) * a.ash; };
  // halo units of this thread: byte offset from the tile's first image (kNone: reads zero), LDS
  // slot and octet
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc(a.x + static_cast<size_t>(img0) * g.H * g.W * g.C + static_cast<size_t>(grp) * g.Cg, 0x7fffffff);
  unsigned aoff[kSplitUnits];
  unsigned aput[kSplitUnits];  // slot | octet << 20
#pragma unroll
  for (int j = 0; j < kSplitUnits; ++j) {
    const int u = t + NT * j;
    int px, oc;
    if (a.lgh >= 0) {
      const int l = u & 15, h = 1 << a.lgh;
      oc = ((l & (h - 1)) << 1) | (l >> 3);
      px = ((u >> 4) << (3 - a.lgh)) + ((l & 7) >> a.lgh);
    } else {
      px = fdiv(u, a.fd_co);
      oc = u - px * a.co;
    }
    const int im = fdiv(px, a.fd_hhw);
    const int p = px - im * (a.hh * a.hw);
    const int hr = fdiv(p, a.fd_hw);
    const int hi = h0 + hr;
    const int wi = w0 + p - hr * a.hw;
    const bool in = px < a.hp;
    const bool ok = in && img0 + im < g.N && hi >= 0 && hi < g.H && wi >= 0 && wi < g.W;
    aoff[j] = ok ? 4u * (static_cast<unsigned>((im * g.H + hi) * g.W + wi) * g.C + 8 * oc) : kNone;
    aput[j] = in ? static_cast<unsigned>(3 * (plane(oc) + px)) | static_cast<unsigned>(oc) << 20 : ~0u;
  }
  // filter units: octet boct[j] of a stage, LDS slot, byte offset of the channel's row (TRANS: of
  // the channel)
  int boct[BU], bslot[BU];
  unsigned boff[BU];
  const int nblk = a.By * a.Bx;
  const int blk_stride = a.ow_taps * a.ow_cg;             // transposed: between filter blocks
  const int ko_stride = MULTI ? blk_stride * nblk : blk_stride;  // and between original channels
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(
      TRANS ? a.w + static_cast<size_t>(grp) * g.Cg * ko_stride
            : a.w + (static_cast<size_t>(grp) * g.Kg * nblk + reg) * a.kdim, 0x7fffffff);
#pragma unroll
  for (int j = 0; j < BU; ++j) {
    const int u = t + NT * j;
    constexpr int H = SO / 2;
    const int r = TRANS ? u % BN : (u >> 4) * (8 / H) + ((u & 7) / H);
    boct[j] = TRANS ? u / BN : (((u & (H - 1)) << 1) | ((u >> 3) & 1));
    bslot[j] = 3 * (boct[j] * BN + (boct[j] >> 1) * BSH + r);
    const int kr = min(n0 + r, g.Kg - 1);
    boff[j] = 4u * (TRANS ? static_cast<unsigned>(kr) : static_cast<unsigned>(kr * nblk) * a.kdim);
  }
  // LDS offset of each (tap, octet) pair's halo values, relative to a position's slot
  for (int o = t; o < a.nst * SO; o += NT) {
    const int tap = fdiv(o, a.fd_co);
    const int r = fdiv(tap, a.fd_s);
    const int off = plane(o - tap * a.co) + r * g.dh * a.hw + (tap - r * g.S) * g.dw;
    tab[o] = o < a.noct ? 48 * off : 0;
  }
  int* const flag = tab + a.nst * SO;
  if (t == 0) *flag = 0;
  // MULTI: 48 bytes of zeros behind the table, at a 16-byte boundary
  const int zoff = (static_cast<int>(reinterpret_cast<char*>(flag + 4) - reinterpret_cast<char*>(lds)) & ~15);
  if (MULTI && t < 12) reinterpret_cast<int*>(reinterpret_cast<char*>(lds) + zoff)[t] = 0;

  // the tile's segments of 16 positions, spread evenly over the WM rows of waves: this wave's
  // first, how many are its own, and whether that is NSEG (else it computes NSEG - 1 and keeps its own)
  const int segs = (a.ti * a.th * a.twp + 15) >> 4;
  const int each = segs / WM, extra = segs - each * WM;
  const int seg0 = wm * each + min(wm, extra);
  const int own = each + (wm < extra ? 1 : 0);
  const bool whole = own >= NSEG;
  const int m0 = 16 * seg0 + (lane & 15);
  int pbase[NSEG];  // byte offset of this lane's positions
#pragma unroll
  for (int i = 0; i < NSEG; ++i) {
    int im, lr, lc;
    const bool ok = decode(m0 + 16 * i, im, lr, lc);
    pbase[i] = ok ? 48 * ((im * a.hh + lr * g.sh) * a.hw + lc * g.sw) : 0;
  }

  v4f va[kSplitUnits][2];
  v4f vb[MULTI ? 2 : 1][BU][2];  // filter values in flight, MULTI: of two stages
  const v4f zero = v4f{0.f, 0.f, 0.f, 0.f};
  auto load_a = [&](int c) {
    const int c0 = 8 * a.co * c;
#pragma unroll
    for (int j = 0; j < kSplitUnits; ++j) {
      const int left = g.Cg - c0 - 8 * static_cast<int>(aput[j] >> 20);
      va[j][0] = buffer_load16(rx, left >= 4 ? aoff[j] : kNone, 4 * c0);
      va[j][1] = buffer_load16(rx, left >= 8 ? aoff[j] + 16u : kNone, 4 * c0);
    }
  };
  float ascale = kSplitScale;  // SO 4: every second chunk's halo is negated
  auto store_a = [&]() {
#pragma unroll
    for (int j = 0; j < kSplitUnits; ++j) {
      if (aput[j] != ~0u) {
        const Split8 s = split8(va[j][0], va[j][1], ascale);
        v4u* const d = sA + (aput[j] & 0xfffffu);
#pragma unroll
        for (int p = 0; p < 3; ++p) d[p] = s.p[p];
      }
    }
  };
  // The filter blocks a tile reaches (MULTI; else one block with every tap): the taps r0.., s0.. of
  // nr x ns that read the block and the block's rows and columns of the input.
  struct Reach {
    int idx, r0, s0, nr, ns, y0, y1, x0, x1, fblk, noct, nst;
    unsigned inv;  // tap / ns = tap * inv >> 16 (tap < 256)
  };
  int bqx0 = 0, bnx = 1, bqy0 = 0, nreach = 1;
  if constexpr (MULTI) {
    const int ylo = max(h0, 0), yhi = min(h0 + a.hh, g.H) - 1, xlo = max(w0, 0), xhi = min(w0 + a.hw, g.W) - 1;
    nreach = 0;
    if (ylo <= yhi && xlo <= xhi) {
      bqy0 = ylo / a.bho;
      bqx0 = xlo / a.bwo;
      bnx = xhi / a.bwo - bqx0 + 1;
      nreach = (yhi / a.bho - bqy0 + 1) * bnx;
    }
  }
  // MULTI: the reach's blocks, 8 ints each behind the zeros: r0 | nr << 8 | s0 << 16 | ns << 24 (0: no
  // tap reads the block), rows y0, y1, columns x0, x1, element offset of the block's filter
  int* const rtab = reinterpret_cast<int*>(reinterpret_cast<char*>(lds) + zoff + 48);
  if constexpr (MULTI) {
    if (t < nreach) {
      const int qy = t / bnx, qx = t - qy * bnx;
      const int y0 = (bqy0 + qy) * a.bho, x0 = (bqx0 + qx) * a.bwo;
      const int y1 = min(y0 + a.bho, g.H) - 1, x1 = min(x0 + a.bwo, g.W) - 1;
      const int ra = y0 - h0 - (a.th - 1), sa = x0 - w0 - (a.tw - 1);
      const int r0 = ra > 0 ? (ra + g.dh - 1) / g.dh : 0, s0 = sa > 0 ? (sa + g.dw - 1) / g.dw : 0;
      const int nr = y1 >= h0 ? min(g.R - 1, (y1 - h0) / g.dh) - r0 + 1 : 0;
      const int ns = x1 >= w0 ? min(g.S - 1, (x1 - w0) / g.dw) - s0 + 1 : 0;
      rtab[8 * t] = nr > 0 && ns > 0 ? r0 | nr << 8 | s0 << 16 | ns << 24 : 0;
      rtab[8 * t + 1] = y0;
      rtab[8 * t + 2] = y1;
      rtab[8 * t + 3] = x0;
      rtab[8 * t + 4] = x1;
      rtab[8 * t + 5] = ((bqy0 + qy) * a.Bx + bqx0 + qx) * blk_stride;
    }
    __syncthreads();
  }
  // block `idx` of the reach or the next one with taps; idx == nreach: none left
  auto set_reach = [&](Reach& b, int idx) {
    b.idx = idx;
    if constexpr (!MULTI) {
      b.noct = a.noct;
      b.nst = a.nst;
    } else {
      int packed = 0;
      for (; b.idx < nreach; ++b.idx) {
        packed = __builtin_amdgcn_readfirstlane(rtab[8 * b.idx]);
        if (packed != 0) break;
      }
      if (b.idx < nreach) {
        b.r0 = packed & 0xff;
        b.nr = (packed >> 8) & 0xff;
        b.s0 = (packed >> 16) & 0xff;
        b.ns = packed >> 24;
        b.y0 = __builtin_amdgcn_readfirstlane(rtab[8 * b.idx + 1]);
        b.y1 = __builtin_amdgcn_readfirstlane(rtab[8 * b.idx + 2]);
        b.x0 = __builtin_amdgcn_readfirstlane(rtab[8 * b.idx + 3]);
        b.x1 = __builtin_amdgcn_readfirstlane(rtab[8 * b.idx + 4]);
        b.fblk = __builtin_amdgcn_readfirstlane(rtab[8 * b.idx + 5]);
        b.noct = b.nr * b.ns * a.co;
        b.nst = (b.noct + SO - 1) / SO;
        b.inv = kInv16[b.ns];
      }
    }
  };
  auto load_b = [&](auto set, int c, int s, const Reach& rb) {
    constexpr int V = MULTI ? decltype(set)::value : 0;
    const int c0 = 8 * a.co * c;
#pragma unroll
    for (int j = 0; j < BU; ++j) {
      const int o = SO * s + boct[j];
      const int tap = fdiv(o, a.fd_co);
      const int ch = c0 + 8 * (o - tap * a.co);
      const int left = o < rb.noct ? g.Cg - ch : 0;
      if constexpr (TRANS) {
        int ft = tap, fblk = 0;
        if constexpr (MULTI) {
          const int tr = static_cast<int>((static_cast<unsigned>(tap) * rb.inv) >> 16);
          ft = (rb.r0 + tr) * g.S + rb.s0 + tap - tr * rb.ns;
          fblk = rb.fblk;
        }
        const unsigned off = boff[j] + 4u * (ch * ko_stride + fblk + (a.ow_taps - 1 - ft) * a.ow_cg);
        const unsigned o0 = left >= 4 ? off : kNone, o1 = left >= 8 ? off : kNone;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vb[V][j][0][e] = buffer_load4(rw, o0, 4 * e * ko_stride);
          vb[V][j][1][e] = buffer_load4(rw, o1, 4 * (e + 4) * ko_stride);
        }
      } else {
        const unsigned off = boff[j] + 4u * (tap * g.Cg + ch);
        vb[V][j][0] = buffer_load16(rw, left >= 4 ? off : kNone, 0);
        vb[V][j][1] = buffer_load16(rw, left >= 8 ? off + 16u : kNone, 0);
      }
    }
  };
  // the values of the set's last load_b
  const float bscale = !MULTI && SO == 8 && (boct[0] & 4) ? -kSplitScale : kSplitScale;
  auto store_b = [&](auto set, int buf, float scale) {
    constexpr int V = MULTI ? decltype(set)::value : 0;
#pragma unroll
    for (int j = 0; j < BU; ++j) {
      const Split8 sp = split8(vb[V][j][0], vb[V][j][1], scale);
#pragma unroll
      for (int p = 0; p < 3; ++p) sB[buf * BSZ + bslot[j] + p] = sp.p[p];
    }
  };

  v4f acc[2][NSEG];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < NSEG; ++i) acc[j][i] = zero;

  const char* const bA = reinterpret_cast<const char*>(sA);
  const char* const bB = reinterpret_cast<const char*>(sB) + 48 * (32 * wn + (lane & 15) + BN * q + BSH * (q >> 1));
  // Stages in order over the chunks, for a wave of NS segments: the filter values of stage i + 1
  // are split and stored, and those of stage i + 2 fetched, inside stage i.  A K-block runs in
  // steps of up to two segments; a step's fragments are read while the step before it computes.
  // The six products of a step sum from zero, smallest first, and are added to the accumulators.
  int lc = 0, ls = 0;  // stage of the next load_b
  Reach lb;
  set_reach(lb, 0);
  const int first_reach = lb.idx;
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  auto fetch = [&](auto set) {
    load_b(set, lc, ls, lb);
    if (++ls == lb.nst) {
      ls = 0;
      if constexpr (MULTI) {
        set_reach(lb, lb.idx + 1);
        if (lb.idx >= nreach) {
          set_reach(lb, 0);
          lc = min(lc + 1, a.nchunk - 1);
        }
      } else {
        lc = min(lc + 1, a.nchunk - 1);  // past the end: loaded, never used
      }
    }
  };
  auto run = [&](auto ns) {
    constexpr int NS = decltype(ns)::value;
    constexpr int HALVES = (NS + 1) / 2;       // steps per K-block
    constexpr int STEPS = SO / 4 * HALVES;     // steps per stage
    int buf = 0;
    for (int c = 0; c < a.nchunk; ++c) {
      const bool more = c + 1 < a.nchunk;
      for (int s = 0; s < a.nst; ++s) {
        int ao[SO / 4];
#pragma unroll
        for (int kb = 0; kb < SO / 4; ++kb) ao[kb] = tab[SO * s + 4 * kb + q];
        const char* const bs = bB + 16 * buf * BSZ;
        v8b fa[2][2][3], fb[2][2][3];
        auto read = [&](int st) {
          const int kb = st / HALVES, i0 = 2 * (st % HALVES);
          if (i0 == 0) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int p = 0; p < 3; ++p)
                fb[kb & 1][j][p] = *reinterpret_cast<const v8b*>(bs + 16 * p + 48 * (4 * kb * BN + 2 * kb * BSH + 16 * j));
          }
#pragma unroll
          for (int i = 0; i < 2; ++i)
            if (i0 + i < NS) {
#pragma unroll
              for (int p = 0; p < 3; ++p)
                fa[st & 1][i][p] = *reinterpret_cast<const v8b*>(bA + pbase[i0 + i] + ao[kb] + 16 * p);
            }
        };
        auto step = [&](auto stc) {
          constexpr int st = decltype(stc)::value;
          constexpr int kb = st / HALVES, i0 = 2 * (st % HALVES);
          if constexpr (st + 1 < STEPS) read(st + 1);
          __builtin_amdgcn_sched_barrier(0x276);  // the reads above, the MFMAs below; the rest may move
          v4f z[2][2];
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            constexpr int kw[6] = {2, 0, 1, 1, 0, 0}, kx[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int i = 0; i < 2; ++i)
              if (i0 + i < NS) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                  z[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kb & 1][j][kw[k]], fa[st & 1][i][kx[k]],
                                                                    k == 0 ? zero : z[j][i], 0, 0, 0);
              }
          }
          if constexpr (st == 0) {
            store_b(even, buf ^ 1, bscale);
            fetch(even);
            if (s == 0) load_a(more ? c + 1 : c);
          }
#pragma unroll
          for (int i = 0; i < 2; ++i)
            if (i0 + i < NS) {
#pragma unroll
              for (int j = 0; j < 2; ++j) acc[j][i0 + i] = kb == 0 ? acc[j][i0 + i] + z[j][i] : acc[j][i0 + i] - z[j][i];
            }
        };
        read(0);
        step(std::integral_constant<int, 0>{});
        if constexpr (HALVES > 1) step(std::integral_constant<int, 1>{});
        if constexpr (SO > 4) {
          if (SO * s + 4 < a.noct) {  // uniform: a second K-block
            step(std::integral_constant<int, HALVES>{});
            if constexpr (HALVES > 1) step(std::integral_constant<int, HALVES + 1>{});
          }
        }
        __syncthreads();
        buf ^= 1;
      }
      if (more) {
        if constexpr (SO == 4) {
          ascale = -ascale;
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < NS; ++i) acc[j][i] = -acc[j][i];
        }
        store_a();
        __syncthreads();
      }
    }
  };
  // MULTI: the chunk's stages block after block, a K-block's fragments read where it is computed
  auto run_blocks = [&]() {
    int prow[NSEG], pcol[NSEG];  // this lane's positions on the input grid, tap (0, 0)
#pragma unroll
    for (int i = 0; i < NSEG; ++i) {
      int im, lr, lcc;
      const bool ok = i < own && decode(m0 + 16 * i, im, lr, lcc);
      prow[i] = ok ? h0 + lr : INT32_MIN / 2;
      pcol[i] = w0 + lcc;
    }
    Reach rb;
    unsigned use[NSEG];  // rows r (bit r) and columns s (bit 16 + s) of the block
    auto enter = [&](int idx) {
      set_reach(rb, idx);
      if (rb.idx >= nreach) return;
#pragma unroll
      for (int i = 0; i < NSEG; ++i) use[i] = 0;
      for (int r = rb.r0; r < rb.r0 + rb.nr; ++r)
#pragma unroll
        for (int i = 0; i < NSEG; ++i)
          use[i] |= static_cast<unsigned>(prow[i] + r * g.dh >= rb.y0 && prow[i] + r * g.dh <= rb.y1) << r;
      for (int s = rb.s0; s < rb.s0 + rb.ns; ++s)
#pragma unroll
        for (int i = 0; i < NSEG; ++i)
          use[i] |= static_cast<unsigned>(pcol[i] + s * g.dw >= rb.x0 && pcol[i] + s * g.dw <= rb.x1) << (16 + s);
    };
    // stage s of the block: the filter buffer and register set of its parity over all stages
    auto stage = [&](auto par, auto other, int c, int s) {
      constexpr int PAR = decltype(par)::value;
      store_b(other, PAR ^ 1, PAR ? kSplitScale : -kSplitScale);  // buffer 1 is negated
      fetch(other);
      if (s == 0 && rb.idx == first_reach) load_a(min(c + 1, a.nchunk - 1));
#pragma unroll
      for (int kb = 0; kb < SO / 4; ++kb) {
        const int o = SO * s + 4 * kb + q;
        if (SO * s + 4 * kb < rb.noct) {  // uniform
          const int tap = fdiv(o, a.fd_co);
          const int tr = static_cast<int>((static_cast<unsigned>(tap) * rb.inv) >> 16);
          const int r = rb.r0 + tr, ss = rb.s0 + tap - tr * rb.ns;
          const int ao = 48 * (plane(o - tap * a.co) + r * g.dh * a.hw + ss * g.dw);
          const bool in = o < rb.noct;
          v8b fb[2][3];
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int p = 0; p < 3; ++p)
              fb[j][p] = *reinterpret_cast<const v8b*>(bB + 16 * (PAR * BSZ + p) + 48 * (4 * kb * BN + 2 * kb * BSH + 16 * j));
#pragma unroll
          for (int i0 = 0; i0 < NSEG; i0 += 2) {
            bool hit[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) hit[i] = in && ((use[i0 + i] >> r) & (use[i0 + i] >> (16 + ss)) & 1u) != 0;
            if (__any(hit[0] || hit[1])) {
              v8b fa[2][3];
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                const int ad = hit[i] ? pbase[i0 + i] + ao : zoff;
#pragma unroll
                for (int p = 0; p < 3; ++p) fa[i][p] = *reinterpret_cast<const v8b*>(bA + ad + 16 * p);
              }
              v4f z[2][2];
#pragma unroll
              for (int k = 0; k < 6; ++k) {
                constexpr int kw[6] = {2, 0, 1, 1, 0, 0}, kx[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                  for (int j = 0; j < 2; ++j)
                    z[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j][kw[k]], fa[i][kx[k]], k == 0 ? zero : z[j][i], 0, 0, 0);
              }
#pragma unroll
              for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[j][i0 + i] = PAR ? acc[j][i0 + i] - z[j][i] : acc[j][i0 + i] + z[j][i];
            }
          }
        }
      }
      __syncthreads();
    };
    int c = 0, s = 0;
    enter(0);
    auto next = [&]() {  // the next stage: of the block, the next block, the next chunk
      if (++s < rb.nst) return true;
      s = 0;
      enter(rb.idx + 1);
      if (rb.idx < nreach) return true;
      if (++c == a.nchunk) return false;
      enter(0);
      store_a();
      __syncthreads();
      return true;
    };
    while (true) {
      stage(even, odd, c, s);
      if (!next()) break;
      stage(odd, even, c, s);
      if (!next()) break;
    }
  };
  // both arms run the same barriers; a tile that reaches no block is zero
  if (!MULTI || first_reach < nreach) {
    fetch(even);
    load_a(0);
    if constexpr (MULTI) fetch(odd);
    store_b(even, 0, MULTI ? kSplitScale : bscale);
    fetch(even);
    store_a();
    __syncthreads();
    if constexpr (MULTI) run_blocks();
    else if (NSEG == 1 || whole) run(std::integral_constant<int, NSEG>{});
    else run(std::integral_constant<int, NSEG == 1 ? 1 : NSEG - 1>{});
  }

  bool bad = false;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < NSEG; ++i) {
      int im, lr, lc;
      const bool ok = i < own && decode(m0 + 16 * i, im, lr, lc);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bad |= ok && !(__builtin_fabsf(acc[j][i][e]) <= kFltMax);
      }
    }
  if (bad) *flag = 1;
  __syncthreads();
  if (*flag != 0) {
    // the tile again with fp32 MFMAs: per tap, 16 channels a step, gathered into LDS
    constexpr int UR = BM * 4 < NT ? 1 : BM * 4 / NT;
    v4f* const fA = reinterpret_cast<v4f*>(lds);
    v4f* const fB = fA + BM * 4;
    int uh[UR], uw[UR];
    const float* ux[UR];
#pragma unroll
    for (int k = 0; k < UR; ++k) {
      int im, lr, lc;
      const bool ok = decode((t + NT * k) >> 2, im, lr, lc);
      uh[k] = ok ? h0 + lr * g.sh : INT32_MIN / 2;
      uw[k] = w0 + lc * g.sw;
      ux[k] = a.x + static_cast<size_t>(ok ? img0 + im : 0) * g.H * g.W * g.C + static_cast<size_t>(grp) * g.Cg;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < NSEG; ++i) acc[j][i] = zero;
    for (int tb = 0; tb < g.R * g.S * (MULTI ? nreach : 1); ++tb) {  // taps, MULTI: of each block
      const int bi = MULTI ? tb / (g.R * g.S) : 0;
      const int tap = tb - bi * (g.R * g.S);
      const int r = fdiv(tap, a.fd_s);
      const int s = tap - r * g.S;
      const int qy = bqy0 + bi / bnx, qx = bqx0 + bi - bi / bnx * bnx;
      const int ylo = MULTI ? qy * a.bho : 0, yhi = MULTI ? min(ylo + a.bho, g.H) : g.H;
      const int xlo = MULTI ? qx * a.bwo : 0, xhi = MULTI ? min(xlo + a.bwo, g.W) : g.W;
      const size_t fblk = MULTI ? static_cast<size_t>(qy * a.Bx + qx) * blk_stride : 0;
      for (int c0 = 0; c0 < g.Cg; c0 += 16) {
        __syncthreads();  // the previous step's reads (and the flag's)
        const int ch = c0 + 4 * (t & 3);
#pragma unroll
        for (int k = 0; k < UR; ++k) {
          const int hi = uh[k] + r * g.dh, wi = uw[k] + s * g.dw;
          const bool ok = ch < g.Cg && hi >= ylo && hi < yhi && wi >= xlo && wi < xhi;
          const v4f v = *reinterpret_cast<const v4f*>(ok ? ux[k] + (static_cast<size_t>(hi) * g.W + wi) * g.C + ch : a.x);
          if (t + NT * k < BM * 4) fA[f32s_slot((t + NT * k) >> 2, t & 3)] = ok ? v : zero;
        }
        for (int u = t; u < BN * 4; u += NT) {
          const int kr = min(n0 + (u >> 2), g.Kg - 1);
          const int cb = c0 + 4 * (u & 3);
          v4f v = zero;
          if (cb < g.Cg) {
            if constexpr (TRANS) {
              const float* p = a.w + (static_cast<size_t>(grp) * g.Cg + cb) * ko_stride +
                               fblk + static_cast<size_t>(a.ow_taps - 1 - tap) * a.ow_cg + kr;
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = p[e * ko_stride];
            } else {
              v = *reinterpret_cast<const v4f*>(a.w + (static_cast<size_t>(grp * g.Kg + kr) * nblk + reg) * a.kdim +
                                                static_cast<size_t>(tap) * g.Cg + cb);
            }
          }
          fB[f32s_slot(u >> 2, u & 3)] = v;
        }
        __syncthreads();
        v4f fb[2], fa[NSEG];
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[j] = fB[f32s_slot(32 * wn + 16 * j + (lane & 15), q)];
#pragma unroll
        for (int i = 0; i < NSEG; ++i) fa[i] = fA[f32s_slot(min(m0 + 16 * i, BM - 1), q)];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < NSEG; ++i)
              acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][k], fa[i][k], acc[j][i], 0, 0, 0);
      }
    }
  } else {
    const float unscale = ascale < 0.0f ? -kSplitUnscale : kSplitUnscale;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < NSEG; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][i][e] = __builtin_fmaf(acc[j][i][e], unscale, 0.0f);  // a zero sum is +0
  }

  // lane (c = lane % 16, q): position c of each segment, channels 4 q .. 4 q + 3 of each 16
  const bool vec = (g.K & 3) == 0 && (g.Kg & 3) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15u) == 0;
  const int bias_y = a.bias_mode == 0 ? rgy : 0;
  const int bias_x = a.bias_mode == 0 ? rgx : 0;
#pragma unroll
  for (int i = 0; i < NSEG; ++i) {
    int im, lr, lc;
    if (i >= own || !decode(m0 + 16 * i, im, lr, lc)) continue;
    const size_t pix = (static_cast<size_t>(img0 + im) * g.Ho + row0 + ty0 + lr) * g.Wo + col0 + tx0 + lc;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int ch = n0 + 32 * wn + 16 * j + 4 * q;
      float* yp = a.y + pix * g.K + static_cast<size_t>(grp) * g.Kg + ch;
      v4f r = acc[j][i];
      if (!TRANS && a.bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = grp * g.Kg + min(ch + e, g.Kg - 1);
          r[e] = __fadd_rn(r[e], a.bias[(static_cast<size_t>(k) * a.By + bias_y) * a.Bx + bias_x]);
        }
      }
      if (vec && ch + 3 < g.Kg) {
        *reinterpret_cast<v4f*>(yp) = r;
        store_gap(r);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ch + e < g.Kg) yp[e] = r[e];
      }
    }
  }
}

// Tile of one launch variant, and its estimated time.
struct SplitPlan {
  int variant;  // index into kVariants, -1: none fits
  int ti, th, tw, twp, hh, hw, hp, hps, co, ash, nchunk, noct, nst;
  int nty, ntx, nti, tn;
  size_t lds;
  long long blocks;
  double cost;
};

struct SplitVariant {
  int nseg, wm, wn;
};
constexpr SplitVariant kVariants[] = {{4, 4, 2}, {4, 2, 2}, {2, 2, 2}, {4, 4, 1}, {1, 4, 2}};

// a reduction and an image to run over; an empty one is all zeros, which the implicit GEMM writes
bool plain_extents(const Geom& g) {
  return g.N > 0 && g.H > 0 && g.W > 0 && g.Cg > 0 && g.Kg > 0 && g.R > 0 && g.S > 0;
}

// Estimated cycles of a launch: rounds of workgroups over the 256 CUs x (K-blocks at the MFMA rate
// of a wave's tile, the staged values, a fixed start and end).
void consider(const Geom& g, int rh, int rw, long long nreg, int v, int ti, int th, int tw, int twp,
              bool blocked_dx, SplitPlan* best) {
  const SplitVariant& V = kVariants[v];
  const int nt = 64 * V.wm * V.wn, bn = 32 * V.wn, so = std::max(4, 2 * V.wm);
  SplitPlan p{};
  p.variant = v;
  p.ti = ti; p.th = th; p.tw = tw; p.twp = twp;
  p.hh = (th - 1) * g.sh + (g.R - 1) * g.dh + 1;
  p.hw = (tw - 1) * g.sw + (g.S - 1) * g.dw + 1;
  const long long hp = static_cast<long long>(ti) * p.hh * p.hw;
  if (hp > kSplitUnits * nt || static_cast<double>(ti) * g.H * g.W * g.C * 4 >= 2147483647.0) return;
  p.hp = static_cast<int>(hp);
  p.nty = (rh + th - 1) / th;
  p.ntx = (rw + tw - 1) / tw;
  p.nti = (g.N + ti - 1) / ti;
  p.tn = (g.Kg + bn - 1) / bn;
  p.blocks = nreg * g.G * p.nty * p.ntx * static_cast<long long>(p.nti) * p.tn;
  const int oct = (g.Cg + 7) / 8;
  int tried = 0;
  for (const int want : {8, 6, 4, 3, 2, 1}) {  // octets of a chunk, evened out over the chunks
    if (want > oct && want != 8 && tried != 0) continue;
    const int chunks = (oct + want - 1) / want;
    const int co = (oct + chunks - 1) / chunks;
    if (co == tried) continue;
    tried = co;
    if (co == 1 && oct > 1) continue;  // a K-block of four taps: its fragment reads conflict in the banks
    const long long noct = static_cast<long long>(g.R) * g.S * co;
    if (hp * co > kSplitUnits * nt || noct > kSplitMaxOct) continue;
    p.co = co;
    p.nchunk = (oct + co - 1) / co;
    p.noct = static_cast<int>(noct);
    p.nst = (p.noct + so - 1) / so;
    p.hps = (p.hp + 15) & ~15;
    p.ash = co >= 6 ? 2 : (co >= 4 ? 4 : 0);
    const int bsz = 3 * (so * bn + (16 / so) * so / 2);
    p.lds = static_cast<size_t>(3 * (co * p.hps + 8) + 2 * bsz) * 16 + static_cast<size_t>(p.nst * so + 1) * 4 +
            (blocked_dx ? 80 + 32 * kSplitMaxReach : 0);
    if (p.lds > kSplitLds) continue;
    // workgroups that share a CU; a stage takes at least its filter values' way through the
    // registers (1200 cycles with 4 waves, 1950 with 8, measured on one image), less when shared
    const int fit = std::max(1, std::min<int>({static_cast<int>(kSplitLds / p.lds), 8 / (V.wm * V.wn), 4}));
    const int per_cu = std::max(1, static_cast<int>(std::min<long long>(fit, (p.blocks + 255) / 256)));
    const double least = (V.wm * V.wn >= 8 ? 1950.0 : 1200.0) / std::sqrt(static_cast<double>(per_cu));
    const double kbs = V.nseg * 12 * 16.0 * V.wm * V.wn / 4 * 1.25;  // SIMD cycles of a K-block
    const double mfma = p.nchunk * ((p.noct + 3) / 4) * kbs;
    const double stage = p.nchunk * (static_cast<double>(p.hp) * co + static_cast<double>(p.nst) * so * bn) * 60.0 / 64;
    double wg = p.nchunk * p.nst * std::max((p.noct + 3) / 4 * kbs / p.nst, least) + stage * 0.7 +
                2500.0 * p.nchunk / per_cu + (2500.0 + 1000.0 * V.nseg) / per_cu;
    if (blocked_dx) {
      // a tile edge on a block edge adds the taps that cross it: (block, tap) pairs and blocks of
      // an average tile; a stage takes at least its filter values' way through the registers
      const double pairs = (g.R + (g.R - 1.0) / p.nty) * (g.S + (g.S - 1.0) / p.ntx);
      const double blks = (1 + (g.R > 1 ? 2.0 : 0.0) / p.nty) * (1 + (g.S > 1 ? 2.0 : 0.0) / p.ntx);
      const double stages = p.nchunk * (pairs * co / so + 0.5 * blks);
      const double bleast = 1.13 * least;
      wg = std::max(mfma, stages * bleast) + 0.24 * std::min(mfma, stages * bleast) + stage * 0.7 +
           2500.0 * p.nchunk / per_cu + 4000.0 / per_cu;
    }
    const double rounds = std::ceil(static_cast<double>(p.blocks) / (256.0 * per_cu)) * per_cu;
    p.cost = std::min(rounds, static_cast<double>(p.blocks) / 256.0 + 0.5 * per_cu) * wg;
    if (best->variant < 0 || p.cost < best->cost) *best = p;
  }
}

// One tap: whether the split is the faster kernel in the chosen tile (us, fp32 GEMM against split; the
// GEMM is taken where it gains more than the 2 to 4% that its short sums cost).  Each stage is as long
// as the latency of its filter values, so it has to hold 8 octets or the reduction 256 channels: tiles
// of 4 waves hold 4 a stage (dx 8 x 56 x 56, 64 -> 128 11.3 / 12.0; 8 x 28 x 28, 256 -> 256 18.0 /
// 16.5), and 256 positions leave room for fewer than 8 octets of halo (112 x 112, 256 -> 16 17.8 /
// 22.4), which pays while its second round is not full (32 x 56 x 56 2 x 2 blocks, 512 -> 32 54.9 /
// 49.0).  A last round of few workgroups is a whole one (dx 8 x 72 x 72, 96 -> 128 in 352: 25.3 / 28.0;
// 96 -> 256 42.1 / 40.2).
bool one_tap_pays(const Geom& g, const SplitPlan& p, bool transposed) {
  const SplitVariant& v = kVariants[p.variant];
  if (v.wn == 1) {
    return p.nchunk * p.nst <= (g.Cg + 63) / 64 || (p.blocks > 256 && (transposed || p.blocks <= 512));
  }
  if (g.Cg >= 256 || v.nseg == 1) return true;
  return v.wm == 4 &&
         (p.blocks <= 256 || 256.0 * ((p.blocks + 255) / 256) <= 1.35 * static_cast<double>(p.blocks));
}

// The tile of a launch, or variant -1 where the fp32 implicit GEMM is the faster kernel (measured
// on a 32 x 56 x 56 layer unless a size is given): with one tap nothing is read twice from the
// halo and a short reduction leaves the split unpaid (1x1 128 -> 256: 100 against 89 us; 512 -> 128
// at 14 x 14: 24.5 against 28; transposed 256 -> 64: 43 against 59), and at most 32 output channels
// at a stride give too few MFMAs per halo value (112 x 112, 32 -> 32: 39 against 35 us, 32 -> 64:
// 24 against 31); four channels fill half an octet (8 x 30 x 30, 4 -> 32: 9.2 against 8.3 us).
SplitPlan make_plan(const Geom& g, int rh, int rw, long long nreg, bool transposed) {
  SplitPlan best{};
  best.variant = -1;
  if (!plain_extents(g) || g.dh <= 0 || g.dw <= 0 || g.sh <= 0 || g.sw <= 0) return best;
  if (g.R * g.S == 1 && g.Cg < (transposed ? 128 : 256)) return best;
  if (g.Kg <= 32 && (g.sh > 1 || g.sw > 1)) return best;
  if (g.Cg < 8 && g.R * g.S <= 9) return best;
  // 32-bit byte offsets: into a group's filter (every block of it) and into an image
  if (static_cast<double>(std::max(g.Kg, g.Cg)) * nreg * g.R * g.S * std::max(g.Kg, g.Cg) * 4 >= 2147483647.0 ||
      static_cast<double>(g.H) * g.W * g.C * 4 >= 2147483647.0) {
    return best;
  }
  for (int v = 0; v < static_cast<int>(sizeof(kVariants) / sizeof(kVariants[0])); ++v) {
    if (kVariants[v].wn == 1 && g.Kg > 32) continue;
    if (kVariants[v].wn == 2 && g.Kg <= 32) continue;
    const int bm = 16 * kVariants[v].nseg * kVariants[v].wm;
    int last = 0;
    for (int j = 1; j <= 12; ++j) {
      const int tw = (rw + j - 1) / j;
      if (tw > bm || tw == last) continue;
      last = tw;
      int th = std::min(rh, bm / tw);
      th = (rh + (rh + th - 1) / th - 1) / ((rh + th - 1) / th);  // even rows of tiles
      const int ti = th == rh && tw == rw ? std::max(1, std::min(g.N, bm / (th * tw))) : 1;
      const int tw16 = (tw + 15) & ~15;  // rows of whole segments: no segment wraps into the next row
      if (tw16 != tw && ti * th * tw16 <= bm) consider(g, rh, rw, nreg, v, ti, th, tw, tw16, false, &best);
      else consider(g, rh, rw, nreg, v, ti, th, tw, tw, false, &best);
      if (tw <= 8) break;
    }
  }
  if (best.variant >= 0 && g.R * g.S == 1 && !one_tap_pays(g, best, transposed)) best.variant = -1;
  return best;
}

template <int MODE, int NSEG, int WM, int WN>
hipError_t launch_variant(const SplitArgs& a, const SplitPlan& p, hipStream_t stream) {
  if (p.lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&f32_split_kernel<MODE, NSEG, WM, WN>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kSplitLds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((f32_split_kernel<MODE, NSEG, WM, WN>), dim3(static_cast<unsigned>(p.blocks)),
                     dim3(64 * WM * WN), p.lds, stream, a);
  return hipGetLastError();
}

template <int MODE>
hipError_t launch_split(const SplitArgs& a, const SplitPlan& p, hipStream_t stream) {
  switch (p.variant) {
    case 0: return launch_variant<MODE, 4, 4, 2>(a, p, stream);
    case 1: return launch_variant<MODE, 4, 2, 2>(a, p, stream);
    case 2: return launch_variant<MODE, 2, 2, 2>(a, p, stream);
    case 3: return launch_variant<MODE, 4, 4, 1>(a, p, stream);
    default:
      if constexpr (MODE != kSplitTransBlocked) return launch_variant<MODE, 1, 4, 2>(a, p, stream);
      return hipErrorInvalidValue;
  }
}

}  // namespace

namespace {

// Along one dimension, the worst window of `len` output positions at multiples of `step` inside a
// region of `rlen`: how many filter blocks (of `blk` input positions) its taps reach, and the taps
// summed over them.  Regions 0 and 1 stand for all: an inner region has neighbours on both sides.
struct Reach1 {
  int taps, blocks;
};
Reach1 worst_reach(int in, int nreg, int rlen, int step, int len, int blk, int R, int d, int pad) {
  Reach1 worst{0, 0};
  for (int q = 0; q < std::min(nreg, 2); ++q)
    for (int o = 0; o < rlen; o += step) {
      const int lo = q * rlen + o - pad, hi = lo + len - 1;  // the window on the input, tap 0
      const int y1 = std::min(hi + (R - 1) * d, in - 1);
      Reach1 now{0, 0};
      for (int y = std::max(lo, 0) / blk * blk; y <= y1; y += blk) {
        const int r0 = y > hi ? (y - hi + d - 1) / d : 0;
        const int r1 = std::min(R - 1, (std::min(y + blk, in) - 1 - lo) / d);
        if (r1 < r0) continue;
        now.taps += r1 - r0 + 1;
        ++now.blocks;
      }
      if (now.taps > worst.taps) worst = now;
    }
  return worst;
}

// Estimated microseconds of the blocked dx: both kernels wait for their worst tile, whose pieces
// (stages of the split kernel, 16-channel chunks of the fp32 GEMM) pass one after the other.  Fitted to
// 422 layers of 1 x 2 to 4 x 4 blocks, 1 to 32 images, 3x3 and 5x5 taps: the GEMM within 4% on
// average (its short sums 3% on top), the split within 11%.
double split_blocked_us(const Geom& g, const BlockGeom& bg, int rh, int rw, const SplitPlan& p) {
  const Reach1 a = worst_reach(g.H, bg.By, rh, p.th, p.th, bg.bho, g.R, g.dh, g.ph);
  const Reach1 b = worst_reach(g.W, bg.Bx, rw, p.tw, p.tw, bg.bwo, g.S, g.dw, g.pw);
  const double so = std::max(4, 2 * kVariants[p.variant].wm);
  const double stages = p.nchunk * (static_cast<double>(a.taps) * b.taps * p.co / so + 0.5 * a.blocks * b.blocks);
  constexpr double fit[4][3] = {{5.5, 1.23, 9.1}, {8.3, 0.95, 3.9}, {6.2, 0.68, 8.9}, {3.0, 1.35, 6.4}};
  const double* f = fit[p.variant];
  return f[0] + f[1] * stages * std::max(1.0, p.blocks / 256.0) + f[2] * p.nchunk;
}
double igemm_blocked_us(const Geom& g, const BlockGeom& bg, int rh, int rw) {
  const int bm = g.Kg <= 32 ? 256 : 128, bn = g.Kg <= 32 ? 32 : 64;
  // its tile: bm (position, image) pairs, the image fastest; whole columns where it wraps a row
  const int pos = (bm + g.N - 1) / g.N;
  const bool in_row = bm % g.N == 0 && rw % pos == 0;
  const int rows = in_row ? 1 : std::min(rh, (pos + rw - 2) / rw + 1);
  const Reach1 a = worst_reach(g.H, bg.By, rh, 1, rows, bg.bho, g.R, g.dh, g.ph);
  const Reach1 b = in_row ? worst_reach(g.W, bg.Bx, rw, pos, pos, bg.bwo, g.S, g.dw, g.pw)
                          : worst_reach(g.W, bg.Bx, rw, rw, rw, bg.bwo, g.S, g.dw, g.pw);
  const double chunks = static_cast<double>(a.taps) * b.taps * g.Cg / 16;
  const double tiles = std::ceil(static_cast<double>(g.N) * rh * rw / bm) * bg.By * bg.Bx * ((g.Kg + bn - 1) / bn) * g.G;
  return 12.1 + 0.857 * chunks * std::max(1.0, tiles / 256);
}

// Blocked dx with one tap: whether the split is the faster kernel in the chosen tile (us, fp32 GEMM
// against split).  Few stages, all latency: small tiles, or tiles of 256 positions of few images that
// fill a round (two of a longer reduction) where the GEMM's tiles take twice as many.
// 32 x 8 x 8, 256 -> 256 in 4 x 4 blocks 20.4 / 18.0; 8 x 28 x 28, 512 -> 256 in 2 x 2 33.4 / 29.6;
// 8 x 56 x 56, 256 -> 256 59.2 / 56.5, 512 -> 256 99 / 109; 32 x 16 x 16, 512 -> 256 in tiles of 16
// images 33.5 / 45.0; 1 x 28 x 28, 256 -> 256 20.1 / 25.2.
bool one_tap_blocked_pays(const Geom& g, const BlockGeom& bg, const SplitPlan& p) {
  if (static_cast<long long>(g.N) * bg.bho * bg.bwo <= 32 || (p.th * p.tw <= 4 && p.ti <= 8)) return true;
  return p.variant == 0 && p.ti <= 4 && p.blocks >= 192 && p.blocks <= (g.Cg >= 256 ? 512 : 256);
}

// Blocked dx: 16 images (or all of fewer) x a few positions per tile, tiles inside regions of
// ceil(Ho / By) x ceil(Wo / Bx), so that most reach one filter block.  Variant -1 where the fp32
// implicit GEMM is the faster kernel: by the two estimates (32 x 14 x 14, 128 -> 64 5x5 in 2 x 2
// blocks 156 us against 215; over 499 layers no call more than 1.11 times the faster kernel's time,
// where the split alone was up to 1.42), and with one tap by one_tap_blocked_pays.
SplitPlan make_blocked_plan(const Geom& g, const BlockGeom& bg, int rh, int rw) {
  SplitPlan best{};
  best.variant = -1;
  const long long nreg = static_cast<long long>(bg.By) * bg.Bx;
  if (!plain_extents(g) || g.dh <= 0 || g.dw <= 0 || g.R > 16 || g.S > 16) return best;
  const bool one_tap = g.R * g.S == 1;
  if (one_tap && g.Cg < 128) return best;
  if (static_cast<double>(g.Kg) * nreg * g.R * g.S * g.Cg * 4 >= 2147483647.0) return best;
  for (int v = 0; v < static_cast<int>(sizeof(kVariants) / sizeof(kVariants[0])); ++v) {
    if ((kVariants[v].wn == 1) != (g.Kg <= 32) || kVariants[v].nseg == 1) continue;
    const int bm = 16 * kVariants[v].nseg * kVariants[v].wm;
    for (const int images : {16, 8, 4, 2, 1}) {
      if (images > g.N && images != 1) continue;
      const int pos = bm / images;
      int last = 0;
      for (int j = 1; j <= 16; ++j) {
        const int tw = (rw + j - 1) / j;
        if (tw > pos || tw == last) continue;
        last = tw;
        int th = std::min(rh, pos / tw);
        th = (rh + (rh + th - 1) / th - 1) / ((rh + th - 1) / th);
        const int hh = th + (g.R - 1) * g.dh, hw = tw + (g.S - 1) * g.dw;
        if ((hh / bg.bho + 2) * (hw / bg.bwo + 2) > kSplitMaxReach) continue;
        consider(g, rh, rw, nreg, v, images, th, tw, tw, true, &best);
        if (tw <= 2) break;
      }
    }
  }
  // more than 9 taps on full tiles of 16 images take up to 1.7 times their estimate
  const double margin = g.R * g.S <= 9 ? 1.05 : 0.75;
  if (best.variant >= 0 &&
      !(one_tap ? one_tap_blocked_pays(g, bg, best)
                : split_blocked_us(g, bg, rh, rw, best) <= margin * igemm_blocked_us(g, bg, rh, rw))) best.variant = -1;
  return best;
}

// The output regions: forward the filter blocks; blocked dx as many of the dx grid.
void split_regions(const Geom& g, const BlockGeom& bg, bool transposed, int* rh, int* rw) {
  const bool blocked_dx = transposed && bg.By * bg.Bx > 1;
  *rh = blocked_dx ? (g.Ho + bg.By - 1) / bg.By : (transposed ? g.Ho : bg.bho);
  *rw = blocked_dx ? (g.Wo + bg.Bx - 1) / bg.Bx : (transposed ? g.Wo : bg.bwo);
}

SplitPlan split_plan(const Geom& g, const BlockGeom& bg, bool transposed) {
  int rh, rw;
  split_regions(g, bg, transposed, &rh, &rw);
  const int nreg = bg.By * bg.Bx;
  SplitPlan p = transposed && nreg > 1 ? make_blocked_plan(g, bg, rh, rw) : make_plan(g, rh, rw, nreg, transposed);
  if (p.variant >= 0 && (p.blocks <= 0 || p.blocks > (1LL << 22))) p.variant = -1;
  return p;
}

}  // namespace

bool plan_f32_split(const Geom& g, const BlockGeom& bg, bool transposed, int32_t* tile) {
  const SplitPlan p = split_plan(g, bg, transposed);
  if (p.variant < 0) return false;
  const SplitVariant& v = kVariants[p.variant];
  const int32_t out[8] = {v.nseg, v.wm, v.wn, p.ti, p.th, p.tw, p.co, p.nchunk};
  std::copy(out, out + 8, tile);
  return true;
}

bool launch_f32_split(const Geom& g, const BlockGeom& bg, const float* x, const float* w, const float* bias,
                      int bias_mode, float* y, bool transposed, hipStream_t stream, hipError_t* err) {
  const int nreg = bg.By * bg.Bx;
  const bool blocked_dx = transposed && nreg > 1;
  const SplitPlan p = split_plan(g, bg, transposed);
  if (p.variant < 0) return false;
  int rh, rw;
  split_regions(g, bg, transposed, &rh, &rw);
  SplitArgs a;
  a.x = x; a.w = w; a.bias = bias; a.y = y; a.g = g;
  a.kdim = g.R * g.S * g.Cg;
  a.tn = p.tn;
  a.tiles = static_cast<int>(static_cast<long long>(p.nty) * p.ntx * p.nti * p.tn);
  a.nty = p.nty; a.ntx = p.ntx;
  a.ti = p.ti; a.th = p.th; a.tw = p.tw; a.hh = p.hh; a.hw = p.hw; a.hp = p.hp; a.hps = p.hps;
  a.twp = p.twp; a.ash = p.ash; a.lgh = p.co == 2 ? 0 : (p.co == 4 ? 1 : (p.co == 8 ? 2 : -1));
  a.co = p.co; a.nchunk = p.nchunk; a.noct = p.noct; a.nst = p.nst;
  a.ow_taps = g.R * g.S;
  a.ow_cg = g.Kg;
  a.rx = bg.Bx; a.nreg = nreg; a.rh = rh; a.rw = rw;
  a.bho = bg.bho; a.bwo = bg.bwo; a.nfast = blocked_dx ? 1 : 0;
  a.By = bg.By; a.Bx = bg.Bx; a.bias_mode = bias_mode;
  a.fd_tn = fastdiv_m(a.tn);
  a.fd_tiles = fastdiv_m(a.tiles);
  a.fd_reg = fastdiv_m(nreg);
  a.fd_rx = fastdiv_m(a.rx);
  a.fd_ntx = fastdiv_m(a.ntx);
  a.fd_nty = fastdiv_m(a.nty);
  a.fd_co = fastdiv_m(a.co);
  a.fd_s = fastdiv_m(g.S);
  a.fd_hw = fastdiv_m(a.hw);
  a.fd_hhw = fastdiv_m(a.hh * a.hw);
  a.fd_twp = fastdiv_m(a.twp);
  a.fd_thw = fastdiv_m(a.th * a.twp);
  a.fd_ti = fastdiv_m(a.ti);
  *err = blocked_dx   ? launch_split<kSplitTransBlocked>(a, p, stream)
         : transposed ? launch_split<kSplitTrans>(a, p, stream)
                      : launch_split<kSplitFwd>(a, p, stream);
  return true;
}

}  // namespace miq
