// fp32 filter gradient on the bf16 matrix cores (conv_f32_split.hip's three-way split, the same
// products and the same fall-back to the fp32 instructions):
//   dw[g Kg + k][by][bx][r][s][ci] = sum over the block's output positions p of
//                                    dy[p][g Kg + k] * x[p stride - pad + (r, s) dil][g Cg + ci]
//
// Work.  A workgroup of 8 waves owns 32 WK output channels x 16 CT WC input channels x up to NB taps
// (CT = 1) of one group and filter block, and a range of position tiles (ti images x th x tw);
// its 32 x 16 NB accumulator tiles per wave stay in registers over the whole range, so x and dy
// are read and split once per workgroup for all of its taps.  The fp32 implicit GEMM gathered x
// once per tap.  WP wave groups share a tile's K-blocks of 32 positions where the layer has too
// few channels for 8 waves; their sums meet in LDS at the end.
//
// Operands.  The reduction runs over positions, but memory (and LDS) hold a position's channels
// together: fragments are read with ds_read_b64_tr_b16, which hands lane n of a 16-lane group the
// four positions 4 q .. 4 q + 3 of channel n.  Position records are [3 pieces][channels] bf16, an
// odd multiple of 32 bytes apart, so the 16 positions of a read fall in distinct bank groups; a
// tap is one byte offset into the halo, whatever the stride or the tile's shape.
//
// The matrix core's sums lean towards minus infinity by a part of their last bit, which over the
// K-blocks of a range adds up where rounding errors cancel: every second K-block computes on negated
// dy and is subtracted.  Relative error of 32 x 56 x 56, 64 -> 64: 4.0e-7 -> 1.3e-7, its mean 0.94 ->
// 0.00 of its rms; of 32 x 112 x 112 7.4e-7 -> 1.7e-7.  The sign costs nothing measurable (60.7 -> 59 us;
// 32 x 112 x 112 stride 2, 32 -> 32 43.9 -> 41): it is a wave's in a tile, so staging multiplies by another
// scalar, and with several wave groups it stays out of the loop.  A negation of the sums every few
// tiles instead took the second to 48, a tile loop for each sign a 2x2 filter from 48 to 283 (spills).
//
// The next tile's values are in flight in registers while a tile computes, and with two LDS buffers
// (where they fit) they are split and stored under its MFMAs.
//
// Measured (us, the split sums' pass apart; before: the fp32 implicit GEMM): 32 x 56 x 56, 64 -> 64
// 3x3 51 (197); 32 x 28 x 28, 128 -> 256 98 with 2 x 4 blocks (374); 32 x 112 x 112 stride 2,
// 32 -> 32 39 (123); four groups of 32 68 with the sums (504). Error against 64 bits 3.0e-7 -> 0.8e-7
// (one 56 x 56 layer). Bound by the MFMAs and their fragment reads (48 of the 63 us of an earlier build, 34 at
// the bare rate), the rest is the loads' and the split's issue. Registers decide: 72 accumulators,
// 48 fragments and 24 to 40 values in flight leave none over, and each pair fewer in flight bought
// 5-9 us through the spills it saved.  What still spills (of 256 registers a wave): with 9 columns and 2
// pairs of x in flight 1 (2 x 4 x 1), 16 (2 x 2 x 2) and 4 (the other two), with 3 pairs 13, 60, 21 and
// 23, with a count of taps other than 9 29, 59, 28 and 30; the smaller instances none.

#include "f32_split.h"

#include <algorithm>
#include <type_traits>

namespace miq {
namespace {

typedef short v4s __attribute__((ext_vector_type(4)));

constexpr int kGradNT = 512;
constexpr int kGradTaps = 9;

struct SGradArgs {
  const float* x;
  const float* dy;
  float* dw;  // partial tiles, splits x K x By x Bx x kdim
  Geom g;
  int By, Bx, bho, bwo;
  int kdim;
  int ti, th, tw;        // images, rows and columns of a tile
  int hh, hw, hp;        // halo rows, columns, positions
  int px, kbs;           // positions of a tile, K-blocks of 32
  int nty, ntx, T;       // tile rows and columns per block, tiles per block
  int tps;               // tiles per split
  int kt, ct, tg;        // channel blocks, input-channel blocks, taps per workgroup
  int inner;             // kt * ct * tap groups
  int recx, recy;        // bytes of a position record
  int bufsz, nbuf;       // bytes of an LDS buffer, how many
  FastDivM fd_inner, fd_g, fd_blk, fd_ct, fd_kt, fd_ntx, fd_nty, fd_hw, fd_hhw, fd_tw, fd_thw, fd_s;
};

__device__ __forceinline__ v4s lds_read_tr(unsigned addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<__attribute__((address_space(3))) v4s*>(addr));
}
__device__ __forceinline__ v8b join(const v4s& a, const v4s& b) {
  return __builtin_bit_cast(v8b, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// staged dy pairs per thread: 128 positions where wave groups share a tile, else 64
constexpr int grad_uy(int wk, int wp) { return (wp > 1 ? 128 : 64) * 4 * wk / kGradNT < 1 ? 1 : (wp > 1 ? 128 : 64) * 4 * wk / kGradNT; }

// whether a tile's K-blocks go round its wave groups (yodd in the kernel)
constexpr bool grad_rotates(int wk, int wc, int wp, int ux) { return wp > 1 && !(wk == 2 && wc == 2) && ux == 3; }

// UX: staged x (position, octet) pairs per thread.  FULL: every workgroup has exactly NB column tiles (taps)
template <int WK, int WC, int WP, int NB, int CT, int UX, bool FULL>
__global__ void __launch_bounds__(kGradNT, 2) f32_split_grad_kernel(SGradArgs a) {
  static_assert(WK * WC * WP == 8 && (CT == 1 || NB == CT), "8 waves");
  constexpr int KR = 32 * WK;
  constexpr int CH = 16 * CT * WC;
  constexpr int UY = grad_uy(WK, WP);
  extern __shared__ v4u lds[];
  const Geom& g = a.g;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int q = lane >> 4, n16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wp = wave / (WK * WC);
  const int wk = (wave - wp * WK * WC) / WC;
  const int wc = wave % WC;

  const int lin = xcd_tile(blockIdx.x, gridDim.x);
  const int o1 = fdiv(lin, a.fd_inner);  // (split * blocks + block) * G + group
  int in = lin - o1 * a.inner;
  const int o2 = fdiv(o1, a.fd_g);
  const int grp = o1 - o2 * g.G;
  const int split = fdiv(o2, a.fd_blk);
  const int nblk = a.By * a.Bx;
  const int blk = o2 - split * nblk;
  const int tgi_kt = fdiv(in, a.fd_ct);
  const int c0 = (in - tgi_kt * a.ct) * CH;  // first input channel of the group
  const int tgi = fdiv(tgi_kt, a.fd_kt);
  const int k0 = (tgi_kt - tgi * a.kt) * KR;
  const int tap0 = tgi * a.tg;
  const int nb = CT > 1 ? NB : min(a.tg, g.R * g.S - tap0);  // column tiles of this workgroup
  const int row0 = (blk / a.Bx) * a.bho, col0 = (blk - (blk / a.Bx) * a.Bx) * a.bwo;
  const int t0 = split * a.tps, t1 = min(a.T, t0 + a.tps);

  // LDS: nbuf x (x records, dy records), the position table, the flag
  const unsigned base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds));
  const int xbytes = a.hp * a.recx;
  int* const tab = reinterpret_cast<int*>(reinterpret_cast<char*>(lds) + a.nbuf * a.bufsz);
  int* const flag = tab + 32 * a.kbs;

  auto decode = [&](int m, int& im, int& lr, int& lc) {  // position m of a tile
    im = fdiv(m, a.fd_thw);
    const int p = m - im * (a.th * a.tw);
    lr = fdiv(p, a.fd_tw);
    lc = p - lr * a.tw;
  };
  for (int m = t; m < 32 * a.kbs; m += kGradNT) {
    int im, lr, lc;
    decode(min(m, a.px - 1), im, lr, lc);
    tab[m] = ((im * a.hh + lr * g.sh) * a.hw + lc * g.sw) * a.recx;
  }
  if (t == 0) *flag = 0;

  // staged pairs of this thread, one octet of positions t / OX + j (512 / OX): offset from the
  // tile's origin and im << 24 | row << 12 | column (kOut: no such position)
  constexpr int OX = CH / 8, OY = KR / 8;
  constexpr int PX = kGradNT / OX, PY = kGradNT / OY;
  constexpr int kOut = 0x7fffffff;
  const int xleft = g.Cg - c0 - 8 * (t % OX), yleft = g.Kg - k0 - 8 * (t % OY);  // channels from the octet on
  int xoff[UX], yoff[UY], xat[UX], yat[UY];
#pragma unroll
  for (int j = 0; j < UX; ++j) {
    const int px = t / OX + PX * j;
    const int im = fdiv(px, a.fd_hhw);
    const int p = px - im * (a.hh * a.hw);
    const int hr = fdiv(p, a.fd_hw), hc = p - hr * a.hw;
    xoff[j] = ((im * g.H + hr) * g.W + hc) * g.C + 8 * (t % OX);
    xat[j] = px < a.hp ? im << 24 | hr << 12 | hc : kOut;
  }
#pragma unroll
  for (int j = 0; j < UY; ++j) {
    const int px = t / OY + PY * j;
    int im, lr, lc;
    decode(px, im, lr, lc);
    yoff[j] = ((im * g.Ho + lr) * g.Wo + lc) * g.K + 8 * (t % OY);
    yat[j] = px < a.px ? im << 24 | lr << 12 | lc : kOut;
  }
  const int xput = (t / OX) * a.recx + 16 * (t % OX), yput = (t / OY) * a.recy + 16 * (t % OY);

  v4f vx[UX][2], vy[UY][2];
  const v4f zero = v4f{0.f, 0.f, 0.f, 0.f};
  auto tile_at = [&](int ti_, int& img0, int& ty0, int& tx0) {
    const int q1 = fdiv(ti_, a.fd_ntx);
    tx0 = (ti_ - q1 * a.ntx) * a.tw;
    const int q2 = fdiv(q1, a.fd_nty);
    ty0 = (q1 - q2 * a.nty) * a.th;
    img0 = q2 * a.ti;
  };
  auto load = [&](int ti_) {
    int img0, ty0, tx0;
    tile_at(ti_, img0, ty0, tx0);
    const int h0 = (row0 + ty0) * g.sh - g.ph, w0 = (col0 + tx0) * g.sw - g.pw;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(
        a.x + static_cast<size_t>(img0) * g.H * g.W * g.C + static_cast<size_t>(grp) * g.Cg + c0, 0x7fffffff);
    const __amdgpu_buffer_rsrc_t ry = make_rsrc(
        a.dy + static_cast<size_t>(img0) * g.Ho * g.Wo * g.K + static_cast<size_t>(grp) * g.Kg + k0, 0x7fffffff);
    const int xorg = (h0 * g.W + w0) * g.C;
    const int yorg = ((row0 + ty0) * g.Wo + col0 + tx0) * g.K;
#pragma unroll
    for (int j = 0; j < UX; ++j) {
      const int hi = h0 + ((xat[j] >> 12) & 0xfff), wi = w0 + (xat[j] & 0xfff);
      const bool ok = img0 + (xat[j] >> 24) < g.N && xat[j] != kOut && static_cast<unsigned>(hi) < static_cast<unsigned>(g.H) &&
                      static_cast<unsigned>(wi) < static_cast<unsigned>(g.W);
      const unsigned off = ok ? 4u * static_cast<unsigned>(xorg + xoff[j]) : kNone;
      vx[j][0] = buffer_load16(rx, xleft >= 4 ? off : kNone, 0);
      vx[j][1] = buffer_load16(rx, xleft >= 8 ? off + 16u : kNone, 0);
    }
#pragma unroll
    for (int j = 0; j < UY; ++j) {
      const bool ok = img0 + (yat[j] >> 24) < g.N && yat[j] != kOut && ty0 + ((yat[j] >> 12) & 0xfff) < a.bho &&
                      tx0 + (yat[j] & 0xfff) < a.bwo;
      const unsigned off = ok ? 4u * static_cast<unsigned>(yorg + yoff[j]) : kNone;
      vy[j][0] = buffer_load16(ry, yleft >= 4 ? off : kNone, 0);
      vy[j][1] = buffer_load16(ry, yleft >= 8 ? off + 16u : kNone, 0);
    }
  };
  // dy is staged negated in every second K-block of 32 positions.  One wave group: counted through the
  // tiles, and mma subtracts those K-blocks' sums.  Several: the odd groups compute the negated
  // K-blocks and reduce() subtracts their sums; a tile's K-blocks go round the groups from another one
  // each tile (ROTATE), or stay with them (the instances that spill on the difference).
  constexpr bool ROTATE = grad_rotates(WK, WC, WP, UX);
  static_assert(PY % 64 == 0 && 64 % OY == 0 && 64 / OY <= 32, "one sign per wave and tile");
  const int yodd = (wave * (64 / OY)) >> 5;
  auto store = [&](int buf, int ti_) {
    const float yscale = (ROTATE || WP == 1 ? yodd ^ ti_ : yodd) & 1 ? -kSplitScale : kSplitScale;
    char* const bx = reinterpret_cast<char*>(lds) + buf * a.bufsz + xput;
    char* const by = reinterpret_cast<char*>(lds) + buf * a.bufsz + xbytes + yput;
#pragma unroll
    for (int j = 0; j < UX; ++j)
      if (xat[j] != kOut) {
        const Split8 s = split8(vx[j][0], vx[j][1], kSplitScale);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<v4u*>(bx + j * PX * a.recx + 2 * CH * p) = s.p[p];
      }
#pragma unroll
    for (int j = 0; j < UY; ++j)
      if (t / OY + PY * j < 32 * a.kbs) {
        const Split8 s = split8(vy[j][0], vy[j][1], yscale);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<v4u*>(by + j * PY * a.recy + 2 * KR * p) = s.p[p];
      }
  };

  // byte offset of each column tile: a tap of the halo, or 16 more input channels
  int toff[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int tap = min(tap0 + (CT > 1 ? 0 : b), g.R * g.S - 1);
    const int r = fdiv(tap, a.fd_s);
    toff[b] = CT > 1 ? 32 * b : (r * g.dh * a.hw + (tap - r * g.S) * g.dw) * a.recx;
  }

  v4f acc[NB][2];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b][0] = acc[b][1] = zero;

  const unsigned xch = base + 32 * CT * wc + 8 * (n16 & 3);
  const unsigned ych = base + xbytes + 64 * wk + 8 * (n16 & 3);
  auto mma = [&](int buf, int ti_) {
    for (int kb = ROTATE ? (wp - ti_) & (WP - 1) : wp; kb < a.kbs; kb += WP) {
      const int m = 32 * kb + 4 * q + (n16 >> 2);
      const unsigned x0 = xch + buf * a.bufsz + tab[m], x1 = xch + buf * a.bufsz + tab[m + 16];
      const unsigned y0 = ych + buf * a.bufsz + m * a.recy, y1 = y0 + 16 * a.recy;
      v8b fy[2][3];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p) fy[i][p] = join(lds_read_tr(y0 + 32 * i + 2 * KR * p), lds_read_tr(y1 + 32 * i + 2 * KR * p));
      v8b fx[2][3];  // a column tile's fragments are read while the one before it computes
      auto read = [&](int b) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          fx[b & 1][p] = join(lds_read_tr(x0 + toff[b] + 2 * CH * p), lds_read_tr(x1 + toff[b] + 2 * CH * p));
      };
      v4f z[2][2];
      auto add = [&](int b, int i) {
        if constexpr (WP > 1) {
          acc[b][i] += z[b & 1][i];
        } else {  // acc +- z, one rounding
          const float sign = (kb ^ ti_) & 1 ? -1.0f : 1.0f;
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[b][i][e] = __builtin_fmaf(z[b & 1][i][e], sign, acc[b][i][e]);
        }
      };
      read(0);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        if (FULL || b < nb) {  // uniform
          if (b + 1 < NB) read(b + 1);
          __builtin_amdgcn_sched_barrier(0);  // the reads above, the MFMAs below
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            constexpr int kx[6] = {2, 0, 1, 1, 0, 0}, ky[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int i = 0; i < 2; ++i)
              z[b & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fy[i][ky[k]], fx[b & 1][kx[k]], k == 0 ? zero : z[b & 1][i], 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {  // the tile before this one is done, this one in flight
            if (b > 0) add(b - 1, i);
            if (b == NB - 1 || (!FULL && b == nb - 1)) add(b, i);
          }
        }
      }
    }
  };
  // the WP wave groups' sums, added in group order into group 0's (`negated`: the odd ones subtracted)
  auto reduce = [&](auto negated) {
    if constexpr (WP > 1) {
      v4f* const r = reinterpret_cast<v4f*>(lds);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        __syncthreads();
        if (wp > 0) {
#pragma unroll
          for (int i = 0; i < 2; ++i) r[(2 * (wave - WK * WC) + i) * 64 + lane] = acc[b][i];
        }
        __syncthreads();
        if (wp == 0) {
#pragma unroll
          for (int o = 1; o < WP; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const v4f v = r[(2 * (wave + (o - 1) * WK * WC) + i) * 64 + lane];
              acc[b][i] = decltype(negated)::value && (o & 1) ? acc[b][i] - v : acc[b][i] + v;
            }
        }
      }
    }
  };

  const int last = t1 - 1;
  load(t0);
  store(0, t0);
  load(min(t0 + 1, last));
  __syncthreads();
  int buf = 0;
  for (int ti_ = t0; ti_ < t1; ++ti_) {
    if (a.nbuf == 2) {
      store(buf ^ 1, ti_ + 1);  // past the last tile: stored, never read
      load(min(ti_ + 2, last));
      mma(buf, ti_);
      buf ^= 1;
    } else {
      mma(0, ti_);
      __syncthreads();
      store(0, ti_ + 1);
      load(min(ti_ + 2, last));
    }
    __syncthreads();
  }
  reduce(std::true_type{});

  bool bad = false;
  if (wp == 0) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (FULL || b < nb) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) bad |= !(__builtin_fabsf(acc[b][i][e]) <= kFltMax);
      }
  }
  if (bad) *flag = 1;
  __syncthreads();
  if (*flag != 0) {
    // the whole range again with fp32 MFMAs, four positions a step, operands straight from memory
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][0] = acc[b][1] = zero;
    for (int ti_ = t0; ti_ < t1; ++ti_) {
      int img0, ty0, tx0;
      tile_at(ti_, img0, ty0, tx0);
      for (int m4 = 4 * wp; m4 < a.px; m4 += 4 * WP) {
        int im, lr, lc;
        decode(min(m4 + q, a.px - 1), im, lr, lc);
        const bool ok = m4 + q < a.px && img0 + im < g.N && ty0 + lr < a.bho && tx0 + lc < a.bwo;
        const int ho = row0 + ty0 + lr, wo = col0 + tx0 + lc;
        const size_t yp = ((static_cast<size_t>(img0 + im) * g.Ho + ho) * g.Wo + wo) * g.K + static_cast<size_t>(grp) * g.Kg;
        float ya[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int k = k0 + 32 * wk + 16 * i + n16;
          ya[i] = ok && k < g.Kg ? a.dy[yp + k] : 0.f;
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if (b < nb) {  // uniform
            const int tap = tap0 + (CT > 1 ? 0 : b);
            const int r = fdiv(tap, a.fd_s), s = tap - r * g.S;
            const int hi = ho * g.sh - g.ph + r * g.dh, wi = wo * g.sw - g.pw + s * g.dw;
            const int c = c0 + 16 * (CT * wc + (CT > 1 ? b : 0)) + n16;
            const bool okx = ok && c < g.Cg && hi >= 0 && hi < g.H && wi >= 0 && wi < g.W;
            const float xa = okx ? a.x[((static_cast<size_t>(img0 + im) * g.H + hi) * g.W + wi) * g.C +
                                       static_cast<size_t>(grp) * g.Cg + c]
                                 : 0.f;
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ya[i], xa, acc[b][i], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();
    reduce(std::false_type{});
  } else {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      acc[b][0] *= kSplitUnscale;
      acc[b][1] *= kSplitUnscale;
    }
  }

  // lane (n16, q) of a tile: output channels 4 q .. 4 q + 3, input channel n16
  if (wp != 0) return;  // after the last barrier
  float* const out = a.dw + static_cast<size_t>(split) * g.K * nblk * a.kdim;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (!FULL && b >= nb) continue;
    const int c = c0 + 16 * (CT * wc + (CT > 1 ? b : 0)) + n16;
    const int col = (tap0 + (CT > 1 ? 0 : b)) * g.Cg + c;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + 32 * wk + 16 * i + 4 * q + e;
        if (c < g.Cg && k < g.Kg) out[(static_cast<size_t>(grp * g.Kg + k) * nblk + blk) * a.kdim + col] = acc[b][i][e];
      }
  }
}

struct GradVariant {
  int wk, wc, wp;
};
constexpr GradVariant kGradVariants[] = {{2, 4, 1}, {2, 2, 2}, {1, 4, 2}, {1, 2, 4}};

struct SGradPlan {
  int variant, nbcols, ct_tiles;  // ct_tiles: 16-channel tiles per wave (2: one tap)
  int ti, th, tw, hh, hw, hp, px, kbs, nty, ntx, nti, kt, ct, ntg, tg, recx, recy, bufsz, nbuf;
  long long T, splits, inner;
  int tps;
  size_t lds;
  double cost;
};

int record_bytes(int channels) {  // an odd multiple of 32 bytes
  const int b = 6 * channels;
  return (b / 32) % 2 ? b : b + 32;
}

// Whether the planned split is the faster kernel.  With at most one workgroup per CU (`gemm` of them)
// the fp32 GEMM is bound by the latency of its (at least 8) chunks and takes 21-25 us whatever the layer,
// or 11 as a single split of at most 64 positions; the split kernel's longer start and tile then lose,
// by more the more taps and idle columns it computes.  Measured (us, fp32 GEMM against split): 3x3,
// 8 x 28 x 28, 64 -> 64 25.8 / 28.0 and 128 -> 128 64 / 36; 5x5, 1 x 14 x 14, 64 -> 64 21.6 / 30.6 and
// 6272 positions 51 / 43; 2x2 29 x 29, 64 -> 64 22.7 / 25.2.  Where half of the GEMM's tile would be idle the
// split wins there too: one tap 21.2 / 12.3 (128 -> 128), few taps and at most 32 output channels 21.7 / 15.9
// (3x3 16 -> 16); and so it does with few taps and at most 128 positions a split, the GEMM's own
// number (2 x 14 x 14, 64 -> 64 22.5 / 21.1, 16 -> 64 21.6 / 19.5).  Over 628 small layers and blocked layers
// and 200 drawn ones every call is within 12% of the faster kernel, where the split alone was up to
// 1.75 times slower.
bool grad_pays(const Geom& g, const BlockGeom& bg, const SGradPlan& p, long long gemm) {
  const int taps = g.R * g.S;
  const long long positions = static_cast<long long>(g.N) * bg.bho * bg.bwo;
  if (taps == 1) return positions > 64 || g.Cg > 64;
  if (taps <= kGradTaps && g.Kg <= 32) return positions > 64;
  return gemm > 256 || (taps <= kGradTaps && positions > 96 && p.tps * p.kbs <= 4);
}

// The tile of a launch, or variant -1 where the fp32 implicit GEMM is the faster kernel: more taps
// than a workgroup takes on a fraction of a 16-channel tile (8 x 224 x 224, 4 -> 64, 7x7 stride 2:
// 372 against 199 us), and few positions at a stride, whose halos hold four values a position
// (19 x 13 x 13, 256 -> 64: 30 against 25 us; 8 x 56 x 56, 64 -> 128: 37 against 45).
SGradPlan grad_plan(const Geom& g, const BlockGeom& bg, long long max_splits, long long gemm) {
  SGradPlan best{};
  best.variant = -1;
  if (g.Cg % 4 || g.Kg % 4 || g.C % 4 || g.K % 4 || g.dh <= 0 || g.dw <= 0) return best;
  if (g.R * g.S > kGradTaps && g.Cg < 16) return best;
  if (g.sh * g.sw > 1 && static_cast<double>(g.N) * bg.bho * bg.bwo < 4096) return best;
  if (static_cast<double>(g.H) * g.W * g.C * 4 >= 2147483647.0 || static_cast<double>(g.Ho) * g.Wo * g.K * 4 >= 2147483647.0)
    return best;
  const int v = g.Kg > 32 ? (g.Cg > 32 ? 0 : 1) : (g.Cg > 32 ? 2 : 3);
  const GradVariant& V = kGradVariants[v];
  const int taps = g.R * g.S;
  const long long positions = static_cast<long long>(g.N) * bg.bho * bg.bwo;
  SGradPlan p{};
  p.variant = v;
  p.ct_tiles = taps == 1 && g.Cg > 16 * V.wc ? 2 : 1;
  const int kr = 32 * V.wk, ch = 16 * p.ct_tiles * V.wc;
  p.ntg = (taps + kGradTaps - 1) / kGradTaps;
  p.tg = (taps + p.ntg - 1) / p.ntg;
  p.kt = (g.Kg + kr - 1) / kr;
  p.ct = (g.Cg + ch - 1) / ch;
  p.inner = static_cast<long long>(p.kt) * p.ct * p.ntg;
  p.recx = record_bytes(ch);
  p.recy = record_bytes(kr);
  for (const int maxpx : {64, 128, 32}) {
    if (maxpx == 128 && V.wp == 1) continue;
    int lasttw = 0;
    for (int j = 1; j <= 16; ++j) {
      const int tw = (bg.bwo + j - 1) / j;
      if (tw > maxpx || tw == lasttw) continue;
      lasttw = tw;
      int th = std::min(bg.bho, maxpx / tw);
      th = (bg.bho + (bg.bho + th - 1) / th - 1) / ((bg.bho + th - 1) / th);
      p.ti = th == bg.bho && tw == bg.bwo ? std::max(1, std::min(g.N, maxpx / (th * tw))) : 1;
      p.th = th; p.tw = tw;
      p.hh = (th - 1) * g.sh + (g.R - 1) * g.dh + 1;
      p.hw = (tw - 1) * g.sw + (g.S - 1) * g.dw + 1;
      p.px = p.ti * th * tw;
      p.kbs = (p.px + 31) / 32;
      const long long hp = static_cast<long long>(p.ti) * p.hh * p.hw;
      // without rotation an odd number of K-blocks per tile leans by one of them, which stays below the
      // fp32 GEMM's error up to about these sizes
      const int ux = p.ct_tiles == 2 || taps != kGradTaps || hp * 2 * V.wc > 2 * kGradNT ? 3 : 2;
      if (V.wp > 1 && !grad_rotates(V.wk, V.wc, V.wp, ux) && (p.kbs & 1) && positions > (p.kbs == 1 ? 1 << 12 : 1 << 20)) continue;
      if (p.hh > 4095 || p.hw > 4095 || p.ti > 126 || hp * (ch / 8) > 3 * kGradNT ||
          32LL * p.kbs * (kr / 8) > grad_uy(V.wk, V.wp) * kGradNT) continue;
      if (static_cast<double>(p.ti) * g.H * g.W * g.C * 4 >= 2147483647.0 ||
          static_cast<double>(p.ti) * g.Ho * g.Wo * g.K * 4 >= 2147483647.0) continue;
      p.hp = static_cast<int>(hp);
      p.bufsz = p.hp * p.recx + 32 * p.kbs * p.recy;
      const size_t tail = static_cast<size_t>(32 * p.kbs + 1) * 4;
      p.nbuf = 2 * static_cast<size_t>(p.bufsz) + tail <= kSplitLds ? 2 : 1;
      p.lds = std::max(static_cast<size_t>(p.nbuf) * p.bufsz + tail, static_cast<size_t>(16 * 1024));
      if (static_cast<size_t>(p.nbuf) * p.bufsz + tail > kSplitLds || p.bufsz * p.nbuf < 16 * 1024) continue;
      p.nty = (bg.bho + th - 1) / th;
      p.ntx = (bg.bwo + tw - 1) / tw;
      p.nti = (g.N + p.ti - 1) / p.ti;
      p.T = static_cast<long long>(p.nti) * p.nty * p.ntx;
      // cycles per tile: the K-blocks' MFMAs, the staged pairs
      const int cols = p.ct_tiles == 2 ? 2 : p.tg;
      const int rounds = (p.kbs + V.wp - 1) / V.wp;
      const double mfma = rounds * cols * 12 * 16.0 * 2;
      const double stage = (static_cast<double>(hp) * ch / 8 + 32.0 * p.kbs * kr / 8) / 512 * 2 * 75 * 4;
      const double tile = (p.nbuf == 2 ? std::max(mfma * 1.3, stage) + 0.3 * std::min(mfma, stage) : mfma * 1.3 + stage) + 500;
      p.cost = tile * p.T;
      if (best.variant < 0 || p.cost < best.cost) best = p;
    }
  }
  if (best.variant < 0) return best;
  // splits: one workgroup per CU, at most as many as the caller's workspace holds
  const long long units = best.inner * g.G * bg.By * bg.Bx;
  long long splits = std::max(1LL, std::min({256 / std::max(1LL, std::min(units, 256LL)), best.T, max_splits}));
  best.tps = static_cast<int>((best.T + splits - 1) / splits);
  best.splits = (best.T + best.tps - 1) / best.tps;
  if (best.splits * units > (1LL << 22) || best.T > (1LL << 30) || !grad_pays(g, bg, best, gemm)) best.variant = -1;
  return best;
}

template <int WK, int WC, int WP, int NB, int CT, int UX, bool FULL>
hipError_t launch_grad_variant(const SGradArgs& a, const SGradPlan& p, unsigned blocks, hipStream_t stream) {
  const auto kern = &f32_split_grad_kernel<WK, WC, WP, NB, CT, UX, FULL>;
  if (p.lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kSplitLds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kGradNT), p.lds, stream, a);
  return hipGetLastError();
}

template <int WK, int WC, int WP>
hipError_t launch_grad_shape(const SGradArgs& a, const SGradPlan& p, int taps, unsigned blocks, hipStream_t stream) {
  if (p.ct_tiles == 2) return launch_grad_variant<WK, WC, WP, 2, 2, 3, true>(a, p, blocks, stream);
  if (taps != kGradTaps) return launch_grad_variant<WK, WC, WP, kGradTaps, 1, 3, false>(a, p, blocks, stream);
  if (p.hp * 2 * WC > 2 * kGradNT) return launch_grad_variant<WK, WC, WP, kGradTaps, 1, 3, true>(a, p, blocks, stream);
  return launch_grad_variant<WK, WC, WP, kGradTaps, 1, 2, true>(a, p, blocks, stream);
}

}  // namespace

bool plan_f32_split_grad(const Geom& g, const BlockGeom& bg, long long max_splits, long long gemm, int32_t* tile) {
  const SGradPlan p = grad_plan(g, bg, max_splits, gemm);
  if (p.variant < 0) return false;
  const GradVariant& v = kGradVariants[p.variant];
  const int32_t out[8] = {v.wk, v.wc, v.wp, p.ti, p.th, p.tw, p.nbuf, static_cast<int32_t>(p.splits)};
  std::copy(out, out + 8, tile);
  return true;
}

bool launch_f32_split_grad(const Geom& g, const BlockGeom& bg, const float* x, const float* dy, float* dw, float* ws,
                           long long max_splits, long long gemm, hipStream_t stream, long long* splits,
                           hipError_t* err) {
  if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy)) & 15u) != 0) return false;
  const SGradPlan p = grad_plan(g, bg, max_splits, gemm);
  if (p.variant < 0) return false;
  SGradArgs a;
  a.x = x; a.dy = dy; a.g = g;
  a.dw = p.splits == 1 ? dw : ws;
  a.By = bg.By; a.Bx = bg.Bx; a.bho = bg.bho; a.bwo = bg.bwo;
  a.kdim = g.R * g.S * g.Cg;
  a.ti = p.ti; a.th = p.th; a.tw = p.tw; a.hh = p.hh; a.hw = p.hw; a.hp = p.hp; a.px = p.px; a.kbs = p.kbs;
  a.nty = p.nty; a.ntx = p.ntx; a.T = static_cast<int>(p.T); a.tps = p.tps;
  a.kt = p.kt; a.ct = p.ct; a.tg = p.tg; a.inner = static_cast<int>(p.inner);
  a.recx = p.recx; a.recy = p.recy; a.bufsz = p.bufsz; a.nbuf = p.nbuf;
  a.fd_inner = fastdiv_m(a.inner);
  a.fd_g = fastdiv_m(g.G);
  a.fd_blk = fastdiv_m(bg.By * bg.Bx);
  a.fd_ct = fastdiv_m(a.ct);
  a.fd_kt = fastdiv_m(a.kt);
  a.fd_ntx = fastdiv_m(a.ntx);
  a.fd_nty = fastdiv_m(a.nty);
  a.fd_hw = fastdiv_m(a.hw);
  a.fd_hhw = fastdiv_m(a.hh * a.hw);
  a.fd_tw = fastdiv_m(a.tw);
  a.fd_thw = fastdiv_m(a.th * a.tw);
  a.fd_s = fastdiv_m(g.S);
  *splits = p.splits;
  const unsigned blocks = static_cast<unsigned>(p.splits * p.inner * g.G * bg.By * bg.Bx);
  const int taps = g.R * g.S;
  switch (p.variant) {
    case 0: *err = launch_grad_shape<2, 4, 1>(a, p, taps, blocks, stream); break;
    case 1: *err = launch_grad_shape<2, 2, 2>(a, p, taps, blocks, stream); break;
    case 2: *err = launch_grad_shape<1, 4, 2>(a, p, taps, blocks, stream); break;
    default: *err = launch_grad_shape<1, 2, 4>(a, p, taps, blocks, stream); break;
  }
  return true;
}

}  // namespace miq
