// The tail launch: the final RMSNorm of the last layer's rows and this GPU's rows of
// the LM head (reference: glm53/gfx950/kernel.py:2220-2350, a `tail` build; host side
// Glm53HeadOp.launch, runner.py:473-545):
//   normed[r]    = bf16(x[r] * rsqrt(mean(x[r]^2) + eps) * g_norm)
//   logits[r][v] = f32(bf16(normed[r] . w_head[v]))
// w_head is SGLang's LM head as loaded, bf16 [vocab_rows][hidden] row-major, read in
// place; the logits are rounded to bf16 as the reference gathers them.
//
// One 512-thread workgroup a CU takes a contiguous range of vocab rows (within one of
// every other's: the launch is HBM-bound, so work is rows) and walks it in 16-row
// tiles, the last one partial: its dead lanes load a live row's addresses, which the
// same instruction already fetches, and store nothing.
// Wave w owns the k slice [w * hidden / 8, (w + 1) * hidden / 8) of every tile: the
// normed rows' B operands for that slice (the rows as the MFMA's columns, up to 16 a
// column group) are built once and stay in registers (part of a second group's in LDS),
// and the tile's W rows stream through a window of WIN 16-byte loads a lane, each refilled
// from the same tile or the next one as its MFMA consumes it.  The norm costs no extra pass over the rows: the x fragments a wave
// loads for its operands give its slice's sums of squares, which the eight waves
// combine through LDS; they and the norm weight are loaded ahead of the first window,
// so the norm runs while the first W bytes are in flight.  A lane (c16, g) loads 16 B
// of row c16 at k = 32 s + 8 g of its slice: a wave instruction reads 64 contiguous
// bytes of each of 16 rows, and two consecutive k-steps fill whole 128-byte lines.  The
// eight waves' 16 x 16 partial tiles are summed in wave order through LDS.
// Above 16 rows the rows are two column groups of one pass: every W fragment feeds two
// MFMAs.  Two passes of 16 streamed the LM head twice, 97.9 us at 32 rows of hidden 6144
// and 19360 vocab rows; the one pass takes 64.8 us (8 rows: 49.8; the bytes at the rate
// of a large copy: 48).
#include <type_traits>

#include "mk2_device.h"
#include "mk2_host.h"

namespace mk2 {

constexpr int TAIL_NT = 512;
constexpr int TAIL_WAVES = TAIL_NT / 64;
constexpr int TAIL_CHUNK = 8;  // tiles whose partials wait in LDS for one barrier

struct TailDev {
  int rows;        // 1..16 NCG
  int hidden;
  int vocab_rows;
  float eps;
  const bf16_t* x;       // [rows][hidden]
  const bf16_t* g;       // [hidden]
  const bf16_t* w;       // [vocab_rows][hidden]
  float* logits;         // [rows][vocab_rows]
  bf16_t* normed;        // [rows][hidden], or null
};

// Where a wave of KS k-steps and NCG column groups of 16 rows keeps its B operands and how
// much of W it holds in flight, within 256 registers a lane and 160 KiB of LDS.  One group:
// everything in registers, a window of one tile (half of one above 24 steps).  Two groups
// are 2 KS steps of four registers; above 16 steps the second group's first LS steps live
// in LDS (8 KiB a step over the eight waves, one conflict-free 16-byte read a lane) and
// the window shrinks to half a tile or less, which still keeps 56-96 KiB a CU in flight.
// LS is the least that spills nothing, which leaves the most LDS to the partials: at KS 24
// and 32 rows a barrier every 5, 2 or 1 tiles took 64.8, 66.7 and 69.9 us.
template <int KS, int NCG>
struct TailPlan {
  static constexpr int LS = NCG == 1 || KS <= 16 ? 0 : KS == 20 ? 8 : KS == 24 ? 8 : KS == 28 ? 12 : 15;
  static constexpr int WIN = NCG == 1 ? (KS <= 24 ? KS : KS / 2) : KS <= 16 ? KS : KS >= 28 ? KS / 4 : KS / 2;
  // tiles a barrier phase, their partials in LDS: 8 KiB a tile and group
  static constexpr int CH = NCG == 1 || LS == 0 ? TAIL_CHUNK : LS == 8 ? 5 : LS == 12 ? 3 : 2;
};

// g_norm is read until the operands are built, the waves' partial tiles are written after:
// with two groups they share their LDS, at the price of a barrier between
template <int KS, int NCG>
struct TailLdsApart {
  uint4 gam[8192 / 8];
  float red[TailPlan<KS, NCG>::CH][TAIL_WAVES][NCG * 256];
};
template <int KS, int NCG>
union TailLdsShared {
  uint4 gam[8192 / 8];
  float red[TailPlan<KS, NCG>::CH][TAIL_WAVES][NCG * 256];
};

template <int KS, int NCG>
__global__ __launch_bounds__(TAIL_NT) void k_tail(TailDev p) {
  using P = TailPlan<KS, NCG>;
  constexpr int WIN = P::WIN, LS = P::LS, CH = P::CH;
  static_assert(KS % WIN == 0, "a window divides the k-steps");
  __shared__ float part[TAIL_WAVES][16 * NCG];  // the waves' sums of squares by row
  __shared__ std::conditional_t<NCG == 1, TailLdsApart<KS, NCG>, TailLdsShared<KS, NCG>> S;
  __shared__ uint4 blds[TAIL_WAVES][LS > 0 ? LS : 1][64];  // the second group's first LS steps
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const int H = p.hidden, G = gridDim.x, b = blockIdx.x, M = p.rows;
  // this workgroup's rows [r0, r1): at least one (G <= vocab_rows)
  const int r0 = (int)((long long)b * p.vocab_rows / G), r1 = (int)((long long)(b + 1) * p.vocab_rows / G);
  const int kw = wave * KS * 32 + 8 * g;  // this lane's first k of its wave's slice
  auto sumsq = [](uint4 q, float ss) {
    // packed dot products of the bf16 pairs with themselves: nothing is unpacked here for
    // the conversion below to keep alive across the barrier
    const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bf16x2 v = __builtin_bit_cast(bf16x2, u[j]);
      ss = __builtin_amdgcn_fdot2_f32_bf16(v, v, ss, false);
    }
    return ss;
  };
  // a row's rstd from the eight waves' slices, in wave order (every lane of the row gets
  // the same bits)
  auto rstd = [&](int row) {
    float tot = part[0][row];
#pragma unroll
    for (int w = 1; w < TAIL_WAVES; ++w) tot += part[w][row];
    return 1.0f / sqrtf(tot / (float)H + p.eps);
  };
  // bf16(x * rstd * g) of a lane's 8 k at step s (zero past the rows)
  auto operand = [&](uint4 x, int s, float rs, bool on, int row) {
    const uint4 gv = S.gam[(kw + 32 * s) >> 3];
    const uint32_t xu[4] = {x.x, x.y, x.z, x.w}, gu[4] = {gv.x, gv.y, gv.z, gv.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = __uint_as_float(xu[j] << 16) * rs * __uint_as_float(gu[j] << 16);
      const float hi = __uint_as_float(xu[j] & 0xFFFF0000u) * rs * __uint_as_float(gu[j] & 0xFFFF0000u);
      o[j] = on ? pack_bf16x2(lo, hi) : 0u;
    }
    const uint4 ov = make_uint4(o[0], o[1], o[2], o[3]);
    if (b == 0 && on && p.normed) *(uint4*)(p.normed + (size_t)row * H + kw + 32 * s) = ov;
    return ov;
  };
  uint4 gq[2];
  auto load_gamma = [&] {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = threadIdx.x + u * TAIL_NT;
      gq[u] = i < H / 8 ? ((const uint4*)p.g)[i] : make_uint4(0, 0, 0, 0);
    }
  };
  auto stage_gamma = [&] {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = threadIdx.x + u * TAIL_NT;
      if (i < H / 8) S.gam[i] = gq[u];
    }
  };
  // the W row of this lane in the tile from row t (the range's last row past its end)
  auto w_row = [&](int t) { return p.w + (size_t)min(t + c16, r1 - 1) * H + kw; };
  const bf16_t* wrow = w_row(r0);
  uint4 wv[WIN];
  auto load_window = [&] {
#pragma unroll
    for (int s = 0; s < WIN; ++s) wv[s] = ld_stream16(wrow + 32 * s);
  };
  // 1. with two groups the second one's operands first, start to end (rows 16 + c16), while
  //    the registers are free: loaded behind the W window they would wait for all of it
  //    (a wave's loads return in order), and held beside the first group's rows they spill
  bf16x8 bq1[NCG == 2 ? KS - LS : 1];
  if constexpr (NCG == 2) {
    const bool live1 = 16 + c16 < M;
    const bf16_t* xr1 = p.x + (size_t)(live1 ? 16 + c16 : 0) * H + kw;
    uint4 x1[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) x1[s] = *(const uint4*)(xr1 + 32 * s);
    load_gamma();
    float ss1 = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) ss1 = sumsq(x1[s], ss1);
    ss1 += __shfl_xor(ss1, 16);
    ss1 += __shfl_xor(ss1, 32);
    if (g == 0) part[wave][16 * (NCG - 1) + c16] = ss1;
    stage_gamma();
    __syncthreads();
    const float rs1 = live1 ? rstd(16 + c16) : 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint4 ov = operand(x1[s], s, rs1, live1, 16 + c16);
      if (s < LS) blds[wave][s][lane] = ov;  // only this lane reads it: no barrier
      else bq1[s < LS ? 0 : s - LS] = __builtin_bit_cast(bf16x8, ov);
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads below stay below: their registers were the rows'
  }
  // 2. this lane's x fragments of row c16, then the first tile's W window: the rows (and
  //    the norm weight) are in hand before the first W bytes arrive
  const bool live = c16 < M;
  const bf16_t* xr = p.x + (size_t)(live ? c16 : 0) * H + kw;
  uint4 xq[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) xq[s] = *(const uint4*)(xr + 32 * s);
  if constexpr (NCG == 1) load_gamma();
  load_window();
  // 3. its sums of squares (the lane's k-steps, the four lanes of its row, the eight
  //    waves) and operands, in place
  float ss = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) ss = sumsq(xq[s], ss);
  ss += __shfl_xor(ss, 16);
  ss += __shfl_xor(ss, 32);
  if (g == 0) part[wave][c16] = ss;
  if constexpr (NCG == 1) stage_gamma();
  __syncthreads();
  const float rs = live ? rstd(c16) : 0.f;
  bf16x8 bq[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) bq[s] = __builtin_bit_cast(bf16x8, operand(xq[s], s, rs, live, c16));
  if constexpr (NCG == 2) __syncthreads();  // the norm weight's LDS is the partials' from here on
  // 4. the tiles, in phases of up to CH: each wave runs its chain for every tile of the
  //    phase and leaves its partial tiles in LDS with no barrier between tiles; the
  //    phase's partials are then summed in wave order and stored
  for (int c0 = r0; c0 < r1; c0 += 16 * CH) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int t = c0 + 16 * i;
      if (t >= r1) break;
      const bool more = t + 16 < r1;
      const bf16_t* nrow = w_row(t + 16);  // this lane's row of the next tile
      f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, wv[s % WIN]);
        acc = mfma_bf16(a, bq[s], acc);
        if constexpr (NCG == 2)
          acc1 = mfma_bf16(a, s < LS ? __builtin_bit_cast(bf16x8, blds[wave][s < LS ? s : 0][lane]) : bq1[s < LS ? 0 : s - LS], acc1);
        const int u = s + WIN;
        if (u < KS)
          wv[s % WIN] = ld_stream16(wrow + 32 * u);
        else if (more)
          wv[s % WIN] = ld_stream16(nrow + 32 * (u - KS));
      }
      // lane (c16, g) holds D[v = 4 g + i][m = c16]
      float* rw = S.red[i][wave];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        rw[(4 * g + j) * 16 + c16] = acc[j];
        if constexpr (NCG == 2) rw[(NCG - 1) * 256 + (4 * g + j) * 16 + c16] = acc1[j];
      }
      wrow = nrow;
    }
    __syncthreads();
    const int nt = min(CH, (r1 - c0 + 15) / 16);
    for (int e = threadIdx.x; e < nt * NCG * 256; e += TAIL_NT) {
      const int i = e / (NCG * 256), m = (e >> 4) % (16 * NCG), v = e & 15;
      const int row = c0 + 16 * i + v, at = (m >> 4) * 256 + v * 16 + (m & 15);
      float s = S.red[i][0][at];
#pragma unroll
      for (int w = 1; w < TAIL_WAVES; ++w) s += S.red[i][w][at];
      if (m < M && row < r1) p.logits[(size_t)m * p.vocab_rows + row] = bf16_to_f32(f32_to_bf16(s));
    }
    __syncthreads();
  }
}

template <int KS>
static void tail_enqueue(const TailDev& d, int grid, hipStream_t st) {
  if (d.rows > 16) k_tail<KS, 2><<<grid, TAIL_NT, 0, st>>>(d);
  else k_tail<KS, 1><<<grid, TAIL_NT, 0, st>>>(d);
}

static int tail_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus[dev] == 0 && hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus[dev] = 0;
  return cus[dev];
}

}  // namespace mk2

using namespace mk2;

extern "C" int mk2_tail_launch(const mk2_tail_args* a, mk2_stream_t stream) {
  clear_error();
  MK2_REQUIRE(a != nullptr, "tail: args is NULL");
  MK2_REQUIRE(a->rows >= 1 && a->rows <= 32, "tail: rows must be in [1, 32], got %d", a->rows);
  MK2_REQUIRE(a->hidden >= 2048 && a->hidden <= 8192 && a->hidden % 1024 == 0,
              "tail: hidden must be a multiple of 1024 in [2048, 8192], got %d", a->hidden);
  MK2_REQUIRE(a->vocab_rows >= 1, "tail: vocab_rows must be positive, got %d", a->vocab_rows);
  MK2_REQUIRE(a->eps > 0.f, "tail: eps must be positive");
  MK2_REQUIRE(a->x && a->g_norm && a->w_head && a->logits, "tail: x, g_norm, w_head and logits must be set");
  MK2_REQUIRE(a->normed != a->x, "tail: normed must not alias x");
  const int cus = tail_cus();
  if (cus <= 0) return set_error(MK2_ELAUNCH, "tail: cannot query the CU count");
  const int grid = a->vocab_rows < cus ? a->vocab_rows : cus;
  hipStream_t st = (hipStream_t)stream;
  const TailDev d{a->rows, a->hidden, a->vocab_rows, a->eps, (const bf16_t*)a->x, (const bf16_t*)a->g_norm,
                  (const bf16_t*)a->w_head, a->logits, (bf16_t*)a->normed};
  switch (a->hidden / 256) {
    case 8: tail_enqueue<8>(d, grid, st); break;
    case 12: tail_enqueue<12>(d, grid, st); break;
    case 16: tail_enqueue<16>(d, grid, st); break;
    case 20: tail_enqueue<20>(d, grid, st); break;
    case 24: tail_enqueue<24>(d, grid, st); break;
    case 28: tail_enqueue<28>(d, grid, st); break;
    default: tail_enqueue<32>(d, grid, st); break;
  }
  return check_launch("tail");
}
