// Sparse-MLA stages of the K2 layer: split attention over gathered FP8 latent-KV
// rows, the merge of the splits, W_UV, and W_o with the residual.
//
// split task (row r, split s): 64 selected positions -> page table -> 576-byte E4M3
// rows, gathered with 16-byte loads into LDS row-major: the QK operand as it lies, the PV
// operand (8 keys of a dim a lane) by transposing LDS reads.  S = q . k on bf16 MFMA (E4M3
// widens exactly), x (scale_k * sm_scale); a split-local softmax per head; P' = p * scale_k
// rounded to bf16; O = P' V on bf16 MFMA.  The split writes O (unnormalized), its max m and sum l.
// merge task (up to 4 rows, head h, half): exact combination of each row's splits ->
// o_lat (bf16), then o[r][h] = W_UV[h] o_lat on bf16 MFMA, the rows as its columns.
// oproj task (16 hidden rows): a = bf16(h + W_o o) on bf16 MFMA.
#pragma once
#include "mk2_device.h"
#include "mla_table.h"

namespace mk2 {

constexpr int MLA_D = 576;        // latent 512 + rope 64
constexpr int MLA_LAT = 512;
constexpr int MLA_HEADS = 16;
constexpr int MLA_SPLIT = 64;     // keys a split task
// LDS row stride of the gathered rows (bytes): 16-byte pieces, and 148 words, so that the
// QK reads (8 bytes of each of 16 rows) and the transposing PV reads (16 bytes of each of 8
// rows) fall in distinct banks
constexpr int MLA_KROW = 592;
constexpr int MLA_NT = 256;

struct MlaDev {
  int rows, v_dim, hidden, topk, stride, nsplit;
  float sm_scale;
  const bf16_t* q;       // [rows][16][576]
  const uint8_t* kv;     // [pages][64][576]
  const float* kv_scale; // [pages][64]; null: unscaled E4M3 (scale 1)
  const int* pt;
  const int* req;
  const int* sel;        // [rows][topk]
  const uint64_t* tsel;  // the same list as tagged words (the persistent layer polls
                         // its split's entries), or null: sel
  const bf16_t* w_uv;    // [16][v_dim][512]
  const uint8_t* w_o;    // tiles of [hidden][16*v_dim]
  const bf16_t* h;       // [rows][hidden] or null
  bf16_t* out;           // [rows][hidden]
  // workspace
  bf16_t* part_o;        // [rows][nsplit][16][512] the splits' P.V, rounded to bf16
  float* part_ml;        // [rows][nsplit][16][2]
  float* o_lat_f32;      // optional [rows][16][512]
  bf16_t* o;             // [rows][16 * v_dim]
  float* ssp;            // optional [rows][hidden/16]: sums of squares of out over 16 columns
};

struct alignas(16) MlaSplitLds {
  uint8_t k[MLA_SPLIT * MLA_KROW];       // gathered rows, row-major
  bf16_t p[MLA_HEADS * (MLA_SPLIT + 8)]; // P' [head][key]
  int row[2][MLA_SPLIT];                 // by task parity: cache row of each key (-1: unused)
  float sc[MLA_SPLIT];                   // per-key scale * sm_scale
  float kscale[MLA_SPLIT];
  alignas(16) float red[4][MLA_HEADS];   // by wave: its keys' maxima by head
  alignas(16) float suml[4][MLA_HEADS];  // and its sums
  int bad;                               // a poll gave up
};
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
// PV's operand from the row-major E4M3 rows: 8 keys (rows of `k`) x 16 dims a 16-lane group,
// lane i of which gets dim d0 + i of keys key0 .. key0 + 7 (lanes 2j, 2j + 1 address key j's
// two 8-byte halves; the read transposes)
MK2_DEV uint2 lds_read_keys8(const uint8_t* k, int key0, int d0, int i) {
  const i32x2 r = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
      (lds_i32x2*)(k + (key0 + (i >> 1)) * MLA_KROW + d0 + 8 * (i & 1)));
  return make_uint2((uint32_t)r.x, (uint32_t)r.y);
}

// ---------------------------------------------------------------- stage: split
// The split tasks t0 .. t1 - 1 (task t: row t / nsplit, split t % nsplit) of one worker: NT =
// 256 or 512 threads, waves 0-3 of which run QK and the softmax (16 keys each), every wave
// gathering and taking a share of the PV dim tiles.  A worker is the workgroup, or (HALF)
// its half threadIdx.x / NT with LDS of its own; the halves keep step, `iters` being the
// larger half's number of tasks.
//
// Without HALF a worker runs one task.  With several tasks a workgroup, QK and the softmax,
// chains of latencies on four waves, leave the other four idle: the halves run two tasks
// at once, neighbours of one row, so that the q operands stay.  A half's tasks also
// overlap: while one computes, the next one's rows are in flight into registers, and on
// its last wave the cache rows of the one after it and the positions of the third.  A
// task's partials are counted out (`done(t)`, by one thread) once the next one's rows have
// arrived, where waiting for the stores costs nothing; the last task's right away.
template <int NT, bool HALF, typename Done, typename Mark = NoMark>
MK2_DEV bool mla_split_tasks(const MlaDev& p, int t0, int t1, int iters, MlaSplitLds* LS, const TagPoll& tp, Done done,
                             Mark mark = Mark()) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x % NT, lane = tid & 63, wave = tid >> 6, g = lane >> 4, c16 = lane & 15;
  const bool qk_wave = wave < 4;
  if (iters <= 0) return true;
  MlaSplitLds& L = LS[HALF ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0];
  auto failed = [&] { return LS[0].bad != 0 || (HALF && LS[1].bad != 0); };
  // q operands for this wave's QK: head c16, dims 8g + 32ks .. +7
  bf16x8 qa[18];
  auto load_q = [&](int r) {
    const bf16_t* qr = p.q + ((size_t)r * MLA_HEADS + c16) * MLA_D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < 18; ++ks) qa[ks] = __builtin_bit_cast(bf16x8, *(const uint4*)(qr + 32 * ks));
  };
  // one wave: a task's 64 positions, an entry a lane, as words of the list (a tagged list's
  // are checked, and polled where they are not out yet: the task starts as soon as its own
  // 64 entries are), then the cache row of a position
  auto list_at = [&](int t) {
    return (size_t)(t / p.nsplit) * p.topk + (t % p.nsplit) * MLA_SPLIT + lane;
  };
  auto list_word = [&](int t) -> uint64_t {
    return p.tsel ? ld_pair(p.tsel + list_at(t)) : (uint64_t)(uint32_t)ldp_i32(p.sel + list_at(t));
  };
  auto list_poll = [&](int t, uint64_t w, bool* bad) {
    if (p.tsel) {
      const uint64_t* src = p.tsel + list_at(t);
      WaitClock wc;
      for (int polls = 1;; polls += 2) {  // two polls in flight
        const uint64_t w1 = ld_pair(src);
        if (poll_done(pair_ready(w, tp), polls, wc, tp, bad)) break;
        w = ld_pair(src);
        if (poll_done(pair_ready(w1, tp), polls + 1, wc, tp, bad)) {
          w = w1;
          break;
        }
      }
    }
    return (int)pair_value(w);
  };
  // (the page's load has no use here to wait for; its row's line is taken ahead of the poll:
  // behind it the 8-row layer was 1 us slower)
  auto line_of = [&](int t) { return mla_line(p.req, t / p.nsplit, p.stride); };
  auto page_of = [&](ptrdiff_t line, int pos) { return mla_page(p.pt, line, p.stride, pos); };
  auto cache_row = [&](int pos, int page) { return mla_cache_row(pos, page, p.stride); };
  // gather: 16-byte piece i % 36 of key i / 36; every load of a thread is issued at once,
  // the rows' scales ahead of them
  constexpr int PIECES = MLA_SPLIT * (MLA_D / 16), PPT = (PIECES + NT - 1) / NT;
  uint4 v[PPT];
  float ksc = 0.f;
  auto gather = [&](const int* row) {
    if (tid < MLA_SPLIT) ksc = row[tid] < 0 ? 0.f : (p.kv_scale ? p.kv_scale[row[tid]] : 1.f);
#pragma unroll
    for (int it = 0; it < PPT; ++it) {
      const int i = tid + it * NT;
      const int rw = i < PIECES ? row[i / 36] : -1;
      v[it] = rw >= 0 ? ld_stream16(p.kv + (size_t)rw * MLA_D + i % 36 * 16) : make_uint4(0, 0, 0, 0);
    }
  };
  // the first task's rows, and the second's positions beside them.  Wave 0 loads its q
  // behind the gather: ahead of its list poll and page-table read they would hold both up
  // (a wave's loads complete in order)
  const bool any = t0 < t1;
  if (any && qk_wave && wave != 0) load_q(t0 / p.nsplit);
  const bool ahead = HALF && wave == NW - 1 && t0 + 1 < t1;  // the wave that resolves later tasks
  uint64_t aw = 0;           // the list words it looks at next
  int apos = -1, apage = 0;  // positions and pages of the task before those
  bool abad = false;
  if (wave == 0) {
    bool bad = false;
    if (any) {
      const ptrdiff_t line = line_of(t0);
      const int pos = list_poll(t0, list_word(t0), &bad);
      L.row[0][lane] = cache_row(pos, page_of(line, pos));
    }
    if (lane == 0) L.bad = bad;  // wave-uniform
  }
  if (ahead) aw = list_word(t0 + 1);
  if (threadIdx.x == 0) mark(0);
  __syncthreads();
  if (failed()) return false;
  if (ahead) {
    const ptrdiff_t line = line_of(t0 + 1);
    apos = list_poll(t0 + 1, aw, &abad);
    apage = page_of(line, apos);
    if (t0 + 2 < t1) aw = list_word(t0 + 2);
  }
  if (any) {
    gather(L.row[0]);
    if (wave == 0) load_q(t0 / p.nsplit);
  }
  for (int i0 = 0, t = t0, par = 0; i0 < (HALF ? iters : 1); ++i0, ++t, par ^= 1) {
    const int r = t / p.nsplit, s = t % p.nsplit;
    const int* row = L.row[par];
    const bool have = t < t1, more = HALF && t + 1 < t1;
    if (have) {
      if (tid < MLA_SPLIT) {
        L.kscale[tid] = ksc;
        L.sc[tid] = ksc * p.sm_scale;
      }
#pragma unroll
      for (int it = 0; it < PPT; ++it) {
        const int i = tid + it * NT;
        if (i < PIECES) *(uint4*)(L.k + i / 36 * MLA_KROW + i % 36 * 16) = v[it];
      }
    }
    if (ahead && more) {  // the next task's rows
      L.row[par ^ 1][lane] = cache_row(apos, apage);
      if (lane == 0 && abad) L.bad = 1;
    }
    if (HALF && i0) drain_memory();  // the previous task's partials are out
    __syncthreads();
    if (HALF && i0 && tid == 0 && t <= t1 && any) done(t - 1);
    if (HALF && failed()) return false;
    if (more) {
      // the pages of the task after it and the list words of the one after that go out ahead
      // of the gather: behind it they would hold this wave, and so the barriers, to its end
      if (ahead && t + 2 < t1) {
        const ptrdiff_t line = line_of(t + 2);
        apos = list_poll(t + 2, aw, &abad);
        apage = page_of(line, apos);
        if (t + 3 < t1) aw = list_word(t + 3);
      }
      gather(L.row[par ^ 1]);
    }
    // QK: wave w < 4 takes keys 16w .. 16w+15 as the MFMA columns
    const int key = (wave & 3) * 16 + c16;
    const bool valid = have && row[key] >= 0;
    float sv[4], m[4];
    if (have && qk_wave) {
      // every LDS read first, then two interleaved accumulator chains
      const uint8_t* krow = L.k + key * MLA_KROW + 8 * g;
      uint2 kw[18];
#pragma unroll
      for (int ks = 0; ks < 18; ++ks) kw[ks] = *(const uint2*)(krow + 32 * ks);
      f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 18; ks += 2) {
        acc0 = mfma_bf16(qa[ks], e4m3x8_to_bf16(kw[ks].x, kw[ks].y), acc0);
        acc1 = mfma_bf16(qa[ks + 1], e4m3x8_to_bf16(kw[ks + 1].x, kw[ks + 1].y), acc1);
      }
      const f32x4 acc = acc0 + acc1;
      // split-local softmax per head (heads 4g + i): the wave's maxima, one 16-byte store a row
      f32x4 mx;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sv[i] = valid ? acc[i] * L.sc[key] : -INFINITY;
        mx[i] = row16_max(sv[i]);
      }
      if (c16 == 0) *(f32x4*)&L.red[wave][4 * g] = mx;
      if (more && (t + 1) / p.nsplit != r) load_q(r + 1);
    }
    __syncthreads();
    if (have && qk_wave) {
      // every LDS read ahead of the first write, the four heads side by side: one head after
      // another, each behind its own reads, took twice as long
      f32x4 rd[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) rd[w] = *(const f32x4*)&L.red[w][4 * g];
      const float ksk = L.kscale[key];
      f32x4 pe, ls;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        m[i] = fmaxf(fmaxf(rd[0][i], rd[1][i]), fmaxf(rd[2][i], rd[3][i]));
        pe[i] = (valid && m[i] != -INFINITY) ? expf(sv[i] - m[i]) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) ls[i] = row16_sum(pe[i]);
#pragma unroll
      for (int i = 0; i < 4; ++i) L.p[(4 * g + i) * (MLA_SPLIT + 8) + key] = f32_to_bf16(pe[i] * ksk);
      if (c16 == 0) *(f32x4*)&L.suml[wave][4 * g] = ls;
    }
    __syncthreads();
    if (have && wave == 0 && c16 == 0) {
      const DevOut out(p.part_ml + ((size_t)r * p.nsplit + s) * MLA_HEADS * 2, MLA_HEADS * 8);
      f32x4 l4 = *(const f32x4*)&L.suml[0][4 * g];
#pragma unroll
      for (int w = 1; w < 4; ++w) l4 += *(const f32x4*)&L.suml[w][4 * g];
#pragma unroll
      for (int i = 0; i < 4; i += 2)
        out.st16((4 * g + i) * 8, make_uint4(__float_as_uint(m[i]), __float_as_uint(l4[i]),
                                                    __float_as_uint(m[i + 1]), __float_as_uint(l4[i + 1])));
    }
    // PV, the dims as the MFMA's rows and the heads as its columns: wave w takes dim tiles
    // TPW*w .. +TPW-1 (16 dims each), 2 key steps of 32
    constexpr int TPW = 32 / NW;
    if (have) {
      bf16x8 pa[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        pa[ks] = __builtin_bit_cast(bf16x8, *(const uint4*)(L.p + c16 * (MLA_SPLIT + 8) + 32 * ks + 8 * g));
      const DevOut out(p.part_o + ((size_t)r * p.nsplit + s) * MLA_HEADS * MLA_LAT, MLA_HEADS * MLA_LAT * 2);
      static_assert(TPW % 2 == 0, "dim tiles go in pairs");
#pragma unroll
      for (int tl = 0; tl < TPW; tl += 2) {
        const int d0 = (wave * TPW + tl) * 16;
        uint32_t w[2][2];  // lane (c16, g): dims 4g .. 4g + 3 of head c16, two tiles, as bf16 pairs
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            const uint2 vw = lds_read_keys8(L.k, 32 * ks + 8 * g, d0 + 16 * tt, c16);
            o = mfma_bf16(e4m3x8_to_bf16(vw.x, vw.y), pa[ks], o);
          }
          w[tt][0] = pack_bf16x2(o[0], o[1]);
          w[tt][1] = pack_bf16x2(o[2], o[3]);
        }
        // the second tile's even lane rows swapped with the first's odd ones: every lane then
        // holds 8 consecutive dims (first tile: g 0, 2; second: g 1, 3), and a head's four
        // lanes store one whole 64-byte piece
        const auto lo = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
        out.st16((c16 * MLA_LAT + d0 + 16 * (g & 1) + 8 * (g >> 1)) * 2, make_uint4(lo[0], hi[0], lo[1], hi[1]));
      }
    }
    if (HALF && i0 + 1 < iters) __syncthreads();  // the next task's rows replace these
  }
  drain_memory();
  __syncthreads();
  if (tid == 0 && any && t1 - t0 == iters) done(t1 - 1);
  return true;
}

// ---------------------------------------------------------------- stage: merge + W_UV
// Task (rows r0 .. r0 + nr - 1, head h, half hf), nr <= MLA_MRG: for each row the exact
// combination of its splits for head h -> o_lat (rounded to bf16, in LDS), then half
// hf of o[r][h] = W_UV[h] o_lat on bf16 MFMA: the half's 16-row W_UV tiles go to waves
// 1, 2, ... over all 512 latent dims, with row r0 + i's o_lat as MFMA column i (the
// W_UV bytes a task moves serve all its rows).  Every row's sums and every MFMA column
// are computed alike whatever the task's rows, and the two halves of (r, h) compute
// the same o_lat bits, so the output does not depend on either split.  A wave's first
// tile is static and loaded before `wait` (the splits' dependency); wave 0, which
// polls the dependency, loads none.
constexpr int MLA_MRG = 4;            // rows a merge task at most
constexpr int MLA_OLROW = MLA_LAT + 8; // LDS row stride (bf16) of o_lat: rows in distinct banks
struct MlaMergeLds {
  float w[MLA_MRG][2 * 1024 + 8];  // per row, per split: exp(m_s - M), then l_s (nsplit <= 1024)
  float hi[MLA_MRG][MLA_LAT];      // the second half of the splits' weighted sums
  float inv[MLA_MRG];              // 1 / sum_s l_s exp(m_s - M)
  bf16_t ol[MLA_MRG][MLA_OLROW];
};

// rows a merge task of a persistent launch takes: about one task a workgroup
MK2_DEV int mla_merge_rows(int rows, int G) { return min(MLA_MRG, max(1, rows * 2 * MLA_HEADS / G)); }

template <int NT, typename Wait = NoWait>
MK2_DEV void mla_merge_uv(const MlaDev& p, int r0, int nr, int h, int hf, MlaMergeLds& L, Wait wait = Wait()) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, c16 = lane & 15;
  const int ns = p.nsplit, nvt = p.v_dim / 16;
  const int vlo = hf ? (nvt + 1) / 2 : 0, vhi = hf ? nvt : (nvt + 1) / 2;  // this half's tiles
  const int vt0 = vlo + wave - 1;  // wave w >= 1 takes tiles vt0, vt0 + NW - 1, ...
  auto load_a = [&](int vt, bf16x8* a) {  // W_UV[h] rows vt*16 + c16, dims 128 kb + 32 g + 8 q
    const bf16_t* wrow = p.w_uv + ((size_t)h * p.v_dim + vt * 16 + c16) * MLA_LAT + 32 * g;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int q = 0; q < 4; ++q) a[kb * 4 + q] = __builtin_bit_cast(bf16x8, ld_stream16(wrow + kb * 128 + 8 * q));
  };
  bf16x8 a[16];
  if (wave >= 1 && vt0 < vhi) load_a(vt0, a);
  if (!wait()) return;
  // the splits' bf16 partials: thread t takes dims 2 (t % 256) and + 1 of every row (one
  // 32-bit load a split) over half of the splits (the first or the second), 16 loads a
  // row in flight; the second half's sums go through LDS and are added to the first's.
  // The first 16 of every row go out right behind the splits' (m, l), so that all
  // arrive in one round trip.
  static_assert(NT == 2 * (MLA_LAT / 2), "two threads a dim pair");
  const int dp = tid % (MLA_LAT / 2), sh = tid / (MLA_LAT / 2);
  const int nh = (ns + 1) / 2, sa = sh * nh, sb = min(ns, sa + nh);
  constexpr int U = 16;
  uint32_t v[MLA_MRG][U];
  auto load_po = [&](int i, int s0) {
    const uint32_t* po = (const uint32_t*)(p.part_o + ((size_t)(r0 + i) * ns * MLA_HEADS + h) * MLA_LAT) + dp;
#pragma unroll
    for (int u = 0; u < U; ++u) v[i][u] = s0 + u < sb ? ldp_u32(po + (size_t)(s0 + u) * (MLA_HEADS * MLA_LAT / 2)) : 0u;
  };
  // (m, l) of split s of row i at flat index f = i * ns + s
  auto ml_at = [&](int f) {
    const int i = f / ns, s = f - i * ns;
    return ldp_8(p.part_ml + (((size_t)(r0 + i) * ns + s) * MLA_HEADS + h) * 2);
  };
  const int nml = nr * ns;
  const uint2 ml0 = tid < nml ? ml_at(tid) : make_uint2(0, 0);
#pragma unroll
  for (int i = 0; i < MLA_MRG; ++i)
    if (i < nr) load_po(i, sa);
  if (tid < nml) {
    const int i = tid / ns, s = tid - i * ns;
    L.w[i][s] = __uint_as_float(ml0.x);
    L.w[i][ns + s] = __uint_as_float(ml0.y);
  }
  for (int f = tid + NT; f < nml; f += NT) {  // more than NT splits in the task
    const uint2 m1 = ml_at(f);
    const int i = f / ns, s = f - i * ns;
    L.w[i][s] = __uint_as_float(m1.x);
    L.w[i][ns + s] = __uint_as_float(m1.y);
  }
  __syncthreads();
  // row i on wave i: M = max_s m_s, the split weights exp(m_s - M), and 1 / sum_s l_s w_s
  if (wave < nr) {
    float* wg = L.w[wave];
    float M = -INFINITY;
    for (int s = lane; s < ns; s += 64) M = fmaxf(M, wg[s]);
    M = wave_max(M);
    float ls = 0.f;
    for (int s = lane; s < ns; s += 64) {
      const float e = wg[s] == -INFINITY ? 0.f : expf(wg[s] - M);
      wg[s] = e;
      ls += wg[ns + s] * e;
    }
    ls = wave_sum(ls);
    if (lane == 0) L.inv[wave] = ls > 0.f ? 1.0f / ls : 0.f;
  }
  __syncthreads();
  float o[MLA_MRG][2];
#pragma unroll
  for (int i = 0; i < MLA_MRG; ++i) {
    o[i][0] = o[i][1] = 0.f;
    if (i >= nr) continue;
    for (int s0 = sa; s0 < sb; s0 += U) {
      if (s0 != sa) load_po(i, s0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float w = s0 + u < sb ? L.w[i][s0 + u] : 0.f;
        o[i][0] += __uint_as_float(v[i][u] << 16) * w;
        o[i][1] += __uint_as_float(v[i][u] & 0xFFFF0000u) * w;
      }
    }
    if (sh == 1) {
      L.hi[i][2 * dp] = o[i][0];
      L.hi[i][2 * dp + 1] = o[i][1];
    }
  }
  __syncthreads();
  if (sh == 0) {
#pragma unroll
    for (int i = 0; i < MLA_MRG; ++i) {
      if (i >= nr) break;
      const float inv = L.inv[i];
      const float f0 = (o[i][0] + L.hi[i][2 * dp]) * inv, f1 = (o[i][1] + L.hi[i][2 * dp + 1]) * inv;
      *(uint32_t*)(L.ol[i] + 2 * dp) = pack_bf16x2(f0, f1);
      if (p.o_lat_f32 && hf == 0) {
        const size_t at = ((size_t)(r0 + i) * MLA_HEADS + h) * MLA_LAT + 2 * dp;
        p.o_lat_f32[at] = f0;
        p.o_lat_f32[at + 1] = f1;
      }
    }
  }
  __syncthreads();
  // column c16: row r0 + c16 (columns past nr repeat the last row and are not stored)
  const bf16_t* olc = L.ol[min(c16, nr - 1)];
  for (int vt = vt0; wave >= 1 && vt < vhi; vt += NW - 1) {
    if (vt != vt0) load_a(vt, a);
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int q = 0; q < 4; ++q) c = mfma_bf16(a[kb * 4 + q], *(const bf16x8*)(olc + kb * 128 + 32 * g + 8 * q), c);
    if (c16 < nr) {  // column c16: v rows 4 g + i of row r0 + c16
      bf16_t* dst = p.o + (size_t)(r0 + c16) * (MLA_HEADS * p.v_dim) + h * p.v_dim + vt * 16 + 4 * g;
      st_dev_8(dst, make_uint2(pack_bf16x2(c[0], c[1]), pack_bf16x2(c[2], c[3])));
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------- stage: W_o
// Tasks (16 hidden rows nt0) and, with NTL = 2, (16 hidden rows nt1; -1: none): both
// tiles' first PF k-blocks a wave are loaded before `wait` (the attention rows'
// dependency), the rest after; the attention rows are loaded once for both.  Without
// a second tile the first is computed twice and stored once.  With `ssp` set, the
// epilogue also leaves each output row's sum of squares over the tile's 16 columns
// (the next RMSNorm's partial sums).
template <int NT, int NCG, int NTL = 1, typename Wait = NoWait>
MK2_DEV void mla_oproj(const MlaDev& p, int nt0, int nt1, float* red, Wait wait = Wait()) {
  constexpr int NW = NT / 64, PF = 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c16 = lane & 15;
  const int K = MLA_HEADS * p.v_dim, KB = K / 128;
  const uint8_t* tiles[NTL];
#pragma unroll
  for (int j = 0; j < NTL; ++j) tiles[j] = p.w_o + (size_t)(j == 0 || nt1 < 0 ? nt0 : nt1) * KB * 64 * 64;
  bf16x8 apf[NTL][PF][4];
#pragma unroll
  for (int j = 0; j < NTL; ++j)
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int kb = wave + u * NW;
      const uint4* t = (const uint4*)(tiles[j] + ((size_t)min(kb, KB - 1) * 64 + lane) * 64);
#pragma unroll
      for (int q = 0; q < 4; ++q) apf[j][u][q] = __builtin_bit_cast(bf16x8, ld_stream16(t + q));
    }
  // the residual rows (the layer's input, static) for the epilogue: entry idx = tid +
  // i * NT of the ntl * 16 * rows outputs
  const int ntl = NTL > 1 && nt1 >= 0 ? 2 : 1;
  constexpr int EPI = (NTL * 16 * 32 + NT - 1) / NT;
  float hres[EPI];
#pragma unroll
  for (int i = 0; i < EPI; ++i) {
    const int idx = threadIdx.x + i * NT;
    hres[i] = 0.f;
    if (p.h && idx < ntl * 16 * p.rows) {
      const int j = idx / (16 * p.rows), jdx = idx - j * 16 * p.rows;
      hres[i] = bf16_to_f32(p.h[(size_t)(jdx >> 4) * p.hidden + (j == 0 ? nt0 : nt1) * 16 + (jdx & 15)]);
    }
  }
  if (!wait()) return;
  f32x4 acc[NTL][NCG];
#pragma unroll
  for (int j = 0; j < NTL; ++j)
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) acc[j][cg] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int kb, bf16x8 (*a)[4]) {
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) {
      const int row = cg * 16 + c16;
      bf16x8 b[4];
      if (row < p.rows) {
        const bf16_t* src = p.o + (size_t)row * K + kb * 128 + 32 * g;
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = __builtin_bit_cast(bf16x8, ldp_16(src + 8 * q));
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
      }
#pragma unroll
      for (int j = 0; j < NTL; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[j][cg] = mfma_bf16(a[j][q], b[q], acc[j][cg]);
    }
  };
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (wave + u * NW < KB) {
      bf16x8 a[NTL][4];
#pragma unroll
      for (int j = 0; j < NTL; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) a[j][q] = apf[j][u][q];
      step(wave + u * NW, a);
    }
  for (int kb = wave + PF * NW; kb < KB; kb += NW) {
    bf16x8 a[NTL][4];
#pragma unroll
    for (int j = 0; j < NTL; ++j) {
      const uint4* t = (const uint4*)(tiles[j] + ((size_t)kb * 64 + lane) * 64);
#pragma unroll
      for (int q = 0; q < 4; ++q) a[j][q] = __builtin_bit_cast(bf16x8, ld_stream16(t + q));
    }
    step(kb, a);
  }
#pragma unroll
  for (int j = 0; j < NTL; ++j)
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) *(f32x4*)(red + (((j * NW + wave) * NCG + cg) * 64 + lane) * 4) = acc[j][cg];
  __syncthreads();
#pragma unroll
  for (int it = 0; it < EPI; ++it) {
    const int idx = threadIdx.x + it * NT;
    if (idx >= ntl * 16 * p.rows) break;
    const int j = idx / (16 * p.rows), jdx = idx - j * 16 * p.rows;
    const int n16 = jdx & 15, row = jdx >> 4, cg = row >> 4, s16 = row & 15;
    const int l = (n16 >> 2) * 16 + s16, i = n16 & 3;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[(((j * NW + w) * NCG + cg) * 64 + l) * 4 + i];
    const size_t o = (size_t)row * p.hidden + (j == 0 ? nt0 : nt1) * 16 + n16;
    if (p.h) v += hres[it];
    const bf16_t ob = f32_to_bf16(v);
    st_dev_u16(p.out + o, ob);
    if (p.ssp) {  // the 16 columns of (tile, row) are one DPP row: 16 * rows and NT are multiples of 16
      const float vb = bf16_to_f32(ob);
      const float ss = row16_sum(vb * vb);
      if (n16 == 0) st_dev_f32(p.ssp + (size_t)row * (p.hidden / 16) + (j == 0 ? nt0 : nt1), ss);
    }
  }
  __syncthreads();
}

}  // namespace mk2
