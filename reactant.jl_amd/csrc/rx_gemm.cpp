#include "rx_gemm.h"

#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <sstream>
#include <stdexcept>

namespace rx {

// f64: the register-staged skeleton on v_mfma_f64_16x16x4_f64
static GemmChoice choose_gemm_f64(int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc) {
  GemmChoice c;
  const int ve = 2, bk = 16;
  if (K < 1 || ((a_kc || b_kc) && K % ve != 0)) return c;
  if (N % 4 != 0 || M < 1 || N < 4) return c;
  if (!a_kc && M % ve != 0) return c;
  if (!b_kc && N % ve != 0) return c;
  if (M * N < 64 * 64) return c;
  if (M >= ((int64_t)1 << 30) || N >= ((int64_t)1 << 30) || K >= ((int64_t)1 << 30)) return c;
  // 4096^3: 256x128 tiles on 8 wavefronts 60-62 TFLOP/s, 128x128 on 4 wavefronts 47, 64x64 52-54;
  // 1024^3: 64x64 32, 128x128 11
  int BM = 64, BN = 64, WM = 2, WN = 2;
  if (((M + 255) / 256) * ((N + 127) / 128) * batch >= 256) { BM = 256; BN = 128; WM = 4; WN = 2; }
  else if (((M + 127) / 128) * ((N + 127) / 128) * batch >= 512) { BM = 128; BN = 128; }
  if (const char* e = getenv("RX_GEMM_TILE_F64")) {  // "BM,BN,WM,WN" for tuning runs
    int v[4];
    if (sscanf(e, "%d,%d,%d,%d", &v[0], &v[1], &v[2], &v[3]) == 4) { BM = v[0]; BN = v[1]; WM = v[2]; WN = v[3]; }
  }
  int rb = 4, cb = 8;
  const int64_t gm = (M + BM - 1) / BM, gn = (N + BN - 1) / BN;
  if (gm * gn < 64) rb = cb = 0;
  else if (gm < rb) { cb = (int)(rb * cb / gm); rb = (int)gm; }
  else if (gn < cb) { rb = (int)(rb * cb / gn); cb = (int)gn; }
  const int pad = 2;
  const int64_t a_sz = a_kc ? (int64_t)BM * (bk + pad) : (int64_t)bk * (BM + pad);
  const int64_t b_sz = b_kc ? (int64_t)BN * (bk + pad) : (int64_t)bk * (BN + pad);
  c.lds_bytes = (unsigned)(2 * (a_sz + b_sz) * 8);
  if (c.lds_bytes > 160 * 1024) return c;
  c.block = WM * WN * 64;
  c.grid[0] = (unsigned)gemm_grid(gm, gn, rb, cb);
  c.grid[1] = (unsigned)batch;
  std::ostringstream t;
  t << BM << ", " << BN << ", " << bk << ", " << WM << ", " << WN << ", " << (a_kc ? "true" : "false") << ", " << (b_kc ? "true" : "false")
    << ", " << M << ", " << N << ", " << K << ", " << rb << ", " << cb;
  c.targs = t.str();
  c.skeleton = "rx_gemm_body_f64";
  c.stype_a = "double";
  c.kind = "gemm_f64";
  c.ok = true;
  return c;
}

// ---------------------------------------------------------------------------
// rx_gemm_body_g (K in groups inside the workgroup): tile, wavefronts, groups and stages
// ---------------------------------------------------------------------------
struct GroupTile { int BM, BN, WM, WN, KG, S, split3 = 0; };   // split3: f32 operands as three bf16 each (rx_gemm_body_x)

// After how many K tiles rx_gemm_body_g adds its sums to totals (0: one running sum per group), and whether those are wide.
// What took these products otherwise sums shortly: the reduction of products of up to eight rows in parts of 16 to 400 k,
// the products cut along K (fewer than 256 64 x 64 tiles, K >= 1024) in slices of 512 k and more.  So for up to eight rows
// sums of 32 k of f32, 16 of f64 and four MFMAs of narrower elements go into wide totals, and for the others sums of 512 k
// into totals of the accumulators' type; no error is larger than that of those plans (f32 3 x 4096 x 784 is closest).
struct GroupFold { int tiles = 0; bool wide = false; };
static GroupFold group_fold(DT dt, int64_t batch, int64_t M, int64_t N, int64_t K, int split, const GroupTile& t) {
  const int es = info(dt).size;
  const int64_t bk = 128 / es, KT = (K + bk - 1) / bk, step = (int64_t)t.KG * split, KTG = (KT + step - 1) / step;
  GroupFold f;
  if (t.split3) return f;
  if (std::min(M, N) <= 8) {
    f.wide = true;
    f.tiles = es == 2 ? 2 : 1;
  } else if (batch == 1 && es <= 4 && ((M + 63) / 64) * ((N + 63) / 64) < 256 && K >= 1024) {
    f.tiles = (int)(512 / bk);
  }
  if (KTG <= (f.wide ? 1 : f.tiles)) f.tiles = 0;
  return f;
}

static bool group_fits(DT dt, int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc, int split, const GroupTile& t, int64_t* lds) {
  const int es = info(dt).size;
  const int64_t bk = 128 / es, KT = (K + bk - 1) / bk, step = (int64_t)t.KG * split, KTG = (KT + step - 1) / step;
  const int NW = t.WM * t.WN;
  if (t.BM % (16 * t.WM) || t.BN % (16 * t.WN) || t.BM / 8 % NW || t.BN / 8 % NW || NW * t.KG > 16) return false;
  if ((a_kc ? K : M) * es % 4 || (b_kc ? K : N) * es % 4) return false;   // operand rows are whole dwords
  const int64_t lim = (int64_t)1 << 31;                                    // 32-bit operand offsets, the last groups' K tiles included
  if (M * K * es >= lim || N * K * es >= lim) return false;
  if ((!a_kc && (K + 2 * bk * step) * M * es >= 2 * lim) || (!b_kc && (K + 2 * bk * step) * N * es >= 2 * lim)) return false;
  if (batch > 65535) return false;                                         // blockIdx.y
  // accumulators and fragments of a wavefront within its share of the register file
  const int na = t.BM / t.WM / 16, nb = t.BN / t.WN / 16;
  const int share = 512 / std::max(1, (NW * t.KG + 3) / 4);
  if (t.split3) {   // rx_gemm_body_x: whole vectors or 4 x 4 blocks per thread, loaded and split registers beside the fragments
    const int nt = NW * 64, nv = (t.BM + t.BN) * 8 / nt;
    if (dt != DT::F32 || split > 1 || t.BM % 32 || t.BN % 32 || t.BM * (a_kc ? 8 : 2) % nt || t.BN * (b_kc ? 8 : 2) % nt) return false;
    if (na * nb * 4 + 10 * nv + 12 * (nb + 1) + 40 > std::min(share, 256)) return false;   // two wavefronts per SIMD
    *lds = std::max<int64_t>((int64_t)t.KG * (t.BM + t.BN) * 192, t.KG > 1 ? (int64_t)t.KG * t.BM * t.BN * 4 : 0);
    return *lds + 128 <= 160 * 1024;   // (128: the wavefronts' votes and the operands' largest magnitudes)
  }
  const GroupFold fold = group_fold(dt, batch, M, N, K, split, t);
  const int words = es == 8 ? 8 : 4;   // of an accumulator block
  if (na * nb * words * (fold.tiles == 0 ? 1 : fold.wide ? 4 : 2) + 8 * (na + nb) + 48 > share) return false;
  if (t.S < 2 && KTG > 1) return false;                                    // a stage to read and one to load
  const int64_t nl = (t.BM + t.BN) / 8 / NW, sd = std::min<int64_t>(t.S, KTG);
  if (nl * (sd - 1) > 63) return false;                                    // outstanding loads that a wait can count
  const int64_t ring = (int64_t)t.KG * sd * (t.BM + t.BN) * 128, sums = t.KG > 1 ? (int64_t)t.KG * t.BM * t.BN * (es == 8 ? 8 : 4) : 0;
  *lds = std::max(ring, sums);
  return *lds <= 160 * 1024;
}

// Time of a launch in microseconds, for comparing tiles: rounds of workgroups over the 256 compute units; per K tile
// the largest of the MFMAs, the operand loads and the LDS fragment reads of the workgroups that share a compute unit
// (with little to overlap them where few wavefronts share a SIMD), or the latency of the loads over the stages in flight;
// the prologue, the epilogue and the groups' sums; bounded below by the operands' traffic from L2 and from memory.
// Constants fitted to 1600 timings of 54 shapes (f32, f64, bf16, e4m3; 1 to 8192 rows; all operand orders): the tile
// with the smallest estimate takes 1.03 times the time of the fastest one (geometric mean).
static double group_estimate(DT dt, int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc, int split, const GroupTile& t, int64_t lds) {
  const int es = info(dt).size, NW = t.WM * t.WN, waves = NW * t.KG;
  const int64_t bk = 128 / es, KT = (K + bk - 1) / bk, step_k = (int64_t)t.KG * split;
  const double KTG = (double)((KT + step_k - 1) / step_k), sd = std::min<double>(t.S, KTG);
  const int64_t T = ((M + t.BM - 1) / t.BM) * ((N + t.BN - 1) / t.BN) * batch * split;
  const int64_t R = std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(160 * 1024 / lds, 16 / waves), 8));
  const int64_t per = (T + 255) / 256, cc = std::min(per, R);          // workgroups of a compute unit in all, and at a time
  const double rounds = per <= cc ? 1.0 : (double)(per / cc) + (double)(per % cc) / (double)cc;
  const double w = (double)waves * (double)cc / 4.0;                   // wavefronts per SIMD
  // flops per clock and compute unit, times what these loops sustain of them
  const double fl = es == 8 ? 128 * 0.93 : es == 4 ? 256.0 : es == 2 ? 4096 * 0.68 : 8192 * 0.64;
  const double mf = (double)t.BM * t.BN * (double)bk * t.KG * 2.0 / fl * (double)cc / std::min(1.0, w);
  const double ld = (double)t.KG * (t.BM + t.BN) * 128.0 / 102.0 * (double)cc;
  const double rd = (double)waves * ((double)t.BM / t.WM + (double)t.BN / t.WN) * 128.0 / 179.0 * (double)cc;
  const double big = std::max(mf, std::max(ld, rd));
  const double step = std::max(1625.0 / std::max(sd - 1.0, 0.5), (big + 0.1 * (mf + ld + rd - big)) * (1.0 + 0.33 / std::max(w, 1.0)) + 170.0);
  double cycles = 4100.0 + rounds * KTG * step + (double)per * (double)t.BM * t.BN * (0.36 + (t.KG > 1 ? 0.15 * t.KG : 0.0)) + (rounds - 1.0) * 5600.0;
  cycles += 0.02 * cycles;
  // Wavefronts that share no fragments, in five rounds of workgroups and more, take 1.35 to 1.9 times what is above (32 x 32 tiles:
  // f32 276 x 4096 x 2048 88 us for 47, 615 x 2048 x 3000 107 for 70, f64 1408 x 1984 x 3840 548 for 392, 832 x 1408 x 704 60 for
  // 35; 32 x 64 tiles: f64 2432 x 1472 x 1920 383 for 241).  With it f32 276 x 4096 x 2048 takes 53 us, f64 2232 x 700 x 3136
  // 203 (320 on 32 x 32 tiles), 1368 x 3524 x 468 90 (105).
  if (es >= 4 && NW <= 2 && t.BM * t.BN >= 1024 && per >= 5) cycles *= 1.5;
  cycles = std::max(cycles, 4100.0 + (double)(T / split) * (t.BM + t.BN) * (double)K * es / 6000.0);
  const double bytes = (double)batch * (double)(M + N) * (double)K * es;
  cycles = std::max(cycles, 4100.0 + bytes / 1700.0);
  // A compute unit has some 250 lines of 128 bytes under way at a time, whole or not: a line, or the part of one that a
  // narrow tile reads of a [k][n] row, costs it 7.5 cycles from memory, 4.5 from the memory-side cache, 2 from L2
  // (16 x 4096 x 25088 bf16: tiles of 16, 32 and 64 columns 84, 98 and 108 us as [k][n], 40, 52 and 77 as [n][k])
  const double line = bytes < 16e6 ? 2.0 : bytes < 128e6 ? 4.5 : 7.5;
  auto lines = [&](bool kc, int64_t rows, int tile) {
    const double tiles = (double)((rows + tile - 1) / tile);
    return kc ? (double)rows * (double)K * es / 128.0 : tiles * (double)K * (double)((tile * es + 127) / 128);
  };
  cycles = std::max(cycles, 4100.0 + (double)batch * (lines(a_kc, M, t.BM) + lines(b_kc, N, t.BN)) * line / (double)std::min<int64_t>(T, 256));
  return cycles / 2400.0;
}

// rx_gemm_body_x: microseconds per K tile of 32 of a workgroup, alone on its compute unit or beside a second one.
// Measured: 128 x 128 2048^3 (one workgroup per compute unit) 107 us, 4096^3 (four) 697, 8192 x 4096 x 1024 (eight) 371; two groups
// 2048^3 98; 128 x 256 4096^3 668, 8192 x 4096 x 1024 370.
static double split3_estimate(int64_t batch, int64_t M, int64_t N, int64_t K, const GroupTile& t) {
  const int64_t T = ((M + t.BM - 1) / t.BM) * ((N + t.BN - 1) / t.BN) * batch, n = (T + 255) / 256, kt = ((K + 31) / 32 + t.KG - 1) / t.KG;
  const double area = (double)t.BM * t.BN / 16384.0;
  if (t.KG > 1) return 11.0 + (double)(n * kt) * 1.45 * t.KG * area;
  if (t.WM * t.WN > 4) return 8.0 + (double)(n * kt) * 1.3 * area;
  return 8.0 + (double)kt * ((double)(n / 2) * 2.75 + (double)(n % 2) * 1.6) * area;
}

// The most tiles that one of the eight XCDs takes of a gm x gn grid walked in blocks of rb x cb (rx_gemm_tile).
static int64_t xcd_tiles(int64_t gm, int64_t gn, int64_t rb, int64_t cb) {
  int64_t load[8] = {}, blk = 0;
  for (int64_t r = 0; r < gm; r += rb)
    for (int64_t c = 0; c < gn; c += cb) load[blk++ % 8] += std::min(rb, gm - r) * std::min(cb, gn - c);
  return *std::max_element(load, load + 8);
}

static GemmChoice group_gemm(DT dt, int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc, int split, const GroupTile& t) {
  GemmChoice c;
  int64_t lds = 0;
  if (!group_fits(dt, batch, M, N, K, a_kc, b_kc, split, t, &lds)) return c;
  const int64_t gm = (M + t.BM - 1) / t.BM, gn = (N + t.BN - 1) / t.BN;
  int rb = 4, cb = 8;
  if (gm * gn < 8) rb = cb = 0;
  // up to two rounds of tiles over the chip: every XCD takes a band of adjacent columns (rows) of tiles, so that narrow
  // tiles that share lines of an operand share an L2
  else if (gm * gn <= 512 && gn >= gm) { rb = (int)gm; cb = (int)((gn + 7) / 8); }
  else if (gm * gn <= 512) { rb = (int)((gm + 7) / 8); cb = (int)gn; }
  else if (gm < rb) { cb = (int)(rb * cb / gm); rb = (int)gm; }
  else if (gn < cb) { rb = (int)(rb * cb / gn); cb = (int)gn; }
  // Dealt one by one where these blocks give an XCD a tenth more rounds of tiles than that does: a 9 x 27 grid in
  // bands of four columns is 36 tiles on an XCD of 32 compute units, two rounds (f64 576 x 3456 x 1024 133 against 70 us, f32 69
  // against 36; f64 704 x 1152 x 2048 135 against 69, 1600 x 2496 x 2944 529 against 363), and a last column of blocks that is
  // mostly empty may fall to the same XCDs again and again (3904 x 320 x 1216 132 against 89).  Otherwise blocks are the better
  // order (f64 2076 x 2008 x 1544 325 against 372), the tiles a little uneven or not (bf16 26 x 1024 x 3000 6.2 against 8.2, f64 192 x
  // 3136 x 2240 70 against 84).
  if (rb > 0) {
    const int64_t most = xcd_tiles(gm, gn, rb, cb), even = (gm * gn + 7) / 8;
    if ((most + 31) / 32 * 10 > (even + 31) / 32 * 11) rb = cb = 0;
  }
  if (const char* e = getenv("RX_GEMM_BLOCK")) { int v[2]; if (sscanf(e, "%d,%d", &v[0], &v[1]) == 2) { rb = v[0]; cb = v[1]; } }
  c.lds_bytes = (unsigned)lds;
  c.block = (unsigned)(t.WM * t.WN * t.KG * 64);
  c.grid[0] = (unsigned)gemm_grid(gm, gn, rb, cb);
  c.grid[1] = (unsigned)(split > 1 ? split : batch);
  c.split = split;
  c.est_us = t.split3 ? split3_estimate(batch, M, N, K, t) : group_estimate(dt, batch, M, N, K, a_kc, b_kc, split, t, lds);
  const std::string el = dt == DT::F64 ? "rx_el_f64" : dt == DT::F32 ? "rx_el_f32" : dt == DT::BF16 ? "rx_el_bf16" : dt == DT::F16 ? "rx_el_f16" : std::min(M, N) <= 8 ? "rx_el_f8b" : "rx_el_f8";
  std::ostringstream o;
  if (!t.split3) o << el << ", ";
  o << t.BM << ", " << t.BN << ", " << t.WM << ", " << t.WN << ", ";
  const GroupFold fold = group_fold(dt, batch, M, N, K, split, t);
  if (!t.split3) o << t.KG << ", " << t.S << ", " << fold.tiles << ", " << (fold.wide ? "true" : "false") << ", ";
  else o << t.KG << ", ";
  o << (a_kc ? "true" : "false") << ", "
    << (b_kc ? "true" : "false") << ", " << M << ", " << N << ", " << K << ", " << rb << ", " << cb;
  c.targs = o.str();
  c.skeleton = t.split3 ? "rx_gemm_body_x" : "rx_gemm_body_g";
  c.kind = dt == DT::F64 ? "gemm_f64" : dt == DT::F32 ? "gemm_f32" : dt == DT::BF16 ? "gemm_bf16" : dt == DT::F16 ? "gemm_f16" : "gemm_f8";
  c.stype_a = t.split3 ? "float" : el + "::elem";
  c.waves = t.split3 ? 2 : 0;   // two workgroups of four wavefronts share a compute unit
  c.ok = true;
  return c;
}

// The tile with the smallest estimate.  RX_GEMM_G=BM,BN,WM,WN,KG,S asks for one (a seventh number, 1: rx_gemm_body_x, which has no S; products it does not fit keep the
// estimate's), RX_GEMM_G=0 leaves this skeleton out.
static GemmChoice choose_group(DT dt, DT out, int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc, int split) {
  GemmChoice best;
  const bool types = (dt == DT::F64 && out == DT::F64) || (dt == DT::F32 && out == DT::F32) || ((dt == DT::BF16 || dt == DT::F16) && (out == dt || out == DT::F32)) ||
                     (dt == DT::F8E4M3FN && (out == DT::F32 || out == DT::BF16 || out == DT::F16));
  if (!types || M < 1 || N < 1 || batch < 1) return best;
  // a few thousand multiplications: the scalar loop is as good
  if (K < 64 || (double)batch * (double)M * (double)N * (double)K < (double)(1 << 19)) return best;
  if (const char* e = getenv("RX_GEMM_G")) {
    GroupTile t;
    if (!strcmp(e, "0")) return best;
    if (sscanf(e, "%d,%d,%d,%d,%d,%d,%d", &t.BM, &t.BN, &t.WM, &t.WN, &t.KG, &t.S, &t.split3) < 6 || t.BM < 16 || t.BN < 16 || t.WM < 1 || t.WN < 1 || t.KG < 1 || t.S < 1 || t.split3 < 0 || t.split3 > 1)
      throw std::runtime_error("RX_GEMM_G wants BM,BN,WM,WN,KG,S");
    best = group_gemm(dt, batch, M, N, K, a_kc, b_kc, split, t);
    if (best.ok) return best;
  }
  static const int tiles[][4] = {{16, 16, 1, 1}, {16, 32, 1, 1}, {32, 16, 1, 1}, {16, 64, 1, 2}, {64, 16, 2, 1}, {32, 32, 1, 1}, {32, 64, 1, 2}, {64, 32, 2, 1},
                                 {32, 64, 2, 2}, {64, 32, 2, 2}, {64, 64, 2, 2}, {64, 96, 2, 2}, {96, 64, 2, 2}, {96, 96, 2, 2}, {64, 128, 2, 2}, {128, 64, 2, 2},
                                 {64, 128, 2, 4}, {128, 64, 4, 2}, {96, 128, 2, 2}, {128, 96, 2, 2}, {128, 128, 2, 2}, {128, 128, 2, 4}, {128, 128, 4, 2},
                                 {160, 128, 2, 2}, {128, 160, 2, 2}, {192, 128, 4, 2}, {128, 192, 2, 4}, {256, 128, 4, 2}, {128, 256, 2, 4}};
  GroupTile pick{};
  double cost = 0;
  for (auto& q : tiles)
    for (int kg = 1; kg <= 16; kg *= 2)
      for (int s = 2; s <= 5; ++s) {
        const GroupTile t{q[0], q[1], q[2], q[3], kg, s};
        int64_t lds = 0;
        if (!group_fits(dt, batch, M, N, K, a_kc, b_kc, split, t, &lds)) continue;
        const double c = group_estimate(dt, batch, M, N, K, a_kc, b_kc, split, t, lds);
        if (cost == 0 || c < cost) { cost = c; pick = t; }
      }
  // f32 products that fill the chip with 128-wide tiles: operands split into bf16 (rx_gemm_body_x)
  if (dt == DT::F32)
    for (const GroupTile& t : {GroupTile{128, 128, 2, 2, 1, 1, 1}, GroupTile{128, 128, 2, 2, 2, 1, 1}, GroupTile{128, 256, 2, 4, 1, 1, 1}, GroupTile{256, 128, 4, 2, 1, 1, 1}}) {
      int64_t lds = 0;
      if (!group_fits(dt, batch, M, N, K, a_kc, b_kc, split, t, &lds)) continue;
      const double c = split3_estimate(batch, M, N, K, t);
      if (cost == 0 || c < cost) { cost = c; pick = t; }
    }
  return cost > 0 ? group_gemm(dt, batch, M, N, K, a_kc, b_kc, split, pick) : best;
}

// The skeletons for tiles that fill the chip (streaming and ping-pong bodies, ring skeleton) and the register-staged one.
static GemmChoice choose_tiled(DT a, DT out, int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc, bool staged_only, int split) {
  GemmChoice c;
  if (split > 1 && (staged_only || batch != 1 || a == DT::F64)) return c;
  if (a == DT::F64 && out == DT::F64) return staged_only ? c : choose_gemm_f64(batch, M, N, K, a_kc, b_kc);
  std::string mma;
  int esize = 0, bk = 0;
  if (a == DT::F32 && out == DT::F32) { mma = "rx_mma_f32"; c.kind = "gemm_f32"; esize = 4; bk = 16; }
  else if (a == DT::BF16 && (out == DT::BF16 || out == DT::F32)) { mma = "rx_mma_bf16"; c.kind = "gemm_bf16"; esize = 2; bk = 64; }
  else if (a == DT::F16 && (out == DT::F16 || out == DT::F32)) { mma = "rx_mma_f16"; c.kind = "gemm_f16"; esize = 2; bk = 64; }
  else if (a == DT::F8E4M3FN && (out == DT::F32 || out == DT::BF16 || out == DT::F16)) { mma = "rx_mma_f8"; c.kind = "gemm_f8"; esize = 1; bk = 128; }
  else return c;
  const int ve = 16 / esize;
  // 16-byte loads along the contracted dimension need whole vectors; a tail shorter than the
  // K step is zero-filled by the register-staged skeleton
  if (K < 1 || ((a_kc || b_kc) && K % ve != 0)) return c;
  if (N % 4 != 0) return c;
  if (!a_kc && M % ve != 0) return c;
  if (!b_kc && N % ve != 0) return c;
  if (M < 1 || N < 4) return c;
  if (M * N < 64 * 64) return c;  // tiny products: the scalar loop is as good
  if (M >= ((int64_t)1 << 30) || N >= ((int64_t)1 << 30) || K >= ((int64_t)1 << 30)) return c;
  // Large problems take 256x256 tiles on 8 wavefronts (each wavefront a 128x64 block of the
  // tile: fewer LDS bytes per MFMA); when that would leave compute units idle, 128x128 on 4.
  // Products that leave most compute units without a 128x128 tile take 64x64 tiles (1000^3 f32:
  // 16 -> 48 TFLOP/s, 1024^3 bf16: 130 -> 240); an operand with at most 64 rows (the output
  // features of a convolution) gets a 64-wide tile so that no MFMA works on padding.
  // A tuning override (RX_GEMM_TILE / _BK / _STAGES / _DIRECT) is honoured or refused with an error: a setting that
  // does not fit must not end in the scalar loop unnoticed.
  bool tuned = false;
  auto refuse = [&](const char* why) {
    throw std::runtime_error(std::string("RX_GEMM_* tuning override cannot be honoured for ") + c.kind + " " + std::to_string(M) + "x" + std::to_string(N) + "x" +
                             std::to_string(K) + ": " + why);
  };
  int BM = 128, BN = 128, WM = 2, WN = 2;
  if (M <= 64 && N > 64) { BM = 64; BN = 128; }
  else if (N <= 64 && M > 64) { BM = 128; BN = 64; }
  else if (M > 128 && N > 128 && ((M + 255) / 256) * ((N + 255) / 256) * batch >= 256) { BM = 256; BN = 256; WM = 2; WN = 4; }
  // 16-bit operands whose 256x256 tiles would leave compute units idle but whose 256x128 tiles fill the chip (the
  // 8192 x 1024 x 4096 layer of the MLP: 256 tiles, one per compute unit): 8 wavefronts, each a 128x32 block of the
  // tile, against 128x128 tiles on 4 wavefronts 75 -> 67 us
  else if (esize == 2 && M >= N && M > 128 && N > 64 && ((M + 255) / 256) * ((N + 127) / 128) * batch >= 256) { BM = 256; BN = 128; WM = 2; WN = 4; }
  else if (esize == 2 && N > M && N > 128 && M > 64 && ((M + 127) / 128) * ((N + 255) / 256) * batch >= 256) { BM = 128; BN = 256; WM = 4; WN = 2; }
  else if (((M + 127) / 128) * ((N + 127) / 128) * batch * split < 128) { BM = 64; BN = 64; }
  if (const char* e = getenv("RX_GEMM_TILE")) {  // "BM,BN,WM,WN" for tuning runs
    int v[4];
    if (sscanf(e, "%d,%d,%d,%d", &v[0], &v[1], &v[2], &v[3]) == 4) { BM = v[0]; BN = v[1]; WM = v[2]; WN = v[3]; tuned = true; }
    else refuse("RX_GEMM_TILE wants BM,BN,WM,WN");
    if (BM < 32 || BN < 32 || WM < 1 || WN < 1 || BM % (32 * WM) != 0 || BN % (32 * WN) != 0 || WM * WN > 16) refuse("tile is not a whole number of 32x32 blocks per wavefront");
  }
  const int ks_step = a == DT::F32 ? 8 : (esize == 2 ? 16 : 64);
  if (const char* e = getenv("RX_GEMM_BK")) {
    const int v = atoi(e);
    if (v <= 0 || v % ks_step != 0) refuse("RX_GEMM_BK is not a multiple of the MFMA k step");
    if (K % v == 0) { bk = v; tuned = true; }   // products whose K it does not divide keep the default
  }
  bool direct = !staged_only;   // global -> LDS direct loads through a ring of LDS stages
  bool direct_forced = false;
  if (const char* e = getenv("RX_GEMM_DIRECT")) { direct = atoi(e) != 0 && !staged_only; direct_forced = atoi(e) != 0 && !staged_only; }
  int stages = 2;
  if (const char* e = getenv("RX_GEMM_STAGES")) { if (atoi(e) < 2) refuse("RX_GEMM_STAGES < 2"); stages = atoi(e); }
  int rb = 4, cb = 8;   // tiles of one XCD's block (rows x columns of the tile grid)
  if (const char* e = getenv("RX_GEMM_BLOCK")) { int v[2]; if (sscanf(e, "%d,%d", &v[0], &v[1]) == 2 && v[0] > 0 && v[1] > 0) { rb = v[0]; cb = v[1]; } }
  // a grid of few tiles (per batch entry) is not worth padding to whole XCD blocks
  if (((M + BM - 1) / BM) * ((N + BN - 1) / BN) < 64) rb = cb = 0;
  // a tile grid with fewer rows (columns) than a block: make the block that flat
  else if ((M + BM - 1) / BM < rb) { const int64_t gm = (M + BM - 1) / BM; cb = (int)(rb * cb / gm); rb = (int)gm; }
  else if ((N + BN - 1) / BN < cb) { const int64_t gn = (N + BN - 1) / BN; rb = (int)(rb * cb / gn); cb = (int)gn; }
  const int nt = WM * WN * 64;
  // 8- and 16-bit operands on the eight-wavefront tiles whose wavefronts own 128 rows (256x256, 256x128): the
  // streaming skeleton on the 16x16 MFMA shapes (kernels/rx_gemm_kernels.h, rx_gemm_body_s).  It wants whole K tiles
  // of 128 bytes and operands below 4 GB (32-bit buffer offsets), and has no K-sliced form; RX_GEMM_STREAM=0 keeps the
  // ring skeleton.
  if (direct && (esize == 1 || esize == 2) && BM == 256 && (BN == 256 || BN == 128) && ((WM == 2 && WN == 4) || (WM == 4 && WN == 2 && BN == 128)) && split == 1 && bk * esize == 128 &&
      K % bk == 0 && stages == 2 && M * K * esize < ((int64_t)1 << 32) && N * K * esize < ((int64_t)1 << 32) &&
      !(getenv("RX_GEMM_STREAM") && atoi(getenv("RX_GEMM_STREAM")) == 0) && !(getenv("RX_GEMM_MFMA32") && atoi(getenv("RX_GEMM_MFMA32")) != 0)) {
    const std::string el = a == DT::F8E4M3FN ? "rx_el_f8" : (a == DT::BF16 ? "rx_el_bf16" : "rx_el_f16");
    // 256x128 tiles: wavefronts of 64x64 (4 + 4 fragments per K tile for 16 MFMA blocks) instead of 128x32 (8 + 2):
    // the 8192 x 1024 x 4096 bf16 layer 68.3 -> 66.6 us
    if (BN == 128 && !tuned) { WM = 4; WN = 2; }
    // three LDS stages where they fit (256x128 tiles: 144 KB): a request then has two K tiles to land instead of one
    int sstages = (BM + BN) * 128 * 3 <= 160 * 1024 ? 3 : 2;
    if (const char* e = getenv("RX_GEMM_STREAM_STAGES")) {
      if ((atoi(e) != 2 && atoi(e) != 3) || (BM + BN) * 128 * atoi(e) > 160 * 1024) refuse("RX_GEMM_STREAM_STAGES is 2, or 3 where three stages fit 160 KB");
      sstages = atoi(e);
    }
    c.lds_bytes = (unsigned)(sstages * (BM + BN) * 128);
    c.block = nt;
    c.grid[0] = (unsigned)gemm_grid((M + BM - 1) / BM, (N + BN - 1) / BN, rb, cb);
    c.grid[1] = (unsigned)batch;
    c.split = 1;
    std::ostringstream t;
    t << el << ", " << BM << ", " << BN << ", " << WM << ", " << WN << ", " << (a_kc ? "true" : "false") << ", " << (b_kc ? "true" : "false") << ", " << M
      << ", " << N << ", " << K << ", " << rb << ", " << cb;
    c.targs = t.str();
    c.stype_a = el + "::elem";
    // 256 x 256 tiles with an even number of K tiles: the ping-pong form of the same tiles (rx_gemm_body_pp: one
    // wavefront of a SIMD multiplies a whole K tile while the other reads its fragments) for 16-bit operands, and for
    // 8-bit operands when B is stored [n][k] (then the requests are shared between the two groups of wavefronts; with
    // one group requesting everything the 8-bit form is slower than the interleaved one).  RX_GEMM_PINGPONG=0 keeps
    // the interleaved form, =1 takes the ping-pong form wherever it exists.
    const int pp = getenv("RX_GEMM_PINGPONG") ? atoi(getenv("RX_GEMM_PINGPONG")) : ((esize == 2 || b_kc) ? 1 : 0);
    if (pp != 0 && BM == 256 && BN == 256 && WM == 2 && WN == 4 && (K / bk) % 2 == 0 && !getenv("RX_GEMM_STREAM_STAGES") && !getenv("RX_GEMM_STREAM_DEPTH")) {
      c.lds_bytes = (unsigned)(2 * (BM + BN) * 128);
      c.skeleton = "rx_gemm_body_pp";
      c.ok = true;
      return c;
    }
    c.skeleton = "rx_gemm_body_s";
    c.depth = 2;
    if (const char* e = getenv("RX_GEMM_STREAM_DEPTH")) {
      if (atoi(e) < 1 || atoi(e) > 3) refuse("RX_GEMM_STREAM_DEPTH is 1, 2 or 3");
      c.depth = atoi(e);
    }
    c.stream_stages = sstages;
    c.stype_a = el + "::elem";
    c.ok = true;
    return c;
  }
  if (direct) {
    const int dbk = bk;
    // 16-bit operands take the 16x16x32 MFMA here (kernels/rx_gemm_kernels.h, rx_mma_16b_16): k step 32
    const bool mfma16 = esize == 2 && dbk % 32 == 0 && !(getenv("RX_GEMM_MFMA32") && atoi(getenv("RX_GEMM_MFMA32")) != 0);
    const std::string dmma = mfma16 ? mma + "_16" : mma;
    const int ks = mfma16 ? 32 : ks_step;
    const int64_t a_ch = (int64_t)BM * dbk / ve, b_ch = (int64_t)BN * dbk / ve;
    const int64_t stage_bytes = ((int64_t)BM + BN) * dbk * esize;
    while (stages > 2 && stage_bytes * stages > 160 * 1024) --stages;
    if (dbk % ks == 0 && K % ((int64_t)dbk * split) == 0 && a_ch % nt == 0 && b_ch % nt == 0 && stage_bytes * stages <= 160 * 1024 &&
        (a_kc ? dbk : BM) % ve == 0 && (b_kc ? dbk : BN) % ve == 0) {
      c.lds_bytes = (unsigned)(stage_bytes * stages);
      c.block = nt;
      const int64_t gm = (M + BM - 1) / BM, gn = (N + BN - 1) / BN;
      c.grid[0] = (unsigned)gemm_grid(gm, gn, rb, cb);
      c.grid[1] = (unsigned)(split > 1 ? split : batch);
      c.split = split;
      std::ostringstream t;
      t << dmma << ", " << BM << ", " << BN << ", " << dbk << ", " << WM << ", " << WN << ", " << stages << ", " << (a_kc ? "true" : "false") << ", "
        << (b_kc ? "true" : "false") << ", " << M << ", " << N << ", " << K << ", " << rb << ", " << cb;
      c.targs = t.str();
      c.skeleton = "rx_gemm_body_dl";
      c.bk = dbk;
      c.stype_a = dmma + "::elem";
      c.ok = true;
      return c;
    }
    if (direct_forced) refuse("the direct-to-LDS skeleton does not tile this shape");
    if (tuned && stage_bytes * 2 > 160 * 1024) refuse("two LDS stages of this tile exceed 160 KB");
  }
  if (split > 1) return c;   // only the direct-to-LDS skeleton slices K
  const int pad = a == DT::F32 ? 4 : (esize == 2 ? 8 : 16);
  const int64_t a_sz = a_kc ? (int64_t)BM * (bk + pad) : (int64_t)bk * (BM + pad);
  const int64_t b_sz = b_kc ? (int64_t)BN * (bk + pad) : (int64_t)bk * (BN + pad);
  c.lds_bytes = (unsigned)(2 * (a_sz + b_sz) * esize);
  if (c.lds_bytes > 160 * 1024) {
    if (tuned) refuse("the register-staged skeleton needs more than 160 KB of LDS for this tile and K step");
    return c;
  }
  c.block = WM * WN * 64;
  const int64_t gm = (M + BM - 1) / BM, gn = (N + BN - 1) / BN;
  c.grid[0] = (unsigned)gemm_grid(gm, gn, rb, cb);
  c.grid[1] = (unsigned)batch;
  std::ostringstream t;
  t << mma << ", " << BM << ", " << BN << ", " << bk << ", " << WM << ", " << WN << ", " << (a_kc ? "true" : "false") << ", " << (b_kc ? "true" : "false")
    << ", " << M << ", " << N << ", " << K << ", " << rb << ", " << cb;
  c.targs = t.str();
  c.skeleton = "rx_gemm_body";
  c.stype_a = mma + "::elem";
  c.ok = true;
  return c;
}

// 9 to 64 rows of 8- and 16-bit elements against up to 4096 columns: the ring skeleton on 64 x 128 tiles, K in enough slices
// for two workgroups per 64 columns and compute unit, reads long matrices at 5 to 7 TB/s where the tiles of the group body
// (whose estimate does not show it) keep to 2 to 3.5; with two more launches it pays from some length on.  Slices and all
// against the group body, bf16, us: matrices stored [k][o] 16 x 2048 x 8192 11.7 and 19.5, 64 x 2048 x 8192 15.0 and 20.3, 32 x 4096 x 8192
// 16.9 and 21.1, 32 x 4096 x 4096 12.6 and 11.7 (15.6 in slices of the group body, which 17 to 32 rows are cut into), 32 x 4096 x 25088 35.9 and 60.5, 32 x 1024 x 8192 11.6 and 8.9, 32 x 1024 x 18432 14.9
// and 17.3; stored [o][k] 64 x 4096 x 18432 32.1 and 39.8, 32 x 4096 x 18432 29.5 and 23.9, 64 x 4096 x 8192 19.6 and 18.7; e4m3
// stored [k][o] 32 x 4096 x 8192 12.4 and 18.1, 32 x 2048 x 8192 11.3 and 11.0.  More than 4096 columns: 32 x 8192 x 8192 63.8
// and 37.0.  With fewer than 128 workgroups (K is no multiple of enough slices) only 33 and more rows: 16 x 1024 x 25088 29.2 and
// 19.5, 64 x 1024 x 25088 31.4 and 44.2.
int ring_slices(DT dt, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc) {
  const int es = info(dt).size;
  const int64_t rows = std::min(M, N), cols = std::max(M, N);
  const bool rows_kc = M < N ? a_kc : b_kc, kc = M < N ? b_kc : a_kc;
  if (es > 2 || !rows_kc || rows < 9 || rows > 64 || cols > 4096) return 1;
  if (es == 1 ? kc || K < 8192 || cols < 3072 : kc ? rows <= 32 || K < 16384 || cols < 900 : K < (rows > 16 && rows <= 32 ? 4096 : 8192) || cols < (K < 16384 ? 1536 : 900)) return 1;
  const int64_t tiles = (cols + 63) / 64;
  int64_t S = 1;
  while (S < 256 && tiles * S < 512 && K / (2 * S) >= 512) S *= 2;
  while (S > 1 && K % (S * (128 / es))) S /= 2;
  if ((cols + 127) / 128 * S < (rows > 32 && !kc ? 64 : 128)) return 1;
  return choose_tiled(dt, DT::F32, 1, M, N, K, a_kc, b_kc, false, (int)S).skeleton == "rx_gemm_body_dl" ? (int)S : 1;
}

GemmChoice choose_gemm(DT a, DT b, DT out, int64_t batch, int64_t M, int64_t N, int64_t K, bool a_kc, bool b_kc, bool staged_only, int split, bool groups) {
  if (a != b) return GemmChoice();
  // a request for one of the other skeletons or for their tiles
  bool asked = false;
  for (const char* e : {"RX_GEMM_TILE", "RX_GEMM_BK", "RX_GEMM_STAGES", "RX_GEMM_DIRECT", "RX_GEMM_STREAM", "RX_GEMM_MFMA32", "RX_GEMM_TILE_F64"}) asked = asked || getenv(e);
  if (staged_only || !groups || asked) return choose_tiled(a, out, batch, M, N, K, a_kc, b_kc, staged_only, split);
  if (split > 1 && batch == 1 && split == ring_slices(a, M, N, K, a_kc, b_kc)) return choose_tiled(a, out, batch, M, N, K, a_kc, b_kc, staged_only, split);
  GemmChoice g = choose_group(a, out, batch, M, N, K, a_kc, b_kc, split);
  if (!g.ok || split > 1) return g.ok ? g : choose_tiled(a, out, batch, M, N, K, a_kc, b_kc, staged_only, split);
  const char* req = getenv("RX_GEMM_G");
  if (req && strcmp(req, "0") && g.ok) return g;
  GemmChoice c = choose_tiled(a, out, batch, M, N, K, a_kc, b_kc, staged_only, split);
  if (!c.ok) return g;
  auto rounds = [&](int64_t bm, int64_t bn) { return (double)((((M + bm - 1) / bm) * ((N + bn - 1) / bn) * batch + 255) / 256); };
  // Eight-wavefront tiles that fill the chip.  The streaming and ping-pong bodies keep the MFMA pipes busier than this
  // skeleton's loop where every round of tiles is full (bf16 4000 x 4096 x 1024 33 against 40 us, e4m3 8192 x 2048 x 5120 72
  // against 98), but a last round of few tiles costs them a whole one (bf16 2443 x 4096 x 4096, 320 tiles: 124 against 102
  // us).  Estimates: 1.33 us per K tile of 128 bytes of a 256 x 256 tile, 0.77 of a 256 x 128 tile, 10.5 and 9.5 us around them.
  // Contractions of fewer than 16 K tiles stay with them: their rounds overlap.
  if (c.skeleton == "rx_gemm_body_pp" || c.skeleton == "rx_gemm_body_s") {
    const double kt = (double)(K * info(a).size / 128);
    const bool sq = c.targs.find(", 256, 256, ") != std::string::npos;
    const double us = rounds(256, sq ? 256 : 128) * (sq ? kt * 1.33 + 10.5 : kt * 0.77 + 9.5) + 3.0;
    return kt >= 16 && g.est_us < us ? g : c;
  }
  // f32, an operand of at most 64 rows against 512 tiles and more (the features of a convolution and its window matrix)
  if (c.skeleton == "rx_gemm_body_dl" && a == DT::F32 && (M <= 64 || N <= 64) && ((M + 63) / 64) * ((N + 63) / 64) >= 1024) return c;
  return g;
}

std::string gemm_instance(const GemmChoice& c, const std::string& kbase, const std::string& epi_params, const std::string& epi_ctor, bool batched,
                          const GemmOperandFn& fa, const GemmOperandFn& fb) {
  std::ostringstream o;
  o << "// dot_general on MFMA: " << c.kind << " <" << c.targs << ">\n";
  const bool fn = !fa.type.empty() || !fb.type.empty();
  o << "extern \"C\" __global__ __launch_bounds__(" << c.block << (c.waves ? ", " + std::to_string(c.waves) : std::string()) << ") void " << kbase << "_gemm(";
  // operands that are read from memory come first, then what the operand functors read, then the epilogue's operands
  std::string params;
  if (fa.type.empty()) params += ", const " + c.stype_a + "* __restrict__ A";
  if (fb.type.empty()) params += ", const " + c.stype_a + "* __restrict__ B";
  params += fa.params + fb.params + epi_params;
  o << params.substr(2) << ") {\n";
  if (!fa.type.empty()) o << "  const " << c.stype_a << "* A = nullptr;\n  " << fa.ctor << "\n";
  if (!fb.type.empty()) o << "  const " << c.stype_a << "* B = nullptr;\n  " << fb.ctor << "\n";
  o << "  " << epi_ctor << "\n";
  o << "  " << c.skeleton << "<" << c.targs << ", " << (batched ? "true" : "false") << ", " << kbase << "_epi";
  if (fn) o << ", " << (fa.type.empty() ? "rx_no_fn" : fa.type) << ", " << (fb.type.empty() ? "rx_no_fn" : fb.type);
  if (c.split > 1) o << ", " << c.split;
  if (c.depth > 0) o << ", " << c.depth;
  if (c.stream_stages > 0) o << ", " << c.stream_stages;
  o << ">(A, B, epi";
  if (fn) o << ", " << (fa.type.empty() ? "rx_no_fn()" : "la") << ", " << (fb.type.empty() ? "rx_no_fn()" : "lb");
  o << ");\n}\n\n";
  return o.str();
}

// The matrix product on the window matrix: 70 TFLOP/s, a layout map of the result, three launches, and the window matrix
// written and read when there are more than 128 features.  Up to 128 it is evaluated while the tiles are loaded, 0.04 us per
// k whatever the number of pixels (28 x 28 images, 128 -> 128: 50 us for one and 48 for four; 14 x 14, 96 -> 96: 37)
static double conv_product_us(int64_t B, int64_t C, int64_t O, int64_t KH, int64_t KW, int64_t HO, int64_t WO) {
  const double flops = 2.0 * (double)B * (double)O * (double)HO * (double)WO * (double)C * (double)(KH * KW);
  const double window_bytes = O > 128 ? 2.0 * 4.0 * (double)B * (double)C * (double)(KH * KW) * (double)HO * (double)WO : 0.0;
  return std::max(flops / 70e6, O > 128 ? 0.0 : 0.04 * (double)(C * KH * KW)) + (window_bytes + 2.0 * 4.0 * (double)B * (double)O * (double)HO * (double)WO) / 5e6 + 5.0 + 8.0;
}

ConvChoice choose_conv(int64_t B, int64_t C, int64_t H, int64_t W, int64_t O, int64_t KH, int64_t KW, int64_t HO, int64_t WO, int64_t pl,
                       int64_t sh, int64_t sw, int64_t dh, int64_t dw) {
  ConvChoice c;
  if (getenv("RX_CONV_DIRECT") && atoi(getenv("RX_CONV_DIRECT")) == 0) return c;
  if (getenv("RX_MFMA") && atoi(getenv("RX_MFMA")) == 0) return c;
  if (B < 1 || C < 1 || O < 1 || HO < 1 || WO < 1 || KH < 1 || KW < 1) return c;
  // four wavefronts of 16 features each: with fewer than 33 features half of them would idle; a tile is whole rows of
  // the result, at most 25 blocks of 16 pixels (100 accumulator registers); taps unroll, so the filter is small
  if (O < 33 || WO > 400 || KH * KW > 49 || KH > H + 64 || KW > W + 64 || sh < 1 || sw < 1 || dh < 1 || dw < 1 || sh > 4 || sw > 4) return c;
  if (B * C * H * W >= ((int64_t)1 << 31) || B * O * HO * WO >= ((int64_t)1 << 31)) return c;
  const int64_t groups = (O + 63) / 64;
  const int slab = C >= 8 ? 8 : 4;
  const int64_t stages = (C + slab - 1) / slab > 1 ? 2 : 1;
  auto lds_of = [&](int64_t tr) {
    const int64_t pr = (tr - 1) * sh + (KH - 1) * dh + 1, off = (pl + 3) / 4 * 4, lastc = (WO - 1) * sw + (KW - 1) * dw - pl;
    const int64_t pw = (off + std::max<int64_t>(lastc + 1, W) + 3) / 4 * 4;
    const int64_t pch = (pr * pw + 47) / 64 * 64 + 16;
    return (stages * slab * pch + stages * KH * KW * (slab / 4) * 4 * 80) * 4;
  };
  // rows per workgroup: least padded work (ragged last tile, ragged last pixel block, workgroups in whole rounds of
  // the 256 compute units) among the tiles that fit
  double best = 0;
  for (int64_t tr = 1; tr <= HO && tr * WO <= 400; ++tr) {
    if (lds_of(tr) > 160 * 1024) break;
    const int64_t tiles = (HO + tr - 1) / tr, npb = (tr * WO + 15) / 16;
    const int64_t wgs = B * tiles * groups;
    const double rounds = (double)((wgs + 255) / 256);
    // time of the slowest compute unit: the MFMAs of its pixel blocks, the filter it reads once per tile (about one pixel block's worth) and the patch loads
    const double cost = rounds * ((double)npb + 1.0) * (1.0 + 0.02 * (double)((tr - 1) * sh + (KH - 1) * dh + 1) / (double)tr);
    if (c.rows == 0 || cost < best) { best = cost; c.rows = (int)tr; }
  }
  if (c.rows == 0) return c;
  if (const char* e = getenv("RX_CONV_ROWS")) {
    const int v = atoi(e);
    if (v >= 1 && v <= HO && (int64_t)v * WO <= 400 && lds_of(v) <= 160 * 1024) c.rows = v;
  }
  // Against the matrix product on the window matrix, whose tiles span images and which can slice the channels: a
  // workgroup of this kernel passes all channels of its 64 features through LDS for one tile of one image, about 1.5 us
  // per slab however few pixels the tile has.  Estimates in microseconds, fitted to 3 x 3 layers of 64 to 512 features
  // on 7 x 7 to 56 x 56 images in batches of 4 and 32 (512 -> 512 on 14 x 14, 4 images: 0.097 ms direct against 0.055;
  // 32 images of 256 -> 256: 0.086 against 0.103): slabs of max(1.5 us, 1.35 x their MFMA time) here, conv_product_us there.
  {
    const int64_t tiles = (HO + c.rows - 1) / c.rows, npb = (c.rows * WO + 15) / 16;
    const double rounds = (double)((B * tiles * groups + 255) / 256);
    const double nslab = (double)((C + slab - 1) / slab), nstep = (double)(KH * KW * (slab / 4));
    const double direct_us = rounds * nslab * std::max(1.5, 1.35 * (double)npb * nstep * 32.0 / 2200.0) + 5.0;
    const double product_us = conv_product_us(B, C, O, KH, KW, HO, WO);
    const char* force = getenv("RX_CONV_DIRECT");   // 2: this kernel wherever it covers the case
    c.us = direct_us;
    if (direct_us > product_us && !(force && atoi(force) == 2)) { c.rows = 0; return c; }
  }
  c.slab = slab;
  c.grid[0] = (unsigned)(B * ((HO + c.rows - 1) / c.rows));
  c.grid[1] = (unsigned)groups;
  c.lds_bytes = (unsigned)lds_of(c.rows);
  c.ok = true;
  return c;
}

ConvSplitChoice choose_conv_split(int64_t B, int64_t C, int64_t H, int64_t W, int64_t O, int64_t KH, int64_t KW, int64_t HO, int64_t WO,
                                  int64_t sh, int64_t sw, int64_t dh, int64_t dw) {
  ConvSplitChoice best;
  if (getenv("RX_MFMA") && atoi(getenv("RX_MFMA")) == 0) return best;
  const int64_t taps = KH * KW, ns = (C + 31) / 32, nob = (O + 127) / 128 * 8;
  // Fewer channels than a slab, or features than two wavefronts' of two groups, would be padding; more taps do not fit the
  // splitting kernel's LDS.
  if (B < 1 || HO < 1 || WO < 1 || C < 32 || O <= 64 || taps > 25 || sh < 1 || sw < 1 || dh < 1 || dw < 1 || sh > 4 || sw > 4) return best;
  if (C * H * W * 4 >= ((int64_t)1 << 31) || H * W >= ((int64_t)1 << 22) || B * O * HO * WO >= ((int64_t)1 << 31) || B * C * H * W >= ((int64_t)1 << 31) || ns * taps * nob * 3072 >= ((int64_t)1 << 31)) return best;
  for (int wf : {4, 2, 1})
    for (int kg : {1, 2, 4, 8}) {
      if (wf * kg != 4 && wf * kg != 8) continue;
      const int64_t fg = (O + 32 * wf - 1) / (32 * wf), nsg = (ns + kg - 1) / kg, nt = 64 * wf;
      for (int64_t parts = 1; parts <= (WO + 7) / 8; ++parts) {
        int64_t tc = (WO + parts - 1) / parts;
        if (WO % 4 == 0) tc = (tc + 3) / 4 * 4;
        for (int64_t tr = 1; tr <= HO && tr * tc <= 112; ++tr) {
          const int64_t npb = (tr * tc + 15) / 16;
          const int64_t pw = (tc - 1) * sw + (KW - 1) * dw + 1, npp = ((tr - 1) * sh + (KH - 1) * dh + 1) * pw;
          const int64_t ni = (npp * 4 + nt - 1) / nt;
          if (npb * 16 + ni * 8 > 160) break;   // registers: sums and the next slab's elements
          const int64_t lds = std::max(kg * npp * 208, kg > 1 ? wf * npb * 2 * kg * 1024 : (int64_t)0);
          if (lds > 160 * 1024 - 256) break;
          const int64_t wgs = B * ((HO + tr - 1) / tr) * ((WO + tc - 1) / tc) * fg;
          // Wavefronts that share a SIMD, rounds of workgroups, cycles of a slab: 12 MFMAs per tap and pixel block, and 300 to
          // stage 8 channels of 64 pixels, at the 1.75 GHz that are left while all matrix cores multiply; or the filter, which
          // every workgroup reads from L2, at 9 TB/s
          const bool pair = wf * kg == 4 && lds <= 80 * 1024 && wgs > 256;
          const double share = wf * kg == 8 || pair ? 2.0 : 1.1, rounds = (double)((wgs + (pair ? 511 : 255)) / (pair ? 512 : 256));
          const double body = rounds * (double)nsg * ((double)(taps * npb) * 192.0 + (double)ni * 300.0) * share / 1750.0;
          const double us = (std::max(body, (double)(wgs * 32 * wf * C * taps) * 6.0 / 9e6) + 8.0 * rounds) * (parts > 1 ? 1.03 : 1.0);
          if (!best.ok || us < best.us - 0.01) {
            best.ok = true;
            best.us = us;
            best.rows = (int)tr;
            best.cols = (int)tc;
            best.wf = wf;
            best.groups = kg;
            best.grid = (unsigned)wgs;
            best.block = (unsigned)(64 * wf * kg);
            best.lds_bytes = (unsigned)lds;
          }
        }
      }
    }
  // The filter: read once, written as 6 bytes an element, at 4 TB/s; the launch is shared by the filters of a module
  best.us += 4.0 + 10.0 * (double)(O * C * taps) / 4e6;
  best.filter_bytes = ns * taps * nob * 3072 + ns * nob * 8;
  best.filter_grid = (unsigned)(ns * nob);
  if (const char* e = getenv("RX_CONV_SPLIT_TILE")) {   // rows, columns, wavefronts of features, groups of channels
    int v[4];
    if (sscanf(e, "%d,%d,%d,%d", &v[0], &v[1], &v[2], &v[3]) == 4 && best.ok) {
      const int64_t pw = (v[1] - 1) * sw + (KW - 1) * dw + 1, npp = ((v[0] - 1) * sh + (KH - 1) * dh + 1) * pw, npb = (v[0] * v[1] + 15) / 16;
      const int64_t lds = std::max(v[3] * npp * 208, v[3] > 1 ? v[2] * npb * 2 * v[3] * 1024 : (int64_t)0);
      if (v[0] < 1 || v[1] < 1 || v[2] < 1 || v[3] < 1 || v[0] * v[1] > 112 || (v[2] * v[3] != 4 && v[2] * v[3] != 8) || lds > 160 * 1024 - 256) throw Error("RX_CONV_SPLIT_TILE cannot be honoured");
      best.rows = v[0]; best.cols = v[1]; best.wf = v[2]; best.groups = v[3];
      best.block = 64 * v[2] * v[3];
      best.lds_bytes = (unsigned)lds;
      best.grid = (unsigned)(B * ((HO + v[0] - 1) / v[0]) * ((WO + v[1] - 1) / v[1]) * ((O + 32 * v[2] - 1) / (32 * v[2])));
    }
  }
  return best;
}

bool conv_split_pays(int64_t B, int64_t C, int64_t H, int64_t W, int64_t O, int64_t KH, int64_t KW, int64_t HO, int64_t WO, int64_t pl, int64_t sh, int64_t sw, int64_t dh, int64_t dw,
                     bool alone) {
  if (getenv("RX_CONV_DIRECT") && atoi(getenv("RX_CONV_DIRECT")) == 0) return false;
  const char* force = getenv("RX_CONV_SPLIT");   // 0: never; 2: wherever the kernel covers the case
  if (force && atoi(force) == 0) return false;
  const ConvSplitChoice c = choose_conv_split(B, C, H, W, O, KH, KW, HO, WO, sh, sw, dh, dw);
  if (!c.ok) return false;
  if (force && atoi(force) == 2) return true;
  const ConvChoice d = choose_conv(B, C, H, W, O, KH, KW, HO, WO, pl, sh, sw, dh, dw);
  const double product = conv_product_us(B, C, O, KH, KW, HO, WO);
  // In us, kernels alone, f32 kernel or product -> this one with the splitting (7 to 15 by itself, 25 for all filters of
  // VGG-11): 8 images of 14 x 14, 512 -> 512: 112 -> 54 + 14; 4 of 28 x 28, 256 -> 256: 53 -> 29 + 11; 8 of 56 x 56, 64 -> 128:
  // 43 -> 23 + 9; 2 of 32 x 32, 64 -> 128: 11.3 -> 6.3 + 6.7; against the product: 4 of 14 x 14, 512 -> 512: 60 -> 34 + 15; one:
  // 21 -> 18 + 14; 8 x 8: 15 -> 14 + 13; 2 of 10 x 10, 160 -> 160: 15 -> 7 + 8.  The product's estimate is a quarter too high.
  double share = 1.0;
  if (alone) {
    // 126 convolutions alone in their modules, 1 to 16 images of 5 x 5 to 64 x 64, 32 to 512 channels: below these shares of the
    // estimates none took longer than before (0.14 to 1.00 of it), above them they took 0.7 to 1.5 of it.  The f32 kernel's
    // estimate is low where its last group of 64 features is not whole, and for 25 taps.  us per call, before -> split: 4 of
    // 41 x 36, 64 -> 192, stride 2: 12 -> 16; 4 of 18 x 44, 64 -> 384, 1 x 1: 6.7 -> 10; 16 of 50 x 27, 32 -> 128: 26 -> 30.
    const int64_t taps = KH * KW;
    if (d.ok) share = O % 64 != 0 || taps > 9 ? 1.0 : taps == 1 ? 0.7 : 0.82;
    else if (taps > 1) share = 0.68;
  }
  return c.us < share * (d.ok ? d.us : 0.8 * product);
}

}  // namespace rx
