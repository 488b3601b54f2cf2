// Float 3x3 convolutions and GEMMs on the bf16 matrix cores. Every float operand is split into three bf16 planes,
// x = h + m + l (each the rounding of what the planes before it leave: 24 significant bits, float's exponent range), and a
// product is taken as l h + m m + m h + h l + h m + h h with float accumulation. The terms left out (m l + l m + l l) are
// at most 2^-23 of the product, where a float product rounds by 2^-24: in sums of 32 terms and more the sums' rounding
// covers them (the error against 64 bits fell in every network measured); a sum that one product carries may be off by
// 1.0e-7 of it instead of 6e-8. Six v_mfma_f32_16x16x32_bf16 take 96 cycles where v_mfma_f32_16x16x4_f32 takes 256 for
// the same products, and the direct sum has neither the transforms' traffic of Winograd F(4x4,3x3) nor its loss of
// accuracy.
//
// A workgroup computes 16 MB pixels x 16 NB channels. Per chunk of 64 input channels it stages the pixel rows (tile and
// a halo of 20, as kgx_igemm.hip) in LDS as three planes, split in registers on the way, in two buffers with one
// barrier per chunk; all nine taps read them there. Four pairs of waves split the chunk's 18 (tap, 32-channel) steps:
// pair w takes steps w, w + 4, w + 8, w + 12 and half of the products of step 16 + w / 2, so a weight fragment is read
// by one pair, straight from memory into registers (packed in fragment order, one 1 KB load each, one step ahead), and
// never passes through LDS. The pairs' sums are added through LDS in order, which the tile's size does not change: a
// row's results do not depend on the batch.
//
// 192 -> 192 channels at 16 boards (96 x 48 tiles, 244 workgroups): 23.7-24.6 us, against 53 us of input transform, 36 point
// GEMMs and output transform (F(4x4,3x3)); 128 -> 128 at 8 boards (48 x 32): 9.3-9.6 against 37 us. The MFMAs are 12 us of
// the first; splitting the operands costs 2.5 us of VALU time, the first stage and the epilogue 4.
// An activation that is infinite, or rounds to infinity as a bf16 (from 3.3962e38), has no planes (inf - inf). A GEMM's
// sum that comes out infinite or NaN is therefore taken again on the float matrix unit (float_sums), which keeps the
// infinities and the top of the range; a 3x3 convolution gives NaN there, as the Winograd transforms do. Weights keep their
// value at the top of the range (their first plane is cut, not rounded, where it would overflow). Below 2^-103 (1e-31) the
// last planes fall under the smallest normal bf16, and an operand keeps fewer bits.
#include "kgx_gemm_epi.h"

#include <cfloat>
#include <climits>

namespace kgx {

namespace {

constexpr int PNT = 512, PCH = 64, PSTEPS = 18, PHALO = POS + 1;
constexpr int PFRAG = 64 * 8;  // elements of a packed weight fragment

// Row tile mt, column tile nt of workgroup g: the column tiles of a row tile on one XCD (workgroup g runs on XCD g mod 8),
// where they share its L2 for the rows.
__host__ __device__ inline void split_tile_of(int g, int ntl, int& mt, int& nt) {
  const int slot = g >> 3, u = slot / ntl;
  nt = slot - u * ntl;
  mt = u * 8 + (g & 7);
}
inline int split_grid(int M, int bm, int ntl) { return round_up((M + bm - 1) / bm, 8) * ntl; }
// The workgroups of the XCD that has most of them, the first: a round of the chip is 32 of these (one per CU), whatever the
// others have. (12 row tiles x 18 column tiles are 216 workgroups, under one round of 256 CUs, but 36 on XCD 0 to 3.)
inline long split_busiest(int M, int N, int bm, int bn) {
  return (long)(((M + bm - 1) / bm + 7) / 8) * ((N + bn - 1) / bn);
}

// x as three bf16 planes, eight values at a time (16 bytes per plane).
__device__ __forceinline__ void split3(const floatx4 (&x)[2], u32x4 (&p)[3]) {
  typedef float floatx2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int k = 0; k < 4; k++) {
    floatx2 v = {x[k >> 1][(k & 1) * 2], x[k >> 1][(k & 1) * 2 + 1]};
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
      p[q][k] = u;
      if (q < 2) {
        v[0] -= __builtin_bit_cast(float, u << 16);
        v[1] -= __builtin_bit_cast(float, u & 0xffff0000u);
      }
    }
  }
}

// The products of 16 rows with a packed 16-column block on v_mfma_f32_16x16x4_f32: ap this lane's row (lane % 16) of A at
// inputs 8 (lane / 16), wp its fragments of W, whose planes add up to the float weights. The steps' shares are summed as
// the wave pairs' are, so that a sum depends on its row and column alone. All lanes of the wave take part.
__device__ __forceinline__ floatx4 float_sums(const float* ap, const bf16* wp, int steps) {
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int w = 0; w < 4; w++) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = w; s < steps; s += 4) {
      const floatx4 a[2] = {*(const floatx4*)(ap + s * 32), *(const floatx4*)(ap + s * 32 + 4)};
      bf16x8 b[3];
#pragma unroll
      for (int q = 0; q < 3; q++) b[q] = *(const bf16x8*)(wp + ((size_t)s * 3 + q) * PFRAG);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float wt = (float)b[0][e] + ((float)b[1][e] + (float)b[2][e]);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e >> 2][e & 3], wt, acc, 0, 0, 0);
      }
    }
    sum += acc;
  }
  return sum;
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) <= FLT_MAX; }
// Whether any of v is infinite or NaN, for one compare a call: adds 0 or NaN to z.
__device__ __forceinline__ float add_zeros(float z, floatx4 v) {
#pragma unroll
  for (int k = 0; k < 4; k++) z = __builtin_fmaf(v[k], 0.f, z);
  return z;
}

template <int MB, int NB, int SC>
__global__ __launch_bounds__(PNT, 1) void conv3_split_kernel(const float* __restrict__ X, int ldx, int IC,
                                                             const bf16* __restrict__ W, int nch, int OC, int M, int ntl,
                                                             ConvOut o) {
  // Two waves per step share: over the rows, or over the columns of the tile that is too short for that.
  constexpr int WM = MB == 6 ? 2 : 1, WN = 2 / WM, WB = MB / WM, WC = NB / WN;
  constexpr int BM = 16 * MB, BN = 16 * NB, AR = BM + 2 * PHALO;
  constexpr int PLB = (AR + 1) * 128, BUF = 3 * PLB;  // bytes of a chunk's plane (its last row zero) and of a chunk
  constexpr int LDC = BN + 4, CB = 4 * BM * LDC * 4;
  __shared__ __align__(128) char smem[2 * BUF > CB ? 2 * BUF : CB];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wid & 3, wr = WM == 2 ? (wid >> 2) * WB * 16 : 0, wc = WN == 2 ? (wid >> 2) * WC : 0;  // steps, row, block
  const int r16 = lane & 15, g4 = lane >> 4;
  int mt, nt;
  split_tile_of(blockIdx.x, ntl, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  if (m0 >= M) return;

  // Staging: 8 channels of one row per task.
  constexpr int SV = (AR * 8 + PNT - 1) / PNT;
  floatx4 st[SV][2];
  auto load = [&](int kc) {
#pragma unroll
    for (int v = 0; v < SV; v++) {
      const int t = tid + PNT * v, row = t >> 3, c = kc * PCH + (t & 7) * 8, gr = m0 - PHALO + row;
      const bool ok = gr >= 0 && gr < M && c < IC;
      const float* p = X + (size_t)min(max(gr, 0), M - 1) * ldx + (c < IC ? c : 0);
      st[v][0] = *(const floatx4*)p;
      st[v][1] = *(const floatx4*)(p + 4);
      if (!ok) st[v][0] = st[v][1] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int v = 0; v < SV; v++) {
      const int t = tid + PNT * v, row = t >> 3;
      u32x4 p[3];
      // (Pinned here: hoisted to the loads, the split would wait for them.)
      asm volatile("" : "+v"(st[v][0]), "+v"(st[v][1]));
      split3(st[v], p);
      if (row < AR) {
        char* d = smem + buf * BUF + row * 128 + (((t & 7) ^ ((row >> 1) & 7)) * 16);
#pragma unroll
        for (int q = 0; q < 3; q++) *(u32x4*)(d + q * PLB) = p[q];
      }
    }
  };
  load(0);

  // Weight fragments (16-column block, chunk, step, plane); blocks past OC are packed as zeros.
  bf16x8 b0[WC][3], b1[WC][3];
  const bf16* const wb = W + (size_t)(nt * NB + wc) * nch * PSTEPS * 3 * PFRAG + lane * 8;
  auto load_b = [&](bf16x8 (&d)[WC][3], int kc, int s) {
#pragma unroll
    for (int j = 0; j < WC; j++)
#pragma unroll
      for (int q = 0; q < 3; q++) d[j][q] = *(const bf16x8*)(wb + (((size_t)j * nch + kc) * PSTEPS + s) * 3 * PFRAG + q * PFRAG);
  };
  load_b(b0, 0, wv);

  // Tap validity of this lane's pixels (bit t: the neighbour at tap t is on the board); others read the zero row.
  unsigned vmask[WB];
#pragma unroll
  for (int i = 0; i < WB; i++) {
    const int m = m0 + wr + i * 16 + r16;
    const int p = m % HW, y = p / POS, x = p - y * POS;
    unsigned bits = m < M ? 0x1ff : 0;
    if (y == 0) bits &= ~0x007u;
    if (y == POS - 1) bits &= ~0x1c0u;
    if (x == 0) bits &= ~0x049u;
    if (x == POS - 1) bits &= ~0x124u;
    vmask[i] = bits;
  }
  if (tid < 48) *(u32x4*)(smem + (tid >> 3) * PLB + AR * 128 + (tid & 7) * 16) = u32x4{0, 0, 0, 0};

  floatx4 acc[WB][WC];
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // The pixel fragments of step s (tap s / 2, channels 32 (s % 2) .. + 32): their addresses, then a plane at a time.
  bf16x8 a[WB][3];
  int aoff[WB];
  auto set_a = [&](int buf, int s) {
    const int t = s >> 1, kc = (s & 1) * 4 + g4, dy = t / 3, shift = (dy - 1) * POS + (t - 3 * dy - 1);
#pragma unroll
    for (int i = 0; i < WB; i++) {
      const int row = (vmask[i] >> t) & 1 ? wr + i * 16 + r16 + PHALO + shift : AR;
      aoff[i] = buf * BUF + row * 128 + ((kc ^ ((row >> 1) & 7)) * 16);
    }
  };
  auto load_a = [&](auto pl) {
    constexpr int q = decltype(pl)::value;
#pragma unroll
    for (int i = 0; i < WB; i++) a[i][q] = *(const bf16x8*)(smem + aoff[i] + q * PLB);
  };
  auto prod = [&](const bf16x8 (&d)[WC][3], auto pa, auto pb) {
#pragma unroll
    for (int i = 0; i < WB; i++)
#pragma unroll
      for (int j = 0; j < WC; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][decltype(pa)::value], d[j][decltype(pb)::value],
                                                            acc[i][j], 0, 0, 0);
  };
  typedef std::integral_constant<int, 0> H;
  typedef std::integral_constant<int, 1> Mi;
  typedef std::integral_constant<int, 2> L;

  // Rolled loops: straight-line code of all steps, each executed once, ran no faster than its instructions arrive in the
  // cold instruction cache (29 against 26 us). Two weight fragment sets take the steps in turn. A plane of the next
  // step's pixel fragments is read as soon as this step's products of it are issued.
  const int half = 16 + (wv >> 1);
  // One of the three thirds of a step's weight fragments (a plane).
  auto load_bp = [&](bf16x8 (&d)[WC][3], int kc, int s, auto pl) {
    constexpr int q = decltype(pl)::value;
#pragma unroll
    for (int j = 0; j < WC; j++) d[j][q] = *(const bf16x8*)(wb + (((size_t)j * nch + kc) * PSTEPS + s) * 3 * PFRAG + q * PFRAG);
  };
  // The scheduler's pattern of a phase: its LDS and memory reads spread between the MFMAs, which issue meanwhile.
  auto spread = [&](auto nm, auto nv) {
#pragma unroll
    for (int k = 0; k < decltype(nm)::value; k++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      if (k < WB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (k < WC) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, decltype(nv)::value, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // The step whose fragments are in d (its H plane of the pixels read here), loading step sn into dn and its pixels.
  auto step = [&](const bf16x8 (&d)[WC][3], bf16x8 (&dn)[WC][3], int kc, int buf, int sn) {
    __builtin_amdgcn_sched_barrier(0);
    load_a(H{});
    set_a(buf, sn);
    load_bp(dn, kc, sn, L{});
    prod(d, L{}, H{});
    spread(std::integral_constant<int, WB * WC / 2>{}, std::integral_constant<int, 8>{});
    load_a(L{});
    load_bp(dn, kc, sn, Mi{});
    prod(d, Mi{}, Mi{});
    prod(d, Mi{}, H{});
    spread(std::integral_constant<int, WB * WC>{}, std::integral_constant<int, 1>{});
    load_a(Mi{});
    load_bp(dn, kc, sn, H{});
    prod(d, H{}, L{});
    prod(d, H{}, Mi{});
    prod(d, H{}, H{});
    spread(std::integral_constant<int, WB * WC * 3 / 2>{}, std::integral_constant<int, 1>{});
  };
  store(0);
#pragma unroll 1
  for (int kc = 0; kc < nch; kc++) {
    const int buf = kc & 1;
    const bool more = kc + 1 < nch;
    lds_barrier();
    if (more) load(kc + 1);
    set_a(buf, wv);
    load_a(L{});
    load_a(Mi{});
#pragma unroll 1
    for (int j = 0; j < 4; j += 2) {
      step(b0, b1, kc, buf, wv + 4 * j + 4);
      step(b1, b0, kc, buf, j == 0 ? wv + 8 : half);
      // The next chunk's planes, at different times in the two waves of a SIMD, so that one's VALU work runs beside
      // the other's MFMAs.
      if (more && (j == 0) == (wid >= 4)) store(buf ^ 1);
    }
    if (wv & 1) {
      prod(b0, L{}, H{});
      prod(b0, Mi{}, Mi{});
      prod(b0, Mi{}, H{});
    } else {
      load_a(H{});
      prod(b0, H{}, L{});
      prod(b0, H{}, Mi{});
      prod(b0, H{}, H{});
    }
    if (more) load_b(b0, kc + 1, wv);
  }
  // The epilogue's inputs, in flight during the exchange of the sums.
  constexpr int G4 = BN / 4, RPE = PNT / G4, EV = (BM + RPE - 1) / RPE;
  const int ec4 = tid % G4, er0 = tid / G4, en = n0 + 4 * ec4, enc = min(en, OC - 4);
  const bool eon = er0 < RPE && en < OC;
  auto epix = [&](int e) { return min(m0 + min(er0 + e * RPE, BM - 1), M - 1); };
  floatx4 yres[EV], es, eb;
  float mkv[EV], rmv[EV];
  if (o.y && o.accumulate) {
#pragma unroll
    for (int e = 0; e < EV; e++) yres[e] = *(const floatx4*)(o.y + (size_t)epix(e) * o.ldy + enc);
  }
  if (o.emit.scale) {
    es = *(const floatx4*)(o.emit.scale + enc);
    eb = *(const floatx4*)(o.emit.bias + enc);
#pragma unroll
    for (int e = 0; e < EV; e++) mkv[e] = o.emit.mask[epix(e)];
  }
  if (o.rowmask) {
#pragma unroll
    for (int e = 0; e < EV; e++) rmv[e] = o.rowmask[epix(e)];
  }
  lds_barrier();  // every wave is done reading the chunks

  float* const Cs = (float*)smem;
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) Cs[(wv * BM + wr + i * 16 + 4 * g4 + r) * LDC + (wc + j) * 16 + r16] = acc[i][j][r];
  lds_barrier();
#pragma unroll
  for (int e = 0; e < EV; e++) {
    const int row = er0 + e * RPE, m = m0 + row;
    if (eon && row < BM && m < M) {
      floatx4 sum = *(const floatx4*)(Cs + row * LDC + 4 * ec4);
#pragma unroll
      for (int q = 1; q < 4; q++) sum += *(const floatx4*)(Cs + (q * BM + row) * LDC + 4 * ec4);
      conv_store4<float, SC >= 0 ? ((SC & SF_EMIT) ? ACT_MISH : ACT_ID) : -1, SC>(o, m, en, sum, yres[e], rmv[e], es, eb,
                                                                                  mkv[e]);
    }
  }
}

// C[M][N] = A[M][K] Bt[N][K]^T with float A split in registers and Bt packed as three planes (fragments [16-column block]
// [32-channel step][plane]). A workgroup computes 16 MB rows x 64 columns; its four pairs of waves split the K steps
// (pair w takes w, w + 4, ...), each reading its own fragments of both operands straight from memory, one step ahead:
// no operand passes through LDS and no barrier stands in the loop, so a product of few tiles (where the latency of
// its serial K loop sets the time) runs a quarter of the steps one after the other. The pairs' sums are added in
// order, whatever the tile. The waves of a pair split the rows (MB = 6) or the columns (MB = 2).
// Against the float matrix unit's 64 x 64 tiles (one 16-channel stage after the other): N = 384 over K = 384 and 1536 at
// 1083 rows 33.0 -> 12.8 us on average; N = 512 over K = 512 and 2048 at 3610 rows 64.2 -> 52.9 on average (80.0 for K = 2048
// here, 25.9 for K = 512 in gemm_split_lds_kernel). Where the rounds are many, both operands' reads from L2 bound it (about
// 64 bytes a cycle and CU): gemm_split_lds_kernel takes those.
template <int MB, int EPI>
__global__ __launch_bounds__(PNT, MB == 2 ? 4 : 2) void gemm_split_kernel(const float* __restrict__ A, const bf16* __restrict__ W, int lda,
                                                            int M, int N, int K, int ntl, GemmArgs g) {
  constexpr int BM = 16 * MB, BN = 64, NB = 4;
  constexpr int WM = MB == 6 ? 2 : 1, WN = 2 / WM, WB = MB / WM, WC = NB / WN;
  constexpr int ELD = BN + 4;
  __shared__ __align__(128) float smem[4 * BM * ELD];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wid & 3, wr = WM == 2 ? (wid >> 2) * WB * 16 : 0, wc = WN == 2 ? (wid >> 2) * WC : 0;
  const int r16 = lane & 15, g4 = lane >> 4;
  int mt, nt;
  split_tile_of(blockIdx.x, ntl, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  if (m0 >= M) return;

  const int steps = K / 32;
  const float* ap[WB];  // this lane's row of each block (rows past M read the last one, never stored)
#pragma unroll
  for (int i = 0; i < WB; i++) ap[i] = A + (size_t)min(m0 + wr + i * 16 + r16, M - 1) * lda + g4 * 8;
  const bf16* const wb = W + (size_t)(nt * NB + wc) * steps * 3 * PFRAG + lane * 8;
  floatx4 raw[WB][2];
  bf16x8 a[WB][3], b0[WC][3], b1[WC][3];
  auto load_a = [&](int s) {
#pragma unroll
    for (int i = 0; i < WB; i++) {
      raw[i][0] = *(const floatx4*)(ap[i] + s * 32);
      raw[i][1] = *(const floatx4*)(ap[i] + s * 32 + 4);
    }
  };
  auto load_b = [&](bf16x8 (&d)[WC][3], int s) {
#pragma unroll
    for (int j = 0; j < WC; j++)
#pragma unroll
      for (int q = 0; q < 3; q++) d[j][q] = *(const bf16x8*)(wb + (((size_t)j * steps + s) * 3 + q) * PFRAG);
  };
  floatx4 acc[WB][WC];
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto prod = [&](const bf16x8 (&d)[WC][3], auto pa, auto pb) {
#pragma unroll
    for (int i = 0; i < WB; i++)
#pragma unroll
      for (int j = 0; j < WC; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][decltype(pa)::value], d[j][decltype(pb)::value],
                                                            acc[i][j], 0, 0, 0);
  };
  typedef std::integral_constant<int, 0> H;
  typedef std::integral_constant<int, 1> Mi;
  typedef std::integral_constant<int, 2> L;
  auto step = [&](const bf16x8 (&d)[WC][3], bf16x8 (&dn)[WC][3], int s) {
#pragma unroll
    for (int i = 0; i < WB; i++) {
      u32x4 p[3];
      split3(raw[i], p);
#pragma unroll
      for (int q = 0; q < 3; q++) a[i][q] = __builtin_bit_cast(bf16x8, p[q]);
    }
    const int sn = min(s + 4, steps - 1);
    load_a(sn);
    load_b(dn, sn);
    __builtin_amdgcn_sched_barrier(0);
    prod(d, L{}, H{});
    prod(d, Mi{}, Mi{});
    prod(d, Mi{}, H{});
    prod(d, H{}, L{});
    prod(d, H{}, Mi{});
    prod(d, H{}, H{});
  };
  load_a(min(wv, steps - 1));
  load_b(b0, min(wv, steps - 1));
#pragma unroll 1
  for (int s = wv; s < steps; s += 8) {
    step(b0, b1, s);
    if (s + 4 < steps) step(b1, b0, s + 4);
  }

  // The inputs of the epilogues that read memory, in flight during the exchange of the sums: thread tid finishes
  // columns 4 (tid % 16) .. + 3 of rows tid / 16 + 32 v (clamped indices; the stores skip what lies outside).
  constexpr int EV = BM * 16 / PNT;
  constexpr bool OWN = EPI == EPI_GEN || EPI == EPI_ACC;
  const ConvOut& o = g.out;
  const int en = n0 + (tid & 15) * 4, enc = min(en, N - 4);
  floatx4 yres[EV], es = {1.f, 1.f, 1.f, 1.f}, eb = {0.f, 0.f, 0.f, 0.f};
  float rmv[EV], mkv[EV];
  if constexpr (OWN) {
    if (EPI == EPI_GEN && o.emit.scale) {
      es = *(const floatx4*)(o.emit.scale + enc);
      eb = *(const floatx4*)(o.emit.bias + enc);
    }
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int m = min(m0 + (tid >> 4) + 32 * v, M - 1);
      yres[v] = o.y && o.accumulate ? *(const floatx4*)(o.y + (size_t)m * o.ldy + enc) : floatx4{0.f, 0.f, 0.f, 0.f};
      rmv[v] = o.rowmask ? o.rowmask[m] : 1.f;
      mkv[v] = EPI == EPI_GEN && o.emit.scale ? o.emit.mask[m] : 1.f;
    }
  }
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        smem[(wv * BM + wr + i * 16 + 4 * g4 + r) * ELD + (wc + j) * 16 + r16] = acc[i][j][r];
  lds_barrier();
#pragma unroll
  for (int v = 0; v < EV; v++) {
    const int e = tid + PNT * v, m = m0 + (e >> 4);
    float* p = smem + (e >> 4) * ELD + (e & 15) * 4;
    floatx4 sum = *(const floatx4*)p;
#pragma unroll
    for (int q = 1; q < 4; q++) sum += *(const floatx4*)(p + q * BM * ELD);
    if (__builtin_expect(__any(!(add_zeros(0.f, sum) == 0.f)), 0)) {
      // The wave's four rows and 64 columns: operand row i is row i / 4 of them, and product q takes columns 4 l + q, so
      // that lane (g4, l) gets column 4 l + q of row g4 as its first output.
      const float* xp = A + (size_t)min(m0 + wid * 4 + 32 * v + (r16 >> 2), M - 1) * lda + g4 * 8;
      const bf16* xw = W + (size_t)(nt * NB + (r16 >> 2)) * steps * 3 * PFRAG + (g4 * 16 + (r16 & 3) * 4) * 8;
#pragma unroll 1
      for (int q = 0; q < 4; q++) {
        const float t = float_sums(xp, xw + q * 8, steps)[0];
#pragma unroll
        for (int k = 0; k < 4; k++)
          if (k == q && !finite(sum[k])) sum[k] = t;
      }
    }
    if constexpr (!OWN) {
      *(floatx4*)p = sum;
    } else if (m < M && en < N) {
      if constexpr (EPI == EPI_ACC) *(floatx4*)(o.y + (size_t)m * o.ldy + en) = sum * rmv[v] + yres[v];
      else conv_store4<float>(o, m, en, sum, yres[v], rmv[v], es, eb, mkv[v]);
    }
  }
  if constexpr (!OWN) {
    lds_barrier();
    gemm_tile_epilogue<float, EPI, BM, BN, PNT>(smem, g, o, m0, n0, M, N, tid);
  }
}

// The same product on 128 x 128 tiles with both operands' planes in LDS, for grids that fill the chip: eight waves of
// 64 x 32 share each 32-channel step's fragments (A split on its way, one task of 8 channels per thread; the packed
// weights straight into LDS), double-buffered with one barrier per step, so an operand byte read from L2 feeds twice to
// four times the MFMAs. The steps run in the order of the wave pairs' shares (0, 4, 8, ..., 1, 5, ...) and each
// share's sum is added to the total when it ends: the sums of gemm_split_kernel, in its order. The next step's A values
// were loaded a whole step before they are split, between this step's products. 3610 rows x 4096 columns over K = 512:
// 140 -> 99 us against the 96 x 64 tile (149 on the float matrix unit), 1536 columns 59 -> 51; bound by the barrier per
// step (the MFMAs are 40 us of the 99).
template <int EPI>
__global__ __launch_bounds__(PNT, 2) void gemm_split_lds_kernel(const float* __restrict__ A, const bf16* __restrict__ W,
                                                                int lda, int M, int N, int K, int ntl, GemmArgs g) {
  constexpr int BM = 128, BN = 128, WB = 4, WC = 2, ELD = BN + 4;
  constexpr int AB = BM / 16 * 3 * 1024, BUF = AB + BN / 16 * 3 * 1024;  // bytes of a step's A planes, of a step
  static_assert(BM * ELD * 4 <= 2 * BUF, "the float tile reuses the steps");
  __shared__ __align__(1024) char smem[2 * BUF];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid >> 2, wn = wid & 3, r16 = lane & 15, g4 = lane >> 4;
  int mt, nt;
  split_tile_of(blockIdx.x, ntl, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  if (m0 >= M) return;

  const int steps = K / 32;
  // Staging of A: thread tid takes channels 8 (tid % 4) .. + 7 of row tid / 4 (rows past M read the last one) into
  // fragment order: [16-row block][plane][lane][16 bytes].
  const int srow = tid >> 2, sch = tid & 3;
  const float* const ap = A + (size_t)min(m0 + srow, M - 1) * lda + sch * 8;
  char* const ad = smem + (srow >> 4) * 3072 + (sch * 16 + (srow & 15)) * 16;
  floatx4 raw[2], nxt[2];  // the next step's values, and the ones after
  auto load_a = [&](floatx4 (&d)[2], int s) {
    d[0] = *(const floatx4*)(ap + s * 32);
    d[1] = *(const floatx4*)(ap + s * 32 + 4);
  };
  auto store_a = [&](int buf) {
    u32x4 p[3];
    asm volatile("" : "+v"(raw[0]), "+v"(raw[1]));  // (split here, not where the values arrive)
    split3(raw, p);
#pragma unroll
    for (int q = 0; q < 3; q++) *(u32x4*)(ad + buf * BUF + q * 1024) = p[q];
  };
  // Wave wid's column block of the packed weights (blocks past the packed ones lie outside the range and read as zero).
  const int cb = n0 / 16 + wid, wbytes = (N + 63) / 64 * 4 * steps * 3 * 1024;
  auto dma_b = [&](int buf, int s) {
#pragma unroll
    for (int q = 0; q < 3; q++)
      lds_load16(W, wbytes, smem + buf * BUF + AB + (wid * 3 + q) * 1024, ((cb * steps + s) * 3 + q) * 1024 + lane * 16);
  };
  floatx4 acc[WB][WC], tot[WB][WC];
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++) acc[i][j] = tot[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto after = [&](int s) { return s + 4 < steps ? s + 4 : (s & 3) + 1; };  // the step after s (4: past the last)

  load_a(raw, 0);
  dma_b(0, 0);
  store_a(0);
  int s1 = after(0);
  load_a(raw, s1);  // (at least four steps: the launch)
#pragma unroll 1
  for (int t = 0, s = 0; t < steps; t++, s = s1, s1 = after(s1)) {
    const int buf = t & 1;
    // (The direct loads are not counted by the compiler.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + 1 < steps) {
      dma_b(buf ^ 1, s1);
      load_a(nxt, t + 2 < steps ? after(s1) : s1);
    }
    bf16x8 a[WB][3], b[WC][3];
    const char* const as = smem + buf * BUF + wm * WB * 3072 + lane * 16;
    const char* const bs = smem + buf * BUF + AB + wn * WC * 3072 + lane * 16;
#pragma unroll
    for (int q = 2; q >= 0; q--) {
#pragma unroll
      for (int i = 0; i < WB; i++) a[i][q] = *(const bf16x8*)(as + i * 3072 + q * 1024);
#pragma unroll
      for (int j = 0; j < WC; j++) b[j][2 - q] = *(const bf16x8*)(bs + j * 3072 + (2 - q) * 1024);
    }
    auto prod = [&](int pa, int pb) {
#pragma unroll
      for (int i = 0; i < WB; i++)
#pragma unroll
        for (int j = 0; j < WC; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa], b[j][pb], acc[i][j], 0, 0, 0);
    };
    prod(2, 0);
    prod(1, 1);
    prod(1, 0);
    if (t + 1 < steps) {
      store_a(buf ^ 1);
      raw[0] = nxt[0];
      raw[1] = nxt[1];
    }
    prod(0, 2);
    prod(0, 1);
    prod(0, 0);
    if (s + 4 >= steps) {  // the share's last step
#pragma unroll
      for (int i = 0; i < WB; i++)
#pragma unroll
        for (int j = 0; j < WC; j++) {
          tot[i][j] += acc[i][j];
          acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }

  constexpr int EV = BM * (BN / 4) / PNT;
  constexpr bool OWN = EPI == EPI_GEN || EPI == EPI_ACC;
  const ConvOut& o = g.out;
  const int en = n0 + (tid & 31) * 4, enc = min(en, N - 4);
  floatx4 yres[EV], es = {1.f, 1.f, 1.f, 1.f}, eb = {0.f, 0.f, 0.f, 0.f};
  float rmv[EV], mkv[EV];
  if constexpr (OWN) {  // (as gemm_split_kernel's)
    if (EPI == EPI_GEN && o.emit.scale) {
      es = *(const floatx4*)(o.emit.scale + enc);
      eb = *(const floatx4*)(o.emit.bias + enc);
    }
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int m = min(m0 + (tid >> 5) + 16 * v, M - 1);
      yres[v] = o.y && o.accumulate ? *(const floatx4*)(o.y + (size_t)m * o.ldy + enc) : floatx4{0.f, 0.f, 0.f, 0.f};
      rmv[v] = o.rowmask ? o.rowmask[m] : 1.f;
      mkv[v] = EPI == EPI_GEN && o.emit.scale ? o.emit.mask[m] : 1.f;
    }
  }
  lds_barrier();  // every wave is done reading the steps
  float* const Et = (float*)smem;
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        Et[((wm * WB + i) * 16 + 4 * g4 + r) * ELD + (wn * WC + j) * 16 + r16] = tot[i][j][r];
  floatx4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WC; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) z[r] = __builtin_fmaf(tot[i][j][r], 0.f, z[r]);
  if (__builtin_expect(__any(!(add_zeros(0.f, z) == 0.f)), 0)) {
#pragma unroll 1
    for (int b = 0; b < WB * WC; b++) {
      const int row = (wm * WB + b / WC) * 16, col = (wn * WC + b % WC) * 16;
      if (n0 + col >= N) continue;
      const floatx4 t = float_sums(A + (size_t)min(m0 + row + r16, M - 1) * lda + g4 * 8,
                                   W + (size_t)((n0 + col) / 16) * steps * 3 * PFRAG + lane * 8, steps);
      for (int r = 0; r < 4; r++) {
        float* p = Et + (row + 4 * g4 + r) * ELD + col + r16;
        if (!finite(*p)) *p = t[r];
      }
    }
  }
  lds_barrier();
  if constexpr (!OWN) {
    gemm_tile_epilogue<float, EPI, BM, BN, PNT>(Et, g, o, m0, n0, M, N, tid);
  } else {
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int row = (tid >> 5) + 16 * v, m = m0 + row;
      if (m < M && en < N) {
        const floatx4 sum = *(const floatx4*)(Et + row * ELD + (tid & 31) * 4);
        if constexpr (EPI == EPI_ACC) *(floatx4*)(o.y + (size_t)m * o.ldy + en) = sum * rmv[v] + yres[v];
        else conv_store4<float>(o, m, en, sum, yres[v], rmv[v], es, eb, mkv[v]);
      }
    }
  }
}

// The three planes of a weight (round to nearest even, but cut where that would be infinite: the next planes hold the rest;
// an infinity is its first plane alone).
__device__ __forceinline__ void split_weight(float v, unsigned short (&p)[3]) {
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const unsigned u = __builtin_bit_cast(unsigned, v), r = u + 0x7fffu + ((u >> 16) & 1u);
    const unsigned h = ((r & 0x7f800000u) == 0x7f800000u ? u : r) & 0xffff0000u;
    p[q] = (unsigned short)(h >> 16);
    v = (u & 0x7fffffffu) == 0x7f800000u ? 0.f : v - __builtin_bit_cast(float, h);
  }
}

// Packs the weights as the kernels read them, eight elements of the three planes per thread, `frags` fragment triples (64
// threads each). GEMM (CONV false): w [N][K] -> [16-column block][step][plane], lane l, element e holding column l % 16,
// input 32 step + 8 (l / 16) + e. Convolution: w [N][K][3][3] -> [16-column block][chunk][step][plane], input channel 64
// chunk + 32 (step % 2) + 8 (l / 16) + e at tap step / 2. Zeros past N and K. On the device: a handle of b10c384h6 took 41 ms to
// create with this on the host, 26 ms with it here; one of b18c384nbt 112 and 19 ms.
template <bool CONV>
__global__ __launch_bounds__(256) void split_pack_kernel(const float* __restrict__ w, int N, int K, int steps, long frags,
                                                         u32x4* __restrict__ out) {
  const long f = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (f >= frags) return;
  const int lane = threadIdx.x & 63;
  const long cb = f / steps;
  const int s = (int)(f - cb * steps), st = CONV ? s % PSTEPS : 0;  // convolution: step s is chunk s / 18, step s % 18
  const long col = cb * 16 + (lane & 15);
  const int k0 = (CONV ? s / PSTEPS * PCH + (st & 1) * 32 : s * 32) + (lane >> 4) * 8;
  unsigned short p[8][3];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const bool on = col < N && k0 + e < K;
    split_weight(on ? w[CONV ? ((size_t)col * K + k0 + e) * 9 + st / 2 : (size_t)col * K + k0 + e] : 0.f, p[e]);
  }
#pragma unroll
  for (int q = 0; q < 3; q++) {
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = p[2 * k][q] | (unsigned)p[2 * k + 1][q] << 16;
    out[(f * 3 + q) * 64 + lane] = v;
  }
}

}  // namespace

// Convolution weights are packed up to a multiple of 192 columns, so that every tile width reads whole blocks.
static long conv_split_steps(int ic) { return (long)((ic + PCH - 1) / PCH) * PSTEPS; }
static long conv_split_frags(int oc, int ic) { return round_up(oc, 192) / 16 * conv_split_steps(ic); }
static long gemm_split_frags(int N, int K) { return (long)round_up(N, 64) / 16 * (K / 32); }

size_t conv_split_bytes(int oc, int ic) { return conv_split_frags(oc, ic) * 3 * PFRAG * sizeof(bf16); }
size_t gemm_split_bytes(int N, int K) { return gemm_split_frags(N, K) * 3 * PFRAG * sizeof(bf16); }

void launch_conv_split_pack(const float* w, int oc, int ic, void* out, hipStream_t s) {
  const long n = conv_split_frags(oc, ic);
  launch_k(split_pack_kernel<true>, (unsigned)((n + 3) / 4), 256, 0, s, w, oc, ic, (int)conv_split_steps(ic), n, (u32x4*)out);
  KGX_CHECK_LAUNCH();
}

void launch_gemm_split_pack(const float* w, int N, int K, void* out, hipStream_t s) {
  const long n = gemm_split_frags(N, K);
  launch_k(split_pack_kernel<false>, (unsigned)((n + 3) / 4), 256, 0, s, w, N, K, K / 32, n, (u32x4*)out);
  KGX_CHECK_LAUNCH();
}

template <int MB, int NB>
static void split_launch(const float* x, int ldx, int IC, const bf16* w, int OC, const ConvOut& o, int M, hipStream_t s) {
  const int ntl = (OC + 16 * NB - 1) / (16 * NB), nch = (IC + PCH - 1) / PCH, grid = split_grid(M, 16 * MB, ntl);
  auto go = [&](auto kernel) { launch_k(kernel, grid, PNT, 0, s, x, ldx, IC, w, nch, OC, M, ntl, o); };
  const int sfl = store_flags(o);
  switch ((sfl & SF_EMIT) && o.emit.act != ACT_MISH ? -1 : sfl) {  // the store cases of igemm_launch
    case SF_EMIT: go(conv3_split_kernel<MB, NB, SF_EMIT>); return;
    case SF_Y: go(conv3_split_kernel<MB, NB, SF_Y>); return;
    case SF_Y | SF_ACC | SF_EMIT: go(conv3_split_kernel<MB, NB, SF_Y | SF_ACC | SF_EMIT>); return;
    case SF_Y | SF_ACC | SF_YDEAD | SF_EMIT: go(conv3_split_kernel<MB, NB, SF_Y | SF_ACC | SF_YDEAD | SF_EMIT>); return;
    default: go(conv3_split_kernel<MB, NB, -1>);
  }
}

// The tile (16 mb pixels x 16 nb channels) whose rounds (of one workgroup per CU: up to 105 KB of LDS) cost least, a round
// taking time in proportion to the tile's 16 x 16 blocks and a fixed part (staging, epilogue) of about six blocks'
// (measured at 192 input channels: 11.3, 23.5 and 30 us for 6, 18 and 24 blocks).
static const int (&conv_split_tile(int M, int OC))[2] {
  static const int tiles[4][2] = {{6, 4}, {6, 3}, {6, 2}, {3, 2}};
  int best = 0;
  long cost = 0;
  for (int k = 0; k < 4; k++) {
    const int mb = tiles[k][0], nb = tiles[k][1];
    const long c = (split_busiest(M, OC, 16 * mb, 16 * nb) + 31) / 32 * (mb * nb + 6);
    if (k == 0 || c < cost) best = k, cost = c;
  }
  return tiles[best];
}

void launch_conv_split(const float* x, int ldx, int IC, const void* w, int OC, const ConvOut& o, int B, hipStream_t s) {
  if (IC % 8 || ldx % 4 || OC % 4 || (o.y && o.ldy % 4) || (o.yt && o.ldyt % 4) || (o.colbias && o.ld_colbias % 4) ||
      (o.emit.scale && o.emit.ld % 4) || ((uintptr_t)x | (uintptr_t)w) % 16 || o.pool.psum)
    throw std::runtime_error("conv_split: channel counts must be multiples of 8 (inputs) and 4 (outputs)");
  const int M = B * HW;
  if (M <= 0) return;
  const bf16* wp = (const bf16*)w;
  const int(&t)[2] = conv_split_tile(M, OC);
  if (t[0] == 3) split_launch<3, 2>(x, ldx, IC, wp, OC, o, M, s);
  else if (t[1] == 2) split_launch<6, 2>(x, ldx, IC, wp, OC, o, M, s);
  else if (t[1] == 3) split_launch<6, 3>(x, ldx, IC, wp, OC, o, M, s);
  else split_launch<6, 4>(x, ldx, IC, wp, OC, o, M, s);
  KGX_CHECK_LAUNCH();
}

bool gemm_split_fits(int N, int K, int dq) { return K % 32 == 0 && N % 4 == 0 && (dq == 0 || 64 % dq == 0); }

// The row tile (32 x 64, 96 x 64 or, with at least four steps, 128 x 128 in LDS) whose rounds take least, by times in
// us of a round of one workgroup per CU of the busiest XCD (two of the 32-row tile) fitted to kernel traces: 96 x 64 over 12
// steps 12.5-12.9 in one round, 21.2 in two, 42.1 in four, over 48 steps 59 in two; 128 x 128 over 12 steps 20.1-20.8 in
// one and 39.6-41.5 in two, over 48 steps 64 in one, over 16 steps 99 in four; 32 x 64 over 12 and 48 steps 7.5 and 19
// at one workgroup per CU, over 12 steps 12.2 at two, over 16 and 64 steps 59 on average in two rounds of two. Counted over
// the whole chip instead (12 x 18 tiles of 96 x 64 are under 256 workgroups, but 36 on four XCDs) the q|k|v projection of 3
// rows of b10c384h6 ran on 96 rows in 22.0 us, where 128 takes 20.8.
int gemm_split_rows(int M, int N, int K) {
  const int steps = K / 32;
  const long w32 = split_busiest(M, N, 32, 64), w96 = split_busiest(M, N, 96, 64), w128 = split_busiest(M, N, 128, 128);
  const double t32 = w32 <= 32 ? 0.26 * steps + 5 : (w32 + 63) / 64 * (0.65 * steps + 5);
  const double t96 = (w96 + 31) / 32 * (0.55 * steps + 4) + 2, t128 = (w128 + 31) / 32 * (1.22 * steps + 5.5);
  // (Its weights' offsets are 32-bit.)
  if (steps >= 4 && t128 < t96 && t128 < t32 && 6.0 * (N + 64) * K < INT_MAX) return 128;
  return t96 <= t32 ? 96 : 32;
}

LaunchGeometry split_geometry(int ks, int M, int N, int K, int g, int& row_tile, int& col_tile) {
  LaunchGeometry r;
  if (ks == 3) {
    const int(&t)[2] = conv_split_tile(M, N);
    r.tile_rows = 16 * t[0];
    r.tile_cols = 16 * t[1];
  } else {
    r.tile_rows = gemm_split_rows(M, N, K);
    r.tile_cols = r.tile_rows == 128 ? 128 : 64;
  }
  const int ntl = (N + r.tile_cols - 1) / r.tile_cols;
  r.grid = split_grid(M, r.tile_rows, ntl);
  split_tile_of(g, ntl, row_tile, col_tile);
  if ((long)row_tile * r.tile_rows >= M) row_tile = col_tile = -1;
  return r;
}

template <int MB, int EPI>
static auto gemm_split_pick() {
  if constexpr (MB == 8) return gemm_split_lds_kernel<EPI>;
  else return gemm_split_kernel<MB, EPI>;
}

template <int MB>
static void gemm_split_launch(const GemmArgs& g, int epi, hipStream_t s) {
  constexpr int BN = MB == 8 ? 128 : 64;
  const int ntl = (g.N + BN - 1) / BN, grid = split_grid(g.M, 16 * MB, ntl);
  auto go = [&](auto kernel) {
    launch_k(kernel, grid, PNT, 0, s, (const float*)g.A, (const bf16*)g.Bt, (int)g.lda, g.M, g.N, g.K, ntl, g);
  };
  switch (epi) {
    case EPI_YT: go(gemm_split_pick<MB, EPI_YT>()); break;
    case EPI_ACC: go(gemm_split_pick<MB, EPI_ACC>()); break;
    case EPI_GLU: go(gemm_split_pick<MB, EPI_GLU>()); break;
    case EPI_QKV: go(gemm_split_pick<MB, EPI_QKV>()); break;
    case EPI_YTMISH: go(gemm_split_pick<MB, EPI_YTMISH>()); break;
    default: go(gemm_split_pick<MB, EPI_GEN>());
  }
}

void launch_gemm_split(const GemmArgs& g, int epi, hipStream_t s) {
  if (!gemm_split_fits(g.N, g.K, g.qkv.dq) || g.lda % 4 || g.lda > INT_MAX || ((uintptr_t)g.A | (uintptr_t)g.Bt) % 16)
    throw std::runtime_error("gemm: shape or alignment does not fit the three-plane product");
  switch (gemm_split_rows(g.M, g.N, g.K)) {
    case 128: gemm_split_launch<8>(g, epi, s); break;
    case 96: gemm_split_launch<6>(g, epi, s); break;
    default: gemm_split_launch<2>(g, epi, s);
  }
}

}  // namespace kgx
