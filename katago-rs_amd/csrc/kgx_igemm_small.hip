// 16-bit 3x3 convolutions of few pixels (a search's single positions and small batches): the implicit GEMM of
// kgx_igemm.hip with its tiles cut for latency instead of throughput.
//
// On 192-pixel x 48-channel tiles one 19x19 board of a 192 -> 192 convolution is 8 workgroups: the launch takes as long
// as one workgroup needs to stream 166 KB of weights and 90 KB of pixels through three dependent stages (11.0 us at
// batch 1, 11.6 us at batch 7, with 8 and 56 of 256 CUs at work). Here a workgroup computes 64 MB pixels x 16 channels
// (72 workgroups at batch 1) and keeps all input channels of its tile in LDS: every load of the launch is issued at
// once, straight into LDS, and one barrier separates them from the matrix instructions: 6.2 us at batch 1, 8.2 us at
// batch 7 (kernel trace), what is left being the launch, one trip to MALL and the epilogue's store.
//
// The arithmetic is that of kgx_igemm.hip's 48-column 3x3, in the same order (two chains per output, each over its half
// of every 64-channel stage's nine-tap steps, then their sum and the same epilogue expressions), so a row's
// results do not depend on which of the two kernels its batch takes.
#include "kgx_device.h"

namespace kgx {

namespace {

constexpr int SN = 16;               // output channels per workgroup
constexpr int SNT = 512;             // eight waves: two step chains of four 16 MB-pixel waves
constexpr int SK = 64;               // channels per stage
constexpr int SSTAGES = 3;           // most stages held in LDS (192 input channels)
constexpr int STB = 9 * SN;          // weight rows per stage
constexpr int SHALO = POS + 1;
constexpr int SLD = SN + 4;          // the epilogue's float tile row stride

__host__ __device__ constexpr int small_rows(int mb) { return 64 * mb + 2 * SHALO; }  // staged pixel rows, multiple of 8

// Pixel tile mt, column tile nt of workgroup g of ntl column tiles.
__host__ __device__ inline void small_tile_of(int g, int ntl, int& mt, int& nt) {
  mt = g / ntl;
  nt = g - mt * ntl;
}

// SC: as igemm_kernel's (kgx_igemm.hip).
template <typename T, int MB, int SC>
__global__ __launch_bounds__(SNT, 2) void conv_small_kernel(const T* __restrict__ X, int ldx, const T* __restrict__ W,
                                                            int icp, int OC, int M, int ntl, int pbn, ConvOut o) {
  typedef typename std::conditional<std::is_same<T, f16>::value, half8, bf16x8>::type frag_t;
  constexpr int BM = 64 * MB, AR = small_rows(MB), WST = STB * 128, AST = AR * 128;  // bytes per stage
  constexpr int ZERO = SSTAGES * (WST + AST), CB = 2 * BM * SLD * 4;
  static_assert(AR % 8 == 0 && CB <= ZERO, "stage rows load in groups of 8; the epilogue tiles reuse the stages");
  __shared__ __align__(1024) char smem[ZERO + 128];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wv >> 2, wm = wv & 3, r16 = lane & 15, g4 = lane >> 4;
  int mt, nt;
  small_tile_of(blockIdx.x, ntl, mt, nt);
  const int m0 = mt * BM, n0 = nt * SN, nk = icp / SK;
  char* const Ab = smem + SSTAGES * WST;

  // Every stage's weight and pixel rows straight into LDS: one instruction fills 8 rows of 128 bytes, lane i row i / 8
  // at stored chunk i % 8 from source chunk (i % 8) ^ (row / 2 % 8), which keeps fragment reads of 16 consecutive rows
  // conflict-free from any first row. Rows off the batch lie outside the buffer's range (a negative offset wraps past
  // it) and read as zero.
  {
    const int rl = lane >> 3, wtile = (n0 / pbn) * 9 * pbn + n0 % pbn;
    const int wbytes = (OC + pbn - 1) / pbn * pbn * 9 * icp * (int)sizeof(T), xbytes = M * ldx * (int)sizeof(T);
    for (int kt = 0; kt < nk; kt++) {
      for (int q = wv; q < (STB + AR) / 8; q += SNT / 64) {
        if (q < STB / 8) {
          const int row = q * 8 + rl, src = wtile + (row / SN) * pbn + row % SN;
          lds_load16(W, wbytes, smem + kt * WST + q * 1024,
                     src * icp * (int)sizeof(T) + kt * 128 + ((lane & 7) ^ ((row >> 1) & 7)) * 16);
        } else {
          const int a8 = q - STB / 8, row = a8 * 8 + rl;
          lds_load16(X, xbytes, Ab + kt * AST + a8 * 1024,
                     (m0 - SHALO + row) * ldx * (int)sizeof(T) + kt * 128 + ((lane & 7) ^ ((row >> 1) & 7)) * 16);
        }
      }
    }
    if (tid < 8) *(u32x4*)(smem + ZERO + tid * 16) = u32x4{0, 0, 0, 0};
  }

  // The epilogue's inputs, in flight with the stages: thread tid finishes channels 4 (tid % 4) .. + 3 of rows tid / 4 +
  // 128 e (clamped indices; the stores skip what lies outside).
  constexpr int EV = (BM + 127) / 128;
  const int ec4 = tid & 3, er0 = tid >> 2, en = n0 + 4 * ec4, enc = min(en, OC - 4);
  auto epix = [&](int e) { return min(m0 + min(er0 + e * 128, BM - 1), M - 1); };
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

  // Tap validity of this lane's pixels (bit t: the neighbour at tap t is on the board); others read the zero row.
  unsigned vmask[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    const int m = m0 + (wm * MB + i) * 16 + r16;
    unsigned bits = 0;
    if (m < M) {
      const int p = m % HW, y = p / POS, x = p - y * POS;
#pragma unroll
      for (int t = 0; t < 9; t++)
        if ((unsigned)(y + t / 3 - 1) < (unsigned)POS && (unsigned)(x + t % 3 - 1) < (unsigned)POS) bits |= 1u << t;
    }
    vmask[i] = bits;
  }

  floatx4 acc[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};

  // The direct loads are not counted by the compiler: wait for all of this wave's loads, then for every wave.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // One chain's nine steps of a stage, step s of 18 being tap s / 2, channels 32 (s % 2) .. + 32: every fragment is read
  // before the first MFMA, so a stage waits for one LDS round trip.
  auto stage = [&](auto gc, int kt) {
    constexpr int S0 = decltype(gc)::value * 9;
    const char *ws = smem + kt * WST, *as = Ab + kt * AST;
    frag_t a[9][MB], b[9];
#pragma unroll
    for (int s = 0; s < 9; s++) {
      const int t = (S0 + s) / 2, kc = ((S0 + s) & 1) * 4 + g4, shift = (t / 3 - 1) * POS + (t % 3 - 1);
      b[s] = *(const frag_t*)(ws + (t * SN + r16) * 128 + (kc ^ ((r16 >> 1) & 7)) * 16);
#pragma unroll
      for (int i = 0; i < MB; i++) {
        const int row = (wm * MB + i) * 16 + r16 + SHALO + shift;
        const char* p = (vmask[i] >> t) & 1 ? as + row * 128 + (kc ^ ((row >> 1) & 7)) * 16 : smem + ZERO + g4 * 16;
        a[s][i] = *(const frag_t*)p;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 9; s++)
#pragma unroll
      for (int i = 0; i < MB; i++) {
        if constexpr (std::is_same<T, f16>::value)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[s][i], b[s], acc[i], 0, 0, 0);
        else acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][i], b[s], acc[i], 0, 0, 0);
      }
  };
  if (grp == 0) {
    for (int kt = 0; kt < nk; kt++) stage(std::integral_constant<int, 0>{}, kt);
  } else {
    for (int kt = 0; kt < nk; kt++) stage(std::integral_constant<int, 1>{}, kt);
  }
  __syncthreads();  // every wave is done reading the stages

  float* const Cs = (float*)smem;
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) Cs[(grp * BM + (wm * MB + i) * 16 + 4 * g4 + r) * SLD + r16] = acc[i][r];
  __syncthreads();

  const int pfv = l2_touch(o.pf, o.pf_bytes, tid);
#pragma unroll
  for (int e = 0; e < EV; e++) {
    const int row = er0 + e * 128, m = m0 + row;
    if (row < BM && m < M && en < OC) {
      floatx4 sum = *(const floatx4*)(Cs + row * SLD + 4 * ec4);
      sum += *(const floatx4*)(Cs + (BM + row) * SLD + 4 * ec4);
      conv_store4<T, SC >= 0 ? ((SC & SF_EMIT) ? ACT_MISH : ACT_ID) : -1, SC>(o, m, en, sum, yres[e], rmv[e], es, eb,
                                                                              mkv[e]);
    }
  }
  l2_touch_keep(pfv);
}

}  // namespace

// MB of the launch over M pixels and OC outputs: the smallest tile whose workgroups all run at once (one per CU:
// its stages take 95 to 145 KB of LDS), 0 where none does (more than 4032 pixels at 192 outputs, batch 11) or the
// channels do not fit the kernel.
int conv_small_mb(int ks, int ic, int icp, int oc, int M) {
  if (ks != 3 || ic != icp || icp > SSTAGES * SK || M < 1) return 0;
  const int ntl = (oc + SN - 1) / SN;
  for (int mb = 1; mb <= 3; mb++)
    if ((M + 64 * mb - 1) / (64 * mb) * ntl <= 256) return mb;
  return 0;
}

static int small_grid(int mb, int OC, int M) { return (M + 64 * mb - 1) / (64 * mb) * ((OC + SN - 1) / SN); }

LaunchGeometry conv_small_geometry(int mb, int oc, int M, int g, int& mt, int& nt) {
  small_tile_of(g, (oc + SN - 1) / SN, mt, nt);
  LaunchGeometry r;
  r.grid = small_grid(mb, oc, M);
  r.tile_rows = 64 * mb;
  r.tile_cols = SN;
  return r;
}

template <typename T, int MB>
static void small_launch(const void* x, int ldx, const void* w, int icp, int OC, const ConvOut& o, int M, int pbn,
                         hipStream_t s) {
  const int ntl = (OC + SN - 1) / SN, grid = small_grid(MB, OC, M);
  auto go = [&](auto kernel) {
    launch_k(kernel, grid, SNT, 0, s, (const T*)x, ldx, (const T*)w, icp, OC, M, ntl, pbn, o);
  };
  const int sfl = store_flags(o);
  switch ((sfl & SF_EMIT) && o.emit.act != ACT_MISH ? -1 : sfl) {  // the store cases of igemm_launch
    case SF_EMIT: go(conv_small_kernel<T, MB, SF_EMIT>); return;
    case SF_Y: go(conv_small_kernel<T, MB, SF_Y>); return;
    case SF_Y | SF_EMIT: go(conv_small_kernel<T, MB, SF_Y | SF_EMIT>); return;
    case SF_Y | SF_ACC | SF_EMIT: go(conv_small_kernel<T, MB, SF_Y | SF_ACC | SF_EMIT>); return;
    case SF_Y | SF_ACC | SF_YDEAD | SF_EMIT: go(conv_small_kernel<T, MB, SF_Y | SF_ACC | SF_YDEAD | SF_EMIT>); return;
    case SF_Y | SF_ACC | SF_EMIT | SF_LO: go(conv_small_kernel<T, MB, SF_Y | SF_ACC | SF_EMIT | SF_LO>); return;
    case SF_Y | SF_ACC | SF_YDEAD | SF_EMIT | SF_LO:
      go(conv_small_kernel<T, MB, SF_Y | SF_ACC | SF_YDEAD | SF_EMIT | SF_LO>);
      return;
    default: go(conv_small_kernel<T, MB, -1>);
  }
}

void launch_conv_small(int prec, int mb, const void* x, int ldx, const void* w, int icp, int OC, const ConvOut& o, int M,
                       int pbn, hipStream_t s) {
  auto go = [&](auto tc) {
    typedef decltype(tc) T;
    if (mb == 1) small_launch<T, 1>(x, ldx, w, icp, OC, o, M, pbn, s);
    else if (mb == 2) small_launch<T, 2>(x, ldx, w, icp, OC, o, M, pbn, s);
    else small_launch<T, 3>(x, ldx, w, icp, OC, o, M, pbn, s);
  };
  if (prec == PREC_F16) go(f16());
  else go(bf16());
}

}  // namespace kgx
