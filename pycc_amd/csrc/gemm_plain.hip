// Plain-matrix MFMA GEMM for gfx950: C[M][N] = alpha * op(A) op(B) + beta * C, C row-major.
//
// Used for every contraction whose operands are ordinary strided matrices -- the packed ladder and
// the six ring GEMM units of the CCSD residual, which carry almost all of its flops. Compared with
// the 2-level-index kernel (gemm.hip) it loads 16-byte vectors, computes addresses once per tile
// and keeps the k loop free of index arithmetic.
//
//   A: A_KC = true  -> A[m * lda + k]  (k contiguous);  false -> A[k * lda + m]  (m contiguous)
//   B: B_NC = true  -> B[k * ldb + n]  (n contiguous);  false -> B[n * ldb + k]  (k contiguous)
//
// Tiles: 128 x 128 per workgroup (4 waves, 2 x 2, each 64 x 64 = 4 x 4 MFMA 16x16 blocks), BK = 16
// (f64) or 32 (f32) so that one tile row is 128 bytes. Operands are double-buffered: the next tile
// is loaded into registers while the current one is consumed from LDS.
#include "common.h"
#include "gemm.h"
#include <cstdlib>
#include <type_traits>

namespace ccx {

typedef double d4p __attribute__((ext_vector_type(4)));
typedef float f4p __attribute__((ext_vector_type(4)));

namespace {

// CCX_PLAIN_TILE=128 or 256 forces the FP32 tile size (measurement of the two variants).
int plain_tile_override() {
  static int v = -1;
  if (v < 0) {
    const char* e = std::getenv("CCX_PLAIN_TILE");
    v = e ? std::atoi(e) : 0;
  }
  return v;
}

template <typename T> struct PAcc;
template <> struct PAcc<double> { typedef d4p type; };
template <> struct PAcc<float> { typedef f4p type; };

__device__ __forceinline__ d4p pmfma(double a, double b, d4p c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4p pmfma(float a, float b, f4p c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int64_t pxcd_remap(int64_t w, int64_t ntiles) {
  const int64_t nx = 8;
  int64_t q = ntiles / nx, r = ntiles % nx;
  int64_t x = w % nx, j = w / nx;
  return x * q + (x < r ? x : r) + j;
}

// One operand tile: R rows (m or n) x BK k's. KC: stored [R][BK + PAD] (k contiguous in LDS) and
// loaded along k; otherwise stored [BK][R + PAD] and loaded along the row index.
template <typename T, int R, int BK, bool KC>
struct alignas(16) PTile {
  static constexpr int VEC = 16 / sizeof(T);
  // Row padding (keeps every LDS row 16-byte aligned). A k-contiguous tile is read along its rows
  // (16 lanes on 16 rows) and VEC suffices; a row-index-contiguous tile is read by 4 lane groups on
  // 4 consecutive k rows, which must then start 16 banks apart: R + 16 elements per row.
  static constexpr int PAD = KC ? VEC : 16;
  static constexpr int NV = R * BK / VEC / 256;         // 16-byte vectors per thread
  T d[KC ? R : BK][(KC ? BK : R) + PAD];
};

template <typename T, int R, int BK, bool KC>
struct PLoader {
  static constexpr int VEC = 16 / sizeof(T);
  static constexpr int NV = R * BK / VEC / 256;
  static constexpr int SEGS = KC ? BK / VEC : R / VEC;  // vectors per stored row
  uint4 v[NV];
  int row[NV], seg[NV];                                 // stored-row index and vector index
  int from[NV];                                         // the row that load_fast reads into it

  // nrows: valid rows; a k-contiguous tile's rows past them read the last one (their results are not stored)
  __device__ __forceinline__ void init(int tid, int64_t nrows) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      int q = tid + 256 * i;
      row[i] = q / SEGS;
      seg[i] = q % SEGS;
      from[i] = KC && row[i] >= nrows ? (int)nrows - 1 : row[i];
    }
  }
  // base points at the tile origin (row 0, k = k0); ld = leading dimension in elements
  __device__ __forceinline__ void load_fast(const T* __restrict__ base, int64_t ld) {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      v[i] = *(const uint4*)(base + (int64_t)from[i] * ld + seg[i] * VEC);
  }
  // guarded: rows beyond nrows / k beyond nk are zero (nrows, nk relative to the tile origin)
  __device__ __forceinline__ void load_safe(const T* __restrict__ base, int64_t ld, int64_t nrows, int64_t nk) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      union { uint4 u; T e[VEC]; } x;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        int64_t r = KC ? row[i] : (int64_t)seg[i] * VEC + e;    // tile row (m / n)
        int64_t k = KC ? (int64_t)seg[i] * VEC + e : row[i];    // tile k
        const T* p = KC ? base + (int64_t)row[i] * ld + seg[i] * VEC + e
                        : base + (int64_t)row[i] * ld + seg[i] * VEC + e;
        x.e[e] = (r < nrows && k < nk) ? *p : T(0);
      }
      v[i] = x.u;
    }
  }
  __device__ __forceinline__ void store(PTile<T, R, BK, KC>& t) {
#pragma unroll
    for (int i = 0; i < NV; ++i) *(uint4*)&t.d[row[i]][seg[i] * VEC] = v[i];
  }
};

// BT = 128: 4 waves of 64 x 64, two workgroups per CU. BT = 256 (FP32 only): 4 waves of 128 x 128
// (256 accumulator registers each), one workgroup per CU, 4x the MFMAs per LDS read and per barrier.
template <typename T, int BK, bool A_KC, bool B_NC, int BT>
__global__ __launch_bounds__(256, BT == 128 ? 2 : 1) void plain_gemm_kernel(PlainGemm<T> p) {
  constexpr int BM = BT, BN = BT, WM = BT / 2, WN = BT / 2, NBI = WM / 16, NBJ = WN / 16;
  typedef typename PAcc<T>::type acc_t;
  __shared__ PTile<T, BM, BK, A_KC> As[2];
  __shared__ PTile<T, BN, BK, !B_NC> Bs[2];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane >> 4, fc = lane & 15;

  const int64_t tiles_m = ceil_div(p.M, BM), tiles_n = ceil_div(p.N, BN);
  int64_t t = pxcd_remap(blockIdx.x, tiles_m * tiles_n);
  const int64_t GM = 8;
  int64_t group = t / (GM * tiles_n);
  int64_t first_m = group * GM;
  int64_t gsize = tiles_m - first_m < GM ? tiles_m - first_m : GM;
  int64_t within = t - group * GM * tiles_n;
  const int64_t tm = first_m + within % gsize, tn = within / gsize;
  const int64_t m0 = tm * BM, n0 = tn * BN;

  // K of this grid row: a split-K chunk may be shorter than p.K
  const int64_t Kb = p.ktot > 0 ? (p.ktot - (int64_t)blockIdx.y * p.K < p.K ? p.ktot - (int64_t)blockIdx.y * p.K : p.K)
                                : p.K;
  const T* A = p.A + blockIdx.y * p.a_b;
  const T* B = p.B + blockIdx.y * p.b_b;
  T* C = p.C + blockIdx.y * p.c_b;

  // tile origins: A at (m0, k), B at (k, n0)
  auto a_at = [&](int64_t k) { return A_KC ? A + m0 * p.lda + k : A + k * p.lda + m0; };
  auto b_at = [&](int64_t k) { return B_NC ? B + k * p.ldb + n0 : B + n0 * p.ldb + k; };
  const int64_t a_rows = p.M - m0, b_rows = p.N - n0;   // valid tile rows (m / n)
  // every load of a whole k-tile is a vector inside the operand
  const bool inside = (a_rows >= BM || A_KC) && (b_rows >= BN || !B_NC);
  // 16-row blocks of this wave that hold outputs
  const int wrows = (int)(a_rows < BM ? a_rows : BM) - wm * WM;
  const int nbi = __builtin_amdgcn_readfirstlane(wrows <= 0 ? 0 : wrows >= WM ? NBI : (wrows + 15) / 16);

  PLoader<T, BM, BK, A_KC> la;
  PLoader<T, BN, BK, !B_NC> lb;
  la.init(tid, a_rows);
  lb.init(tid, b_rows);
  acc_t acc[NBI][NBJ];
#pragma unroll
  for (int i = 0; i < NBI; ++i)
#pragma unroll
    for (int j = 0; j < NBJ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  // The k loop, compiled three times: FAST (K a multiple of BK, every load a full in-bounds vector), with all
  // of the tile's rows or (!WHOLE) only the 16-row blocks that hold outputs, and checked. A ladder of 528 pair
  // rows ends in a tile of 16: with checked loads and all products it cost as much as two whole ones. Keeping the checked loads out of the FAST loop lets the
  // prefetch of tile k + 1 stay in flight while tile k is multiplied (a shared loop forces a full
  // wait on the loads at the join of the two load paths).
  auto kloop = [&](auto fast_tag, auto whole_tag) {
    constexpr bool FAST = decltype(fast_tag)::value, WHOLE = decltype(whole_tag)::value;
    auto load = [&](int64_t k0) {
      const int64_t nk = Kb - k0;
      if constexpr (FAST) {
        la.load_fast(a_at(k0), p.lda);
      } else {
        la.load_safe(a_at(k0), p.lda, a_rows, nk);
      }
      if constexpr (FAST) lb.load_fast(b_at(k0), p.ldb);
      else lb.load_safe(b_at(k0), p.ldb, b_rows, nk);
    };
    load(0);
    la.store(As[0]);
    lb.store(Bs[0]);
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = 0; k0 < Kb; k0 += BK) {
      const bool has_next = k0 + BK < Kb;
      if (has_next) load(k0 + BK);
#pragma unroll
      for (int ks = 0; ks < BK; ks += 4) {
        T a[NBI], b[NBJ];
#pragma unroll
        for (int i = 0; i < NBI; ++i)
          a[i] = A_KC ? As[buf].d[wm * WM + i * 16 + fc][ks + fr] : As[buf].d[ks + fr][wm * WM + i * 16 + fc];
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
          b[j] = B_NC ? Bs[buf].d[ks + fr][wn * WN + j * 16 + fc] : Bs[buf].d[wn * WN + j * 16 + fc][ks + fr];
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
          if (!WHOLE && i >= nbi) break;
#pragma unroll
          for (int j = 0; j < NBJ; ++j) acc[i][j] = pmfma(a[i], b[j], acc[i][j]);
        }
      }
      if (has_next) {
        la.store(As[buf ^ 1]);
        lb.store(Bs[buf ^ 1]);
      }
      __syncthreads();
      buf ^= 1;
    }
  };
  if (Kb > 0) {
    if (inside && Kb % BK == 0 && a_rows >= BM) kloop(std::true_type{}, std::true_type{});
    else if (inside && Kb % BK == 0) kloop(std::true_type{}, std::false_type{});
    else kloop(std::false_type{}, std::true_type{});
  }

#pragma unroll
  for (int j = 0; j < NBJ; ++j) {
    const int64_t n = n0 + wn * WN + j * 16 + fc;
    if (n >= p.N) continue;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // output row of register r (f64: 4r + fr, f32: 4 fr + r; see gemm.hip)
        const int64_t m = m0 + wm * WM + i * 16 + (sizeof(T) == 8 ? 4 * r + fr : 4 * fr + r);
        if (m >= p.M) continue;
        T* dst = C + m * p.ldc + n;
        T val = p.alpha * acc[i][j][r];
        if (p.beta != T(0)) val += p.beta * *dst;
        *dst = val;
      }
  }
}

// 256 x 256 tiles for large FP32 GEMMs (enough tiles to fill the 256 CUs several times over).
template <typename T>
bool plain_big_tiles(const PlainGemm<T>& p) {
  if (sizeof(T) != 4 || plain_tile_override() == 128) return false;
  return plain_tile_override() == 256 || ceil_div(p.M, 256) * ceil_div(p.N, 256) * p.batch >= 1024;
}

template <typename T, bool A_KC, bool B_NC>
void launch_plain(const PlainGemm<T>& p, hipStream_t s) {
  constexpr int BK = sizeof(T) == 8 ? 16 : 32;
  if constexpr (sizeof(T) == 4) {
    if (plain_big_tiles(p)) {
      int64_t tiles = ceil_div(p.M, 256) * ceil_div(p.N, 256);
      plain_gemm_kernel<T, BK, A_KC, B_NC, 256><<<dim3((unsigned)tiles, (unsigned)p.batch), 256, 0, s>>>(p);
      CCX_HIP(hipGetLastError());
      return;
    }
  }
  {
    int64_t tiles = ceil_div(p.M, 128) * ceil_div(p.N, 128);
    plain_gemm_kernel<T, BK, A_KC, B_NC, 128><<<dim3((unsigned)tiles, (unsigned)p.batch), 256, 0, s>>>(p);
  }
  CCX_HIP(hipGetLastError());
}

typedef double d2p __attribute__((ext_vector_type(2)));

// 16 bytes per lane from global memory into LDS at lds + 16 lane, no register in between. The load takes the LDS address
// from m0, which it sees one wait state after a scalar write: the s_nop is that state, which the compiler cannot add here.
__device__ __forceinline__ void dma16(const double* g, const double* lds) {
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const double*)lds;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is reserved, named all the same
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(__builtin_amdgcn_readfirstlane(base)), "v"(g) : "memory", "m0");
#pragma clang diagnostic pop
}

// The (T) products (kcat64): 128 x 16 NBJ tiles, 4 waves of 32 rows by all 16 NBJ columns. A stage is
// 8 k values of every row; its operands go from global memory straight into LDS
// (global_load_lds_dwordx4) through 4 buffers, so that three stages are in flight while one feeds
// 4 NBJ MFMAs (64 cycles each) per wave, with one barrier per stage. LDS rows are 64 bytes with the
// 16-byte chunk c of row r at c ^ (r / 2 % 4): neither the DMA nor the fragment reads (8 lanes to a
// cycle, eight rows of one chunk) conflict. Every wave issues the same number of DMA instructions
// per stage (blocks past NBJ land in rows of sB that are never read), so that one immediate count
// waits for a stage. Rows past v^2 or v load a valid row; their results are not stored.
// Bound by the FP64 MFMA rate (a library product reaches 72.8 TFLOP/s): 67 TFLOP/s of padded work at K =
// 960, 63 at v = 112 K = 256, 58 at v = 107 K = 240 (40 triples, ends of the short k loop exposed).
// Fragments loaded straight from global memory: 56, 53, 51; two buffers: 65, 62, 56; registers and
// LDS with checked loads (v = 107, K padded to 256): 35.
template <int NBJ>
__global__ __launch_bounds__(256, 2) void kcat64_kernel(Kcat64 p, int64_t tiles_m, int64_t tiles_n) {
  constexpr int NB = (NBJ + 3) / 4, D = 2 + NB, ST = 4, BLK = 16 * 8;   // doubles per 16-row block
  __shared__ __attribute__((aligned(1024))) double sA[ST][8][BLK];
  __shared__ __attribute__((aligned(1024))) double sB[ST][4 * NB][BLK];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane >> 4, fc = lane & 15;
  int64_t b, tm, tn;
  kcat_tile(pxcd_remap(blockIdx.x, gridDim.x), tiles_m, tiles_n, b, tm, tn);
  const int64_t e = b / 3;
  const int4 blk = kcat_blocks(p.tri[e], (int)(b - 3 * e), p.n);
  const int64_t v = p.v, vv = v * v, Kp = p.Kp, ldc = p.ldc, m0 = tm * 128, n0 = tn * (16 * NBJ);
  // DMA lane: row lane / 4 of its block, chunk (lane % 4) ^ (row / 2 % 4)
  const int dr = lane >> 2, dc = (lane & 3) ^ ((dr >> 1) & 3);
  const double *pA[2], *pA2[2], *pB[NB], *pB2[NB];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t r = m0 + 16 * (2 * wave + i) + dr, m = r < vv ? r : vv - 1, x = m / v, y = m - x * v;
    pA[i] = p.A + (blk.x * vv + m) * Kp + 2 * dc;
    pA2[i] = p.A + (blk.y * vv + y * v + x) * Kp + 2 * dc;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int64_t r = n0 + 16 * (wave + 4 * i) + dr, n = r < v ? r : v - 1;
    pB[i] = p.B + (blk.z * v + n) * Kp + 2 * dc;
    pB2[i] = p.B + (blk.w * v + n) * Kp + 2 * dc;
  }
  d4p acc[2][NBJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NBJ; ++j) acc[i][j] = d4p{0, 0, 0, 0};
  const int half = (int)(Kp / 8), nst = 2 * half;
  int st = 0;
  auto issue = [&](int q) {   // stage st into buffer q, then on to the next (past the last: the last again)
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16(pA[i], &sA[q][2 * wave + i][0]);
#pragma unroll
    for (int i = 0; i < NB; ++i) dma16(pB[i], &sB[q][wave + 4 * i][0]);
    if (++st == half) {
#pragma unroll
      for (int i = 0; i < 2; ++i) pA[i] = pA2[i];
#pragma unroll
      for (int i = 0; i < NB; ++i) pB[i] = pB2[i];
    } else if (st < nst) {
#pragma unroll
      for (int i = 0; i < 2; ++i) pA[i] += 8;
#pragma unroll
      for (int i = 0; i < NB; ++i) pB[i] += 8;
    }
  };
  const int fo = fc * 8 + ((fr ^ ((fc >> 1) & 3)) * 2);   // fragment: row fc, chunk fr
#pragma unroll
  for (int q = 0; q < ST - 1; ++q) issue(q);
  auto step = [&](auto buf) {
    constexpr int q = decltype(buf)::value;
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((ST - 2) * D) : "memory");
    issue((q + ST - 1) % ST);
    d2p fa[2], fb[NBJ];
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[i] = *(const d2p*)&sA[q][2 * wave + i][fo];
#pragma unroll
    for (int j = 0; j < NBJ; ++j) fb[j] = *(const d2p*)&sB[q][j][fo];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < NBJ; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][j] = pmfma(fa[i][h], fb[j][h], acc[i][j]);
  };
  constexpr std::integral_constant<int, 0> b0{};
  constexpr std::integral_constant<int, 1> b1{};
  constexpr std::integral_constant<int, 2> b2{};
  constexpr std::integral_constant<int, 3> b3{};
  int s = 0;
  for (; s + 4 <= nst; s += 4) {
    step(b0);
    step(b1);
    step(b2);
    step(b3);
  }
  if (s < nst) {   // nst is even
    step(b0);
    step(b1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the DMA into LDS ends before the work-group does

  double* C = p.C + b * vv * ldc;
#pragma unroll
  for (int j = 0; j < NBJ; ++j) {
    const int64_t n = n0 + 16 * j + fc;
    if (n >= v) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + 16 * (2 * wave + i) + 4 * r + fr;
        if (m < vv) C[m * ldc + n] = acc[i][j][r];
      }
  }
}

}  // namespace

template <typename T>
bool plain_gemm_ok(const PlainGemm<T>& p) {
  const int64_t VEC = 16 / sizeof(T);
  if (p.M <= 0 || p.N <= 0 || p.batch < 1 || p.batch > 65535) return false;
  if (ceil_div(p.M, 128) * ceil_div(p.N, 128) >= (1ll << 31)) return false;
  auto aligned = [&](const void* q) { return ((uintptr_t)q % 16) == 0; };
  if (!aligned(p.A) || !aligned(p.B)) return false;
  if (p.lda % VEC || p.ldb % VEC) return false;
  if (p.batch > 1 && (p.a_b % VEC || p.b_b % VEC)) return false;
  return true;
}

template <typename T>
void plain_gemm(const PlainGemm<T>& p, hipStream_t s) {
  CCX_CHECK(plain_gemm_ok(p), ERR_INTERNAL, "plain_gemm called on an unsupported layout");
  if (p.a_kc && p.b_nc) launch_plain<T, true, true>(p, s);
  else if (p.a_kc) launch_plain<T, true, false>(p, s);
  else if (p.b_nc) launch_plain<T, false, true>(p, s);
  else launch_plain<T, false, false>(p, s);
}

void kcat64(const Kcat64& p, hipStream_t s) {
  if (p.ntri == 0 || p.v == 0) return;
  const int64_t tm = ceil_div(p.v * p.v, 128), tn = ceil_div(p.v, 128), nbj = ceil_div(ceil_div(p.v, tn), 16);
  CCX_CHECK(p.Kp % 8 == 0 && p.Kp > 0 && p.ldc >= p.v && ((uintptr_t)p.A | (uintptr_t)p.B) % 16 == 0,
            ERR_INTERNAL, "kcat64 layout");
  const int64_t blocks = tm * tn * 3 * p.ntri;
  CCX_CHECK(blocks < (int64_t(1) << 31), ERR_ARG, "(T) GEMM grid too large");
  const dim3 g((unsigned)blocks);
  switch (nbj) {
    case 1: kcat64_kernel<1><<<g, 256, 0, s>>>(p, tm, tn); break;
    case 2: kcat64_kernel<2><<<g, 256, 0, s>>>(p, tm, tn); break;
    case 3: kcat64_kernel<3><<<g, 256, 0, s>>>(p, tm, tn); break;
    case 4: kcat64_kernel<4><<<g, 256, 0, s>>>(p, tm, tn); break;
    case 5: kcat64_kernel<5><<<g, 256, 0, s>>>(p, tm, tn); break;
    case 6: kcat64_kernel<6><<<g, 256, 0, s>>>(p, tm, tn); break;
    case 7: kcat64_kernel<7><<<g, 256, 0, s>>>(p, tm, tn); break;
    default: kcat64_kernel<8><<<g, 256, 0, s>>>(p, tm, tn); break;
  }
  CCX_HIP(hipGetLastError());
}

template bool plain_gemm_ok<double>(const PlainGemm<double>&);
template bool plain_gemm_ok<float>(const PlainGemm<float>&);
template void plain_gemm<double>(const PlainGemm<double>&, hipStream_t);
template void plain_gemm<float>(const PlainGemm<float>&, hipStream_t);

}  // namespace ccx
