// MFMA tensor-contraction GEMM for gfx950.
//
// The tile kernel serves every contraction that is not a plain matrix product of many tiles (gemm_plain.hip): M and N
// are 2-level indices (two tensor indices with independent strides), K has a third, outer level, and there is one
// batch index, so e.g. 'jnfb,mnef->mbej' runs without materialising permuted copies. It comes as 128 x 128 tiles of 8
// waves (64 x 32 each) and 64 x 64 tiles of 4, alone or several contractions to a launch (GemmQueue).
//
// Lane layout of the 16x16x4 MFMAs used here (measured on gfx950):
//   A (16x4):  lane l holds A[l % 16][l / 16]
//   B (4x16):  lane l holds B[l / 16][l % 16]
//   C (16x16): lane l, register r holds C[row][l % 16] with
//              row = 4 * (l / 16) + r   for v_mfma_f32_16x16x4f32
//              row = 4 * r + (l / 16)   for v_mfma_f64_16x16x4f64
#include "common.h"
#include "gemm.h"
#include "tile_blocks.h"
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

namespace ccx {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T> struct AccT;
template <> struct AccT<double> { typedef d4 type; };
template <> struct AccT<float> { typedef f4 type; };

__device__ __forceinline__ d4 mfma16(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma16(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int64_t off2(const Idx2& d, int64_t i) {
  // all extents are < 2^31, so 32-bit division is exact here
  uint32_t q = (uint32_t)i / (uint32_t)d.n2;
  uint32_t r = (uint32_t)i - q * (uint32_t)d.n2;
  return (int64_t)q * d.s1 + (int64_t)r * d.s2;
}

// Map the hardware workgroup id (dispatched round-robin over the 8 XCDs) to a logical tile id so
// that each XCD receives one contiguous run of logical tiles (and so shares operands in its L2).
__device__ __forceinline__ int64_t xcd_remap(int64_t w, int64_t ntiles) {
  const int64_t nx = 8;
  int64_t q = ntiles / nx, r = ntiles % nx;
  int64_t x = w % nx, j = w / nx;
  return x * q + (x < r ? x : r) + j;
}

// ---- the tile kernel -------------------------------------------------------------------------------
// C[b][m][n] = alpha sum_(x, k) A[b][m][x, k] B[b][x, k][n] + beta C: M, N and K are 2-level indices, x an
// outer third level of K (its strides a_x, b_x), b the batch.
//
// What bounds it: a 16x16x4 FP64 MFMA holds a SIMD for 64 cycles, so the matrix cores, as long as some wave always has
// one to issue: 8 waves of 64 x 32 per 128 x 128 work-group, two work-groups per CU (4 waves per SIMD, 128 registers).
// Measured at 8192^3: 59-62 TF; 70-74 TF with the global loads and LDS writes left out, each of which costs the
// matrix cores about 10% however early it is issued (a third LDS stage, two k-tiles in flight and 32-wide k-tiles
// changed nothing), so loads and LDS writes are pairs wherever those are contiguous (57 TF with 8-byte ones). Addresses
// come from an odometer per k-tile, so any strides, odd extents and remainders run the same loop: 2793^3 with odd
// leading dimensions takes 0.76 ms (0.99 with guarded 8-byte loads). Rows past M or N read row M - 1 or N - 1
// (their outputs are not stored); k past its end reads a valid k and is zeroed on its way into LDS.
//
// LDS: a k-fast tile is [rows][BK + 2] (FP32: BK + 1) and a row-fast one [BK][rows + 16]: the two k rows of a half wave's
// fragment read start 4 (k-fast: rows start 36 banks) or 32 banks apart, so reads are free of conflicts.

// i / d for 0 <= i < 2^31 by multiply-high (d >= 1).
struct FastIdx {
  uint32_t n2, mul, sh;
  int64_t s1, s2;
};
static FastIdx fast_idx(const Idx2& x) {
  FastIdx f;
  CCX_CHECK(x.n2 >= 1 && x.n2 < (1ll << 31), ERR_INTERNAL, "index extent");
  f.n2 = (uint32_t)x.n2;
  f.sh = 0;
  while ((1ull << f.sh) < f.n2) ++f.sh;
  f.mul = (uint32_t)((((1ull << f.sh) - f.n2) << 32) / f.n2 + 1);
  f.s1 = x.s1;
  f.s2 = x.s2;
  return f;
}
__device__ __forceinline__ int64_t off2(const FastIdx& d, uint32_t i) {
  const uint32_t q = (__umulhi(i, d.mul) + i) >> d.sh;
  const uint32_t r = i - q * d.n2;
  return (int64_t)q * d.s1 + (int64_t)r * d.s2;
}

template <typename T>
struct TileGemm {
  uint32_t M, N, K;         // under 2^31: rows, columns and k's of a tile that reaches past them stay under 2^32
  int kx, splits, chunk;    // chunk: k-tiles per split, counted over x and k
  FastIdx am, ak, bk, bn, cm, cn;
  int64_t a_x, b_x, a_b, b_b, c_b;
  T alpha, beta;
  const T* A;
  const T* B;
  T* C;
  T* work;   // [split][batch][M][N] partial sums when splits > 1
};

// two neighbouring elements, aligned as one: read from memory by one load, written to LDS by one instruction
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) Two {
  T x, y;
};
// a pair of doubles in LDS, where rows are 16-byte aligned
struct alignas(16) Two16 {
  double x, y;
};

// One operand's tile, and its fragments: MFMA step s of a 16-wide k-tile holds k = 4 s + lane / 16, so every sum runs
// over k upwards whatever the tile.
template <typename T, int R, int BK, bool KF>
struct GTile {
  alignas(16) T d[KF ? R : BK][KF ? BK + (sizeof(T) == 8 ? 2 : 1) : R + 16];
  __device__ __forceinline__ T& at(int r, int k) { return KF ? d[r][k] : d[k][r]; }
  // f[h][b]: row r0 + 16 b + fc, MFMA step k8 / 4 + h
  template <int NB>
  __device__ __forceinline__ void frags(T (&f)[2][NB], int r0, int k8, int fr, int fc) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < NB; ++b) f[h][b] = at(r0 + 16 * b + fc, k8 + 4 * h + fr);
  }
};

// One operand's loader: a thread owns NE pieces of V values of the R x BK tile, V along k (k-fast) or along the
// rows; k-fast: one k and NE rows, else one row piece and NE k's. Addresses are a uniform base plus a lane
// offset in bytes (Off: 32 bits where the operand spans less than 4 GiB), k by an odometer over its (n2, s1, s2):
// a k-tile costs a lane one step of it and an add per load. Where a whole wave holds one k (row-fast, V R >= 64
// lanes) that k stays in scalar registers.
// V = 2 reads two elements at a time. It needs the inner index contiguous and pairs that do not straddle its blocks: an
// even n2 or a single level. An odd extent ends in a pair that starts one early (`late`: its second half counts).
template <typename T, int R, int BK, bool KF, int NT, typename Off, int V>
struct GLoader {
  static constexpr int LANES = (KF ? BK : R) / V;   // pieces along the contiguous index
  static constexpr int NE = R * BK / V / NT, STEP = NT / LANES;
  static constexpr bool UK = !KF && LANES >= 64;    // k uniform in a wave
  static constexpr int NO = KF || UK ? 1 : NE;      // odometers
  int kl, rl;
  Off roff[KF ? NE : 1], koff[NO];
  uint32_t kr[NO];
  bool row_late;
  // one k-tile's values on their way to LDS
  struct Load {
    T v[NE][V];
    uint32_t ok;   // bit i: piece i's k is inside
    bool late, whole;
  };
  __device__ __forceinline__ void init(const FastIdx& rix, uint32_t row0, uint32_t nrows, int tid) {
    const int along = tid % LANES * V, across = tid / LANES;
    kl = KF ? along : UK ? __builtin_amdgcn_readfirstlane(across) : across;
    rl = KF ? across : along;
    row_late = false;
#pragma unroll
    for (int i = 0; i < (KF ? NE : 1); ++i) {
      uint32_t r = row0 + rl + i * STEP;
      if (!KF && V == 2) row_late = r == nrows - 1;
      r = r < nrows - (KF ? 1 : V) ? r : nrows - (KF ? 1 : V);
      roff[i] = (Off)(off2(rix, r) * (int64_t)sizeof(T));
    }
  }
  __device__ __forceinline__ void seek(const FastIdx& kix, uint32_t k0) {
    if (UK) return;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const uint32_t k = k0 + kl + i * STEP, q = (__umulhi(k, kix.mul) + k) >> kix.sh;
      kr[i] = k - q * kix.n2;
      koff[i] = (Off)(((int64_t)q * kix.s1 + (int64_t)kr[i] * kix.s2) * (int64_t)sizeof(T));
    }
  }
  __device__ __forceinline__ void step(const FastIdx& kix, uint32_t k0) {   // BK further, to the tile at k0
    if (UK) return;
    if (kix.n2 < (uint32_t)BK) {
      seek(kix, k0);
      return;
    }
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      kr[i] += BK;
      koff[i] += (Off)(BK * kix.s2 * (int64_t)sizeof(T));
      if (kr[i] >= kix.n2) {
        kr[i] -= kix.n2;
        koff[i] += (Off)((kix.s1 - (int64_t)kix.n2 * kix.s2) * (int64_t)sizeof(T));
      }
    }
  }
  static __device__ __forceinline__ void get(T (&v)[V], const char* p) {
    if constexpr (V == 2) {
      const Two<T> q = *(const Two<T>*)p;
      v[0] = q.x;
      v[1] = q.y;
    } else {
      v[0] = *(const T*)p;
    }
  }
  // rows_in: every row of the tile is inside
  __device__ __forceinline__ void load(Load& l, const T* __restrict__ base, const FastIdx& kix, uint32_t k0, uint32_t K,
                                       bool rows_in) {
    l.ok = 0;
    l.late = row_late;
    l.whole = rows_in && k0 + BK <= K;
    if constexpr (KF) {
      const uint32_t k = k0 + kl;
      Off ko = koff[0];
      if (V == 2) l.late = k == K - 1;
      if (k > K - V) ko = V == 2 && k < K ? ko - (Off)sizeof(T) : 0;
      if (k < K) l.ok = ~0u;
#pragma unroll
      for (int i = 0; i < NE; ++i) get(l.v[i], (const char*)base + (Off)(roff[i] + ko));
    } else {
#pragma unroll
      for (int i = 0; i < NE; ++i) {
        const uint32_t k = k0 + kl + i * STEP;
        if (k < K) l.ok |= 1u << i;
        if constexpr (UK) get(l.v[i], (const char*)(base + off2(kix, k < K ? k : K - 1)) + roff[0]);
        else get(l.v[i], (const char*)base + (Off)(roff[0] + (k < K ? koff[i] : (Off)0)));
      }
    }
  }
  __device__ __forceinline__ void put(const T (&x)[V], int i, GTile<T, R, BK, KF>& t) {
    T* dst = KF ? &t.at(rl + i * STEP, kl) : &t.at(rl, kl + i * STEP);
    if constexpr (V == 2 && sizeof(T) == 8) *(Two16*)dst = Two16{x[0], x[1]};
    else if constexpr (V == 2) *(Two<T>*)dst = Two<T>{x[0], x[1]};
    else *dst = x[0];
  }
  __device__ __forceinline__ void store(const Load& l, GTile<T, R, BK, KF>& t) {
    if (l.whole) {
#pragma unroll
      for (int i = 0; i < NE; ++i) put(l.v[i], i, t);
    } else {
      asm volatile("");   // keeps this a branch (it is uniform): as selects it would cost every k-tile
#pragma unroll
      for (int i = 0; i < NE; ++i) {
        const bool in = (l.ok >> i) & 1u, late = V == 2 && l.late;
        T x[V];
        x[0] = in ? (late ? l.v[i][V - 1] : l.v[i][0]) : T(0);
        if (V == 2) x[V - 1] = in && !late ? l.v[i][V - 1] : T(0);
        put(x, i, t);
      }
    }
  }
};

// One work-group's tile `t` (of tiles_m x tiles_n), batch entry and split.
template <typename T, int BM, int BN, int WM, int WN, int BK, bool AKF, bool BKF, typename Off, int V>
__device__ __forceinline__ void tile_body(const TileGemm<T>& p, int64_t t, int bidx, int sidx, int64_t nbatch,
                                          GTile<T, BM, BK, AKF>* As, GTile<T, BN, BK, BKF>* Bs) {
  constexpr int NWN = BN / WN, NT = 64 * (BM / WM) * NWN, NBI = WM / 16, NBJ = WN / 16;
  typedef typename AccT<T>::type acc_t;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / NWN, wn = wave % NWN;

  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  // 8 tile-rows together, so that concurrently running tiles share A and B panels
  const int64_t group = t / (8 * tiles_n);
  const int first_m = (int)group * 8, gsize = tiles_m - first_m < 8 ? tiles_m - first_m : 8;
  const int within = (int)(t - group * 8 * tiles_n);
  const uint32_t m0 = (uint32_t)(first_m + within % gsize) * BM, n0 = (uint32_t)(within / gsize) * BN;

  const int ntk = (p.K + BK - 1) / BK;   // k-tiles of one x
  int kt = sidx * p.chunk;               // first and end k-tile of this split, over x and k
  const int kt_end = kt + p.chunk < ntk * p.kx ? kt + p.chunk : ntk * p.kx;
  const int x0 = ntk ? kt / ntk : 0;
  uint32_t k0 = (uint32_t)(kt - x0 * ntk) * BK;
  const T* __restrict__ A = p.A + bidx * p.a_b + x0 * p.a_x;
  const T* __restrict__ B = p.B + bidx * p.b_b + x0 * p.b_x;

  GLoader<T, BM, BK, AKF, NT, Off, V> la;
  GLoader<T, BN, BK, BKF, NT, Off, V> lb;
  la.init(p.am, m0, p.M, tid);
  lb.init(p.bn, n0, p.N, tid);

  acc_t acc[NBI][NBJ];
#pragma unroll
  for (int i = 0; i < NBI; ++i)
#pragma unroll
    for (int j = 0; j < NBJ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  const int fr = lane >> 4, fc = lane & 15;
  const bool m_in = m0 + BM <= p.M, n_in = n0 + BN <= p.N;
  // This wave's 16 x 16 blocks: rows r0 + 16 i, columns c0 + 16 j, i < ni, j < nj
  int r0 = wm * WM, c0 = wn * WN, ni = NBI, nj = NBJ;
  if constexpr (BM == 64 && BN == 64) {
    const WaveBlocks b = wave_blocks(m_in ? 4 : (p.M - m0 + 15) >> 4, n_in ? 4 : (p.N - n0 + 15) >> 4,
                                     __builtin_amdgcn_readfirstlane(wave));
    r0 = b.r0;
    c0 = b.c0;
    ni = b.ni;
    nj = b.nj;
  }
  const bool all = ni == NBI && nj == NBJ;

  if (kt < kt_end) {
    typename decltype(la)::Load va;
    typename decltype(lb)::Load vb;
    la.seek(p.ak, k0);
    lb.seek(p.bk, k0);
    auto load = [&] {
      la.load(va, A, p.ak, k0, p.K, m_in);
      lb.load(vb, B, p.bk, k0, p.K, n_in);
    };
    // to the next k-tile; past the last one the last is loaded again (no branch around the loads)
    auto next = [&] {
      if (kt + 1 >= kt_end) return;
      k0 += BK;
      if (k0 >= p.K) {
        k0 = 0;
        A += p.a_x;
        B += p.b_x;
        la.seek(p.ak, 0);
        lb.seek(p.bk, 0);
      } else {
        la.step(p.ak, k0);
        lb.step(p.bk, k0);
      }
    };
    load();
    la.store(va, As[0]);
    lb.store(vb, Bs[0]);
    __syncthreads();
    // one k-tile, from LDS buffer `buf` (a constant where it is called: LDS addresses stay immediate offsets)
    auto body = [&](int buf) {
      next();
      load();
#pragma unroll
      for (int kg = 0; kg < BK; kg += 8) {
        // BI x BJ blocks: only rows that the wave owns are read (r0 and c0 go up to 48, so that a second block's rows
        // may lie past the tile, in the buffer that is being written or past the work-group's LDS)
        auto products = [&](auto bi, auto bj) {
          constexpr int BI = decltype(bi)::value, BJ = decltype(bj)::value;
          T a[2][BI], b[2][BJ];
          As[buf].frags(a, r0, kg, fr, fc);
          Bs[buf].frags(b, c0, kg, fr, fc);
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < BI; ++i)
#pragma unroll
              for (int j = 0; j < BJ; ++j) acc[i][j] = mfma16(a[h][i], b[h][j], acc[i][j]);
        };
        constexpr std::integral_constant<int, 1> one{};
        if constexpr (BM == 64 && BN == 64) {
          if (all) products(std::integral_constant<int, NBI>{}, std::integral_constant<int, NBJ>{});
          else if (ni == 2 && nj == 1) products(std::integral_constant<int, 2>{}, one);
          else if (ni == 1 && nj == 2) products(one, std::integral_constant<int, 2>{});
          else if (ni == 1 && nj == 1) products(one, one);
        } else {
          products(std::integral_constant<int, NBI>{}, std::integral_constant<int, NBJ>{});
        }
      }
      la.store(va, As[buf ^ 1]);
      lb.store(vb, Bs[buf ^ 1]);
      __syncthreads();
      ++kt;
    };
    while (kt + 1 < kt_end) {
      body(0);
      body(1);
    }
    if (kt < kt_end) body(0);
  }

  // output row of register r within a 16x16 block (see the layout note at the top)
  auto row = [&](int i, int r) { return m0 + r0 + i * 16 + (sizeof(T) == 8 ? 4 * r + fr : 4 * fr + r); };
  if (p.splits == 1) {
    T* C = p.C + bidx * p.c_b;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t m = row(i, r);
        if (i >= ni || m >= p.M) continue;
        T* Cm = C + off2(p.cm, m);
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
          const uint32_t n = n0 + c0 + j * 16 + fc;
          if (j >= nj || n >= p.N) continue;
          T* dst = Cm + off2(p.cn, n);
          T v = p.alpha * acc[i][j][r];
          if (p.beta != T(0)) v += p.beta * *dst;
          *dst = v;
        }
      }
  } else {
    T* W = p.work + ((int64_t)sidx * nbatch + bidx) * p.M * p.N;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t m = row(i, r);
        if (i >= ni || m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
          const uint32_t n = n0 + c0 + j * 16 + fc;
          if (j < nj && n < p.N) W[(int64_t)m * p.N + n] = acc[i][j][r];
        }
      }
  }
}

template <typename T, int BM, int BN, int WM, int WN, int BK, bool AKF, bool BKF, typename Off, int V>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN), 4) void tile_gemm_kernel(TileGemm<T> p) {
  __shared__ GTile<T, BM, BK, AKF> As[2];
  __shared__ GTile<T, BN, BK, BKF> Bs[2];
  const int64_t tiles = (int64_t)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  const int64_t t = blockIdx.x + (int64_t)gridDim.x * blockIdx.z;
  if (t >= tiles) return;
  tile_body<T, BM, BN, WM, WN, BK, AKF, BKF, Off, V>(p, xcd_remap(t, tiles), blockIdx.y / p.splits,
                                                     blockIdx.y % p.splits, gridDim.y / p.splits, As, Bs);
}

// Several small independent FP64 contractions in one launch (GemmQueue): 64 x 64 tiles, block b belongs to the
// contraction with first[i] <= b < first[i + 1]. What bounds them one by one is the launch: at o=5 v=19 and
// o=9 v=61 a contraction takes 4.5 us to be launched and 4 to 15 to run a handful of work-groups.
constexpr int GROUP = 12;
struct GemmGroup {
  int n;
  int first[GROUP + 1];
  int form[GROUP];      // 1: A k-fast, 2: B k-fast, 4: pairs
  int batch[GROUP];
  TileGemm<double> g[GROUP];
};
template <bool AKF, bool BKF, int V>
__device__ __forceinline__ void group_body(const TileGemm<double>& p, int nbatch, int local, char* lds) {
  typedef GTile<double, 64, 16, AKF> TA;
  typedef GTile<double, 64, 16, BKF> TB;
  const int tiles = (int)((p.M + 63) / 64) * (int)((p.N + 63) / 64), y = local / tiles;
  tile_body<double, 64, 64, 32, 32, 16, AKF, BKF, uint32_t, V>(p, local - y * tiles, y / p.splits, y % p.splits, nbatch,
                                                               (TA*)lds, (TB*)(lds + 2 * sizeof(TA)));
}
__global__ __launch_bounds__(256, 4) void tile_group_kernel(const GemmGroup a) {
  constexpr size_t ROWS = sizeof(GTile<double, 64, 16, false>), KFAST = sizeof(GTile<double, 64, 16, true>);
  __shared__ alignas(16) char lds[4 * (ROWS > KFAST ? ROWS : KFAST)];
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
  const int local = blockIdx.x - a.first[i], nb = a.batch[i];
  const TileGemm<double> g = a.g[i];   // one copy, in scalar registers
  switch (a.form[i]) {
    case 0: group_body<false, false, 1>(g, nb, local, lds); break;
    case 1: group_body<true, false, 1>(g, nb, local, lds); break;
    case 2: group_body<false, true, 1>(g, nb, local, lds); break;
    case 3: group_body<true, true, 1>(g, nb, local, lds); break;
    case 4: group_body<false, false, 2>(g, nb, local, lds); break;
    case 5: group_body<true, false, 2>(g, nb, local, lds); break;
    case 6: group_body<false, true, 2>(g, nb, local, lds); break;
    default: group_body<true, true, 2>(g, nb, local, lds); break;
  }
}

// The split-K sums of a group: 64 outputs and 4 groups of splits per block (more than FIXED_K_SPLITS splits), or 256
// outputs with their partials in order.
struct SumGroup {
  int n;
  int first[GROUP + 1];
  int64_t batch[GROUP];
  TileGemm<double> g[GROUP];
};
__global__ __launch_bounds__(256) void sum_group_kernel(const SumGroup a) {
  __shared__ double part[4][64];
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
  const TileGemm<double>& p = a.g[i];
  const int local = blockIdx.x - a.first[i];
  const int64_t total = a.batch[i] * p.M * p.N;
  const bool wide = p.splits > FIXED_K_SPLITS;
  const int G = wide ? 4 : 1, g = wide ? threadIdx.x >> 6 : 0;
  const int64_t e = wide ? (int64_t)local * 64 + (threadIdx.x & 63) : (int64_t)local * 256 + threadIdx.x;
  double s = 0;
  if (e < total) {
    const double* w = p.work + e;
    int k = g;
    for (; k + 7 * G < p.splits; k += 8 * G) {
      double x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = w[(int64_t)(k + u * G) * total];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += x[u];
    }
    for (; k < p.splits; k += G) s += w[(int64_t)k * total];
  }
  if (wide) {
    part[g][threadIdx.x & 63] = s;
    __syncthreads();
    if (g > 0) return;
    s = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
  }
  if (e >= total) return;
  const uint32_t mn = p.M * p.N, b = (uint32_t)(e / mn), r = (uint32_t)(e - (int64_t)b * mn);
  const uint32_t m = r / p.N;
  double* dst = p.C + b * p.c_b + off2(p.cm, m) + off2(p.cn, r - m * p.N);
  double v = p.alpha * s;
  if (p.beta != 0.0) v += p.beta * *dst;
  *dst = v;
}

template <typename T, int BM, int BN, int WM, int WN, typename Off, int V>
static void launch_tile(const TileGemm<T>& p, int64_t batch, bool akf, bool bkf, hipStream_t s) {
  constexpr int BK = 16, NT = 64 * (BM / WM) * (BN / WN);
  // a launch has under 2^32 threads along x (outputs of a row or two with 2^30 columns have more): z takes the rest
  const int64_t tiles = ceil_div(p.M, BM) * ceil_div(p.N, BN), gx = std::min<int64_t>(tiles, ((1ll << 32) - 1) / NT);
  const dim3 grid((unsigned)gx, (unsigned)(batch * p.splits), (unsigned)ceil_div(tiles, gx));
  if (akf && bkf) tile_gemm_kernel<T, BM, BN, WM, WN, BK, true, true, Off, V><<<grid, NT, 0, s>>>(p);
  else if (akf) tile_gemm_kernel<T, BM, BN, WM, WN, BK, true, false, Off, V><<<grid, NT, 0, s>>>(p);
  else if (bkf) tile_gemm_kernel<T, BM, BN, WM, WN, BK, false, true, Off, V><<<grid, NT, 0, s>>>(p);
  else tile_gemm_kernel<T, BM, BN, WM, WN, BK, false, false, Off, V><<<grid, NT, 0, s>>>(p);
  CCX_HIP(hipGetLastError());
}

template <typename T, typename Off, int V>
static void launch_tile(int tile, const TileGemm<T>& p, int64_t batch, bool akf, bool bkf, hipStream_t s) {
  if (tile == 64) launch_tile<T, 64, 64, 32, 32, Off, V>(p, batch, akf, bkf, s);
  else launch_tile<T, 128, 128, 64, 32, Off, V>(p, batch, akf, bkf, s);
}

// Largest element offset of a 2-level index over `extent` values; negative when a stride is.
static int64_t span(const Idx2& d, int64_t extent) {
  if (d.s1 < 0 || d.s2 < 0) return -1;
  const int64_t q = (extent - 1) / d.n2;
  return q * d.s1 + (std::min(extent, d.n2) - 1) * d.s2;
}

// C = alpha * sum_s work[s] + beta * C, in a fixed summation order (deterministic).
//
// Bound by the latency of its loads when the output is small and the split count large (13 x 13 sums
// of 252 partials): a thread that walks its element's partials alone has one chain of them. A block
// therefore takes 64 consecutive elements and RED_G wave-groups; group g sums the partials g,
// g + G, ... with 8 loads in flight, and the groups' sums meet in LDS in the order of g. G = 1 keeps
// one thread per element, its partials in ascending order, 8 loads in flight (FP32 takes only this form,
// whose rounding does not depend on the launch). Measured (FP64): 169 elements of 252 splits 64 -> 5 us,
// 1313 elements of 71 splits 20 -> 4.6 us (of which 4 us is what any launch takes in the trace); 1.7 M
// elements of 9 splits stay at 27 us, 5.1 TB/s.
template <typename T, int G>
__global__ __launch_bounds__(G == 1 ? 256 : 64 * G) void splitk_reduce_kernel(GemmParams<T> p, const T* __restrict__ work,
                                                                             int splits) {
  const int64_t total = p.batch * p.M * p.N;
  __shared__ T part[G == 1 ? 1 : G][G == 1 ? 1 : 64];
  const int g = G == 1 ? 0 : threadIdx.x >> 6;
  const int64_t e = G == 1 ? blockIdx.x * (int64_t)256 + threadIdx.x : blockIdx.x * (int64_t)64 + (threadIdx.x & 63);
  T s = 0;
  if (e < total) {
    const T* w = work + e;
    int k = g;
    for (; k + 7 * G < splits; k += 8 * G) {
      T x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = w[(int64_t)(k + u * G) * total];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += x[u];
    }
    for (; k < splits; k += G) s += w[(int64_t)k * total];
  }
  if constexpr (G > 1) {
    part[g][threadIdx.x & 63] = s;
    __syncthreads();
    if (g > 0) return;
    s = 0;
#pragma unroll
    for (int u = 0; u < G; ++u) s += part[u][threadIdx.x];
  }
  if (e >= total) return;
  const uint32_t mn = (uint32_t)(p.M * p.N);
  const uint32_t b = p.batch == 1 ? 0u : (uint32_t)(e / mn);
  const uint32_t r = (uint32_t)(e - (int64_t)b * mn);
  const uint32_t m = r / (uint32_t)p.N, n = r - m * (uint32_t)p.N;
  T* dst = p.C + b * p.c_b + off2(p.cm, m) + off2(p.cn, n);
  T v = p.alpha * s;
  if (p.beta != T(0)) v += p.beta * *dst;
  *dst = v;
}

// G so that the launch has about 1024 waves or each group 4 partials left, whichever comes first.
template <typename T>
static void splitk_reduce(const GemmParams<T>& p, const T* work, int splits, hipStream_t s) {
  const int64_t total = p.batch * p.M * p.N;
  CCX_CHECK(p.M * p.N < (1ll << 32) && ceil_div(total, 64) < (1ll << 31), ERR_ARG, "split-K output too large");
  const int64_t waves = ceil_div(total, 64);
  if (sizeof(T) == 8 && waves < 256 && splits >= 32)
    splitk_reduce_kernel<T, 16><<<(unsigned)waves, 1024, 0, s>>>(p, work, splits);
  else if (sizeof(T) == 8 && waves < 1024 && splits > FIXED_K_SPLITS)
    splitk_reduce_kernel<T, 4><<<(unsigned)waves, 256, 0, s>>>(p, work, splits);
  else
    splitk_reduce_kernel<T, 1><<<(unsigned)ceil_div(total, 256), 256, 0, s>>>(p, work, splits);
  CCX_HIP(hipGetLastError());
}

// Plain GEMM, split along K into workspace partials when its tile grid cannot fill the chip.
template <typename T>
static void plain_dispatch(const PlainGemm<T>& q, Workspace& ws, hipStream_t s) {
  const int64_t BKp = sizeof(T) == 8 ? 16 : 32;
  const int64_t tiles = ceil_div(q.M, 128) * ceil_div(q.N, 128);
  int64_t splits = 1;
  if (q.batch == 1 && tiles < 768) {
    splits = std::min<int64_t>(ceil_div(1024, tiles), std::min<int64_t>(q.K / (BKp * 16), 64));
    const size_t one = (size_t)q.M * q.N * sizeof(T);
    splits = std::min<int64_t>(splits, (int64_t)(ws.limit / one));
  }
  if (splits > 1) {
    const int64_t kchunk = ceil_div(ceil_div(q.K, splits), BKp) * BKp;
    splits = ceil_div(q.K, kchunk);
  }
  if (std::getenv("CCX_TRACE"))
    std::fprintf(stderr, "[ccx]   -> plain %s%s batch %lld splits %lld\n", q.a_kc ? "N" : "T", q.b_nc ? "N" : "T",
                 (long long)q.batch, (long long)splits);
  if (splits <= 1) {
    plain_gemm<T>(q, s);
    return;
  }
  const int64_t kchunk = ceil_div(ceil_div(q.K, splits), BKp) * BKp;
  T* work = (T*)ws.get((size_t)splits * q.M * q.N * sizeof(T));
  PlainGemm<T> w = q;
  w.batch = splits;
  w.ktot = q.K;
  w.K = kchunk;
  w.a_b = q.a_kc ? kchunk : kchunk * q.lda;
  w.b_b = q.b_nc ? kchunk * q.ldb : kchunk;
  w.C = work;
  w.ldc = q.N;
  w.c_b = q.M * q.N;
  w.alpha = T(1);
  w.beta = T(0);
  plain_gemm<T>(w, s);
  GemmParams<T> r;
  r.M = q.M;
  r.N = q.N;
  r.C = q.C;
  r.cm = Idx2{q.M, 0, q.ldc};
  r.cn = Idx2{q.N, 0, 1};
  r.alpha = q.alpha;
  r.beta = q.beta;
  splitk_reduce<T>(r, work, (int)splits, s);
}

// Single stride of a 2-level index over `extent` values, or -1 when it is not a plain stride.
static int64_t plain_stride(const Idx2& d, int64_t extent) {
  if (extent <= 1) return 0;
  if (extent <= d.n2) return d.s2;
  if (d.s1 == d.n2 * d.s2) return d.s2;
  return -1;
}

// Express the contraction as a plain strided GEMM when every operand is an ordinary matrix.
template <typename T>
static bool as_plain(const GemmParams<T>& p, PlainGemm<T>& q) {
  const int64_t am = plain_stride(p.am, p.M), ak = plain_stride(p.ak, p.K);
  const int64_t bk = plain_stride(p.bk, p.K), bn = plain_stride(p.bn, p.N);
  const int64_t cm = plain_stride(p.cm, p.M), cn = plain_stride(p.cn, p.N);
  if (am < 0 || ak < 0 || bk < 0 || bn < 0 || cm < 0 || cn < 0 || p.K < 1) return false;
  q = PlainGemm<T>{};
  q.batch = p.batch;
  q.alpha = p.alpha;
  q.beta = p.beta;
  if (cn == 1 || p.N == 1) {          // C row-major
    q.M = p.M; q.N = p.N; q.K = p.K;
    q.A = p.A; q.B = p.B; q.C = p.C;
    q.a_b = p.a_b; q.b_b = p.b_b; q.c_b = p.c_b;
    q.ldc = cm;
    if (ak == 1) { q.a_kc = true; q.lda = am; } else if (am == 1) { q.a_kc = false; q.lda = ak; } else return false;
    if (bn == 1) { q.b_nc = true; q.ldb = bk; } else if (bk == 1) { q.b_nc = false; q.ldb = bn; } else return false;
  } else if (cm == 1) {               // C column-major: C^T = B^T A^T
    q.M = p.N; q.N = p.M; q.K = p.K;
    q.A = p.B; q.B = p.A; q.C = p.C;
    q.a_b = p.b_b; q.b_b = p.a_b; q.c_b = p.c_b;
    q.ldc = cn;
    if (bk == 1) { q.a_kc = true; q.lda = bn; } else if (bn == 1) { q.a_kc = false; q.lda = bk; } else return false;
    if (am == 1) { q.b_nc = true; q.ldb = ak; } else if (ak == 1) { q.b_nc = false; q.ldb = am; } else return false;
  } else {
    return false;
  }
  if (q.lda < 1 || q.ldb < 1 || q.ldc < 1) return false;
  return plain_gemm_ok(q);
}

// Whether p runs on the plain-matrix kernel: enough 128 x 128 tiles to fill the 256 CUs
template <typename T>
static bool takes_plain(const GemmParams<T>& p, PlainGemm<T>& q) {
  return p.kx == 1 && ceil_div(p.M, 128) * ceil_div(p.N, 128) * p.batch >= 240 && as_plain(p, q);
}

// Tile and split count of an FP64 contraction: the cheapest of both tiles and a few split counts under a model of the
// launch. It is fitted to the times of every tile and split count of 150 contractions from 5 x 5 x 1805 to 5632^3 (plain
// and compound, one row to square, K from 13 to 410571); the plan that it takes is 0.8% from the best of them in the
// mean and 7% at most (1024^3: 128 x 128 in 4, 57 us; 64 x 64 unsplit 77; 1313^3 125 to 130 against 158; 3072^3 1042
// against 1129; 1 x 40000 x 2400: 64 x 64 in 4, 154 us, in 30 187, unsplit 198). A launch costs 5 us; a k-tile takes 0.26
// (64 x 64) or 0.49 us (128 x 128) a round of resident work-groups plus its flops at 0.205 or 0.252 TF a CU, and at least
// the latency of its loads, 1.05 us a round; the operands come at 5.7 TB/s beside it; partial sums, which mostly stay in
// the caches, move at 7.4 TB/s behind a launch that gains its 8 us (4 to 9 fit alike; with 4 products of 10 us were split).
//
// Where an operand is not contiguous along either index that its lanes could walk (two summed indices, each contiguous in
// another operand), every lane reads a line of its own, which later k-tiles have to find in cache. Past two 64 x 64
// work-groups a CU that fails for these, whose panels are read twice as often (5120^3 of o=32 v=160: 20.1 ms, 128 x 128 6.0
// to 6.6; 576 x 576 x 22500 1.5 and 0.96), and it fails the sooner the longer the work-groups that share a panel run apart: 4% per doubling of a split's
// k-tiles over 40, which gives 2048^3 two parts and 4960^3 five (8.8 ms unsplit, in 4 8.0, in 8 7.6).
struct Plan {
  int tile = 128, splits = 1, chunk = 0;
};
// CU time of a contraction on 64 x 64 tiles, of which only the 16 x 16 blocks that hold outputs are computed
static double tile64_us(const GemmParams<double>& p) {
  const double blocks = (double)ceil_div(p.M, 16) * (double)ceil_div(p.N, 16) * (double)p.batch;
  return blocks * (double)std::max<int64_t>(1, ceil_div(p.K, 16) * p.kx) * (2.0 * 16 * 16 * 16 / 0.24e6);
}
static Plan plan_f64(const GemmParams<double>& p, size_t limit) {
  static const int counts[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64, 96, 128, 192, 256};
  const int64_t ntk = std::max<int64_t>(1, ceil_div(p.K, 16) * p.kx);
  // lanes walk k wherever rows are not contiguous (form_of)
  const bool strided = (p.am.s2 != 1 && p.ak.s2 != 1) || (p.bn.s2 != 1 && p.bk.s2 != 1);
  const bool cached = strided && p.M > 64 && p.N > 64;
  const double t_load = 8.0 * (double)p.batch * ((double)(p.K * p.kx) * (double)(p.M + p.N) + (double)p.M * (double)p.N) / 5.7e6;
  Plan best;
  double t_best = 0.0;
  for (int tile : {128, 64}) {
    const int64_t tiles = ceil_div(p.M, tile) * ceil_div(p.N, tile) * p.batch;
    const double t_ktile = tile == 64 ? 1.17 * tile64_us(p) / (double)(tiles * ntk) : 2.0 * tile * tile * 16 / 0.252e6;
    const int per_cu = tile == 128 ? 2 : 4;   // resident work-groups (LDS)
    for (int want : counts) {
      const int64_t chunk = ceil_div(ntk, want), splits = ceil_div(ntk, chunk);
      if (want > 1 && (chunk < 4 || splits * p.batch > 65535)) break;
      const double bytes = 8.0 * (double)splits * (double)p.batch * (double)p.M * (double)p.N;
      if (want > 1 && bytes > (double)limit) break;
      if (cached && tile == 64 && tiles * splits > 512) break;
      const int64_t on_cu = ceil_div(tiles * splits, 256);
      const double rounds = (double)ceil_div(on_cu, per_cu), busy = (double)on_cu * t_ktile;
      const double work = (double)chunk * (tile == 64 ? std::max(1.05 * rounds, 0.26 * rounds + busy) : 0.49 * rounds + busy);
      double t = 5.0 + std::max(work, t_load) + 0.05 * std::min(work, t_load);
      if (splits > 1) t += 8.0 + 2.0 * bytes / 7.4e6;
      if (cached && chunk > 40) t *= 1.0 + 0.04 * std::log2((double)chunk / 40.0);
      if (t_best == 0.0 || t < t_best) {
        t_best = t;
        best.tile = tile;
        best.splits = (int)splits;
        best.chunk = (int)chunk;
      }
    }
  }
  return best;
}

// The K partition by the shape alone, where it is part of the result: FP32 sums, and FP64 sums that are rounded to FP32
// or split FP16 operands. About 1024 work-groups, at least 8 k-tiles per split, at most 256 splits.
template <typename T>
static Plan plan_fixed(const GemmParams<T>& p, size_t limit) {
  Plan r;
  r.tile = p.M <= 64 || p.N <= 64 ? 64 : 128;
  const int64_t ntk = ceil_div(p.K, 16) * p.kx;
  const int64_t tiles = ceil_div(p.M, r.tile) * ceil_div(p.N, r.tile) * p.batch;
  int64_t splits = 1, kchunk = p.K;
  if (p.K > 0 && tiles < 1024) {
    splits = std::max<int64_t>(1, std::min<int64_t>(ceil_div(1024, tiles), std::min<int64_t>(p.K * p.kx / 128, 256)));
    splits = std::max<int64_t>(1, std::min<int64_t>(splits, 65535 / p.batch));
  }
  if (splits > 1) {
    kchunk = ceil_div(ntk, splits);
    splits = ceil_div(ntk, kchunk);
    const size_t one = (size_t)p.batch * p.M * p.N * sizeof(T);
    if ((size_t)splits * one > limit) {   // keep the workspace bounded; fall back to fewer splits
      splits = (int64_t)std::max<size_t>(1, limit / one);
      kchunk = ceil_div(ntk, splits);
      splits = ceil_div(ntk, kchunk);
    }
  }
  if (splits <= 1) kchunk = ntk;
  r.splits = (int)std::max<int64_t>(splits, 1);
  r.chunk = (int)kchunk;
  return r;
}
static Plan plan(const GemmParams<float>& p, const Workspace& ws) {
  Plan f = plan_fixed(p, ws.limit);
  // the tile is free: 128 x 128 reach 100 TF of padded work at 2793^3, 64 x 64 93, so these where they pad 7% less (190
  // x 13671 x 10878: 862 to 615 us; 549^3: 22 to 17)
  if (f.tile == 128 && 25 * ceil_div(p.M, 64) * ceil_div(p.N, 64) < 93 * ceil_div(p.M, 128) * ceil_div(p.N, 128)) f.tile = 64;
  return f;
}
// Splits of a member of a group whose work is `group_us` over the whole chip: chains of k-tiles of half that time (1.4
// us a k-tile with two work-groups on the CU), so that the blocks of all members pack, but no shorter than 4 us, and
// partial sums that move (4 TB/s) in a third of it. A 549 x 549 x 549 product among small ones then splits in 3:
// 53 to 39 us for that launch (each member planned for an equal share of the chip left it unsplit).
static Plan plan_member(const GemmParams<double>& p, size_t limit, double group_us) {
  Plan r;
  r.tile = 64;
  const int64_t ntk = std::max<int64_t>(1, ceil_div(p.K, 16) * p.kx);
  const double one = 8.0 * (double)p.batch * (double)p.M * (double)p.N;
  const double target = std::max(8.0, group_us);
  const int64_t room = std::min<int64_t>((int64_t)((double)limit / one), 65535 / p.batch);
  const int64_t cheap = (int64_t)(target / 3 * 4.0e6 / (2.0 * one));
  int64_t splits = ceil_div(ntk, std::max<int64_t>(4, (int64_t)(target / 2.8)));
  splits = std::max<int64_t>(1, std::min({splits, room, std::max<int64_t>(cheap, 1), (int64_t)256}));
  r.chunk = (int)ceil_div(ntk, splits);
  r.splits = (int)ceil_div(ntk, r.chunk);
  return r;
}
// group_us: the work of the group that it is launched in, 0 for a launch of its own
static Plan plan(const GemmParams<double>& p, const Workspace& ws, double group_us = 0.0) {
  if (ws.fixed_k) {
    Plan f = plan_fixed(p, ws.limit);
    if (f.splits <= FIXED_K_SPLITS) {   // the tile is free
      if (ceil_div(p.M, 128) * ceil_div(p.N, 128) * p.batch * f.splits < 512 || group_us > 0) f.tile = 64;
      return f;
    }
  }
  return group_us > 0 ? plan_member(p, ws.limit, group_us) : plan_f64(p, ws.limit);
}

// How a contraction is loaded: which operands are k-fast, lane offsets in 32 bits, pairs.
struct Form {
  bool akf, bkf, off32, two;
};
template <typename T>
static Form form_of(const GemmParams<T>& p, int tile) {
  Form f;
  // A is "k-fast" when its inner k index is contiguous (coalesced loads along k); otherwise the
  // loader walks along m. Same for B with n.
  f.akf = !(p.am.s2 == 1 && p.ak.s2 != 1);
  f.bkf = !(p.bn.s2 == 1 && p.bk.s2 != 1);
  // lane offsets in 32 bits: what a lane adds to the uniform base stays under 4 GiB -- the rows, and k where it is
  // not the same in a whole wave (k-fast, and pairs of rows in a 64-wide tile)
  auto narrow = [&](const Idx2& r, int64_t nr, const Idx2& k, bool with_k) {
    const int64_t a = span(r, nr), b = with_k ? span(k, std::max<int64_t>(p.K, 1)) : 0;
    return a >= 0 && b >= 0 && (a + b + 1) * (int64_t)sizeof(T) <= (1ll << 32);
  };
  f.off32 = narrow(p.am, p.M, p.ak, f.akf) && narrow(p.bn, p.N, p.bk, f.bkf);
  // pairs along the contiguous index of both operands
  auto pairs = [](const Idx2& d, int64_t n) { return d.s2 == 1 && n >= 2 && (d.n2 % 2 == 0 || n <= d.n2); };
  f.two = f.off32 &&
          (tile == 128 || (narrow(p.am, p.M, p.ak, true) && narrow(p.bn, p.N, p.bk, true))) &&
          pairs(f.akf ? p.ak : p.am, f.akf ? p.K : p.M) && pairs(f.bkf ? p.bk : p.bn, f.bkf ? p.K : p.N);
  return f;
}

template <typename T>
static TileGemm<T> describe(const GemmParams<T>& p, const Plan& pl) {
  TileGemm<T> g;
  g.M = (uint32_t)p.M;
  g.N = (uint32_t)p.N;
  g.K = (uint32_t)p.K;
  g.kx = (int)p.kx;
  g.splits = pl.splits;
  g.chunk = pl.chunk;
  g.am = fast_idx(p.am);
  g.ak = fast_idx(p.ak);
  g.bk = fast_idx(p.bk);
  g.bn = fast_idx(p.bn);
  g.cm = fast_idx(p.cm);
  g.cn = fast_idx(p.cn);
  g.a_x = p.a_x;
  g.b_x = p.b_x;
  g.a_b = p.a_b;
  g.b_b = p.b_b;
  g.c_b = p.c_b;
  g.alpha = p.alpha;
  g.beta = p.beta;
  g.A = p.A;
  g.B = p.B;
  g.C = p.C;
  g.work = nullptr;
  return g;
}

template <typename T>
static void check_extents(const GemmParams<T>& p) {
  CCX_CHECK(p.M < (1ll << 31) && p.N < (1ll << 31) && p.K < (1ll << 31) && p.K * p.kx < (1ll << 31), ERR_ARG,
            "gemm extent too large");
  CCX_CHECK(p.batch < 65536, ERR_ARG, "gemm batch too large");
}

// p as the planner and the kernels take it: an empty sum (K = 0: C = beta C) has any index of extent one, which the
// empty loop over k never reads, so that nobody divides by an extent of zero.
template <typename T>
static GemmParams<T> summable(GemmParams<T> p) {
  if (p.K == 0 || p.kx == 0) {
    p.K = 0;
    p.kx = 1;
    p.a_x = p.b_x = 0;
    p.ak = p.bk = Idx2{1, 0, 0};
  }
  return p;
}

template <typename T>
void tc_gemm(const GemmParams<T>& given, Workspace& ws, hipStream_t s) {
  const GemmParams<T> p = summable(given);
  if (p.M == 0 || p.N == 0 || p.batch == 0) return;
  PlainGemm<T> q;
  if (takes_plain(p, q)) {
    plain_dispatch<T>(q, ws, s);
    return;
  }
  check_extents(p);
  const Plan pl = plan(p, ws);
  CCX_CHECK(ceil_div(p.M, pl.tile) * ceil_div(p.N, pl.tile) < (1ll << 31), ERR_ARG, "gemm grid too large");
  TileGemm<T> g = describe(p, pl);
  if (pl.splits > 1) g.work = (T*)ws.get((size_t)pl.splits * p.batch * p.M * p.N * sizeof(T));
  const Form f = form_of(p, pl.tile);
  if (std::getenv("CCX_TRACE"))
    std::fprintf(stderr, "[ccx]   -> tile %d%s%s batch %lld splits %d\n", pl.tile, f.akf ? " Ak" : " Am",
                 f.bkf ? " Bk" : " Bn", (long long)p.batch, pl.splits);
  if (f.two) launch_tile<T, uint32_t, 2>(pl.tile, g, p.batch, f.akf, f.bkf, s);
  else if (f.off32) launch_tile<T, uint32_t, 1>(pl.tile, g, p.batch, f.akf, f.bkf, s);
  else launch_tile<T, int64_t, 1>(pl.tile, g, p.batch, f.akf, f.bkf, s);
  if (pl.splits > 1) splitk_reduce<T>(p, g.work, pl.splits, s);
}

// ---- GemmQueue ------------------------------------------------------------------------------------
namespace {
// addresses [lo, hi) that an operand spans
struct Range {
  uintptr_t lo = 0, hi = 0;
  bool meets(const Range& o) const { return lo < o.hi && o.lo < hi; }
};
Range range_of(const double* base, std::initializer_list<std::pair<int64_t, int64_t>> dims) {
  int64_t lo = 0, hi = 0;   // (extent, stride)
  for (auto& d : dims) {
    const int64_t e = (d.first - 1) * d.second;
    (e < 0 ? lo : hi) += e;
  }
  return Range{(uintptr_t)(base + lo), (uintptr_t)(base + hi + 1)};
}
Range range_of(const double* base, const Idx2& r, int64_t nr, const Idx2& c, int64_t nc, int64_t nx, int64_t sx, int64_t nb,
               int64_t sb) {
  return range_of(base, {{std::min(nr, r.n2), r.s2}, {(nr - 1) / r.n2 + 1, r.s1}, {std::min(nc, c.n2), c.s2},
                         {(nc - 1) / c.n2 + 1, c.s1}, {nx, sx}, {nb, sb}});
}
}  // namespace

struct GemmQueue::Op {
  GemmParams<double> p;
  Range a, b, c;
  int part;
};
struct GemmQueue::Elt {
  EltOp op;
  Range a, c;
};

GemmQueue::GemmQueue(Workspace& w, hipStream_t st) : ws(w), s(st) {}
GemmQueue::~GemmQueue() {}

void GemmQueue::axpby(const EltOp& e, int64_t n) {
  if (n == 0) return;
  Elt x{e, Range{}, Range{}};
  auto range = [&](const double* p, const int64_t* str) {
    int64_t hi = 0;
    for (int k = 0; k < e.rank; ++k) hi += (e.ext[k] - 1) * str[k];
    return Range{(uintptr_t)p, (uintptr_t)(p + hi + 1)};
  };
  if (e.A) x.a = range(e.A, e.sa);
  x.c = range(e.C, e.sc);
  bool clash = false;   // it runs before the queued contractions, and beside the queued elementwise ones
  for (auto& o : ops) clash = clash || x.c.meets(o.a) || x.c.meets(o.b) || x.c.meets(o.c) || x.a.meets(o.c);
  for (auto& o : elts) clash = clash || x.c.meets(o.a) || x.c.meets(o.c) || x.a.meets(o.c);
  if (clash) flush();
  elts.push_back(x);
}

void GemmQueue::gemm(const GemmParams<double>& given, int part) {
  const GemmParams<double> p = summable(given);
  if (p.M == 0 || p.N == 0 || p.batch == 0) return;
  check_extents(p);
  Op o{p, Range{}, Range{}, range_of(p.C, p.cm, p.M, p.cn, p.N, 1, 0, p.batch, p.c_b), part};
  if (p.K > 0) {
    o.a = range_of(p.A, p.am, p.M, p.ak, p.K, p.kx, p.a_x, p.batch, p.a_b);
    o.b = range_of(p.B, p.bn, p.N, p.bk, p.K, p.kx, p.b_x, p.batch, p.b_b);
  }
  for (auto& q : ops) {
    const bool apart = part && q.part && part != q.part;   // the caller's word that the outputs do not meet
    if ((!apart && o.c.meets(q.c)) || o.c.meets(q.a) || o.c.meets(q.b) || o.a.meets(q.c) || o.b.meets(q.c)) {
      flush();
      break;
    }
  }
  const int64_t tiles = ceil_div(p.M, 64) * ceil_div(p.N, 64) * p.batch;
  // With fixed_k, the plain kernel's too: it has a partition of K of its own, so that whether such a contraction takes
  // it must not depend on what else is queued.
  PlainGemm<double> plain;
  if (tiles > GROUP_TILES || 2.0 * p.M * p.N * p.K * p.kx * p.batch > GROUP_FLOPS || !form_of(p, 64).off32 ||
      (ws.fixed_k && takes_plain(p, plain))) {
    // it fills the chip by itself: now, before the queued ones, which it does not meet
    bool clash = false;
    for (auto& e : elts) clash = clash || o.a.meets(e.c) || o.b.meets(e.c) || o.c.meets(e.c) || o.c.meets(e.a);
    if (clash) flush();
    tc_gemm<double>(p, ws, s);
    return;
  }
  ops.push_back(o);
}

void GemmQueue::flush() {
  if (!elts.empty()) {
    std::vector<EltOp> e;
    for (auto& x : elts) e.push_back(x.op);
    elts.clear();
    elementwise(e, s);
  }
  std::vector<Op> todo;
  todo.swap(ops);
  for (size_t at = 0; at < todo.size();) {
    if (todo.size() - at == 1) {
      tc_gemm<double>(todo[at].p, ws, s);
      return;
    }
    const size_t left = std::min<size_t>(todo.size() - at, GROUP);
    double work_us = 0.0;   // of the group, spread over the chip
    for (size_t i = at; i < at + left; ++i) work_us += tile64_us(todo[i].p) / 256;
    struct Item {
      const Op* o;
      Plan pl;
    };
    std::vector<Item> items;
    size_t bytes = 0;
    for (; items.size() < left; ++at) {
      const GemmParams<double>& p = todo[at].p;
      const Plan pl = plan(p, ws, work_us);
      const size_t w = pl.splits > 1 ? (size_t)pl.splits * p.batch * p.M * p.N * sizeof(double) : 0;
      if (!items.empty() && bytes + w > ws.limit) break;
      bytes += w;
      items.push_back(Item{&todo[at], pl});
    }
    std::stable_sort(items.begin(), items.end(), [](const Item& x, const Item& y) { return x.pl.chunk > y.pl.chunk; });
    double* work = bytes ? (double*)ws.get(bytes) : nullptr;
    GemmGroup a{};
    SumGroup r{};
    for (const Item& it : items) {
      const GemmParams<double>& p = it.o->p;
      TileGemm<double> g = describe(p, it.pl);
      const Form f = form_of(p, 64);
      const int64_t outputs = p.batch * p.M * p.N;
      if (it.pl.splits > 1) {
        g.work = work;
        work += it.pl.splits * outputs;
        r.g[r.n] = g;
        r.batch[r.n] = p.batch;
        r.first[r.n + 1] = r.first[r.n] + (int)ceil_div(outputs, it.pl.splits > FIXED_K_SPLITS ? 64 : 256);
        ++r.n;
      }
      a.g[a.n] = g;
      a.batch[a.n] = (int)p.batch;
      a.form[a.n] = (f.akf ? 1 : 0) + (f.bkf ? 2 : 0) + (f.two ? 4 : 0);
      a.first[a.n + 1] = a.first[a.n] + (int)(ceil_div(p.M, 64) * ceil_div(p.N, 64) * p.batch * it.pl.splits);
      ++a.n;
    }
    tile_group_kernel<<<(unsigned)a.first[a.n], 256, 0, s>>>(a);
    CCX_HIP(hipGetLastError());
    if (r.n) {
      sum_group_kernel<<<(unsigned)r.first[r.n], 256, 0, s>>>(r);
      CCX_HIP(hipGetLastError());
    }
  }
}

template void tc_gemm<double>(const GemmParams<double>&, Workspace&, hipStream_t);
template void tc_gemm<float>(const GemmParams<float>&, Workspace&, hipStream_t);

}  // namespace ccx
