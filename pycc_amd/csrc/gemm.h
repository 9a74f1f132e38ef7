// Tensor-contraction GEMM launcher (see gemm.hip).
#pragma once
#include "common.h"
#include <algorithm>
#include <string>
#include <vector>

namespace ccx {

// Grow-only device scratch owned by a context; `limit` bounds what split-K may request. A fixed
// workspace wraps memory it does not own (size = limit): it never allocates or frees, and a request
// beyond its size is an error.
constexpr int FIXED_K_SPLITS = 8;
struct Workspace {
  void* ptr = nullptr;
  size_t size = 0;
  size_t limit = size_t(1) << 30;
  bool fixed = false;
  // FP64 sums over K in up to FIXED_K_SPLITS parts are partitioned by the shape alone, and the parts added in order: a
  // context whose FP64 results become FP32 or split FP16 operands then rounds the same operands whatever else is queued
  // beside them. (Two rules: one of the tile kernel and one of the plain-matrix kernel, whose contractions are never
  // grouped in such a context. Sums in more parts, of few outputs, follow the launch that they are in.)
  bool fixed_k = false;
  static Workspace wrap(void* p, size_t bytes) {
    Workspace w;
    w.ptr = p;
    w.size = w.limit = bytes;
    w.fixed = true;
    return w;
  }
  void* get(size_t bytes) {
    if (bytes > size) {
      CCX_CHECK(!fixed, ERR_ARG,
                "workspace request of " + std::to_string(bytes) + " bytes exceeds the fixed scratch of " +
                    std::to_string(size) + " bytes");
      if (ptr) CCX_HIP(hipFree(ptr));
      ptr = nullptr;
      size = 0;
      CCX_HIP(hipMalloc(&ptr, bytes));
      size = bytes;
    }
    return ptr;
  }
  void release() {
    if (ptr && !fixed) (void)hipFree(ptr);
    ptr = nullptr;
    size = 0;
  }
};

template <typename T>
void tc_gemm(const GemmParams<T>& p, Workspace& ws, hipStream_t s);

// One elementwise operation of a queue: C = alpha A + beta C over rank <= 6 dimensions (A null: no term).
struct EltOp {
  int rank;
  int64_t ext[6], sa[6], sc[6], total;
  double alpha, beta;
  const double* A;
  double* C;
};
// Independent elementwise operations in as few launches as they fit (contract.hip).
void elementwise(const std::vector<EltOp>& e, hipStream_t s);

// Small FP64 contractions and elementwise operations gathered into few launches. An operation is queued while it does
// not meet a queued one (none reads or writes what another writes; ranges of addresses decide) and flush() runs
// first when it does, so the results are those of the calls in program order. A contraction over GROUP_TILES 64 x 64
// tiles or GROUP_FLOPS flops fills the chip by itself and is launched when it is added. `part`: two operations with
// different nonzero parts write disjoint elements even where their ranges overlap. Whoever launches a kernel of another
// kind that meets a queued operation flushes first; a queue ends with flush().
constexpr int64_t GROUP_TILES = 8192;
constexpr double GROUP_FLOPS = 4e10;
class GemmQueue {
 public:
  GemmQueue(Workspace& ws, hipStream_t s);
  ~GemmQueue();
  GemmQueue(const GemmQueue&) = delete;
  GemmQueue& operator=(const GemmQueue&) = delete;
  void gemm(const GemmParams<double>& p, int part = 0);
  void axpby(const EltOp& e, int64_t n);
  void flush();

 private:
  struct Op;
  struct Elt;
  Workspace& ws;
  hipStream_t s;
  std::vector<Op> ops;
  std::vector<Elt> elts;
};

// Plain strided matrices (gemm_plain.hip): C[b][m * ldc + n] = alpha op(A) op(B) + beta C.
template <typename T>
struct PlainGemm {
  int64_t M = 0, N = 0, K = 0, batch = 1;
  const T* A = nullptr;
  const T* B = nullptr;
  T* C = nullptr;
  int64_t lda = 0, ldb = 0, ldc = 0;
  int64_t a_b = 0, b_b = 0, c_b = 0;
  bool a_kc = true;   // A[m * lda + k] (else A[k * lda + m])
  bool b_nc = true;   // B[k * ldb + n] (else B[n * ldb + k])
  T alpha = 1, beta = 0;
  // split-K: when ktot > 0, grid.y runs over K chunks of length K (the last one shorter), each
  // chunk is a "batch" entry (a_b / b_b advance by one chunk) and ktot is the total K.
  int64_t ktot = 0;
};
template <typename T>
bool plain_gemm_ok(const PlainGemm<T>& p);
template <typename T>
void plain_gemm(const PlainGemm<T>& p, hipStream_t s);
// Blocks of the K-concatenated product s = 0, 1, 2 (Y1, Y2, Y3) of the triple (i, j, k) = (t.x, t.y,
// t.z): (p, p2, q n + r, q2 n + r2) of [A_p | A_p2^s] . [B_(q,r) | B_(q2,r2)].
__host__ __device__ inline int4 kcat_blocks(int4 t, int s, int n) {
  const int i = t.x, j = t.y, k = t.z;
  if (s == 0) return int4{i, j, j * n + k, i * n + k};
  if (s == 1) return int4{i, k, k * n + j, i * n + j};
  return int4{j, k, k * n + i, j * n + i};
}

// Tile t of nprod such products, three to a triple: the tiles of one triple's products at the same
// rows (tm) are neighbours, so that the A rows that they share meet in an XCD's L2. Each triple
// starts at another tm (a golden-section sequence): the XCDs, which are at different triples, would
// otherwise read the same A rows at the same time.
__device__ inline void kcat_tile(int64_t t, int64_t tiles_m, int64_t tiles_n, int64_t& b, int64_t& tm, int64_t& tn) {
  const int64_t per = 3 * tiles_m * tiles_n, e = t / per, r = t - e * per;
  const int64_t m = r / (3 * tiles_n), r2 = r - m * 3 * tiles_n, q = r2 / tiles_n;
  tm = m + (((int64_t)((uint32_t)e * 2654435769u) * tiles_m) >> 32);
  if (tm >= tiles_m) tm -= tiles_m;
  b = 3 * e + q;
  tn = r2 - q * tiles_n;
}

// The FP64 (T) products of ntri triples: C[3 e + s][m][z] = sum_kk [A_p | A_p2^s][m][kk] [B | B2][z][kk]
// with the blocks of kcat_blocks(tri[e], s, n); A_p is v^2 rows and B_(q,r) v rows of Kp (a multiple
// of 8), A^s is A with its row index m = x v + y read as y v + x, C blocks are v^2 rows of ldc.
struct Kcat64 {
  int64_t v, Kp, ldc;
  int n;
  int64_t ntri;
  const double *A, *B;
  double* C;
  const int4* tri;
};
void kcat64(const Kcat64& p, hipStream_t s);

}  // namespace ccx
