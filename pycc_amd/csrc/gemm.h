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
  // context whose FP64 results become FP32 or split FP16 operands then rounds the same operands however a
  // launch is planned.
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
  bool empty() const;

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
  // K concatenation (plain_gemm_kcat; A k-contiguous, FP64): k in [K1, K) reads A2 at k - K1 and
  // row (m mod sw) sw + m / sw, the (x, y) -> (y, x) swap of a row m = x sw + y (M = sw^2); batch b
  // adds b a2_b to A2.
  const T* A2 = nullptr;
  int64_t K1 = 0, sw = 0, a2_b = 0;
};
template <typename T>
bool plain_gemm_ok(const PlainGemm<T>& p);
template <typename T>
void plain_gemm(const PlainGemm<T>& p, hipStream_t s);
// C_b = alpha [A | A2_b swapped] B_b^T + beta C_b over K = K concatenated at K1 (FP64, A and B
// k-contiguous, fields A2 .. a2_b above; K1 a multiple of 16).
void plain_gemm_kcat(const PlainGemm<double>& p, hipStream_t s);

}  // namespace ccx
