// Primitives between the reference's host layout p[i][j][k][pl] and the device
// planes a[pl][k][j][i] (hg_set_prims, hg_get_prims and the other calls that
// move a whole state).
//
// The transposition runs on the device, straight from and to pinned host
// memory, and the host only copies contiguous pieces between that and the
// caller's array.  In this order a row i is one contiguous run of Q = m2 m3 8
// numbers; q = (j m3 + k) 8 + pl.  A state is cut into pieces of 32 rows by up
// to 8192 numbers (2 MiB): 32 rows so that the device side reads and writes
// 256 contiguous bytes.  Host threads take the pieces in turn, each with its
// own pinned slot: while one waits for its kernel the others copy, and the
// first touch of a fresh array's pages, the larger half of a large get, is
// spread over them.  A state of up to 2 MiB is one piece, one kernel and one
// wait.
//
// 256x128x64 with 6 ghost layers (182 MB): 4.2 ms in, 5.5 ms out, where one
// thread transposing on the host around a pageable copy took 71 and 77; 128^2
// with 3 (1.1 MB) 55 and 69 us against 135 and 240, 32^2 (92 kB) 20 and 20
// against 18 and 20.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

#include "harmgpu.h"
#include "hg_host.h"

using namespace hg;

namespace {

constexpr int TI = 32, TQ = 64;             // tile of the transposition
constexpr int64_t PIECE_Q = 8192;           // numbers of a row in one piece
constexpr size_t SLOT = (size_t)TI * PIECE_Q * sizeof(double);

// device offset of number q of row i = 0
__device__ __forceinline__ int64_t plane_of(const Dims &d, int64_t q) {
  const int64_t r = q >> 3;
  const int64_t j = r / d.m3, k = r - j * d.m3;
  return (q & 7) * d.spl + k * d.sk + j * d.sj;
}

// rows i0 .. i0 + ni - 1, numbers q0 .. q0 + nq - 1: host[(i - i0) nq + (q - q0)]
template <bool TO_DEVICE>
__global__ void __launch_bounds__(256) k_transpose(double *__restrict__ dev, double *__restrict__ host, Dims d, int i0,
                                                   int ni, int64_t q0, int64_t nq) {
  __shared__ double tile[TQ][TI + 1];
  const int64_t qb = (int64_t)blockIdx.x * TQ;
  const int ib = blockIdx.y * TI;
  const int t = threadIdx.x;
  // a thread's 8 numbers are all loaded before the first is stored: a state of
  // one piece waits once for the bus, not 8 times
  constexpr int NR = TI / 4, NQ = TQ / 8;
  const int64_t qh = qb + (t & 63);
  const int ih = t >> 6, id = ib + (t & 31), qd = t >> 5;
  double v[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
  static_assert(NR == 8 && NQ == 8, "256 threads");
  if (TO_DEVICE) {
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (ib + ih + 4 * r < ni && qh < nq) v[r] = host[(int64_t)(ib + ih + 4 * r) * nq + qh];
#pragma unroll
    for (int r = 0; r < NR; r++) tile[t & 63][ih + 4 * r] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NQ; r++)
      if (id < ni && qb + qd + 8 * r < nq) dev[plane_of(d, q0 + qb + qd + 8 * r) + i0 + id] = tile[qd + 8 * r][t & 31];
  } else {
#pragma unroll
    for (int r = 0; r < NQ; r++)
      if (id < ni && qb + qd + 8 * r < nq) v[r] = dev[plane_of(d, q0 + qb + qd + 8 * r) + i0 + id];
#pragma unroll
    for (int r = 0; r < NQ; r++) tile[qd + 8 * r][t & 31] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (ib + ih + 4 * r < ni && qh < nq) host[(int64_t)(ib + ih + 4 * r) * nq + qh] = tile[t & 63][ih + 4 * r];
  }
}

struct Piece {
  int i0, ni;
  int64_t q0, nq;
};

// one piece through one slot; the host's part before (to the device) or after
// the kernel
template <bool TO_DEVICE>
hipError_t move_piece(const Dims &d, double *dev, double *host, const Piece &p, HostSlot &s) {
  const int64_t Q = (int64_t)d.m2 * d.m3 * NPR;
  double *row = host + (int64_t)p.i0 * Q + p.q0, *slot = (double *)s.mem;
  const size_t len = (size_t)p.nq * sizeof(double);
  if (TO_DEVICE)
    for (int i = 0; i < p.ni; i++) memcpy(slot + i * p.nq, row + i * Q, len);
  hipLaunchKernelGGL(k_transpose<TO_DEVICE>, dim3((unsigned)((p.nq + TQ - 1) / TQ), (unsigned)((p.ni + TI - 1) / TI)),
                     dim3(256), 0, 0, dev, slot, d, p.i0, p.ni, p.q0, p.nq);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipEventRecord(s.done, 0);
  if (e == hipSuccess) e = hipEventSynchronize(s.done);
  if (!TO_DEVICE && e == hipSuccess)
    for (int i = 0; i < p.ni; i++) memcpy(row + i * Q, slot + i * p.nq, len);
  return e;
}

template <bool TO_DEVICE>
int move_state(hg_ctx *c, double *dev, double *host) {
  const Dims &d = c->d;
  const int64_t Q = (int64_t)d.m2 * d.m3 * NPR;
  std::vector<Piece> pieces;
  if ((size_t)d.m1 * Q * sizeof(double) <= SLOT) {
    pieces.push_back({0, d.m1, 0, Q});
  } else {
    for (int64_t q = 0; q < Q; q += PIECE_Q)
      for (int i = 0; i < d.m1; i += TI)
        pieces.push_back({i, d.m1 - i < TI ? d.m1 - i : TI, q, Q - q < PIECE_Q ? Q - q : PIECE_Q});
  }
  // two calls on one context share its slots
  std::lock_guard<std::mutex> lk(c->slots_mu);
  // the kernels run where the state is, whichever device the caller has set
  int caller = c->device;
  (void)hipGetDevice(&caller);
  hipError_t e = caller == c->device ? hipSuccess : hipSetDevice(c->device);
  const size_t bytes = pieces.size() == 1 ? (size_t)d.m1 * Q * sizeof(double) : SLOT;
  size_t want = pieces.size() < (size_t)HOST_SLOTS ? pieces.size() : (size_t)HOST_SLOTS;
  for (size_t k = 0; k < want && e == hipSuccess; k++) {
    HostSlot &s = c->slots[k];
    if (!s.mem) {
      if (!s.done) e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
      if (e == hipSuccess) e = hipHostMalloc(&s.mem, bytes, hipHostMallocDefault);
      if (e != hipSuccess) {
        s.mem = nullptr;
        if (k == 0) break;
        want = k;  // fewer slots, fewer threads
        e = hipSuccess;
        (void)hipGetLastError();
      }
    }
  }
  if (e == hipSuccess) {
    std::atomic<size_t> next{0};
    std::vector<hipError_t> err(want, hipSuccess);
    auto work = [&](size_t k) {
      if (k) err[k] = hipSetDevice(c->device);  // a new thread starts on device 0
      for (size_t n; err[k] == hipSuccess && (n = next.fetch_add(1)) < pieces.size();)
        err[k] = move_piece<TO_DEVICE>(d, dev, host, pieces[n], c->slots[k]);
    };
    std::vector<std::thread> team;
    try {
      team.reserve(want);
      for (size_t k = 1; k < want; k++) team.emplace_back(work, k);
    } catch (...) {
      // no further threads: those there are take every piece
    }
    work(0);
    for (auto &t : team) t.join();
    for (hipError_t k : err)
      if (e == hipSuccess) e = k;
  }
  if (caller != c->device) (void)hipSetDevice(caller);
  if (e != hipSuccess) {
    set_error("copying a state: %s", hipGetErrorString(e));
    return 1;
  }
  return 0;
}

}  // namespace

int hg::copy_prims(hg_ctx *c, double *dev, const double *host) {
  return move_state<true>(c, dev, const_cast<double *>(host));
}

int hg::fetch_prims(hg_ctx *c, const double *dev, double *host) {
  return move_state<false>(c, const_cast<double *>(dev), host);
}

void hg::slots_free(hg_ctx *c) {
  for (HostSlot &s : c->slots) {
    if (s.mem) (void)hipHostFree(s.mem);
    if (s.done) (void)hipEventDestroy(s.done);
  }
}
