// fs_xfer.hip - copies between the caller's host arrays and device memory.
//
// The caller's arrays are pageable, and the runtime copies such memory through its own staging
// buffer with one thread: 10 GB/s, so that reading back 32 M particles (1.5 GB) took 150 ms, as
// long as seven substeps with multigrid. Here each copy goes through pinned slots of the context,
// two per lane, in pieces of XFER_PIECE bytes: while the link fills one slot of a lane, a host
// thread empties the other. Up to XFER_LANES lanes work side by side, each a host thread, so that
// the page faults of a fresh destination and the host's copies, not the link, are what they share.
// In mixed precision the pieces cross the link in FP32 and the host thread widens or narrows them
// (the same rounding as on the device), which halves the bytes on the link and needs no FP64 copy
// in device memory.
//
// The threads live for one call. A lane waits for its own events before it returns, so no slot is
// in use between calls and the caller's arrays are never held on to.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <string>
#include <thread>
#include <vector>
#include <xmmintrin.h>

#include "fs_ctx.h"

namespace {

constexpr size_t XFER_PIECE = (size_t)1 << 20;      // device bytes per piece
constexpr size_t XFER_PER_LANE = (size_t)2 << 20;   // bytes of a copy that are worth another lane

struct Job {
  char* dev;
  char* host;
  size_t n;       // elements of `edev` bytes on the device
  size_t piece0;  // its first piece in the call
};

// Conversions as the device makes them (round to nearest, denormals kept), whatever the caller has set.
struct DefaultFp {
  unsigned csr = _mm_getcsr();
  DefaultFp() { _mm_setcsr(0x1F80); }
  ~DefaultFp() { _mm_setcsr(csr); }
};
void widen(double* d, const float* s, size_t n) {
  const DefaultFp fp;
  for (size_t i = 0; i < n; i++) d[i] = (double)s[i];
}
void narrow(float* d, const double* s, size_t n) {
  const DefaultFp fp;
  for (size_t i = 0; i < n; i++) d[i] = (float)s[i];
}

// One lane over its pieces (lane, lane + nlanes, ..) of all jobs.
hipError_t run_lane(fs_ctx* c, const std::vector<Job>& jobs, size_t npieces, size_t edev, size_t ehost, bool to_host,
                    XferLane& L, int lane, int nlanes) {
  hipError_t e = hipSetDevice(c->device);
  if (e != hipSuccess) return e;
  const size_t per = XFER_PIECE / edev;  // elements per piece
  struct Piece {
    char *dev, *host;
    size_t n;
  };
  auto piece = [&](size_t p) {
    size_t j = 0;
    while (j + 1 < jobs.size() && p >= jobs[j + 1].piece0) j++;
    const size_t at = (p - jobs[j].piece0) * per;
    return Piece{jobs[j].dev + at * edev, jobs[j].host + at * ehost, std::min(per, jobs[j].n - at)};
  };
  bool busy[2] = {false, false};
  auto wait = [&](int s) {
    if (!busy[s]) return hipSuccess;
    busy[s] = false;
    return hipEventSynchronize(L.ev[s]);
  };
  auto finish = [&](hipError_t st) {  // leave no slot in flight
    for (int s = 0; s < 2; s++) {
      const hipError_t w = wait(s);
      if (st == hipSuccess) st = w;
    }
    return st;
  };
  if (to_host) {
    auto issue = [&](size_t p, int s) {
      const Piece q = piece(p);
      hipError_t r = hipMemcpyAsync(L.slot[s], q.dev, q.n * edev, hipMemcpyDeviceToHost, c->stream);
      if (r == hipSuccess) r = hipEventRecord(L.ev[s], c->stream);
      busy[s] = r == hipSuccess;
      return r;
    };
    size_t next = lane;
    for (int s = 0; s < 2 && next < npieces; s++, next += nlanes)
      if ((e = issue(next, s)) != hipSuccess) return finish(e);
    int s = 0;
    for (size_t p = lane; p < npieces; p += nlanes, s ^= 1) {
      if ((e = wait(s)) != hipSuccess) return finish(e);
      const Piece q = piece(p);
      if (edev == ehost) std::memcpy(q.host, L.slot[s], q.n * edev);
      else widen(reinterpret_cast<double*>(q.host), static_cast<const float*>(L.slot[s]), q.n);
      if (next < npieces) {
        if ((e = issue(next, s)) != hipSuccess) return finish(e);
        next += nlanes;
      }
    }
    return finish(hipSuccess);
  }
  int s = 0;
  for (size_t p = lane; p < npieces; p += nlanes, s ^= 1) {
    if ((e = wait(s)) != hipSuccess) return finish(e);
    const Piece q = piece(p);
    if (edev == ehost) std::memcpy(L.slot[s], q.host, q.n * edev);
    else narrow(static_cast<float*>(L.slot[s]), reinterpret_cast<const double*>(q.host), q.n);
    e = hipMemcpyAsync(q.dev, L.slot[s], q.n * edev, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipEventRecord(L.ev[s], c->stream);
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(c->stream);  // the copy may be queued without its event
      return finish(e);
    }
    busy[s] = true;
  }
  return finish(hipSuccess);
}

int open_lane(fs_ctx* c, XferLane& L) {
  if (!L.slot[0]) {
    FS_HIP(c, hipHostMalloc(&L.slot[0], 2 * XFER_PIECE, hipHostMallocDefault));
    L.slot[1] = static_cast<char*>(L.slot[0]) + XFER_PIECE;
  }
  for (int s = 0; s < 2; s++) {
    if (!L.ev_ok[s]) FS_HIP(c, hipEventCreateWithFlags(&L.ev[s], hipEventDisableTiming));
    L.ev_ok[s] = true;
  }
  return FS_OK;
}

int transfer(fs_ctx* c, const FsXfer* x, int nx, size_t edev, size_t ehost, bool to_host) {
  const size_t per = XFER_PIECE / edev;
  size_t npieces = 0, bytes = 0;
  hipError_t e = hipSuccess;
  try {
    std::vector<Job> jobs;
    for (int q = 0; q < nx; q++) {
      if (!x[q].host || x[q].n == 0) continue;
      jobs.push_back({static_cast<char*>(x[q].dev), static_cast<char*>(x[q].host), x[q].n, npieces});
      npieces += (x[q].n + per - 1) / per;
      bytes += x[q].n * ehost;
    }
    if (npieces == 0) {
      FS_HIP(c, hipStreamSynchronize(c->stream));
      return FS_OK;
    }
    const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
    const int nlanes = (int)std::min<size_t>({(size_t)FS_XFER_LANES, (size_t)hw, npieces, 1 + bytes / XFER_PER_LANE});
    for (int l = 0; l < nlanes; l++) FS_TRY(open_lane(c, c->xfer[l]));
    std::vector<hipError_t> st(nlanes, hipSuccess);
    std::vector<std::thread> th;
    th.reserve(nlanes);
    // the pieces of a thread that cannot be started are done here, after the lane of this thread
    int started = 1;
    for (; started < nlanes; started++) {
      const int l = started;
      try {
        th.emplace_back([&, l] { st[l] = run_lane(c, jobs, npieces, edev, ehost, to_host, c->xfer[l], l, nlanes); });
      } catch (const std::exception&) {
        break;
      }
    }
    st[0] = run_lane(c, jobs, npieces, edev, ehost, to_host, c->xfer[0], 0, nlanes);
    for (int l = started; l < nlanes; l++)
      st[l] = run_lane(c, jobs, npieces, edev, ehost, to_host, c->xfer[l], l, nlanes);
    for (std::thread& t : th) t.join();
    for (int l = 0; l < nlanes && e == hipSuccess; l++) e = st[l];
  } catch (const std::exception& ex) {
    c->set_error(std::string("transfer: ") + ex.what());
    return FS_DEVICE_ERROR;
  }
  FS_HIP(c, e);
  return FS_OK;
}

}  // namespace

int fs_xfer_to_host(fs_ctx* c, const FsXfer* x, int nx, size_t edev, size_t ehost) {
  return transfer(c, x, nx, edev, ehost, true);
}
int fs_xfer_to_device(fs_ctx* c, const FsXfer* x, int nx, size_t edev, size_t ehost) {
  return transfer(c, x, nx, edev, ehost, false);
}

void fs_xfer_release(fs_ctx* c) {
  for (XferLane& L : c->xfer) {
    if (L.slot[0]) (void)hipHostFree(L.slot[0]);
    L.slot[0] = L.slot[1] = nullptr;
    for (int s = 0; s < 2; s++) {
      if (L.ev_ok[s]) (void)hipEventDestroy(L.ev[s]);
      L.ev_ok[s] = false;
    }
  }
}

int64_t fs_first_outside(const double* p, int64_t n, const double ext[3]) {
  // blocks of whole triples, so that a block's axes are those of its index
  auto first = [&](int64_t a, int64_t b) {
    for (int64_t i = a; i < b; i += 3)
      for (int d = 0; d < 3; d++)
        if (!(p[i + d] >= 0.0 && p[i + d] <= ext[d])) return i + d;
    return n;
  };
  const int64_t per = (int64_t)3 << 17;
  const int nt = (int)std::min<int64_t>({(int64_t)FS_XFER_LANES, (n + per - 1) / per,
                                         (int64_t)std::max(1u, std::thread::hardware_concurrency())});
  if (nt <= 1) return first(0, n);
  std::atomic<int64_t> found(n);
  std::atomic<int64_t> next(0);
  auto work = [&] {
    for (int64_t a = next.fetch_add(per); a < found.load(); a = next.fetch_add(per)) {
      const int64_t f = first(a, std::min(n, a + per));
      for (int64_t o = found.load(); f < o && !found.compare_exchange_weak(o, f);) {
      }
    }
  };
  std::vector<std::thread> th;
  try {
    for (int t = 1; t < nt; t++) th.emplace_back(work);
  } catch (const std::exception&) {  // the threads there are do the rest
  }
  work();
  for (std::thread& t : th) t.join();
  return found.load();
}

int fs_upload_real(fs_ctx* c, DBuf& dst, const double* src, size_t n) {
  const FsXfer x{dst.p, const_cast<double*>(src), n};
  return fs_xfer_to_device(c, &x, 1, c->rsz, sizeof(double));
}
int fs_download_real(fs_ctx* c, const DBuf& src, double* dst, size_t n) {
  const FsXfer x{src.p, dst, n};
  return fs_xfer_to_host(c, &x, 1, c->rsz, sizeof(double));
}
