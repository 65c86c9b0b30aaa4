// Pieces shared by the C-ABI translation units (hplx_api.hip, mxp_api.hip):
// the context object, error reporting, palg validation and the panel-loop
// progress lines.
#pragma once

#include <chrono>
#include <cstdarg>
#include <cstdio>

#include "hplx_internal.hpp"

struct hplx_ctx {
  hplx::Ctx c;
};

namespace hplx {

inline int fail(Ctx& c, int code, const char* fmt, ...) {
  char    buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  c.last_error = buf;
  return code;
}

#define HIPCHK(C, expr)                                                    \
  do {                                                                     \
    hipError_t e_ = (expr);                                                \
    if(e_ != hipSuccess)                                                   \
      return hplx::fail((C), HPLX_ERR_HIP, "%s failed: %s (%s:%d)", #expr, \
                        hipGetErrorString(e_), __FILE__, __LINE__);        \
  } while(0)

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Timing-disabled event i of the context's cross-stream pool (created on
// first use).
inline int sync_event(Ctx& c, size_t i, hipEvent_t* e) {
  while(c.ev_sync.size() <= i) {
    hipEvent_t x;
    const hipError_t r = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    if(r != hipSuccess)
      return fail(c, HPLX_ERR_HIP, "hipEventCreateWithFlags: %s",
                  hipGetErrorString(r));
    c.ev_sync.push_back(x);
  }
  *e = c.ev_sync[i];
  return HPLX_SUCCESS;
}

// Room for the times of a factorisation of `panels` panels: of its updates
// (buf 0), or of its interchanges and panels (buf 1).  Nothing is counted in a
// buffer from here on, whether or not it is replaced.
inline int reserve_stamps(Ctx& c, int buf, int panels) {
  if(buf == 0) {
    c.ev_pairs   = 0;
    c.gemm_flops = 0.0;
  } else {
    c.swap_pairs = c.panel_pairs = 0;
    c.swap_bytes = c.panel_bytes = 0.0;
  }
  StampBuf& b = c.stamps[buf];
  if(panels <= b.panels) return HPLX_SUCCESS;
  if(b.t) (void)hipFree(b.t);
  b = StampBuf();
  HIPCHK(c, hipMalloc(&b.t, sizeof(long long) * 2 * kStampPairs * panels));
  b.panels = panels;
  return HPLX_SUCCESS;
}

// Pair i of the updates (kind 0), the interchanges (1) or the panels (2).
inline long long* stamp_at(const Ctx& c, int kind, int i) {
  const StampBuf& b = c.stamps[kind > 0];
  return b.t + 2 * (static_cast<size_t>(kind == 2 ? 2 : 0) * b.panels + i);
}

// The durations (ms) of the first n pairs of a kind, read on the context's own
// stream (the null stream would wait for every other blocking stream).
inline int stamp_times(Ctx& c, int kind, int n, std::vector<double>* ms) {
  ms->assign(n, 0.0);
  if(n == 0) return HPLX_SUCCESS;
  int khz = 0;
  HIPCHK(c, hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c.device));
  std::vector<long long> t(2 * static_cast<size_t>(n));
  HIPCHK(c, hipMemcpyAsync(t.data(), stamp_at(c, kind, 0), sizeof(long long) * t.size(),
                           hipMemcpyDeviceToHost, c.stream));
  HIPCHK(c, hipStreamSynchronize(c.stream));
  for(int i = 0; i < n; ++i)
    (*ms)[i] = static_cast<double>(t[2 * i + 1] - t[2 * i]) / khz;
  return HPLX_SUCCESS;
}

inline int use(hplx_ctx* ctx) {
  if(!ctx) return HPLX_ERR_INVALID;
  hipError_t e = hipSetDevice(ctx->c.device);
  if(e != hipSuccess)
    return fail(ctx->c, HPLX_ERR_HIP, "hipSetDevice: %s", hipGetErrorString(e));
  return HPLX_SUCCESS;
}

// The P=Q=1 configurations this library builds (HPL_T_palg values):
// HPLX_SUCCESS, or an error code with its message in msg.  No device needed.
inline int palg_status(const hplx_palg* p, char* msg, size_t len) {
  if(!p) {
    std::snprintf(msg, len, "null palg");
    return HPLX_ERR_INVALID;
  }
  if(!valid_fact(p->pfact) || !valid_fact(p->rfact)) {
    std::snprintf(msg, len, "unknown panel factorisation (pfact=%d rfact=%d)",
                  p->pfact, p->rfact);
    return HPLX_ERR_INVALID;
  }
  // L1notran picks how the reference stores its copy of the panel's top
  // block (src/HPL_pddriver.cpp:166-199); the factors here stay in A, so
  // both forms run the same kernels.  U in non-transposed form is refused,
  // as the reference refuses it (src/HPL_pdinfo.cpp:979-986).
  if(p->L1notran != 0 && p->L1notran != 1) {
    std::snprintf(msg, len, "L1notran=%d (0 or 1)", p->L1notran);
    return HPLX_ERR_INVALID;
  }
  if(p->Unotran != 0) {
    std::snprintf(msg, len, "U in non-transposed form is not supported");
    return HPLX_ERR_UNSUPPORTED;
  }
  if(p->equil != 0) {
    std::snprintf(msg, len, "equilibration is not supported");
    return HPLX_ERR_UNSUPPORTED;
  }
  if(p->nbmin < 1 || p->nbdiv < 2) {
    std::snprintf(msg, len, "nbmin=%d nbdiv=%d", p->nbmin, p->nbdiv);
    return HPLX_ERR_INVALID;
  }
  // the reference refuses both in HPL_pdinfo (src/HPL_pdinfo.cpp:930-935
  // "Value of DEPTH must be 1", :950-955 "Value of SWAP must be 1")
  if(p->depth != 1) {
    std::snprintf(msg, len, "look-ahead depth must be 1 (got %d)", p->depth);
    return HPLX_ERR_UNSUPPORTED;
  }
  if(p->fswap != HPLX_SWAP01) {
    std::snprintf(msg, len,
                  "only long swapping (HPLX_SWAP01) is implemented (got %d)",
                  p->fswap);
    return HPLX_ERR_UNSUPPORTED;
  }
  return HPLX_SUCCESS;
}

inline int check_palg(Ctx& c, const hplx_palg* p) {
  char      msg[256];
  const int r = palg_status(p, msg, sizeof(msg));
  return r ? fail(c, r, "%s", msg) : HPLX_SUCCESS;
}

// Progress lines of a panel loop (HPLX_PROGRESS=<panels>, the counterpart of
// the reference's HPL_PROGRESS_REPORT build option): reports panels the
// device has finished, at most kLag panels behind what is queued, so the
// host never runs further ahead than that while it reports.
class Progress {
 public:
  static constexpr int kLag = 8;
  Progress(Ctx& c, int npanels, int nb, int n)
      : c_(c), npanels_(npanels), nb_(nb), n_(n),
        t0_(std::chrono::steady_clock::now()) {}

  hipError_t init() {
    if(c_.progress_every <= 0) return hipSuccess;
    while(static_cast<int>(c_.ev_prog.size()) < 2 * kLag) {
      hipEvent_t e;
      hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
      if(r != hipSuccess) return r;
      c_.ev_prog.push_back(e);
    }
    return hipSuccess;
  }

  // panel k's work has been queued; s: the stream its last step is on
  hipError_t panel_queued(int k, hipStream_t s) {
    if(c_.progress_every <= 0) return hipSuccess;
    hipError_t r = hipEventRecord(c_.ev_prog[k % (2 * kLag)], s);
    if(r != hipSuccess) return r;
    const int done = k - kLag;
    if(done < 0) return hipSuccess;
    r = hipEventSynchronize(c_.ev_prog[done % (2 * kLag)]);
    if(r != hipSuccess) return r;
    if(done % c_.progress_every == 0) {
      const double el =
          std::chrono::duration<double>(std::chrono::steady_clock::now() - t0_)
              .count();
      std::fprintf(stderr, "[hplx] panel %d/%d done (column %d of %d) %.2f s\n",
                   done + 1, npanels_, (done + 1) * nb_, n_, el);
      std::fflush(stderr);
    }
    return hipSuccess;
  }

 private:
  Ctx&                                  c_;
  int                                   npanels_, nb_, n_;
  std::chrono::steady_clock::time_point t0_;
};

}  // namespace hplx
