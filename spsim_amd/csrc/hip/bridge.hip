// Host-array bridge used by the reference-shaped C API (see host/bridge.h).
// Every call stages host arrays into HBM on a private stream, runs the device
// entry points and copies the results back before returning. The stream, the
// device buffer and the pinned staging buffer of a call are kept for the next
// one: creating them took most of a small call (a 64 x 64 shot of 500 atoms is
// four calls, 590 us with a stream and up to nine hipMalloc/hipFree each).
#include <algorithm>
#include <cstring>
#include <mutex>

#include "../host/bridge.h"
#include "common.hpp"
#include "epilogue.hpp"
#include "sf_kernels.hpp"

namespace spsim {
namespace {

// What a call works with. Sessions are handed out one per call, so calls of
// several threads never share one (they still follow each other where the entry
// points that they call use the library workspace); idle ones wait in a list of
// at most kMaxIdle, their buffers at most kKeepBytes each, until spsim_hip_release.
struct Session {
  int device = -1;
  hipStream_t s = nullptr;
  char *dev = nullptr, *pin = nullptr;
  size_t dev_bytes = 0;
};

constexpr int kMaxIdle = 8;
constexpr size_t kKeepBytes = (size_t)64 << 20;
constexpr size_t kStageBytes = (size_t)4 << 20;  // inputs, and outputs, up to this size travel in one copy

std::mutex g_session_mu;
Session g_idle[kMaxIdle];
int g_idle_count = 0;

void destroy(Session &x) {
  if (x.dev) (void)hipFree(x.dev);
  if (x.pin) (void)hipHostFree(x.pin);
  if (x.s) (void)hipStreamDestroy(x.s);
  x = Session{};
}

int acquire(Session *x) {
  int device = 0;
  SPSIM_HIP_TRY(hipGetDevice(&device));
  {
    std::lock_guard<std::mutex> lk(g_session_mu);
    for (int i = g_idle_count - 1; i >= 0; --i)
      if (g_idle[i].device == device) {
        *x = g_idle[i];
        g_idle[i] = g_idle[--g_idle_count];
        g_idle[g_idle_count] = Session{};
        return SPSIM_HIP_OK;
      }
  }
  x->device = device;
  SPSIM_HIP_TRY(hipStreamCreateWithFlags(&x->s, hipStreamNonBlocking));
  SPSIM_HIP_TRY(hipHostMalloc((void **)&x->pin, 2 * kStageBytes, hipHostMallocDefault));
  return SPSIM_HIP_OK;
}

void give_back(Session &x) {
  if (x.s && x.pin && x.dev_bytes <= kKeepBytes) {
    std::lock_guard<std::mutex> lk(g_session_mu);
    if (g_idle_count < kMaxIdle) {
      g_idle[g_idle_count++] = x;
      x = Session{};
      return;
    }
  }
  destroy(x);
}

// One call: its host inputs and outputs and device scratch, declared first
// (in, out, scratch), then placed and copied in by start(), copied out by
// finish(). A null or empty array is a null device pointer.
class Call {
 public:
  ~Call() {
    if (running_) (void)hipStreamSynchronize(x_.s);  // a failed call: nothing may still use the buffers
    if (x_.device >= 0) give_back(x_);
  }
  template <class T>
  void in(const T *host, size_t n, T **dev) {
    add(ins_, nin_, const_cast<T *>(host), host ? n * sizeof(T) : 0, (void **)dev);
  }
  template <class T>
  void out(T *host, size_t n, T **dev) {
    add(outs_, nout_, host, host ? n * sizeof(T) : 0, (void **)dev);
  }
  template <class T>
  void scratch(size_t n, T **dev) {
    add(tmps_, ntmp_, nullptr, n * sizeof(T), (void **)dev);
  }
  int start() {
    SPSIM_TRY(acquire(&x_));
    size_t at = 0;
    place(ins_, nin_, &at);
    in_bytes_ = at;
    out_at_ = at;
    place(outs_, nout_, &at);
    out_bytes_ = at - out_at_;
    place(tmps_, ntmp_, &at);
    if (at > x_.dev_bytes) {
      if (x_.dev) (void)hipFree(x_.dev);
      x_.dev = nullptr;
      x_.dev_bytes = 0;
      const hipError_t e = hipMalloc((void **)&x_.dev, at);
      if (e != hipSuccess) return fail(SPSIM_HIP_ERR_NOMEM, "hipMalloc(%zu) failed: %s", at, hipGetErrorString(e));
      x_.dev_bytes = at;
    }
    point(ins_, nin_);
    point(outs_, nout_);
    point(tmps_, ntmp_);
    running_ = true;
    if (in_bytes_ && in_bytes_ <= kStageBytes) {
      for (int i = 0; i < nin_; ++i)
        if (ins_[i].bytes) std::memcpy(x_.pin + ins_[i].at, ins_[i].host, ins_[i].bytes);
      SPSIM_HIP_TRY(hipMemcpyAsync(x_.dev, x_.pin, in_bytes_, hipMemcpyHostToDevice, x_.s));
    } else {
      for (int i = 0; i < nin_; ++i)
        if (ins_[i].bytes)
          SPSIM_HIP_TRY(hipMemcpyAsync(x_.dev + ins_[i].at, ins_[i].host, ins_[i].bytes, hipMemcpyHostToDevice, x_.s));
    }
    return SPSIM_HIP_OK;
  }
  hipStream_t stream() const { return x_.s; }
  int finish() {
    const bool staged = out_bytes_ && out_bytes_ <= kStageBytes;
    if (staged) {
      SPSIM_HIP_TRY(hipMemcpyAsync(x_.pin + kStageBytes, x_.dev + out_at_, out_bytes_, hipMemcpyDeviceToHost, x_.s));
    } else {
      for (int i = 0; i < nout_; ++i)
        if (outs_[i].bytes)
          SPSIM_HIP_TRY(hipMemcpyAsync(outs_[i].host, x_.dev + outs_[i].at, outs_[i].bytes, hipMemcpyDeviceToHost,
                                       x_.s));
    }
    SPSIM_HIP_TRY(hipStreamSynchronize(x_.s));
    running_ = false;
    if (staged)
      for (int i = 0; i < nout_; ++i)
        if (outs_[i].bytes) std::memcpy(outs_[i].host, x_.pin + kStageBytes + (outs_[i].at - out_at_), outs_[i].bytes);
    return SPSIM_HIP_OK;
  }

 private:
  static constexpr int kMax = 12;
  struct Array {
    void *host;
    size_t bytes, at;
    void **dev;
  };
  static void add(Array *list, int &n, void *host, size_t bytes, void **dev) {
    *dev = nullptr;
    list[n++] = Array{host, bytes, 0, dev};
  }
  static void place(Array *list, int n, size_t *at) {
    for (int i = 0; i < n; ++i) {
      list[i].at = *at;
      *at += (list[i].bytes + 255) / 256 * 256;
    }
  }
  void point(Array *list, int n) {
    for (int i = 0; i < n; ++i)
      if (list[i].bytes) *list[i].dev = x_.dev + list[i].at;
  }
  Session x_;
  Array ins_[kMax], outs_[kMax], tmps_[kMax];
  int nin_ = 0, nout_ = 0, ntmp_ = 0;
  size_t in_bytes_ = 0, out_at_ = 0, out_bytes_ = 0;
  bool running_ = false;
};

int run_stage(const spsim_hip_detector *det, Stage st, const float *h0, const float *h1, const float *h2,
              size_t n_in, uint64_t seed, uint64_t pattern, float *out, size_t n_out) {
  DetConst d;
  SPSIM_TRY(make_det_const(det, &d));
  SPSIM_TRY(ensure_device(nullptr));
  if (!out) return fail(SPSIM_HIP_ERR_INVALID, "output is NULL");
  Call c;
  float *d0, *d1, *d2, *dout;
  c.in(h0, n_in, &d0);
  c.in(h1, n_in, &d1);
  c.in(h2, n_in, &d2);
  c.out(out, n_out, &dout);
  SPSIM_TRY(c.start());
  SPSIM_TRY(launch_stage(st, d, d0, d1, d2, seed, (uint32_t)pattern, dout, c.stream()));
  return c.finish();
}

size_t raw_count(const spsim_hip_detector *det) {
  return det ? (size_t)det->nx * det->ny * (det->nz > 0 ? det->nz : 1) : 0;
}
size_t bin_count(const spsim_hip_detector *det) {
  if (!det || det->bin_x < 1 || det->bin_y < 1) return 0;
  const int nz = det->nz > 0 ? det->nz : 1, bz = det->bin_z > 0 ? det->bin_z : 1;
  return (size_t)(det->nx / det->bin_x) * (det->ny / det->bin_y) * (nz / bz);
}

}  // namespace

void bridge_release() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return;
  std::lock_guard<std::mutex> lk(g_session_mu);
  for (int i = g_idle_count - 1; i >= 0; --i)
    if (g_idle[i].device == device) {
      destroy(g_idle[i]);
      g_idle[i] = g_idle[--g_idle_count];
      g_idle[g_idle_count] = Session{};
    }
}

}  // namespace spsim

extern "C" {

int spsim_bridge_hkl_detector(int nx, int ny, float width, float height, float distance, float center_x,
                              float center_y, int spherical, float wavelength, float *out) {
  using namespace spsim;
  SPSIM_TRY(ensure_device(nullptr));
  const size_t n = (size_t)(nx > 0 ? nx : 0) * (ny > 0 ? ny : 0) * 3;
  Call c;
  float *d;
  c.out(out, n, &d);
  SPSIM_TRY(c.start());
  SPSIM_TRY(
      spsim_hip_hkl_detector(nx, ny, width, height, distance, center_x, center_y, spherical, wavelength, d, c.stream()));
  return c.finish();
}

int spsim_bridge_hkl_detector_3d(int nx, int ny, int nz, float width, float height, float depth, float center_x,
                                 float center_y, float center_z, float distance, float wavelength, float *out) {
  using namespace spsim;
  SPSIM_TRY(ensure_device(nullptr));
  const size_t n = (size_t)(nx > 0 ? nx : 0) * (ny > 0 ? ny : 0) * (nz > 0 ? nz : 0) * 3;
  Call c;
  float *d;
  c.out(out, n, &d);
  SPSIM_TRY(c.start());
  SPSIM_TRY(spsim_hip_hkl_detector_3d(nx, ny, nz, width, height, depth, center_x, center_y, center_z, distance,
                                      wavelength, d, c.stream()));
  return c.finish();
}

int spsim_bridge_rotate_hkl(float *list, int npix, const double *rot9) {
  using namespace spsim;
  SPSIM_TRY(ensure_device(nullptr));
  if (npix <= 0) return SPSIM_HIP_OK;
  Call c;
  float *d, *rotated;
  c.in((const float *)list, (size_t)npix * 3, &d);
  c.out(list, (size_t)npix * 3, &rotated);
  SPSIM_TRY(c.start());
  SPSIM_TRY(spsim_hip_rotate_hkl(d, npix, rot9, rotated, c.stream()));
  return c.finish();
}

// One structure-factor launch on host arrays: the spectrum kernel when
// nsamples > 0, else the grid kernel when nx > 0, else the per-pixel kernel.
static int structure_factor_impl(const float *hkl, int npix, int nx, int ny, const spsim_hip_atom *atoms,
                                 const float *atom_b, const spsim_hip_segment *segs, int nsegs, int natoms,
                                 const float *ff, float b_global, Complex *F, float *I, int nsamples = 0,
                                 const double *scales = nullptr, const double *weights = nullptr) {
  using namespace spsim;
  SPSIM_TRY(ensure_device(nullptr));
  if (npix <= 0) return SPSIM_HIP_OK;
  Call c;
  float *dq, *dff, *db, *dF, *dI;
  spsim_hip_atom *da;
  spsim_hip_segment *ds;
  c.in(hkl, (size_t)npix * 3, &dq);
  c.in(atoms, (size_t)natoms, &da);
  c.in(atom_b, (size_t)natoms, &db);
  c.in(segs, (size_t)nsegs, &ds);
  c.in(ff, (size_t)SPSIM_HIP_NSPECIES * SPSIM_HIP_FF_STRIDE, &dff);
  c.out((float *)F, (size_t)npix * 2, &dF);
  c.out(I, (size_t)npix, &dI);
  SPSIM_TRY(c.start());
  if (nsamples > 0)
    SPSIM_TRY(spsim_hip_sf_spectrum(dq, npix, da, db, ds, nsegs, natoms, dff, b_global, nullptr, nsamples, scales,
                                    weights, dF, dI, nullptr, c.stream()));
  else if (nx > 0)
    SPSIM_TRY(
        spsim_hip_sf_grid(dq, nx, ny, da, db, ds, nsegs, natoms, dff, b_global, nullptr, dF, dI, nullptr, c.stream()));
  else
    SPSIM_TRY(
        spsim_hip_sf_pattern(dq, npix, da, db, ds, nsegs, natoms, dff, b_global, nullptr, dF, dI, nullptr, c.stream()));
  return c.finish();
}

int spsim_bridge_structure_factor(const float *hkl, int npix, const spsim_hip_atom *atoms, const float *atom_b,
                                  const spsim_hip_segment *segs, int nsegs, int natoms, const float *ff, float b_global,
                                  Complex *F, float *I) {
  return structure_factor_impl(hkl, npix, 0, 0, atoms, atom_b, segs, nsegs, natoms, ff, b_global, F, I);
}

int spsim_bridge_structure_factor_spectrum(const float *hkl, int npix, const spsim_hip_atom *atoms,
                                           const float *atom_b, const spsim_hip_segment *segs, int nsegs,
                                           int natoms, const float *ff, float b_global, int nsamples,
                                           const double *scales, const double *weights, Complex *F, float *I) {
  if (nsamples < 1) return spsim::fail(SPSIM_HIP_ERR_INVALID, "nsamples=%d", nsamples);
  return structure_factor_impl(hkl, npix, 0, 0, atoms, atom_b, segs, nsegs, natoms, ff, b_global, F, I, nsamples,
                               scales, weights);
}

int spsim_bridge_structure_factor_grid(const float *hkl, int nx, int ny, const spsim_hip_atom *atoms,
                                       const float *atom_b, const spsim_hip_segment *segs, int nsegs, int natoms,
                                       const float *ff, float b_global, Complex *F, float *I) {
  if (nx < 0 || ny < 0) return spsim::fail(SPSIM_HIP_ERR_INVALID, "negative detector size");
  return structure_factor_impl(hkl, nx * ny, nx, ny, atoms, atom_b, segs, nsegs, natoms, ff, b_global, F, I);
}

int spsim_bridge_structure_factor_nfft(const float *hkl, int npix, const spsim_hip_atom *atoms,
                                       const spsim_hip_segment *segs, int nsegs, int natoms, const float *ff,
                                       float b_global, double eps, Complex *F, float *I) {
  using namespace spsim;
  SPSIM_TRY(ensure_device(nullptr));
  if (npix <= 0) return SPSIM_HIP_OK;
  Call c;
  float *dq, *dff, *dF, *dI;
  spsim_hip_atom *da;
  spsim_hip_segment *ds;
  c.in(hkl, (size_t)npix * 3, &dq);
  c.in(atoms, (size_t)natoms, &da);
  c.in(segs, (size_t)nsegs, &ds);
  c.in(ff, (size_t)SPSIM_HIP_NSPECIES * SPSIM_HIP_FF_STRIDE, &dff);
  c.out((float *)F, (size_t)npix * 2, &dF);
  c.out(I, (size_t)npix, &dI);
  SPSIM_TRY(c.start());
  SPSIM_TRY(spsim_hip_sf_nfft(dq, npix, da, nullptr, ds, nsegs, natoms, dff, b_global, nullptr, eps, dF, dI, nullptr,
                              c.stream()));
  return c.finish();
}

int spsim_bridge_thomson(const spsim_hip_detector *det, float *out) {
  using namespace spsim;
  return run_stage(det, Stage::kThomson, nullptr, nullptr, nullptr, 0, 0, 0, out, raw_count(det));
}

int spsim_bridge_solid_angle(const spsim_hip_detector *det, float *out) {
  using namespace spsim;
  return run_stage(det, Stage::kSolidAngle, nullptr, nullptr, nullptr, 0, 0, 0, out, raw_count(det));
}

int spsim_bridge_photons(const spsim_hip_detector *det, const float *thomson, const float *solid_angle,
                         const float *I, float *out) {
  using namespace spsim;
  if (!thomson || !solid_angle || !I) return fail(SPSIM_HIP_ERR_INVALID, "photons: input is NULL");
  return run_stage(det, Stage::kPhotons, thomson, solid_angle, I, raw_count(det), 0, 0, out, raw_count(det));
}

int spsim_bridge_poisson(const spsim_hip_detector *det, const float *photons, uint64_t seed, uint64_t pattern,
                         float *out) {
  using namespace spsim;
  if (!photons) return fail(SPSIM_HIP_ERR_INVALID, "poisson: photons is NULL");
  return run_stage(det, Stage::kPoisson, photons, nullptr, nullptr, raw_count(det), seed, pattern, out, raw_count(det));
}

int spsim_bridge_electrons(const spsim_hip_detector *det, const float *count, float *out) {
  using namespace spsim;
  if (!count) return fail(SPSIM_HIP_ERR_INVALID, "electrons: count is NULL");
  return run_stage(det, Stage::kElectrons, count, nullptr, nullptr, raw_count(det), 0, 0, out, raw_count(det));
}

int spsim_bridge_real_output(const spsim_hip_detector *det, const float *electrons, uint64_t seed, uint64_t pattern,
                             float *out) {
  using namespace spsim;
  if (!electrons) return fail(SPSIM_HIP_ERR_INVALID, "real output: electrons is NULL");
  return run_stage(det, Stage::kRealOutput, electrons, nullptr, nullptr, raw_count(det), seed, pattern, out,
                   bin_count(det));
}

int spsim_bridge_noiseless_output(const spsim_hip_detector *det, const float *photons, float *out) {
  using namespace spsim;
  if (!photons) return fail(SPSIM_HIP_ERR_INVALID, "noiseless output: photons is NULL");
  return run_stage(det, Stage::kNoiselessOutput, photons, nullptr, nullptr, raw_count(det), 0, 0, out, bin_count(det));
}

int spsim_bridge_detector_chain(const spsim_hip_detector *det, const float *I, uint64_t seed, uint64_t pattern,
                                float *thomson, float *solid_angle, float *photons, float *count, float *electrons,
                                float *real_output, float *noiseless_output) {
  using namespace spsim;
  DetConst d;
  SPSIM_TRY(make_det_const(det, &d));
  SPSIM_TRY(ensure_device(nullptr));
  const size_t n = raw_count(det), nb = bin_count(det);
  Call c;
  float *dI, *o[7];
  float *host[7] = {thomson, solid_angle, photons, count, electrons, real_output, noiseless_output};
  const size_t sizes[7] = {n, n, n, n, n, nb, nb};
  c.in(I, n, &dI);
  for (int i = 0; i < 7; ++i) c.out(host[i], sizes[i], &o[i]);
  SPSIM_TRY(c.start());
  SPSIM_TRY(launch_chain(d, dI, 1, seed, pattern, o[0], o[1], o[2], o[3], o[4], o[5], o[6], c.stream()));
  return c.finish();
}

int spsim_bridge_shot(const spsim_hip_detector *det, const double *rot9, const spsim_hip_atom *atoms,
                      const spsim_hip_segment *segs, int nsegs, int natoms, const float *ff, float b_global,
                      uint64_t seed, uint64_t pattern, float *hkl, Complex *F, float *I, float *thomson,
                      float *solid_angle, float *photons, float *count, float *electrons, float *real_output,
                      float *noiseless_output) {
  using namespace spsim;
  DetConst d;
  SPSIM_TRY(make_det_const(det, &d));
  SPSIM_TRY(ensure_device(nullptr));
  const size_t n = raw_count(det), nb = bin_count(det);
  if (n == 0 || det->nz > 1) return fail(SPSIM_HIP_ERR_INVALID, "a shot needs a 2-D detector");
  Call c;
  float *dff, *dq0, *dq, *dF, *dI, *o[7];
  spsim_hip_atom *da;
  spsim_hip_segment *ds;
  float *host[7] = {thomson, solid_angle, photons, count, electrons, real_output, noiseless_output};
  const size_t sizes[7] = {n, n, n, n, n, nb, nb};
  c.in(atoms, (size_t)natoms, &da);
  c.in(segs, (size_t)nsegs, &ds);
  c.in(ff, (size_t)SPSIM_HIP_NSPECIES * SPSIM_HIP_FF_STRIDE, &dff);
  c.out(hkl, 3 * n, &dq);
  c.out((float *)F, 2 * n, &dF);
  c.out(I, n, &dI);
  for (int i = 0; i < 7; ++i) c.out(host[i], sizes[i], &o[i]);
  c.scratch(3 * n, &dq0);
  SPSIM_TRY(c.start());
  SPSIM_TRY(spsim_hip_hkl_detector(det->nx, det->ny, det->width, det->height, det->distance, det->center_x,
                                   det->center_y, det->spherical, det->wavelength, dq0, c.stream()));
  SPSIM_TRY(spsim_hip_rotate_hkl(dq0, (int)n, rot9, dq, c.stream()));
  SPSIM_TRY(spsim_hip_sf_grid(dq, det->nx, det->ny, da, nullptr, ds, nsegs, natoms, dff, b_global, nullptr, dF, dI,
                              nullptr, c.stream()));
  SPSIM_TRY(launch_chain(d, dI, 1, seed, pattern, o[0], o[1], o[2], o[3], o[4], o[5], o[6], c.stream()));
  return c.finish();
}

}  // extern "C"
