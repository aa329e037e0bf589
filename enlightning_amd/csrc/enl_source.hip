// Source injection: enlightning::addSource (enlightning.C:2140-2307), the
// lightning-channel file reader (enlightning::readLightningInput,
// enlightning.C:2333-2389) and the microphones' pressure read
// (enlightning::recordAudio, enlightning.C:2392-2506) for the device.
//
// addSource writes the mass source of every interior cell of a patch:
//   PULSE POINT      amp * exp(-log 2 / s^2 * (x0^2 + x1^2))
//   PULSE SINE       amp * exp(-log 2 / s^2 * (x0 - A sin(f x1))^2)
//   PULSE LIGHTNING  per channel segment, the Gaussian of the distance to the
//                    segment (a cap around each end point on its side of the
//                    segment's normal through it, the perpendicular distance
//                    between them), merged into the cell's value v as
//                    v + t - (v / amp) * t, segment by segment
//   DRIVEN POINT     the POINT pulse times sin(omega * (it + 1 - t0) * dt)
// (x0, x1 the cell centre relative to src_pos, s = src_spread).  The
// per-segment quantities (angle, the slope of the normal lines, sin and cos
// of the angle, the orientation) are formed on the host with the reference's
// expressions; the device evaluates the per-cell expressions in the
// reference's order without contraction.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

#include "enl_batch.h"
#include "enl_kernels.h"

namespace enl {

namespace {

constexpr int kPoint = 10, kSine = 20, kLightning = 30;  // enlightning.C:55-57
constexpr int kPulse = 10, kDriven = 20;                 // enlightning.C:60-61
constexpr double kPi = 3.14159265358979323846264338;     // enlightning.C:70

// One channel segment with its host-formed quantities.
struct Segment {
  double x0, y0, x1, y1;  // end points (p_lightning_coords[4k .. 4k+3])
  double slope;           // tan(PI/2 - theta)
  double sn, cs;          // sin(theta), cos(theta)
  int orientation;        // 1 or 2 (0: no cell qualifies)
};

struct SourceArgs {
  double* out;  // interior cell (0, 0)
  long sy;      // row stride of out
  int nx, ny;
  double xlo0, xlo1, dx0, dx1;
  int type;
  double amp, k;  // k = -log(2.0) / SQUARE(spread)
  double pos0, pos1, sine_amp, sine_freq;
  double drive;  // DRIVEN: the sin(...) factor; PULSE: unused
  bool driven;
  const Segment* seg;
  int nseg;
};

// The source of the cell centred at (xc0, xc1); v is its present value
// (LIGHTNING merges into it).
__device__ inline double source_value(const SourceArgs& a, double xc0, double xc1, double v) {
  if (a.type == kPoint) {
    const double x0 = xc0 - a.pos0, x1 = xc1 - a.pos1;
    v = a.amp * exp(a.k * (x0 * x0 + x1 * x1));
    if (a.driven) v = v * a.drive;
    return v;
  }
  if (a.type == kSine) {
    const double x0 = xc0 - a.pos0, x1 = xc1 - a.pos1;
    const double d = x0 - a.sine_amp * sin(a.sine_freq * x1);
    return a.amp * exp(a.k * (d * d));
  }
  for (int k = 0; k < a.nseg; k++) {
    const Segment s = a.seg[k];
    const double line0 = s.slope * (xc0 - s.x0) + s.y0;
    const double line1 = s.slope * (xc0 - s.x1) + s.y1;
    if ((s.orientation == 1 && xc1 >= line0) || (s.orientation == 2 && xc1 <= line0)) {
      const double dx = xc0 - s.x0, dy = xc1 - s.y0;
      const double t = a.amp * exp(a.k * (dx * dx + dy * dy));
      v = v + t - (v / a.amp) * t;
    }
    if ((s.orientation == 1 && xc1 <= line1) || (s.orientation == 2 && xc1 >= line1)) {
      const double dx = xc0 - s.x1, dy = xc1 - s.y1;
      const double t = a.amp * exp(a.k * (dx * dx + dy * dy));
      v = v + t - (v / a.amp) * t;
    }
    if ((s.orientation == 1 && xc1 < line0 && xc1 > line1) || (s.orientation == 2 && xc1 > line0 && xc1 < line1)) {
      const double d = s.sn * (xc0 - s.x0) + s.cs * (xc1 - s.y0);
      const double t = a.amp * exp(a.k * (d * d));
      v = v + t - (v / a.amp) * t;
    }
  }
  return v;
}

__global__ void __launch_bounds__(256) source_kernel(SourceArgs a) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (long)a.nx * a.ny) return;
  const int i = (int)(q % a.nx), j = (int)(q / a.nx);
  double* o = a.out + (long)i + (long)j * a.sy;
  *o = source_value(a, a.xlo0 + a.dx0 * ((double)i + 0.5), a.xlo1 + a.dx1 * ((double)j + 0.5),
                    a.type == kLightning ? *o : 0.0);
}

// The same for every patch of a hierarchy in one launch, in chunks (kChunk)
// whose ghosts stand still: one launch per patch, ~700 at a 512^2 base, took
// 4 ms for a source that costs some 10 us to evaluate; one of (the largest
// patch's cells, at most 256 workgroups) x patches left a large patch short
// of waves (a channel of 24 segments on 2048^2 in one patch 0.34 ms by the
// patch, 0.73 so, 0.35 in chunks; on 1024 patches 36, 0.29 and 0.29 ms).
__global__ void __launch_bounds__(kChunk) batch_source_kernel(double* pool, const PatchDev* __restrict__ pd,
                                                              const int* __restrict__ chunk_patch, SourceArgs a) {
  const PatchDev& p = pd[chunk_patch[blockIdx.x]];
  const unsigned n = (unsigned)((int)blockIdx.x - p.chunk0) * kChunk + threadIdx.x;
  const unsigned row = n / (unsigned)p.sy;
  const int i = (int)(n - row * (unsigned)p.sy) - p.g, j = (int)row - p.g;
  if (i < 0 || i >= p.nx || j < 0 || j >= p.ny) return;
  double* o = pool + p.src + n;
  *o = source_value(a, p.xlo + p.dx * ((double)i + 0.5), p.ylo + p.dy * ((double)j + 0.5),
                    a.type == kLightning ? *o : 0.0);
}

// Segments of the channel with the quantities of enlightning.C:2215-2232.
std::vector<Segment> segments(const double* c, int n) {
  std::vector<Segment> v((size_t)n);
  for (int k = 0; k < n; k++) {
    const double x0 = c[4 * k], y0 = c[4 * k + 1], x1 = c[4 * k + 2], y1 = c[4 * k + 3];
    const double theta = -std::atan((y1 - y0) / (x1 - x0));
    int orientation = 0;
    if ((x0 > x1 && y0 > y1) || (x0 <= x1 && y0 >= y1))
      orientation = 1;
    else if ((x0 >= x1 && y0 <= y1) || (x0 < x1 && y0 < y1))
      orientation = 2;
    Segment& s = v[(size_t)k];
    s.x0 = x0;
    s.y0 = y0;
    s.x1 = x1;
    s.y1 = y1;
    s.slope = std::tan(kPi / 2.0 - theta);
    s.sn = std::sin(theta);
    s.cs = std::cos(theta);
    s.orientation = orientation;
  }
  return v;
}

// Pressure at each microphone inside the patch (enlightning::recordAudio,
// enlightning.C:2414-2436): cell i = (int)((x - xlo) / dx) of the interior
// array, the bounds inclusive as in the reference.
__global__ void __launch_bounds__(64) mic_kernel(const double* pres, long sy, int nx, int ny, double xlo0,
                                                 double xlo1, double xhi0, double xhi1, double dx0, double dx1,
                                                 int nmics, const double* mx, const double* my, double* out,
                                                 int* hit) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nmics) return;
  const double x = mx[k], y = my[k];
  if (x >= xlo0 && x <= xhi0 && y >= xlo1 && y <= xhi1) {
    const int i = (int)((x - xlo0) / dx0), j = (int)((y - xlo1) / dx1);
    // the reference reads cell (i, j) even on the upper bound (i == nx);
    // the device clamps it into the patch instead of reading past it
    const int ic = i < nx ? i : nx - 1, jc = j < ny ? j : ny - 1;
    out[k] = pres[(long)ic + (long)jc * sy];
    hit[k] = 1;
  } else {
    hit[k] = 0;
  }
}

// Values at up to kGather places of the pool, the places in the kernel's
// arguments (no upload).
constexpr int kGather = 128;
struct GatherAt {
  long at[kGather];
};
__global__ void __launch_bounds__(kGather) gather_kernel(const double* pool, GatherAt g, int n, double* out) {
  if ((int)threadIdx.x < n) out[threadIdx.x] = pool[g.at[threadIdx.x]];
}

// What a source's cells need of it; LIGHTNING segments are uploaded by
// upload_segments.
int source_args(const enl_source_t* src, int iteration, int pulse_time0, double dt, SourceArgs* out) {
  SourceArgs& a = *out;
  a.type = src->type;
  a.amp = src->amp;
  a.k = -std::log(2.0) / (src->spread * src->spread);
  a.pos0 = src->pos[0];
  a.pos1 = src->pos[1];
  a.sine_amp = src->sine_amp;
  a.sine_freq = src->sine_freq;
  a.driven = src->mode == kDriven;
  a.drive = a.driven ? std::sin(src->omega * (double)(iteration + 1 - pulse_time0) * dt) : 0.0;
  a.seg = nullptr;
  a.nseg = 0;
  if (src->mode != kPulse && src->mode != kDriven) return set_error(-2, "unknown source mode %d", src->mode);
  if (src->type != kPoint && src->type != kSine && src->type != kLightning)
    return set_error(-2, "unknown source type %d", src->type);
  // enlightning.C:2301-2302
  if (a.driven && src->type != kPoint) return set_error(-2, "DRIVEN SINE or LIGHTNING source mode not implemented");
  if (src->type == kLightning && (src->nseg < 0 || (src->nseg > 0 && !src->coords)))
    return set_error(-3, "lightning segments missing");
  return 0;
}

// The channel's segments into stream-ordered device memory (a->seg, freed by
// the caller with hipFreeAsync).
int upload_segments(const enl_source_t* src, SourceArgs* a, hipStream_t s) {
  const std::vector<Segment> h = segments(src->coords, src->nseg);
  Segment* dseg = nullptr;
  hipError_t e = hipMallocAsync((void**)&dseg, sizeof(Segment) * h.size(), s);
  if (e == hipSuccess) e = hipMemcpyAsync(dseg, h.data(), sizeof(Segment) * h.size(), hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);  // h goes out of scope
  if (e != hipSuccess) {
    if (dseg) (void)hipFreeAsync(dseg, s);
    return check_hip(e, "lightning segments upload");
  }
  a->seg = dseg;
  a->nseg = src->nseg;
  return 0;
}

}  // namespace

}  // namespace enl

using namespace enl;

extern "C" {

int enl_add_source(int ifirst0, int ilast0, int ifirst1, int ilast1, const double* patch_xlo, const double* dx,
                   const enl_source_t* src, int iteration, int pulse_time0, double dt, double* source, long sy) {
  if (ilast0 < ifirst0 || ilast1 < ifirst1)
    return set_error(-2, "invalid box [%d,%d]x[%d,%d]", ifirst0, ilast0, ifirst1, ilast1);
  if (!patch_xlo || !dx || !src) return set_error(-3, "null argument");
  if (!source || !is_device_ptr(source)) return set_error(-4, "enl_add_source needs a device source array");
  const int nx = ilast0 - ifirst0 + 1, ny = ilast1 - ifirst1 + 1;
  if (sy < nx) return set_error(-2, "source row stride below the patch width");
  SourceArgs a;
  a.out = source;
  a.sy = sy;
  a.nx = nx;
  a.ny = ny;
  a.xlo0 = patch_xlo[0];
  a.xlo1 = patch_xlo[1];
  a.dx0 = dx[0];
  a.dx1 = dx[1];
  int rc = source_args(src, iteration, pulse_time0, dt, &a);
  if (rc) return rc;
  if (src->type == kLightning && src->nseg == 0) return 0;
  hipStream_t s = lib_stream();
  if (src->type == kLightning && (rc = upload_segments(src, &a, s))) return rc;
  const long cells = (long)nx * ny;
  hipLaunchKernelGGL(source_kernel, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, s, a);
  hipError_t e = hipGetLastError();
  if (a.seg) {
    hipError_t f = hipFreeAsync((void*)a.seg, s);
    if (e == hipSuccess) e = f;
  }
  return check_hip(e, "source launch");
}

int enl_batch_add_source(void* handle, const enl_source_t* src, int iteration, int pulse_time0, double dt) {
  Batch* b = (Batch*)handle;
  if (!b) return set_error(-2, "null batch");
  if (!src) return set_error(-3, "null argument");
  SourceArgs a = {};
  int rc = source_args(src, iteration, pulse_time0, dt, &a);
  if (rc) return rc;
  if (src->type == kLightning && src->nseg == 0) return 0;
  hipStream_t s = lib_stream();
  if (src->type == kLightning && (rc = upload_segments(src, &a, s))) return rc;
  hipLaunchKernelGGL(batch_source_kernel, chunk_grid(b), dim3(kChunk), 0, s, b->pool, b->dp, b->chunk_patch, a);
  hipError_t e = hipGetLastError();
  if (a.seg) {
    hipError_t f = hipFreeAsync((void*)a.seg, s);
    if (e == hipSuccess) e = f;
  }
  return check_hip(e, "batched source launch");
}

int enl_batch_sample_mics(void* handle, int nmics, const double* mic_x, const double* mic_y, int max_entries, int* mic,
                          int* level, int* pid, double* value) {
  Batch* b = (Batch*)handle;
  if (!b) return set_error(-2, "null batch");
  if (nmics < 0 || max_entries < 0) return set_error(-2, "enl_batch_sample_mics: bad counts");
  if (nmics == 0) return 0;
  if (!mic_x || !mic_y || (max_entries > 0 && !(mic && level && pid && value))) return set_error(-3, "null argument");
  // per level and patch in order, the microphones within its bounds (inclusive)
  std::vector<long> at;
  int n = 0;
  for (int lev = 0; lev < b->nlevels; lev++)
    for (int p = 0; p < b->npatch; p++) {
      const PatchDev& pd = b->hp[p];
      if (pd.level != lev) continue;
      const double lo0 = pd.xlo, lo1 = pd.ylo;
      // the upper bounds from the origin of the index space: with an origin
      // of 0 they are (bi0 + nx) * dx to the last bit, the next patch's xlo
      const double hi0 = (lo0 - pd.bi0 * pd.dx) + (double)(pd.bi0 + pd.nx) * pd.dx;
      const double hi1 = (lo1 - pd.bj0 * pd.dy) + (double)(pd.bj0 + pd.ny) * pd.dy;
      for (int k = 0; k < nmics; k++) {
        const double x = mic_x[k], y = mic_y[k];
        if (!(x >= lo0 && x <= hi0 && y >= lo1 && y <= hi1)) continue;
        if (n < max_entries) {
          const int i = (int)((x - lo0) / pd.dx), j = (int)((y - lo1) / pd.dy);
          // the last cell for a microphone on the upper bound, as mic_kernel
          const int ic = std::min(i, pd.nx - 1), jc = std::min(j, pd.ny - 1);
          at.push_back(pd.state[0] + 5 * pd.sk + (ic + pd.g) + (long)(jc + pd.g) * pd.sy);
          mic[n] = k;
          level[n] = lev;
          pid[n] = p;
        }
        n++;
      }
    }
  if (at.empty()) return n;
  int rc = reserve(b, &b->stage, &b->stage_cap, sizeof(double) * at.size());
  if (rc) return rc;
  hipStream_t s = lib_stream();
  double* out = (double*)b->stage;
  for (size_t o = 0; o < at.size(); o += kGather) {
    GatherAt g = {};
    const int m = (int)std::min<size_t>(kGather, at.size() - o);
    for (int k = 0; k < m; k++) g.at[k] = at[o + k];
    hipLaunchKernelGGL(gather_kernel, dim3(1), dim3(kGather), 0, s, b->pool, g, m, out + o);
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(value, out, sizeof(double) * at.size(), hipMemcpyDeviceToHost, s);
  const hipError_t e2 = hipStreamSynchronize(s);
  rc = check_hip(e != hipSuccess ? e : e2, "enl_batch_sample_mics");
  return rc ? rc : n;
}

int enl_sample_mics(int ifirst0, int ilast0, int ifirst1, int ilast1, const double* patch_xlo, const double* patch_xhi,
                    const double* dx, int nmics, const double* mic_x, const double* mic_y, const double* pres, long sy,
                    double* out, int* hit) {
  if (ilast0 < ifirst0 || ilast1 < ifirst1)
    return set_error(-2, "invalid box [%d,%d]x[%d,%d]", ifirst0, ilast0, ifirst1, ilast1);
  if (nmics <= 0) return 0;
  if (!patch_xlo || !patch_xhi || !dx) return set_error(-3, "null argument");
  const void* dev[5] = {mic_x, mic_y, pres, out, hit};
  for (int i = 0; i < 5; i++)
    if (!dev[i] || !is_device_ptr(dev[i])) return set_error(-4, "enl_sample_mics needs device arrays");
  const int nx = ilast0 - ifirst0 + 1, ny = ilast1 - ifirst1 + 1;
  if (sy < nx) return set_error(-2, "pressure row stride below the patch width");
  hipLaunchKernelGGL(mic_kernel, dim3((unsigned)((nmics + 63) / 64)), dim3(64), 0, lib_stream(), pres, sy, nx, ny,
                     patch_xlo[0], patch_xlo[1], patch_xhi[0], patch_xhi[1], dx[0], dx[1], nmics, mic_x, mic_y, out,
                     hit);
  return check_hip(hipGetLastError(), "mic gather launch");
}

// enlightning::readLightningInput: one segment per line read with
// fgets(line, 80) and sscanf("%f %f %f %f"); a line that does not parse
// repeats the previous segment's values (zeros before the first).
int enl_read_lightning(const char* path, double* coords, int max_segments) {
  if (!path) return set_error(-3, "null path");
  FILE* fr = fopen(path, "rt");
  if (!fr) return set_error(-6, "can't open '%s' for reading", path);
  char line[80];
  float x1 = 0, y1 = 0, x2 = 0, y2 = 0;
  int n = 0;
  while (fgets(line, 80, fr) != NULL) {
    (void)sscanf(line, "%f %f %f %f", &x1, &y1, &x2, &y2);
    if (coords && n < max_segments) {
      coords[4 * n] = x1;
      coords[4 * n + 1] = y1;
      coords[4 * n + 2] = x2;
      coords[4 * n + 3] = y2;
    }
    n++;
  }
  fclose(fr);
  if (n < 1) return set_error(-6, "file '%s' is empty", path);
  return n;
}

}  // extern "C"
