// fd2_device.h -- device-side optical-photon transport for gfx950.
//
// The per-photon physics of fastDETECT2 as the reference C path defines it
// (main/kernel_cuda_c_ver1_0.cu, C branches), in FP32 with per-lane state in
// registers.  The control flow (including every random draw, resample loop
// and the stale-state quirks) follows the reference step for step because
// the draw order decides each photon's fate; the arithmetic is plain FP32
// (no double anywhere on the GPU).
//
// Geometry of the reference ("on-the-fly" columns): every column is an
// infinite vertical cylinder of radius R; the first one is centred on the
// event's (x,y); after crosstalk or a flight between columns the next column
// is centred at pos - R*n for a sampled inward normal n.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/fd2.h"
#include "fd2_ff.h"
#include "fd2_math.h"

namespace fd2 {

// Arithmetic policies of the transport code below.
//   MathDevice    the production kernel's FP32 arithmetic (fd2_math.h):
//                 azimuths in turns, reciprocal square roots, the Fresnel
//                 branch from cosines and sines (Snell's law).
//   MathFaithful  the reference C path's own arithmetic: float state, each
//                 double <math.h> expression evaluated with float pairs
//                 (fd2_ff.h) and rounded to float as the reference rounds
//                 it, the C library's acosf/asinf restated, the angles
//                 themselves in the Fresnel branch.  Used by the trajectory
//                 test's kernel only; no FP64 instruction either way.
// The control flow, draw order and every float operation the reference
// writes in float are the same under both.
struct MathDevice {
  static constexpr bool kFaithful = false;
};
struct MathFaithful {
  static constexpr bool kFaithful = true;
};

// The reference's azimuths are u * twopipen (main/kernel_cuda_c_ver1_0.cu:56);
// here they are the turn u itself, in quarters (fd2_sincos_quarters).
// The reference compares floats against the double constant eps =
// 8.1929093e-6 (and 1 +- eps, R - 1e-5, asin(nIC/nC)).  Each such test is
// done here against the float threshold that gives the same answer for every
// float operand: x < c  <=>  x < lt(c), x > c  <=>  x > gt(c), with lt(c) the
// smallest float >= c and gt(c) the largest float <= c.
// Safety cap on one photon's loop passes (in-column steps plus the
// boundary_analysis / top-surface loops the reference leaves unbounded); a
// photon past it is ended as lost.  Typical photons need well under 10^3.
constexpr int32_t kMaxLoops = 1 << 20;

// eps as float thresholds (see above): x < eps, x > eps, and |v| < 1 - eps,
// |v| > 1 + eps for norms
constexpr float kEpsLt = 0x1.12e890p-17f, kEpsGt = 0x1.12e88ep-17f;
constexpr float kNormLo = 0x1.fffeeep-1f, kNormHi = 0x1.000088p+0f;

// Per-geometry transport constants, derived once on the host.  ColumnGeom is
// what the in-column pass reads: with one geometry per launch it comes in one
// scalar load per pass (loaded where they are used, the constants made about
// 16 loads per pass, each with its own wait).
struct ColumnGeom {
  float xdet, ydet, R;
  float half_h;          // H/2
  float top_absfrac, beta, sensor_refl;
  float neg_inv_bulk;    // -1/bulk; +0 (all bits clear): no bulk absorption
  float r_sq;            // R*R
  float nudge_sq;        // rn > R - 1e-5  <=>  rn^2 > nudge_sq, rn the rounded root
  float top20;           // lower edge of the band of certain crosstalk, H/2 - 0.2 H
  float den_up, inv_up;  // crosstalk slopes' divisors 2*top20 and -H, and their
  float den_dn, inv_dn;  // correctly rounded reciprocals
  float dist_max;        // dist_to_surface's short form holds up to this distance:
                         // 2^27, or NaN (never) unless R and H/2 are in [2^-8, 2^20]
};
static_assert(sizeof(ColumnGeom) == 64, "one 16-dword scalar load");

struct GeomDev : ColumnGeom {
  float H, n1, n2, d_min, d_max;
  float lbx, lby, ubx, uby;
  // total internal reflection, theta1 > asin(n2/n1) inside a column and
  // theta1 > asin(n1/n2) from the gap, as cos(theta1) < threshold: the
  // smallest float >= cos(asin(.)) (NaN from the gap when n1/n2 > 1)
  float cos_tir_in, cos_tir_gap;
  float ratio12, ratio21;  // n1/n2, n2/n1
  float dspan;         // d_max - d_min
  int32_t pixel, xdim, ydim, num_hist;
  int32_t gap_fresnel; // (n1/n2) >= 1.57: gap side recomputes Pr/Pt
  float inv_pixel;     // 1/pixel when pixel is a power of two (x/pixel ==
                       // x*inv_pixel exactly), else 0
  // MathFaithful: total internal reflection as theta1 > the largest float
  // <= asin(n2/n1) (inside) or asin(n1/n2) (gap; NaN, never, when n1 > n2)
  float t1_tir_in, t1_tir_gap;
  unsigned long long* prf;   // xdim*ydim
  uint32_t* hist;            // num_hist
};

// ------------------------------------------------------------------ RNG

__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0,
                                              uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    uint32_t lo0 = 0xD2511F53u * c[0], hi0 = __umulhi(0xD2511F53u, c[0]);
    uint32_t lo1 = 0xCD9E8D57u * c[2], hi1 = __umulhi(0xCD9E8D57u, c[2]);
    uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// Production stream: xoshiro128+ (Blackman & Vigna 2018) per photon, its
// 128-bit state = Philox4x32-10(counter (photon, event >> 32, 0, 0),
// key (seed, event mod 2^32)): distinct for all 2^64 event numbers, and the
// same as a 32-bit event key below 2^32.  The + scrambler (the sum of two
// state words) is the generator's authors' choice for floating-point
// output: its weak low bits never reach u(), which keeps the high 24.  The
// ** scrambler's two integer multiplies per draw cost 2% of the transport's
// time (mono25x50: 134.7 -> 132.0 ms per launch).
struct CounterRng {
  uint32_t s0, s1, s2, s3;
  __device__ __forceinline__ void seed(uint32_t key0, uint64_t event,
                                       uint32_t photon) {
    uint32_t c[4] = {photon, (uint32_t)(event >> 32), 0u, 0u};
    philox4x32_10(c, key0, (uint32_t)event);
    s0 = c[0]; s1 = c[1]; s2 = c[2]; s3 = c[3];
    if ((s0 | s1 | s2 | s3) == 0u) s0 = 0x9E3779B9u;
  }
  __device__ __forceinline__ uint32_t next() {
    const uint32_t out = s0 + s3;
    const uint32_t t = s1 << 9;
    const uint32_t x = s3 ^ s1;
    const uint32_t n1 = fd2_xor3(s1, s2, s0);
    s2 = fd2_xor3(s2, s0, t);
    s0 = fd2_xor3(s0, s3, s1);
    s1 = n1;
    s3 = (x << 11) | (x >> 21);
    return out;
  }
  // (k + 1)/2^24 of the high 24 bits k: in (0,1], exact in float (k is exact
  // and the fused sum is representable); u4 = 4u, the same draw in quarter
  // turns
  __device__ __forceinline__ float u() {
    return fmaf((float)(next() >> 8), 0x1p-24f, 0x1p-24f);
  }
  __device__ __forceinline__ float u4() {
    return fmaf((float)(next() >> 8), 0x1p-22f, 0x1p-22f);
  }
};

// Trajectory-test stream: RANECU (L'Ecuyer 1988) exactly as
// main/kernel_cuda_c_ver1_0.cu:3694-3711, float result in (0,1].
struct RanecuRng {
  int32_t s0, s1;
  __device__ __forceinline__ float u() {
    int32_t q1 = s0 / 53668;
    s0 = 40014 * (s0 - q1 * 53668) - q1 * 12211;
    int32_t q2 = s1 / 52774;
    s1 = 40692 * (s1 - q2 * 52774) - q2 * 3791;
    if (s0 < 0) s0 += 2147483563;
    if (s1 < 0) s1 += 2147483399;
    int32_t z = s0 - s1;
    if (z < 1) z += 2147483562;
    return (float)z * (float)(1.0 / 2147483563.0);
  }
  __device__ __forceinline__ float u4() { return 4.0f * u(); }
};

// a^e mod m with 64-bit products (the reference's jump-ahead,
// main/kernel_cuda_c_ver1_0.cu:3516-3572)
__device__ __forceinline__ uint32_t powmod_u32(uint32_t a, uint64_t e,
                                               uint32_t m) {
  uint64_t r = 1, b = a % m;
  while (e) {
    if (e & 1u) r = (r * b) % m;
    b = (b * b) % m;
    e >>= 1;
  }
  return (uint32_t)r;
}

__device__ __forceinline__ void ranecu_init(RanecuRng& g, int batch,
                                            int32_t seed_input) {
  uint64_t leap = (uint64_t)(batch + 1) * (uint64_t)(50000 * 1000);
  uint64_t s = (uint64_t)(uint32_t)seed_input;
  g.s0 = (int32_t)((s * powmod_u32(40014u, leap, 2147483563u)) % 2147483563u);
  g.s1 = (int32_t)((s * powmod_u32(40692u, leap, 2147483399u)) % 2147483399u);
}

// ----------------------------------------------------------- tallies

// Orders a wave's LDS accesses of before with those of after, where one lane
// reads what another wrote: a wave's LDS operations complete in order, so this
// is only the statement of it to the compiler (no instruction).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Tally atomics (PRF, history counts, radial bins) through
// global (address space 1) pointers.  The tally pointers are read from the
// geometry table, so the compiler cannot tell their address space and would
// issue flat atomics; a flat operation counts against lgkmcnt as well as
// vmcnt, and the wave's next wait for an LDS or scalar load would then wait
// for the atomic to reach L2 (on every detection, at the pencil beam's few
// hot pixels).  A global atomic without return counts against vmcnt only.
template <class T>
__device__ __forceinline__ void tally_add(T* p, T v) {
  __hip_atomic_fetch_add((__attribute__((address_space(1))) T*)p, v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
}

// How a photon ended (kNone: by a step of length -99, the reference's own mark
// of a photon lost inside dist_to_surface).
enum Fate : int {
  kNone = 0, kDetect = 1, kDetectOut = 2, kAbsTop = 3, kAbsBulk = 4,
  kLost = 5, kOutOfCol = 6, kTheta1 = 7,
  // what follows an in-column pass of a photon that has not ended: the wall's
  // Fresnel branch, a restart, the next pass, a sample of a direction.  A hit
  // of the pass's draw changes kHit of the code: detected or reflected by the
  // sensor, absorbed or sampled at the top, wall or crosstalk.
  kHit = 32,
  kWall = 16, kTrapped = 17, kAlive = kDetectOut ^ kHit, kSampleTop = kAbsTop ^ kHit,
  kSample = kWall ^ kHit
};
static_assert(kAlive < kSampleTop && kSampleTop < kSample, "samples are the highest codes");
__device__ __forceinline__ bool ended(int fate) { return fate < kWall; }
static_assert(kDetectOut - 1 == FD2_C_DETECT && kAbsTop - 1 == FD2_C_ABS_TOP &&
              kAbsBulk - 1 == FD2_C_ABS_BULK && kLost - 1 == FD2_C_LOST &&
              kOutOfCol - 1 == FD2_C_OUTOFCOL && kTheta1 - 1 == FD2_C_THETA1,
              "fates in counter order");
// counter of an ended photon whose pixel is not known yet (kDetectOut)
__device__ __forceinline__ int fate_counter(int fate) {
  return fate == kNone ? (int)FD2_C_REGEN : fate - 1;
}

// photon state, all in registers.  The event's position and history stay
// in the event record; the caller passes them where they are needed.
// `st` is the photon's loop passes so far (kMaxLoops cap, 21 bits) and where
// its next pass starts: kStResume after a reflection by the sensor (its next
// in-column step is due; the count is one less, as that pass counts again),
// kStNewColumn when a crosstalk's neighbour-column
// sample is due, with the samples rejected so far (<= 100) in bits 24-30.  One
// word, so that a photon moves through the queues without packing.
constexpr uint32_t kStLoops = 0x1fffffu, kStResume = 1u << 21, kStNewColumn = 1u << 31;
constexpr int kStRejected = 24;
struct Photon {
  float px, py, pz;   // position (the detection point once detected)
  float ux, uy, uz;   // direction cosines
  float nx, ny, nz;   // surface normal
  float xc, yc;       // current column axis (the event's first column at start)
  uint32_t st;
  int fate;           // set when the photon ends
};

// A new photon of event ev at its emission point.  The first column is
// centred on the event (x - col_dx, y): the reference re-centres at the
// first dist_to_surface of a photon (main/kernel_cuda_c_ver1_0.cu:985-989),
// and nothing reads the centre before that.
__device__ __forceinline__ void start_photon(Photon& p, const fd2_event& ev) {
  p.px = ev.x;
  p.py = ev.y;
  p.pz = ev.z;
  p.xc = ev.x - ev.col_dx;
  p.yc = ev.y;
  p.st = 0;
  p.fate = kNone;
  p.nx = p.ny = p.nz = 0.0f;
}

// Detection: pixel floor((x-lb)/pitch), inside iff lb <= x <= ub
// (main/kernel_cuda_c_ver1_0.cu:3402-3419).  A detected photon ends with
// fate kDetectOut; when the kernels count it, this gives its pixel and makes
// the fate kDetect if it lies in the image.
struct Pixel {
  int i, j;
};
__device__ __forceinline__ Pixel detected_pixel(Photon& p, const GeomDev& g) {
  const float ax = p.px - g.lbx, ay = p.py - g.lby;
  float qx, qy;
  if (g.inv_pixel != 0.0f) {
    qx = ax * g.inv_pixel;
    qy = ay * g.inv_pixel;
  } else {
    qx = ax / (float)g.pixel;
    qy = ay / (float)g.pixel;
  }
  const Pixel x{(int)floorf(qx), (int)floorf(qy)};
  if (p.px <= g.ubx && p.py <= g.uby && p.px >= g.lbx && p.py >= g.lby &&
      x.i >= 0 && x.i < g.xdim && x.j >= 0 && x.j < g.ydim)
    p.fate = kDetect;
  return x;
}

// PRF index (row-major, xdim x ydim) of a pixel
__device__ __forceinline__ int32_t pix_index(const Pixel& x, const GeomDev& g) {
  return x.i * g.ydim + x.j;
}

// ------------------------------------------------------- vector helpers

template <class M = MathDevice>
__device__ __forceinline__ void renorm(float& x, float& y, float& z,
                                       const ColumnGeom& g) {
  if constexpr (M::kFaithful) {  // (float)sqrt((double)s) is sqrtf(s)
    const float nrm = sqrtf(x * x + y * y + z * z);
    if (nrm < kNormLo || nrm > kNormHi) {
      x = x / nrm;
      y = y / nrm;
      z = z / nrm;
    }
  } else {
    float nrm = fd2_sqrt_unit(x * x + y * y + z * z);
    if (nrm < kNormLo || nrm > kNormHi) {
      const float inv = 1.0f / nrm;
      x = x * inv;
      y = y * inv;
      z = z * inv;
    }
  }
}

// trans_dir_cos (main/kernel_cuda_c_ver1_0.cu:3169-3205)
template <class M = MathDevice>
__device__ __forceinline__ void reflect(Photon& p, const ColumnGeom& g) {
  float ca = -p.ux * p.nx + -p.uy * p.ny + -p.uz * p.nz;
  p.ux = 2.0f * ca * p.nx + p.ux;
  p.uy = 2.0f * ca * p.ny + p.uy;
  p.uz = 2.0f * ca * p.nz + p.uz;
  renorm<M>(p.ux, p.uy, p.uz, g);
}

// refraction with sin(theta1) = s1, sin(theta2) = s2, cos(theta2) = c2
__device__ __forceinline__ void refract(Photon& p, float s1, float s2, float c2,
                                        const GeomDev& g) {
  float ca = -p.ux * p.nx + -p.uy * p.ny + -p.uz * p.nz;
  float ratio = s2 / s1;
  p.ux = -p.nx * c2 - ratio * (p.ux + ca * p.nx);
  p.uy = -p.ny * c2 - ratio * (p.uy + ca * p.ny);
  p.uz = -p.nz * c2 - ratio * (p.uz + ca * p.nz);
  renorm(p.ux, p.uy, p.uz, g);
}

// refraction from the angles theta1, theta2, MathFaithful:
// d' = -n cos(t2) - (sin t2 / sin t1)(d + (-d.n) n), each component a double
// expression rounded to float
__device__ __forceinline__ void refract_angles(Photon& p, float t1, float t2,
                                               const GeomDev& g) {
  const float ca = -p.ux * p.nx + -p.uy * p.ny + -p.uz * p.nz;
  const fd2_ff ct = fd2x_cos(t2);
  const fd2_ff ratio = fd2x_div(fd2x_sin(t2), fd2x_sin(t1));
  p.ux = fd2x_refract_component(p.nx, p.ux + ca * p.nx, ct, ratio);
  p.uy = fd2x_refract_component(p.ny, p.uy + ca * p.ny, ct, ratio);
  p.uz = fd2x_refract_component(p.nz, p.uz + ca * p.nz, ct, ratio);
  renorm<MathFaithful>(p.ux, p.uy, p.uz, g);
}

// x, y direction cosines rr (cos, sin) of the azimuth 2 pi u of a new draw
// u: in quarter turns (MathDevice), or theta = (float)(u * twopipen) and the double products
// (MathFaithful, main/kernel_cuda_c_ver1_0.cu:582-584)
template <class M, class Rng>
__device__ __forceinline__ void azimuth(float rr, Rng& rng, float& x, float& y) {
  if constexpr (M::kFaithful) {
    fd2x_polar(rr, fd2x_mul_dconst(rng.u(), FD2X_TWOPI_D), &x, &y);
  } else {
    float sn, cs;
    fd2_sincos_quarters(rng.u4(), &sn, &cs);
    x = rr * cs;
    y = rr * sn;
  }
}

// RoughSurface (main/kernel_cuda_c_ver1_0.cu:3261-3300): perturbation with
// z = 2s-1 and radius sqrt(1-s^2) (s, not z), normalised, then
// n <- normalise(beta*p + n).  rough_offset draws the normalised p.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ void rough_offset(Rng& rng, float& qx, float& qy, float& qz) {
  float s = rng.u();
  qz = fmaf(2.0f, s, -1.0f);  // 2 s - 1, one rounding either way
  if constexpr (M::kFaithful) {
    // theta = s * 2.0f * pi with the double pi (K:3275), the double
    // cos/sin products and sqrt(pow + pow + pow) (K:3277-3285)
    const float rr = sqrtf(1.0f - s * s);
    s = rng.u();
    fd2x_polar(rr, fd2x_mul_dconst(s * 2.0f, FD2X_PI_D), &qx, &qy);
    const float nb = fd2x_norm3(qx, qy, qz);
    qx = qx / nb;
    qy = qy / nb;
    qz = qz / nb;
  } else {
    azimuth<M>(fd2_sqrt_01(1.0f - s * s), rng, qx, qy);
    float inv = fd2_rsqrt(qx * qx + qy * qy + qz * qz);
    qx = qx * inv;
    qy = qy * inv;
    qz = qz * inv;
  }
}

template <class Rng, class M = MathDevice>
__device__ __forceinline__ void rough(Rng& rng, float& nx, float& ny, float& nz,
                                      float beta) {
  float qx, qy, qz;
  rough_offset<Rng, M>(rng, qx, qy, qz);
  const float rx = beta * qx + nx, ry = beta * qy + ny;
  // a normal in the plane (the constant 0) adds nothing
  const float rz = __builtin_constant_p(nz) && nz == 0.0f ? beta * qz : beta * qz + nz;
  if constexpr (M::kFaithful) {
    const float nb = fd2x_norm3(rx, ry, rz);
    nx = rx / nb;
    ny = ry / nb;
    nz = rz / nb;
  } else {
    float inv = fd2_rsqrt(rx * rx + ry * ry + rz * rz);
    nx = rx * inv;
    ny = ry * inv;
    nz = rz * inv;
  }
}

// isotropic direction at photon termination / trapped restart
// (main/kernel_cuda_c_ver1_0.cu:578-592)
// (MathFaithful: the radius is sqrt(1.0 - r*r) in double, K:581)
template <class Rng, class M = MathDevice>
__device__ __forceinline__ void emit_dir(Rng& rng, Photon& p, const ColumnGeom& g) {
  float r = rng.u() * 2.0f - 1.0f;
  p.uz = r;
  float rr;
  if constexpr (M::kFaithful)
    rr = fd2x_sqrt_one_minus(r * r);
  else
    rr = fd2_sqrt_01(1.0f - r * r);
  azimuth<M>(rr, rng, p.ux, p.uy);
  renorm<M>(p.ux, p.uy, p.uz, g);
}

// first photon of an event: |2u-1| > 0.01 by rejection
// (main/hybridMANTIS_c_ver1_0.c:257-277)
template <class Rng, class M = MathDevice>
__device__ __forceinline__ void emit_first_dir(Rng& rng, Photon& p,
                                               const ColumnGeom& g) {
  float r = rng.u() * 2.0f - 1.0f;
  while (fabsf(r) <= 0.01f) r = rng.u() * 2.0f - 1.0f;
  p.uz = r;
  float rr = fd2_sqrt_01(1.0f - r * r);
  azimuth<M>(rr, rng, p.ux, p.uy);
  renorm<M>(p.ux, p.uy, p.uz, g);
}

// ---------------------------------------------------------- transport

__device__ __forceinline__ bool outside_xy(const Photon& p, const ColumnGeom& g) {
  float eps = kEpsLt;  // opaque: the compiler would make one comparison of a
  asm volatile("" : "+s"(eps));  // minimum, with two more instructions
  return (p.px < kEpsLt) | (p.px > g.xdet) | (p.py < eps) | (p.py > g.ydet);
}

__device__ __forceinline__ bool out_of_slab(const Photon& p, const ColumnGeom& g) {
  return outside_xy(p, g) || fabsf(p.pz) > g.half_h;
}

// Optional per-step trace (FP64 re-trace check): 14 floats per step.
struct StepSink {
  float* buf;
  int32_t* count;
  int32_t max_steps;
  int32_t photon;
  bool on;
};

// dist_to_surface (main/kernel_cuda_c_ver1_0.cu:966-1185): move to the
// nearer of the column wall (larger ray/cylinder root) and the plane
// z = +-H/2; lost check; out-of-column nudge (back 0.5 um along -d, halving
// on overshoot, at most 10+10 tries).  Returns the distance, or -99 when the
// photon was lost or left its column (fate set).
//
// MathDevice: straight-line code for directions and distances of ordinary
// size, with the correctly rounded root, reciprocal and quotient of
// fd2_math.h; a lane outside its limits (in about one step of 2^20) takes the
// IEEE operations in a branch that a wave nearly always skips.  Inside the
// limits both roots are ordered, so the wall distance is the first, and the
// direction is not along the axis.  The limit on the plane's distance is one on
// the quotient itself: a photon far outside the layer (its distance to the plane
// then overflows or is infinite) would get NaN from the short form.  A numerator
// other than 0 is at least 2^-33 (H/2 >= 2^-8), so a quotient up to 2^27 also
// means |uz| >= 2^-60, the short quotient's own limit.  The radii are compared by their squares:
// rn > r_nudge is s > nudge_sq for the rounded root rn of s, and a candidate's
// root can only exceed the current one when its square does.
template <bool TRACE, class M = MathDevice>
__device__ __forceinline__ float dist_to_surface(Photon& p, const ColumnGeom& g,
                                                 StepSink* sink) {
  const float H2 = g.half_h;
  const float t0 = p.px, t1 = p.py, t2 = p.pz;
  const float xc = p.xc, yc = p.yc;
  const float dx0 = p.px - xc, dy0 = p.py - yc;
  const float qa = p.ux * p.ux + p.uy * p.uy;
  const float qb = 2.0f * (dx0 * p.ux + dy0 * p.uy);
  const float qc = dx0 * dx0 + dy0 * dy0 - g.r_sq;
  const float disc = qb * qb - 4.0f * qa * qc;
  // the plane z = +H/2 (going up) or -H/2 (going down) when it is nearer
  // than the wall, or when the direction is along the axis
  const float zpl = __builtin_copysignf(H2, p.uz);
  float dcyl, dpl = 0.0f;
  bool plane = false, general = true;
  if constexpr (!M::kFaithful) {
    dcyl = (fd2_sqrt_pos(disc) - qb) * fd2_recip(2.0f * qa);
    dpl = fd2_div(zpl - p.pz, p.uz);
    plane = !(dpl >= dcyl);
    // dcyl is NaN for a negative, zero or infinite discriminant
    general = !((qa >= 0x1p-32f) & (dcyl <= g.dist_max) & (fabsf(dpl) <= g.dist_max));
  }
  if (M::kFaithful || __builtin_expect(general, 0)) {
    float r1, r2;
    if constexpr (M::kFaithful) {  // double root and quotients (K:992-998)
      fd2x_roots(qb, disc, 2.0f * qa, &r1, &r2);
    } else {
      const float sq = sqrtf(disc);
      const float inv2a = 1.0f / (2.0f * qa);
      r1 = (-qb + sq) * inv2a;
      r2 = (-qb - sq) * inv2a;
    }
    dcyl = 999.0f;
    if (r1 >= r2)
      dcyl = r1;
    else if (r2 > r1)
      dcyl = r2;
    plane = false;
    if (p.uz > 0.0f || p.uz < 0.0f) {
      dpl = (zpl - p.pz) / p.uz;
      const bool axial = fabsf(p.ux) < kEpsLt && fabsf(p.uy) < kEpsLt &&
                         fabsf(p.uz - (p.uz > 0.0f ? 1.0f : -1.0f)) < kEpsLt;
      plane = axial || !(dpl >= dcyl);
    }
  }
  const float d = plane ? dpl : dcyl;
  p.pz = plane ? zpl : t2 + d * p.uz;
  p.px = t0 + d * p.ux;
  p.py = t1 + d * p.uy;

  int code = kNone;
  uint32_t decisions = 0, iters = 0;  // traced nudge moves (1) / halvings (0)
  const bool lost = out_of_slab(p, g);
  if (lost) code = kLost;
  const float dx = p.px - xc, dy = p.py - yc;
  float s = dx * dx + dy * dy;
  if (!lost & (s > g.nudge_sq)) {
    float step = 0.5f;
    int moved = 0, shrunk = 0;
    // one try; a candidate farther out halves the step instead.  The move is
    // the ordinary outcome, so the other one undoes it in a branch.
    auto nudge = [&]() {
      const float ox = p.px, oy = p.py, os = s;
      p.px = ox - step * p.ux;
      p.py = oy - step * p.uy;
      const float ex = p.px - xc, ey = p.py - yc;
      s = ex * ex + ey * ey;
      bool farther = false;
      if (__builtin_expect(s > os, 0)) {
        farther = sqrtf(s) > sqrtf(os);
        if (farther) {
          p.px = ox;
          p.py = oy;
          s = os;
          step = step * 0.5f;
          ++shrunk;
        }
      }
      if (TRACE && !farther) decisions |= 1u << iters;
      if (TRACE) ++iters;
      ++moved;
    };
    nudge();  // nearly always enough
    if (__builtin_expect(s > g.nudge_sq, 0)) {
      do nudge(); while (s > g.nudge_sq && moved - shrunk < 10 && shrunk < 10);
      if (s > g.nudge_sq) code = kOutOfCol;
    }
    if (outside_xy(p, g)) code = code > (int)kLost ? code : (int)kLost;
  }
  if (TRACE && sink->on) {
    const int slot = atomicAdd(sink->count, 1);
    if (slot < sink->max_steps) {
      float* o = sink->buf + (size_t)slot * 14;
      o[0] = t0; o[1] = t1; o[2] = t2;
      o[3] = p.ux; o[4] = p.uy; o[5] = p.uz;
      o[6] = xc; o[7] = yc;
      o[8] = p.px; o[9] = p.py; o[10] = p.pz;
      o[11] = __int_as_float(code == kLost ? 1 : code == kOutOfCol ? 2 : 0);
      o[12] = __int_as_float(sink->photon);
      o[13] = __uint_as_float(decisions | (iters << 20) | ((uint32_t)plane << 25));
    }
  }
  p.fate = code;
  return code != kNone ? -99.0f : d;
}

// isotropic (main/kernel_cuda_c_ver1_0.cu:702-732): in-column step, then
// bulk absorption at -ln(u)/mu (drawn even when the step was lost).
// true = photon ended.
template <class Rng, bool TRACE, class M = MathDevice>
__device__ __forceinline__ bool isotropic(Rng& rng, Photon& p, const ColumnGeom& g,
                                          StepSink* sink) {
  const float ds = dist_to_surface<TRACE, M>(p, g, sink);
  const bool ended = fabsf(ds - (-99.0f)) < kEpsLt;
  const bool bulk = __float_as_uint(g.neg_inv_bulk) != 0u;
  bool absorbed = false;
  if (M::kFaithful && bulk) {  // (float)((double)(-1/mu) * log(u)), K:712
    const float da = fd2x_scaled_log(g.neg_inv_bulk, rng.u());
    absorbed = ds >= da && ds >= 0.0f;
  } else if (bulk) {
    const float u = rng.u();
    // -ln u >= 1 - u, so the absorption length da = -ln(u)/bulk exceeds a
    // step shorter than (1 - u)/bulk less a 2^-20 margin (which covers the
    // logarithm's error and the roundings, checked for every u the kernel
    // draws); only the remaining steps need the logarithm, and the outcome
    // is the same
    if (__builtin_expect(!(ds < ((1.0f - u) * -g.neg_inv_bulk) * 0.99999904632568359375f), 0)) {
      const float da = g.neg_inv_bulk * fd2_log(u);
      absorbed = ds >= da && ds >= 0.0f;
    }
  } else {
    absorbed = ds >= 999999.0f;
  }
  if (absorbed) p.fate = kAbsBulk;
  return ended || absorbed;
}

// fd2_acos(x) < 0 || fd2_acos(x) > 1.57 from comparisons.  The arc cosine
// crosses 1.57 at x = cos(1.57) = 7.9633e-4; over all floats x in [-1, 1],
// fd2_acos(x) >= 0, x <= 7.90e-4 gives an angle above 1.57 and x >= 8.03e-4
// one at or below it, and between the two fd2_acos is its |x| <= 1/2 branch
// (fd2_acos_small), evaluated only for a cosine in that band (about one in
// 10^5).  |x| > 1 and NaN give a NaN angle, which is neither.
__device__ __forceinline__ bool angle_over_157(float x) {
  const bool below = x <= 7.90e-4f;
  bool over = below && x >= -1.0f;
  if (__builtin_expect(x < 8.03e-4f && !below, 0)) {
    asm volatile("");  // kept a branch
    over = fd2_acos_small(x) > 1.57f;
  }
  return over;
}

// acos(x) < 0 || acos(x) > 1.57 under either arithmetic (MathFaithful: the C
// library's acosf, K:2531, :1904)
template <class M>
__device__ __forceinline__ bool angle_over(float x) {
  if constexpr (M::kFaithful) {
    const float a = fd2x_acosf(x);
    return a < 0.0f || a > 1.57f;
  } else {
    return angle_over_157(x);
  }
}

// New column orientation (transmit/boundary_analysis/refl_bottom,
// main/kernel_cuda_c_ver1_0.cu:2452-2488, 2501-2538, 1769-1804, 3036-3070):
// n = -d perturbed with beta = 1, projected on xy and renormalised, then
// perturbed with beta (always for refl_bottom); accept when
// acos(-d.n) <= 1.57.  One sample; true = accepted (p.n is the sample
// either way).
template <class Rng, class M = MathDevice>
__device__ __forceinline__ bool column_normal_sample(Rng& rng, Photon& p, const ColumnGeom& g,
                                                     float mx, float my, float mz,
                                                     bool always_rough) {
  float nx, ny, nz = 0.0f;
  if constexpr (M::kFaithful) {
    // RoughSurface(beta = 1) of -d, then the xy projection renormalised
    nx = mx;
    ny = my;
    float tz = mz;
    rough<Rng, M>(rng, nx, ny, tz, 1.0f);
    const float den = sqrtf(nx * nx + ny * ny);
    nx = nx / den;
    ny = ny / den;
  } else {
    // -d perturbed with beta = 1 and projected on xy: the xy part of p + m
    // is normalised directly (the same direction as normalising p + m first)
    float qx, qy, qz;
    rough_offset(rng, qx, qy, qz);
    nx = qx + mx;
    ny = qy + my;
    const float inv = fd2_rsqrt(nx * nx + ny * ny);
    nx = nx * inv;
    ny = ny * inv;
  }
  if (always_rough || g.beta > 0.0f) rough<Rng, M>(rng, nx, ny, nz, g.beta);
  p.nx = nx;
  p.ny = ny;
  p.nz = nz;
  return !angle_over<M>(mx * nx + my * ny + mz * nz);
}

// Samples until accepted, while the caller's counter < 100.  true = photon
// killed (theta1).
template <class Rng, class M = MathDevice>
__device__ __forceinline__ bool column_normal(Rng& rng, Photon& p,
                                              const GeomDev& g, float mx,
                                              float my, float mz, int& tries,
                                              bool always_rough) {
  while (!column_normal_sample<Rng, M>(rng, p, g, mx, my, mz, always_rough)) {
    if (tries >= 100) {
      p.fate = kTheta1;
      return true;
    }
    tries++;
  }
  return false;
}

__device__ __forceinline__ bool at_top_up(const Photon& p, const ColumnGeom& g) {
  return fabsf(p.pz - g.half_h) < kEpsLt && p.uz > 0.0f;
}

// refl_bottom (main/kernel_cuda_c_ver1_0.cu:2985-3087).  true = ended.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ bool refl_bottom(Rng& rng, Photon& p,
                                            const GeomDev& g) {
  const float tx = p.px, ty = p.py, tz = p.pz;
  const float mx = -p.ux, my = -p.uy, mz = -p.uz;
  const float d = rng.u() * g.dspan + g.d_min;
  const float dtop = (g.half_h - tz) / p.uz;
  p.px = tx + p.ux * d;
  p.py = ty + p.uy * d;
  p.pz = tz + p.uz * d;
  if (outside_xy(p, g)) {
    p.fate = kLost;
    return true;
  }
  if (p.pz > g.half_h) {
    if (dtop < d && dtop > kEpsGt) {
      p.px = tx + p.ux * dtop;
      p.py = ty + p.uy * dtop;
      p.pz = g.half_h;
      return false;
    }
    p.fate = kLost;
    return true;
  }
  int tries = 0;
  return column_normal<Rng, M>(rng, p, g, mx, my, mz, tries, true);
}

// sensor plane reached between columns: reflect + refl_bottom, or detect.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ bool gap_sensor(Rng& rng, Photon& p,
                                           const GeomDev& g) {
  if (rng.u() < g.sensor_refl) {
    p.nx = 0.0f;
    p.ny = 0.0f;
    p.nz = 1.0f;
    reflect<M>(p, g);
    return refl_bottom<Rng, M>(rng, p, g);
  }
  p.fate = kDetectOut;
  return true;
}

// transmit with flagCCT = 0 (main/kernel_cuda_c_ver1_0.cu:2421-2865):
// flight of U(dmin,dmax) between columns against the detector's top
// (reflector/absorber), bottom (sensor) and sides, then the next column's
// orientation.  true = ended.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ bool transmit_gap(Rng& rng, Photon& p,
                                          const GeomDev& g) {
  const float H2 = g.half_h;
  float tx = p.px, ty = p.py, tz = p.pz;
  float mx = -p.ux, my = -p.uy, mz = -p.uz;
  int tries1 = 0, tries2 = 0;
  float d = rng.u() * g.dspan + g.d_min;
  p.px = tx + p.ux * d;
  p.py = ty + p.uy * d;
  p.pz = tz + p.uz * d;
  float dtop = (H2 - tz) / p.uz;
  float dbot = (-H2 - tz) / p.uz;
  if (outside_xy(p, g)) {
    p.fate = kLost;
    return true;
  }
  if (p.pz < -H2 || p.pz > H2) {
    if (dtop < d && dtop > kEpsGt) {
      p.px = tx + p.ux * dtop;
      p.py = ty + p.uy * dtop;
      p.pz = H2;
    } else if (dbot < d && dbot > kEpsGt) {
      p.px = tx + p.ux * dbot;
      p.py = ty + p.uy * dbot;
      p.pz = -H2;
      if (gap_sensor<Rng, M>(rng, p, g)) return true;
      if (at_top_up(p, g)) goto top;
    } else {
      p.fate = kLost;
      return true;
    }
  }
  if (column_normal<Rng, M>(rng, p, g, mx, my, mz, tries1, false)) return true;
  if (fabsf(p.px) < kEpsLt || fabsf(p.px - g.xdet) < kEpsLt ||
      fabsf(p.py) < kEpsLt || fabsf(p.py - g.ydet) < kEpsLt) {
    p.fate = kLost;
    return true;
  }
top:
  if (++p.st > (uint32_t)kMaxLoops) {
    p.fate = kLost;
    return true;
  }
  if (at_top_up(p, g)) {
    p.nx = 0.0f;
    p.ny = 0.0f;
    p.nz = -1.0f;
    if (g.top_absfrac > 0.0f && rng.u() < g.top_absfrac) {
      p.fate = kAbsTop;
      return true;
    }
    p.uz = -fabsf(rng.u() * 2.0f - 1.0f);
    azimuth<M>(fd2_sqrt_01(1.0f - p.uz * p.uz), rng, p.ux, p.uy);
    tx = p.px;
    ty = p.py;
    tz = p.pz;
    mx = -p.ux;
    my = -p.uy;
    mz = -p.uz;
    d = rng.u() * g.dspan + g.d_min;
    dbot = (-H2 - tz) / p.uz;
    p.px = tx + p.ux * d;
    p.py = ty + p.uy * d;
    p.pz = tz + p.uz * d;
    if (outside_xy(p, g)) {
      p.fate = kLost;
      return true;
    }
    if (p.pz < -H2 || p.pz > H2) {
      if (dbot < d && dbot > kEpsGt) {
        p.px = tx + p.ux * dbot;
        p.py = ty + p.uy * dbot;
        p.pz = -H2;
        if (gap_sensor<Rng, M>(rng, p, g)) return true;
        if (at_top_up(p, g)) goto top;
      } else {
        p.fate = kLost;
        return true;
      }
    }
    if (column_normal<Rng, M>(rng, p, g, mx, my, mz, tries2, false)) return true;
  }
  if (fabsf(p.pz - (-H2)) < kEpsLt) {
    if (gap_sensor<Rng, M>(rng, p, g)) return true;
    if (at_top_up(p, g)) goto top;
  }
  return false;
}

// boundary_analysis (main/kernel_cuda_c_ver1_0.cu:1582-1958), split up: the
// top reflector (K:1610-1634), the crosstalk decision (K:1639-1652) and the
// neighbour column's orientation after a crosstalk (K:1655-1673) in
// hot_step, the wall's Fresnel branch (K:1677-1955) in prpt_loop below.
// Running the last later for a lane changes nothing for that photon: all its
// state and its random stream go with it.

// Crosstalk probability, piecewise linear in depth: 1 in the top fifth, z/(2
// top20) + 1/2 from there to the middle, (z + H/2)/(-H) + 1 below.  z lies in
// [-H/2, H/2] or is NaN (then no crosstalk).
template <class M>
__device__ __forceinline__ float crosstalk(float z, const ColumnGeom& g) {
  // both pieces from the uniform constants: selecting the constants instead
  // takes more instructions
  const float zl = z + g.half_h;
  float qu, ql;
  if constexpr (M::kFaithful) {
    qu = z / g.den_up;
    ql = zl / g.den_dn;
  } else {
    qu = fd2_div_by(z, g.den_up, g.inv_up);
    ql = fd2_div_by(zl, g.den_dn, g.inv_dn);
  }
  const float c = z >= 0.0f ? qu + 0.5f : ql + 1.0f;
  return z >= g.top20 ? 1.0f : c;
}

// Fresnel reflection/refraction at a column wall and the flights between
// columns it leads to (K:1677-1955).
//
// The reference runs this as one goto loop whose locals persist across its
// passes: the resample/retry counters, the stale Pr/Pt of the gap side
// without Fresnel recomputation, and the stale theta2 that a refraction
// then uses.  The Fresnel branch (K:1811-1871) is evaluated from cos(theta1)
// (the dot product the reference takes acos of) and Snell's law without the
// angles themselves: sin(theta1) = sqrt(1 - cos^2), sin(theta2) =
// (n_from/n_to) sin(theta1), cos(theta2) = sqrt(1 - sin^2), Pr =
// fd2_fresnel_r (Pr + Pt = 1, so no normalisation); theta2 persists as its
// sine and cosine.  PrptState holds them so that, with stop_at_gap, the loop stops
// before each flight through the gap (after the refraction out of a column,
// and after a reflection off the outside of the next column) and returns
// kPrGap; a later call with inside = false continues with that flight.  The
// photon's arithmetic and draws are the same whether or not it stops there.
struct PrptState {
  uint32_t tries;  // theta, smooth, reperturb, normal counters, 8 bits each
  float pr;        // reflection probability
  float s2, c2;    // sin, cos of theta2
};
// the reference starts with Pr = 0 and theta2 = 0
__device__ __forceinline__ PrptState prpt_initial() { return PrptState{0u, 0.0f, 0.0f, 1.0f}; }
enum PrptResult : int { kPrAlive = 0, kPrEnded = 1, kPrGap = 2 };

//
// MathFaithful keeps the reference's angles instead: theta1 = acosf of the
// dot product, theta2 from asinf, Pr and Pt from the angle sums and
// differences, normalised by their sum on every pass (stale values
// included, as the reference does).  Its state is local: that arithmetic
// runs only in the whole-branch form (ba_prpt), never with stop_at_gap.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ int prpt_loop(Rng& rng, Photon& p, const GeomDev& g, PrptState& st,
                                         bool inside, bool stop_at_gap) {
  const float R = g.R;
  int theta_tries = (int)(st.tries & 0xffu), smooth_tries = (int)((st.tries >> 8) & 0xffu);
  int reperturb = (int)((st.tries >> 16) & 0xffu), normal_tries = (int)(st.tries >> 24);
  float pr = st.pr, s2 = st.s2, c2 = st.c2, s1 = 0.0f;
  float pt = 0.0f, t1 = 0.0f, t2 = 0.0f;  // MathFaithful: Pt, theta1, theta2
  float onx, ony, onz, odx, ody, odz;
  float mx, my, mz;

  if (!inside) {
    if (transmit_gap<Rng, M>(rng, p, g)) return kPrEnded;
  }

prpt:
  if (++p.st > (uint32_t)kMaxLoops) {
    p.fate = kLost;
    return kPrEnded;
  }
  if (inside) {
    const float ax = p.xc - p.px, ay = p.yc - p.py;
    if constexpr (M::kFaithful) {  // K:1686-1690
      const float mag = sqrtf(ax * ax + ay * ay);
      p.nx = ax / mag;
      p.ny = ay / mag;
    } else {
      const float inv = fd2_rsqrt(ax * ax + ay * ay);
      p.nx = ax * inv;
      p.ny = ay * inv;
    }
    p.nz = 0.0f;
    if (g.beta > 0.0f) rough<Rng, M>(rng, p.nx, p.ny, p.nz, g.beta);
  } else {
    p.xc = p.px + R * (-p.nx);
    p.yc = p.py + R * (-p.ny);
  }
  onx = p.nx; ony = p.ny; onz = p.nz;
  odx = p.ux; ody = p.uy; odz = p.uz;

reperturb_point:
  p.nx = onx; p.ny = ony; p.nz = onz;
  p.ux = odx; p.uy = ody; p.uz = odz;
  mx = -p.ux; my = -p.uy; mz = -p.uz;
  if (reperturb != 0) {
    if (g.beta > 0.0f) rough<Rng, M>(rng, p.nx, p.ny, p.nz, g.beta);
    if (!inside) {
      p.xc = p.px + R * (-p.nx);
      p.yc = p.py + R * (-p.ny);
    }
  }

no_perturbation:
  {
    float c1 = mx * p.nx + my * p.ny + mz * p.nz;  // cos(theta1)
    if (c1 > 1.0f || c1 < 0.0f) {
      if (!inside) {
        if (column_normal<Rng, M>(rng, p, g, mx, my, mz, normal_tries, false))
          return kPrEnded;
      }
      if (theta_tries < 100) {
        theta_tries++;
        goto prpt;
      }
      p.fate = kTheta1;
      return kPrEnded;
    }
    if constexpr (M::kFaithful) {
      // K:1757-1871: theta1 = acosf; TIR against asin of the index ratio;
      // theta1 < eps becomes 0.00042; theta2 = asinf((float)(ratio *
      // sin(theta1))); Pr and Pt from the angles; then both normalised
      t1 = fd2x_acosf(c1);
      bool fresnel = false;
      float snell = 0.0f;
      if (inside) {
        if (t1 > g.t1_tir_in) {
          pr = 1.0f;
          pt = 0.0f;
        } else {
          if (t1 < kEpsLt) t1 = 0.00042f;
          snell = g.ratio12;
          fresnel = true;
        }
      } else if (!g.gap_fresnel) {
        if (t1 > g.t1_tir_gap) {
          pr = 1.0f;
          pt = 0.0f;
        }
      } else {
        snell = t1 < kEpsLt ? g.ratio12 : g.ratio21;
        if (t1 < kEpsLt) t1 = 0.00042f;
        fresnel = true;
      }
      if (fresnel) {
        t2 = fd2x_asinf(fd2x_scaled_sin(snell, t1));
        fd2x_fresnel(t1, t2, &pr, &pt);
      }
      const float tot = pr + pt;
      pr = pr / tot;
      pt = pt / tot;
      goto fresnel_draw;
    }
    s1 = fd2_sqrt_01(1.0f - c1 * c1);
    // theta1 < eps (c1 == 1) is replaced by 0.00042 rad where the reference
    // computes Pr from the angles
    float snell = 0.0f;  // n_from / n_to; 0: Pr is not recomputed
    if (inside) {
      if (c1 < g.cos_tir_in)
        pr = 1.0f;
      else
        snell = g.ratio12;
    } else if (!g.gap_fresnel) {
      if (c1 < g.cos_tir_gap) pr = 1.0f;
    } else {
      snell = c1 >= 1.0f ? g.ratio12 : g.ratio21;
    }
    if (snell != 0.0f) {
      if (c1 >= 1.0f) {
        c1 = FD2_COS_00042;
        s1 = FD2_SIN_00042;
      }
      s2 = snell * s1;
      c2 = fd2_sqrt_01(fmaxf(1.0f - s2 * s2, 0.0f));
      pr = fd2_fresnel_r(c1, s1, c2, s2);
    }
  }

fresnel_draw:
  if (rng.u() < pr) {
    reflect<M>(p, g);
    if (angle_over<M>(onx * p.ux + ony * p.uy + onz * p.uz)) {
      reperturb++;
      if (reperturb < 4) goto reperturb_point;
      p.nx = onx; p.ny = ony; p.nz = onz;
      p.ux = odx; p.uy = ody; p.uz = odz;
      mx = -p.ux; my = -p.uy; mz = -p.uz;
      reperturb = 0;
      if (smooth_tries < 25) {
        smooth_tries++;
        goto no_perturbation;
      }
      p.fate = kTheta1;
      return kPrEnded;
    }
    if (!inside) goto gap_flight;
    return kPrAlive;
  }
  if constexpr (M::kFaithful)
    refract_angles(p, t1, t2, g);
  else
    refract(p, s1, s2, c2, g);
  if (!inside) return kPrAlive;
  inside = false;
gap_flight:
  if (stop_at_gap) {
    st.tries = (uint32_t)theta_tries | ((uint32_t)smooth_tries << 8) |
               ((uint32_t)reperturb << 16) | ((uint32_t)normal_tries << 24);
    st.pr = pr;
    st.s2 = s2;
    st.c2 = c2;
    return kPrGap;
  }
  if (transmit_gap<Rng, M>(rng, p, g)) return kPrEnded;
  goto prpt;
}

// The whole branch in one call.  true = ended.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ bool ba_prpt(Rng& rng, Photon& p, const GeomDev& g) {
  PrptState st = prpt_initial();
  return prpt_loop<Rng, M>(rng, p, g, st, true, false) == kPrEnded;
}

// One algo() pass of the reference (main/kernel_cuda_c_ver1_0.cu:553-655)
// fused with the boundary interaction that follows it: in-column step and
// sensor check, then (if alive and not trapped) boundary_analysis up to its
// Fresnel branch, which the caller runs (fate kWall: ba_prpt).
//
// Crosstalk moves the photon to a neighbour column whose orientation is
// sampled from -d until a sample passes the angle test, at most 101 samples
// (K:2452-2488).  A pass takes one sample: a rejected photon is left in
// state kStNewColumn with its rejected samples counted and its next pass samples
// again instead of stepping, so its draws and arithmetic are the same, and
// lanes that need one sample do not wait in a loop for lanes that need
// several.  The top reflector's new direction (one lane of a wave in two
// passes out of five) draws the same polar/azimuth pair as a sample's
// perturbation and shares its code.
//
// The pass is bound by instruction issue, and for the last photons of a launch
// by its latency.  Selects instead of branches of one or two instructions, the
// short root, reciprocal and quotient, comparisons of squares instead of roots,
// one draw for the three decisions, and one outcome code (the fate) instead of
// flags.  On mono25x50 (100,000 histories at 25 keV, 1.1e8 photons) the first
// three took the kernel from 972 to 810 vector instructions per photon and from
// 132 to 118 ms, and the last two, with the column's constants in the kernel's
// arguments, from 108.1 to 105.5 ms.
template <class Rng, bool TRACE, class M = MathDevice>
__device__ __forceinline__ void hot_step(Rng& rng, Photon& p, const ColumnGeom& g,
                                         StepSink* sink) {
  const bool again = (int32_t)p.st < 0;  // kStNewColumn: only a sample
  // a pass resumed after a sensor reflection is the rest of the previous
  // pass: no loop count, no second sensor check
  const bool resumed = p.st >= kStResume;
  if (!again) p.st = (p.st + 1u) & kStLoops;
  p.fate = again ? kSample : kLost;
  if (!again & (p.st <= (uint32_t)kMaxLoops)) {
    const bool gone = isotropic<Rng, TRACE, M>(rng, p, g, sink);
    // what the photon has reached: the sensor plane, nothing (it moves within
    // a plane z = const), the top reflector inside a column, else the wall
    const bool sensor = !resumed & (fabsf(p.pz - (-g.half_h)) < kEpsLt);
    const bool flat = !sensor & (fabsf(p.uz) < kEpsLt);
    const bool top = (fabsf(p.pz - g.half_h) < kEpsLt) & (p.uz > 0.0f);
    // one draw decides: specular reflection by the sensor
    // (main/kernel_cuda_c_ver1_0.cu:3372-3427, else detected), absorption at
    // the top, crosstalk at the wall
    if (!gone) {
      int fate = kTrapped;
      if (!flat) {
        float cct = crosstalk<M>(p.pz, g);
        asm volatile("" : "+v"(cct));  // not in a branch of its own
        const float limit = sensor ? g.sensor_refl : top ? g.top_absfrac : cct;
        int flip = 0;
        if (sensor | !top | (g.top_absfrac > 0.0f)) flip = rng.u() < limit ? (int)kHit : 0;
        fate = (sensor ? (int)kDetectOut : top ? (int)kSampleTop : (int)kWall) ^ flip;
        if (sensor & (flip != 0)) {
          // the reference follows the reflection with another in-column step
          // inside the same pass; here that step is the start of the next
          // pass, so its code exists once
          p.nx = 0.0f;
          p.ny = 0.0f;
          p.nz = 1.0f;
          reflect<M>(p, g);
          p.st = (p.st - 1u) | kStResume;
        }
      }
      p.fate = fate;
    }
  }
  if (__builtin_expect(p.fate >= kSampleTop, 1)) {
    const bool top = p.fate == kSampleTop;
    float qx, qy, w, nx, ny, nz = 0.0f;
    const float mx = -p.ux, my = -p.uy, mz = -p.uz;
    if constexpr (M::kFaithful) {
      if (top) {
        w = rng.u() * 2.0f - 1.0f;
        azimuth<M>(fd2_sqrt_unit(1.0f - w * w), rng, qx, qy);
      }
    } else {
      const float s = rng.u();
      w = fmaf(2.0f, s, -1.0f);  // exact
      const float c = top ? w : s;
      azimuth<M>(fd2_sqrt_01(1.0f - c * c), rng, qx, qy);
    }
    if (top) {
      p.ux = qx;
      p.uy = qy;
      p.uz = -fabsf(w);
    } else {
      // neighbour column with a random orientation, direction kept
      bool over;
      if constexpr (M::kFaithful) {
        over = !column_normal_sample<Rng, M>(rng, p, g, mx, my, mz, false);
        nx = p.nx;
        ny = p.ny;
      } else {
        // rough_offset's normalisation, then the xy part of p + m normalised
        float inv = fd2_rsqrt(qx * qx + qy * qy + w * w);
        nx = qx * inv + mx;
        ny = qy * inv + my;
        inv = fd2_rsqrt(nx * nx + ny * ny);
        nx = nx * inv;
        ny = ny * inv;
        if (g.beta > 0.0f) rough<Rng, M>(rng, nx, ny, nz, g.beta);
        over = angle_over<M>(mx * nx + my * ny + mz * nz);
      }
      const bool last = over & (p.st >= kStNewColumn + (100u << kStRejected));
      p.xc = over ? p.xc : p.px - g.R * nx;
      p.yc = over ? p.yc : p.py - g.R * ny;
      p.st = over ? (p.st | kStNewColumn) + (1u << kStRejected) : p.st & kStLoops;
      p.fate = last ? kTheta1 : kAlive;
    }
  }
}

// the whole pass, for kernels that do not defer the Fresnel branch
template <class Rng, bool TRACE, class M = MathDevice>
__device__ __forceinline__ void photon_step(Rng& rng, Photon& p, const GeomDev& g,
                                            StepSink* sink) {
  hot_step<Rng, TRACE, M>(rng, p, g, sink);
  if (p.fate == kWall) p.fate = ba_prpt<Rng, M>(rng, p, g) ? p.fate : (int)kAlive;
}

// trapped photon (|dcos.z| < eps): restart from the event with a new
// direction; the column centre and rebound count are kept (C branch,
// main/kernel_cuda_c_ver1_0.cu:609-644).  The normal drawn there is never
// read before being overwritten, so only its two draws are consumed.
template <class Rng, class M = MathDevice>
__device__ __forceinline__ void restart_trapped(Rng& rng, Photon& p,
                                                const ColumnGeom& g, const fd2_event& ev) {
  emit_dir<Rng, M>(rng, p, g);
  p.px = ev.x;
  p.py = ev.y;
  p.pz = ev.z;
  if (g.beta > 0.0f) {
    (void)rng.u();
    (void)rng.u();
  }
}

}  // namespace fd2
