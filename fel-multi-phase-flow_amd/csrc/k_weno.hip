// k_weno.hip -- momentum advection, WENO5 in derivative form.
//
// Reference: srcs/cal_advu_weno5.f:1-257 with srcs/weno5.h:1-71.  Interior
// cells get the three upwind-weighted derivatives of each velocity
// component; the ghost shell is zeroed (the reference's clearing pass,
// cal_advu_weno5.f:44-52), so the outputs are written exactly once.
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "felgpu.hpp"

namespace fel {

// srcs/weno5.h:24-71 (nonlinear weights with the 1e-80 floor of
// cal_advu_weno5.f:31), expressions in the reference's order.
//
// T = double is the reference's FP64 arithmetic.  T = float (the FP32 mode)
// evaluates the same weights from differences scaled by the power of two
// that brings their largest magnitude to [1, 2): the weights are homogeneous
// of degree 0 in that scale, so the scaling changes nothing but keeps the
// degree-8 products of the smoothness indicators inside the FP32 range; the
// stencil derivatives use the unscaled differences.  The scale is that of the
// five differences the upwind side reads: a sixth, much larger one beside them
// would push the weight sums under their floor.
// 1/x for the weights: IEEE division in FP64 (and the tangent mode); in the
// FP32 mode the hardware reciprocal (v_rcp_f32, 1 ulp), whose rounding is
// far below the FP32 mode's accuracy bar and which replaces a ten-instruction
// division sequence in a compute-bound kernel.  The weight sums are floored
// at 1e-30 and, after the scaling, lie far above the smallest normal float.
// FAST (FP64): the quotient by Newton's iteration from the hardware reciprocal
// with the final residual correction (Markstein), which is the correctly
// rounded 1/x where no step leaves the normal range; the weight sums are at
// least 1e-80, and one of 1e300 or more (or NaN) sets `odd`.  (The one divisor
// for which the iteration may end a unit low, a significand of all ones, does
// not: gfx950's approximation of it is the rounded quotient already, at every
// exponent, and the steps keep it.)
template <bool FAST, class T>
__device__ __forceinline__ T weight_rcp(T x, bool& odd) {
  if constexpr (is_f32<T>) {
    return __builtin_amdgcn_rcpf(x);
  } else if constexpr (FAST) {
    odd |= !(x < 1.0e300);
    T r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(fma(-x, r, 1.0), r, r);
  } else {
    return T(1.0) / x;
  }
}

// p x + y with p a power of two, where the reference rounds p x and then the
// sum: p x is exact, so one fused operation gives the same bits.
template <class T>
__device__ __forceinline__ T pow2_fma(double p, T x, T y) {
  if constexpr (std::is_floating_point_v<T>) return fma(T(p), x, y);
  else return x * T(p) + y;
}

// One upwind-biased side of srcs/weno5.h: w1*df1 + w2*df2 + w3*df3 of the
// side whose differences are (d5, d3, d1, e1, e3) -- the m side (dfm5,
// dfm3, dfm1, dfp1, dfp3), the p side mirrored (dfp5, dfp3, dfp1, dfm1,
// dfm3) -- with the candidate derivatives from those differences and the
// smoothness indicators from their scaled copies (s5, s3, s1, t1, t3);
// expressions in the reference's order.
template <bool FAST, class T>
__device__ __forceinline__ T weno_side(T d5, T d3, T d1, T e1, T e3, T s5, T s3, T s1, T t1,
                                       T t3, bool& odd) {
  const T c3 = T(3.0), c5 = T(5.0), c7 = T(7.0), c11 = T(11.0), c13 = T(13.0);
  const T df_1 = pow2_fma(2.0, d5, -(d3 * c7)) + d1 * c11;
  const T df_2 = pow2_fma(2.0, e1, -d3 + d1 * c5);
  const T df_3 = pow2_fma(2.0, d1, e1 * c5) - e3;
  T a, b;
  a = pow2_fma(-2.0, s3, s5) + s1;
  b = pow2_fma(-4.0, s3, s5) + s1 * c3;
  const T sm_1 = a * a * c13 + b * b * c3;
  a = pow2_fma(-2.0, s1, s3) + t1;
  b = s3 - t1;
  const T sm_2 = a * a * c13 + b * b * c3;
  a = pow2_fma(-2.0, t1, s1) + t3;
  b = pow2_fma(-4.0, t1, s1 * c3) + t3;
  const T sm_3 = a * a * c13 + b * b * c3;
  T a_1 = sm_2 * sm_3, a_2 = sm_1 * sm_3, a_3 = sm_1 * sm_2;
  a_1 = a_1 * a_1;
  a_2 = a_2 * a_2;
  a_3 = a_3 * a_3;
  a_2 = a_2 * T(6.0);
  a_3 = a_3 * c3;
  const T deninv = weight_rcp<FAST>(a_1 + a_2 + a_3 + guard<T>(1.0e-80), odd);
  const T w_1 = a_1 * deninv, w_3 = a_3 * deninv;
  const T w_2 = T(1.0) - w_1 - w_3;
  return w_1 * df_1 + w_2 * df_2 + w_3 * df_3;
}

// srcs/weno5.h:24-71: (velm1 * m side + velp1 * p side) / 12 with velm1 =
// vel + |vel| and velp1 = vel - |vel|, vel = vel4 / 4, from the values
// f(-3..3).  For vel != 0 one of the two factors is an exact zero and its side
// is not evaluated: the sum is the other term's value, the same bits (up to
// the sign of a zero result), and in the tangent mode the zero factor's
// derivative is zero too.  vel = 0 (or NaN) evaluates both sides as written.
//
// The p side of f is minus the m side of its mirror image, sign for sign, and
// both factors are 2 |vel| up to that sign.  So the upwind half of the values
// is selected per lane and one polynomial is evaluated: a branch on the sign
// runs both sides, one after the other, in every wavefront whose 64 cells hold
// both signs.  The powers of two in 2 |vel| = |vel4| / 2 go into the constant.
//
// FAST: without branches on a lane; for vel = 0 the m side stands for both, which
// is the same zero while both sides are finite.  `odd` is set where they may not
// be: with a value of 1e30 or more (below it the products of eight differences,
// scaled ones in FP32, stay in range), looked for in wavefronts that hold a zero
// velocity, and wherever the side that is formed sets it through its weights' sum.
template <bool FAST, class T>
__device__ __forceinline__ T weno_up(T fm3, T fm2, T fm1, T f0, T fp1, T fp2, bool& odd) {
  const T d5 = fm2 - fm3, d3 = fm1 - fm2, d1 = f0 - fm1, e1 = fp1 - f0, e3 = fp2 - fp1;
  if constexpr (is_f32<T>) {
    const T mx = fmax(fmax(fmax(fabs(d5), fabs(d3)), fmax(fabs(d1), fabs(e1))), fabs(e3));
    // scale by the exact power of two that brings the largest difference to
    // [1, 2): the weights are invariant to it, and unlike 1/mx (which
    // overflows for mx below ~2.9e-39) it stays finite for subnormal mx
    const int e = mx > T(0.0) ? -ilogbf(mx) : 0;
    return weno_side<FAST>(d5, d3, d1, e1, e3, T(ldexpf(d5, e)), T(ldexpf(d3, e)),
                           T(ldexpf(d1, e)), T(ldexpf(e1, e)), T(ldexpf(e3, e)), odd);
  } else {
    return weno_side<FAST>(d5, d3, d1, e1, e3, d5, d3, d1, e1, e3, odd);
  }
}

template <bool FAST, class T>
__device__ __forceinline__ T weno5(T fm3, T fm2, T fm1, T f0, T fp1, T fp2, T fp3, T vel4,
                                   bool& odd) {
  const T r12 = T(1.0) / T(12.0), r24 = T(0.5) * r12;
  const bool down = vel4 < T(0.0);
  if constexpr (FAST) {
    const bool still = !(fabs(vel4) > T(0.0));
    if (__builtin_amdgcn_ballot_w64(still) != 0) {
      bool small = true;
      for (const T x : {fm3, fm2, fm1, f0, fp1, fp2, fp3}) small = small && fabs(x) < T(1.0e30);
      odd |= still && !small;
    }
  }
  const T side = weno_up<FAST>(down ? fp3 : fm3, down ? fp2 : fm2, down ? fp1 : fm1, f0,
                               down ? fm1 : fp1, down ? fm2 : fp2, odd);
  if constexpr (FAST) {
    return (fabs(vel4) * side) * r24;
  } else {
    if (down || vel4 > T(0.0)) return (fabs(vel4) * side) * r24;
    const T vel00 = vel4 * T(0.25), velab = fabs(vel00);
    const T velm1 = vel00 + velab, velp1 = vel00 - velab;
    return (velm1 * side - velp1 * weno_up<FAST>(fp3, fp2, fp1, f0, fm1, fm2, odd)) * r12;
  }
}

// The value at a byte offset from a row's start.  The rows are the same for
// all lanes of a wavefront (64 cells along x), so their addresses are scalar
// and a load needs no vector address arithmetic.
template <class T>
__device__ __forceinline__ T at(const T* row, uint32_t off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(row) + off);
}

template <class T>
__device__ __forceinline__ void put(T* row, uint32_t off, T x) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(row) + off) = x;
}

template <bool FAST, class T>
__device__ __forceinline__ T weno_dir(const T* __restrict__ f, uint32_t off, ptrdiff_t st, T vel4,
                                      bool& odd) {
  return weno5<FAST>(at(f - 3 * st, off), at(f - 2 * st, off), at(f - st, off), at(f, off),
                     at(f + st, off), at(f + 2 * st, off), at(f + 3 * st, off), vel4, odd);
}

// The WENO5 derivative from a register queue f(k-3..k+3) of the cell's own
// column (the z direction).
template <bool FAST, class T>
__device__ __forceinline__ T weno_q(const T* q, T vel4, bool& odd) {
  return weno5<FAST>(q[0], q[1], q[2], q[3], q[4], q[5], q[6], vel4, odd);
}

// Interior cells, k-marching: one thread per (i,j) column of one component
// over up to kWenoK planes.  The own column's component at k-3..k+3 lives in a
// register queue, so the z-direction stencil loads one new plane per step
// instead of seven; the in-plane (x, y) stencils and the transport velocities
// are loaded from the same plane, which the block's other lanes share in cache.
//
// Bound by the FP64 units: about 95 operations a derivative, issued in 75% of
// the cycles.  Measured at 512x128x256 with velocities of both signs everywhere:
// 606-625 us in FP64, 331-342 us in FP32 and 1.52 ms in the tangent mode; a
// branch per side and all components in one thread took 810 us, 464 us and
// 2.10 ms, the one polynomial per lane alone 657 us in FP64.  In a flow whose
// wavefronts mostly hold one sign (the droplet impact) the branch cost little:
// 636 -> 612 us.  One component per thread holds 90 registers instead of 124,
// which keeps 5 wavefronts on a SIMD instead of 4 and triples the threads of a
// small grid (7.6 -> 4.6 us at 32x8x32); the three columns of one place run side
// by side on one XCD, whose L2 they share.  Planes per thread: 633, 606 and 606
// us with 4, 8 and 16.
constexpr int kWenoK = 8;

template <int COMP, class T>
__device__ __forceinline__ void weno_column(ptrdiff_t Y, ptrdiff_t Z, T dxinv, T dyinv, T dzinv,
                                            const T* __restrict__ u, const T* __restrict__ v,
                                            const T* __restrict__ w, T* __restrict__ out,
                                            uint32_t off, int planes) {
  const ptrdiff_t X = 1;
  // towards the component's face
  const ptrdiff_t S = COMP == 0 ? X : (COMP == 1 ? Y : Z);
  const T* __restrict__ f = COMP == 0 ? u : (COMP == 1 ? v : w);
  T q[7];
#pragma unroll
  for (int m = 0; m < 6; m++) q[m + 1] = at(f + (m - 3) * Z, off);
  for (int n = 0; n < planes; n++, f += Z, u += Z, v += Z, w += Z, out += Z) {
    // one address register: the lanes' offset is made opaque, or its widening
    // to 64 bits leaves the loop and every load adds it to the row again
    uint32_t o = off;
    asm volatile("" : "+v"(o));
#pragma unroll
    for (int m = 0; m < 6; m++) q[m] = q[m + 1];
    q[6] = at(f + 3 * Z, o);
    // The transport velocity is the mean of two face means; its halvings are
    // exact and left to weno5 (sums of two sums, four times the mean).
    // (srcs/cal_advu_weno5.f:80-120, 147-187, 214-254)
    auto cell = [&](auto fast, bool& odd) {
      constexpr bool F = decltype(fast)::value;
      const T vx = COMP == 0 ? (at(u - X, o) + q[3]) + (q[3] + at(u + X, o))
                             : (at(u - X, o) + at(u - X + S, o)) + (at(u, o) + at(u + S, o));
      const T vy = COMP == 1 ? (at(v - Y, o) + q[3]) + (q[3] + at(v + Y, o))
                             : (at(v - Y, o) + at(v - Y + S, o)) + (at(v, o) + at(v + S, o));
      const T vz = COMP == 2 ? (q[2] + q[3]) + (q[3] + q[4])
                             : (at(w - Z, o) + at(w - Z + S, o)) + (at(w, o) + at(w + S, o));
      T a = weno_dir<F>(f, o, X, vx, odd) * dxinv;
      a = a + weno_dir<F>(f, o, Y, vy, odd) * dyinv;
      return a + weno_q<F>(q, vz, odd) * dzinv;
    };
    T a;
    bool odd = false;
    if constexpr (std::is_floating_point_v<T>) {
      a = cell(std::true_type{}, odd);
      if (odd) a = cell(std::false_type{}, odd);
    } else {
      a = cell(std::false_type{}, odd);
    }
    put(out, o, a);
  }
}

template <class T>
__global__ void __launch_bounds__(256) weno_march_kernel(Dims d, T dxinv, T dyinv, T dzinv,
                                                         const T* __restrict__ u,
                                                         const T* __restrict__ v,
                                                         const T* __restrict__ w,
                                                         T* __restrict__ au, T* __restrict__ av,
                                                         T* __restrict__ aw, int gx, int gy,
                                                         int kc) {
  const int L = xcd_tile((int)blockIdx.x, (int)gridDim.x);
  const int comp = L % 3, tile = L / 3;
  const int bx = tile % gx, t = tile / gx, by = t % gy, bz = t / gy;
  const int i = 1 + bx * 64 + (int)threadIdx.x;
  const int j = 1 + by * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  if (i > d.ni || j > d.nj) return;
  const int k0 = 1 + bz * kc, planes = min(d.nk - k0 + 1, kc);
  const ptrdiff_t Y = d.sx, Z = (ptrdiff_t)d.sx * d.sy, c = d.ix(1 + bx * 64, j, k0);
  const uint32_t off = (uint32_t)(threadIdx.x * sizeof(T));
  if (comp == 0)
    weno_column<0>(Y, Z, dxinv, dyinv, dzinv, u + c, v + c, w + c, au + c, off, planes);
  else if (comp == 1)
    weno_column<1>(Y, Z, dxinv, dyinv, dzinv, u + c, v + c, w + c, av + c, off, planes);
  else
    weno_column<2>(Y, Z, dxinv, dyinv, dzinv, u + c, v + c, w + c, aw + c, off, planes);
}

// The reference clears the outputs over the padded image and fills the
// interior (cal_advu_weno5.f:44-52): interior by the marching kernel, the
// ghost shell zeroed separately, so every output element is written once.
template <class T>
void advect_weno5(const Dims d, double dxinv, double dyinv, double dzinv, const T* __restrict__ u,
                  const T* __restrict__ v, const T* __restrict__ w, T* __restrict__ au,
                  T* __restrict__ av, T* __restrict__ aw) {
  const int gx = (d.ni + 63) / 64, gy = (d.nj + 3) / 4;
  const int kc = march_planes(3 * gx * gy, d.nk, kWenoK), gz = (d.nk + kc - 1) / kc;
  weno_march_kernel<T><<<dim3(3 * gx * gy * gz), dim3(64, 4, 1), 0, stream()>>>(
      d, T(dxinv), T(dyinv), T(dzinv), u, v, w, au, av, aw, gx, gy, kc);
  FEL_CHECK(hipGetLastError());
  launch_shell(d, [=] __device__(int i, int j, int k) {
    const int c = d.ix(i, j, k);
    au[c] = T(0.0);
    av[c] = T(0.0);
    aw[c] = T(0.0);
  });
}

// Result reuse.  The timestep asks for the advection of (u,v,w) and then of
// (uo,vo,wo) (srcs/main.f90:532-533); uo..wo are copies of the previous
// step's u..w (main.f90:686-688), whose advection the previous step already
// computed into adv_u..adv_w.  Content versions identify that case exactly:
// before adv_u..adv_w are overwritten, their buffers (holding the advection
// of the inputs whose versions they were computed from) are parked in a
// stash, and a later request whose inputs carry those same versions gets the
// parked buffers swapped in instead of a recomputation -- the same bits, no
// kernel.  Anything not provably identical is recomputed.
namespace {

struct WenoKey {
  uint64_t ver[3];
  int ni, nj, nk;
  double dx, dy, dz;
  bool operator==(const WenoKey& o) const {
    return ver[0] == o.ver[0] && ver[1] == o.ver[1] && ver[2] == o.ver[2] && ni == o.ni &&
           nj == o.nj && nk == o.nk && dx == o.dx && dy == o.dy && dz == o.dz;
  }
};

struct WenoHeld {  // what one output triple holds, valid while its versions are unchanged
  const void* out[3];
  uint64_t out_ver[3];
  WenoKey key;
};

struct WenoStash {
  bool valid = false;
  WenoKey key{};
  void* buf[3] = {nullptr, nullptr, nullptr};
  size_t bytes = 0;
};

std::vector<WenoHeld> g_held;
WenoStash g_stash;

bool reuse_disabled() { return !result_reuse(); }

WenoHeld* held_for(const void* const* out) {
  for (auto& h : g_held)
    if (h.out[0] == out[0] && h.out[1] == out[1] && h.out[2] == out[2]) return &h;
  return nullptr;
}

void record_held(const void* const* out, size_t n, const WenoKey& k) {
  WenoHeld* h = held_for(out);
  if (!h) {
    g_held.push_back(WenoHeld{});
    h = &g_held.back();
    for (int m = 0; m < 3; m++) h->out[m] = out[m];
  }
  for (int m = 0; m < 3; m++) h->out_ver[m] = content_version(out[m], n);
  h->key = k;
}

}  // namespace

template <class T>
void weno_compute(const Dims d, double dxinv, double dyinv, double dzinv, const double* u,
                  const double* v, const double* w, double* adv_u, double* adv_v, double* adv_w) {
  Call c("cal_advu_weno5_");
  const T* du = c.in_t<T>(u, d.n3, "u");
  const T* dv = c.in_t<T>(v, d.n3, "v");
  const T* dw = c.in_t<T>(w, d.n3, "w");
  T* au = c.out_t<T>(adv_u, d.n3, "adv_u");
  T* av = c.out_t<T>(adv_v, d.n3, "adv_v");
  T* aw = c.out_t<T>(adv_w, d.n3, "adv_w");
  advect_weno5<T>(d, dxinv, dyinv, dzinv, du, dv, dw, au, av, aw);
  c.finish();
}

void weno_release() {
  for (int m = 0; m < 3; m++)
    if (g_stash.buf[m]) FEL_CHECK(hipFree(g_stash.buf[m]));
  g_stash = WenoStash{};
  g_held.clear();
}

}  // namespace fel

using namespace fel;

extern "C" {

// srcs/cal_advu_weno5.f:1-2
void cal_advu_weno5_(const int* ni, const int* nj, const int* nk, const double* dxinv,
                     const double* dyinv, const double* dzinv, const double* u, const double* v,
                     const double* w, double* adv_u, double* adv_v, double* adv_w) {
  const Dims d = make_dims(*ni, *nj, *nk);
  const size_t n = (size_t)d.n3;
  const void* out[3] = {adv_u, adv_v, adv_w};
  const void* in[3] = {u, v, w};
  WenoKey key{{content_version(u, n), content_version(v, n), content_version(w, n)},
              *ni, *nj, *nk, *dxinv, *dyinv, *dzinv};
  bool track = !reuse_disabled();
  for (int m = 0; m < 3 && track; m++) {
    if (key.ver[m] == 0 || content_version(out[m], n) == 0) track = false;
    for (int q = 0; q < 3; q++)
      if (out[m] == in[q] || (q != m && out[m] == out[q])) track = false;
  }
  if (track) {
    WenoHeld* h = held_for(out);
    bool h_valid = h != nullptr;
    for (int m = 0; m < 3 && h_valid; m++)
      if (h->out_ver[m] != content_version(out[m], n)) h_valid = false;
    if (g_stash.valid && g_stash.key == key) {
      // the parked buffers hold exactly this result: swap them in
      for (int m = 0; m < 3; m++) g_stash.buf[m] = exchange_device_buffer(out[m], n, g_stash.buf[m]);
      g_stash.valid = h_valid;
      if (h_valid) g_stash.key = h->key;
      Call c("cal_advu_weno5_");  // the outputs change: fresh versions
      with_flow([&](auto t) {
        for (int m = 0; m < 3; m++) c.out_t<decltype(t)>(out[m], n, "adv");
      });
      c.finish();
      record_held(out, n, key);
      return;
    }
    if (h_valid) {
      // park what the outputs hold before overwriting them
      const size_t bytes = n * (size_t)elem_size(out[0]);
      if (g_stash.bytes != bytes) {
        for (int m = 0; m < 3; m++) {
          if (g_stash.buf[m]) FEL_CHECK(hipFree(g_stash.buf[m]));
          FEL_CHECK(hipMalloc(&g_stash.buf[m], bytes));
        }
        g_stash.bytes = bytes;
      }
      for (int m = 0; m < 3; m++) g_stash.buf[m] = exchange_device_buffer(out[m], n, g_stash.buf[m]);
      g_stash.valid = true;
      g_stash.key = h->key;
    }
  }
  with_flow([&](auto t) {
    weno_compute<decltype(t)>(d, *dxinv, *dyinv, *dzinv, u, v, w, adv_u, adv_v, adv_w);
  });
  if (track) record_held(out, n, key);
}

}  // extern "C"
