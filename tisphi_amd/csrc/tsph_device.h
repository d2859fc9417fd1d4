// tsph_device.h — device-side data layout and per-pair arithmetic of the
// MI355X SPH engine (gfx950, wave64).
//
// Data layout in HBM (structure of arrays, one entry per particle slot of
// the engine's particle capacity; every scene owns a contiguous range):
//   cell   int32   scene-local flattened cell id  (ix*gny + iy)*gnz + iz
//   pos    float4  cell-local offset x,y,z (metres) and m_V
//   vel    float4  velocity and density
//   vtmp   float4  v_tmp and density_tmp (leap-frog half state)
//   mass   float, type int8, id0/obj int32, stress (6 comps, component-major)
// Positions are an integer cell plus an FP32 offset from the cell corner:
// the pair vector x_i - x_j = (c_i - c_j)*grid + (o_i - o_j) keeps ~1e-9 m
// resolution anywhere in the domain.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tsph {

constexpr int kFluid = 1, kSoil = 2, kRigid = 11, kDummy = -1, kRep = -2;
constexpr int kWC = 1, kMUI = 2, kDP = 3;
constexpr int kWave = 64;

__device__ __forceinline__ bool is_flow(int t) { return t == kFluid || t == kSoil; }
__device__ __forceinline__ bool is_real(int t) { return t > 0; }
__device__ __forceinline__ bool is_bdy(int t) { return t == kDummy || t == kRep; }
// Particles the WC pair passes treat as walls (dummy extrapolation, flow
// neighbours only): boundary and rigid (solver_sph_wc.py:90).
__device__ __forceinline__ bool is_solid(int t) { return is_bdy(t) || t == kRigid; }
constexpr int kMaxRigid = 4;  // dynamic rigid objects per scene

// Stress components xx,yy,zz,xy,yz,zx.
__device__ __forceinline__ constexpr int sidx(int a, int b) {
  return a == b ? a : ((a + b) == 1 ? 3 : ((a + b) == 3 ? 4 : 5));
}

// Per-scene parameters (host fills from tsph_scene_desc; float copies are
// the float64 values rounded once, like the reference's compile-time
// constants folded into float32 code).
struct SceneDev {
  int32_t active, dim, method, boundary, kernel, ti, xsph, iexp;
  int32_t gn[3];
  int32_t tile_first, n_tiles;
  int32_t pbase, n, cbase, ncell;
  int32_t sbase, total;  // particles of the scenes with lower cells, of all scenes
  double grid, vds[3], dstart[3], dend[3], radius, dt_d;
  float g, rs2, h1, kW, kC, eps;
  float kG, kGc;  // gradient factors: -5 kW h1^2 (Wendland C2), kC h1^2 (cubic)
  float rs2c;     // stencil-cell culling threshold 1.0001 rs2
  int kcorr;      // kernelCorrection: 1 CSPM, 2 MLS switch (zero corrected gradient)
  int rep;        // add the repulsive-particle force (boundary 3 / 4; WC, muI)
  float rep_k, rep_d, rep_h;  // 0.01 c^2, particle diameter, 0.75 h
  float dt, half_dt, dt6, rho0, visc_c1, visc_c2, grav[3];
  float stiffness, exponent, vsound2, coh, mu, young, h2;
  double alpha, kc, G, K, sin_psi, eps_f;
  // dynamic rigid objects (isDynamic blocks): object ids and rest centres
  // of mass (calc_rigid_rest_m, solver_sph_base.py:467-470, 517-518)
  int32_t nrig, rig_obj[kMaxRigid];
  double rig_cm0[kMaxRigid][3];
};

// Index of particle p's object among the scene's dynamic rigid objects, -1
// for a static rigid or any other particle.
__device__ __forceinline__ int rigid_slot(const SceneDev& S, int type, int obj) {
  if (type != kRigid) return -1;
  // constant indices only: a runtime index into the scene record would put
  // the whole record on the stack of every kernel that calls this
  int r = -1;
#pragma unroll
  for (int k = kMaxRigid - 1; k >= 0; --k)
    if (k < S.nrig && S.rig_obj[k] == obj) r = k;
  return r;
}

// Particle state that survives a step (double-buffered; the counting sort
// moves it from one buffer to the other).
struct PState {
  int32_t* cell;
  float4* pos;
  float4* vel;
  float4* vtmp;
  float* mass;
  int8_t* type;
  int32_t* id0;
  int32_t* obj;
  float* sig_f;    // 6 x cap, muI stress
  double* sig_d;   // 6 x cap, DP stress
  double* seq;     // strain_equ
  double* seqp;    // strain_equ_p
  int32_t* flag;   // flag_retmap
};

// Per-step work arrays (single-buffered).
struct PWork {
  int32_t* key;      // global cell key (pre-sort order)
  int32_t* slot;     // arrival slot inside the cell (histogram atomics)
  int32_t* tmp;      // scan position -> particle
  int32_t* sid;      // particle -> scene slot (static per scene range)
  float* p;          // pressure
  float* Lc;          // inverse CSPM_L, row-major 3x3, entry c at [c*cap + p]
  float4* vp;        // WC pair record of a particle: v_tmp, p / density_tmp^2;
                     // sign bit of .w set for a boundary particle
  float* cspm;       // Shepard factor
  float* drho;       // d_density
  float4* dv;        // d_vel
  float* sigt_f;     // stress_tmp in float (muI; DP mirror), one record (rec6) per particle
  float* sigq;       // records: stress_tmp / density_tmp^2, density_tmp
  double* sigt_d;    // 6 x cap, DP stress_tmp
  double* dsig_d;    // 6 x cap, DP d_stress
  float* gradv;      // 9 x cap, velocity gradient of a DP soil particle
  double* dseq;      // d_strain_equ
  double* dseqp;     // d_strain_equ_p
  float4* xs;        // XSPH sums
  float* drho_rk;    // RK4 accumulators
  float4* dv_rk;
  double* dsig_rk;
  int32_t* count;    // cell histogram (cell capacity)
  uint8_t* cflow;    // 1 if the cell holds a flow (fluid/soil) particle
  int32_t* start;    // exclusive scan (cell capacity + 1)
  int32_t* bsum;     // scan block sums
  unsigned long long* status;  // per slot: escaped, NaN
  double* gpart;     // globals partials per tile (4 each)
  uint32_t* nl;      // neighbour lists, blocked per 64-particle tile (nl_base / nl_at)
  int32_t* nlc;      // neighbour count per particle (> nl_cap: walk instead)
  int32_t* tflag;    // per tile: what the pair passes find there (kTile*)
  // colour feed (allocated on first use)
  double* val;       // colour value per particle (current order)
  float4* rgb;       // colour per particle (current order)
  double* x0;        // 3 x cap initial position, indexed by scene base + id0
  float4* c0;        // initial colour, indexed by scene base + id0
  double* crange;    // per slot: vmax, vmin of the last v_maxmin
  // shape matching of dynamic rigid objects (allocated with the first one)
  double* rigpart;   // per tile and object: 16 partial sums
  double* rigout;    // per slot and object: centre of mass (3), rotation (9)
};

struct KArgs {
  const SceneDev* __restrict__ scenes;
  const int2* __restrict__ tiles;  // (slot, first particle) per 64-particle tile
  PState cur, alt;
  PWork w;
  int32_t cap;     // particle capacity
  int32_t ccap;    // cell capacity
  int32_t stride;  // component stride of 6-vectors (== cap)
  int32_t nl_cap;  // neighbour-list capacity per particle
  uint32_t nl_pad; // list entry of the null particle (pads lists to kNlPad)
};

// ---------------------------------------------------------- pair distance
// |x_ij| from r2 >= 0: v_sqrt_f32 (within an ulp), then the neighbouring
// float whose square is on the right side of r2 (the residual sign decides,
// with exact fused multiply-adds).  Equal bit for bit to the correctly
// rounded sqrtf for every r2 >= 2^-96 (checked over all those floats by
// tsph_check_sqrt); below 2^-96 it returns a value under 1e-8, which the
// kernels below map to 0 exactly as they map sqrtf's (r > 1e-8 test).  It
// drops sqrtf's rescaling of tiny arguments and its special-value fixup:
// 7 of its 16 instructions per pair.
__device__ __forceinline__ float pair_dist(float r2) {
  const float s = __builtin_amdgcn_sqrtf(r2);
  const float sd = __int_as_float(__float_as_int(s) - 1);
  const float su = __int_as_float(__float_as_int(s) + 1);
  const float rd = fmaf(-sd, s, r2);
  const float ru = fmaf(-su, s, r2);
  float r = rd <= 0.0f ? sd : s;
  r = ru > 0.0f ? su : r;
  return r;
}

// ------------------------------------------------------------- kernels W
// Wendland C2 (solver_sph_base.py:334-358) and cubic spline (:298-330).
__device__ __forceinline__ float kernel_W(const SceneDev& S, float rn) {
  float q = rn * S.h1;
  if (!(rn > S.eps && q <= 2.0f)) return 0.0f;
  if (S.kernel == 1) {
    float q1 = 1.0f - 0.5f * q;
    float q2 = q1 * q1;
    return S.kW * (q2 * q2) * (1.0f + 2.0f * q);
  }
  if (q <= 1.0f) {
    float qq = q * q;
    return S.kC * (0.5f * (qq * q) - qq + (float)(2.0 / 3.0));
  }
  float t = 2.0f - q;
  return S.kC / 6.0f * (t * t * t);
}
// grad W = fac * x_ij with fac = W'(r)/r.  With q = r h1, q h1 / r = h1^2,
// so W'(r)/r = -5 kW h1^2 q1^3 (Wendland C2), kC h1^2 (1.5 q - 2) (cubic,
// q <= 1) and -0.5 kC h1^2 (2 - q)^2 / q (cubic, q > 1).
__device__ __forceinline__ float kernel_gradfac(const SceneDev& S, float rn) {
  float q = rn * S.h1;
  if (!(rn > S.eps && q <= 2.0f)) return 0.0f;
  if (S.kernel == 1) {
    float q1 = 1.0f - 0.5f * q;
    return S.kG * ((q1 * q1) * q1);
  }
  if (q <= 1.0f) return S.kGc * (1.5f * q - 2.0f);
  float t = 2.0f - q;
  return S.kGc * (-0.5f * t * t) / q;
}

// The same two functions with the kernel type fixed at compile time and no
// branch (both cubic pieces are formed and one is selected): identical
// values, but a pair loop built on them is straight-line code, so the
// loads of several neighbours can be in flight together.
// 1 - q / 2 clamped to [0, 1] (the instruction's output modifier): q <= 2
// exactly where 1 - q / 2 >= 0, and beyond it W = 0 and W'(r)/r = +-0 follow
// from the zero, so the Wendland functions need no test of q.
__device__ __forceinline__ float wendland_q1(float q) {
  return __builtin_amdgcn_fmed3f(1.0f - 0.5f * q, 0.0f, 1.0f);
}
template <int KT>
__device__ __forceinline__ float kernel_W_t(const SceneDev& S, float rn) {
  const float q = rn * S.h1;
  float w;
  if (KT == 1) {
    const float q1 = wendland_q1(q);
    const float q2 = q1 * q1;
    w = S.kW * (q2 * q2) * (1.0f + 2.0f * q);
    return rn > S.eps ? w : 0.0f;
  } else {
    const float qq = q * q;
    const float wi = S.kC * (0.5f * (qq * q) - qq + (float)(2.0 / 3.0));
    const float t = 2.0f - q;
    const float wo = S.kC / 6.0f * (t * t * t);
    w = q <= 1.0f ? wi : wo;
  }
  return (rn > S.eps && q <= 2.0f) ? w : 0.0f;
}
template <int KT>
__device__ __forceinline__ float kernel_gradfac_t(const SceneDev& S, float rn) {
  const float q = rn * S.h1;
  float f;
  if (KT == 1) {
    const float q1 = wendland_q1(q);
    f = S.kG * ((q1 * q1) * q1);
    return rn > S.eps ? f : 0.0f;
  } else {
    const float fi = S.kGc * (1.5f * q - 2.0f);
    const float t = 2.0f - q;
    const float fo = S.kGc * (-0.5f * t * t) / q;
    f = q <= 1.0f ? fi : fo;
  }
  return (rn > S.eps && q <= 2.0f) ? f : 0.0f;
}

// kernel_deriv_corr (solver_sph_base.py:375-384) with kernelCorrection 1:
// the gradient times the particle's stored inverse CSPM_L.
__device__ __forceinline__ void corr_load(const float* __restrict__ Lc, int stride, int p,
                                          float m[9]) {
#pragma unroll
  for (int c = 0; c < 9; ++c) m[c] = Lc[(size_t)c * stride + p];
}
__device__ __forceinline__ void corr_apply(const float m[9], float g[3]) {
  const float o0 = (m[0] * g[0] + m[1] * g[1]) + m[2] * g[2];
  const float o1 = (m[3] * g[0] + m[4] * g[1]) + m[5] * g[2];
  const float o2 = (m[6] * g[0] + m[7] * g[1]) + m[8] * g[2];
  g[0] = o0;
  g[1] = o1;
  g[2] = o2;
}
// Inverse of calc_CSPM_L (solver_sph_base.py:410-423): adjugate times 1/det
// when |det| > eps (2D: the upper 2x2 block, the rest zero); M keeps I
// otherwise.
template <int DIM>
__device__ __forceinline__ void corr_invert(const float L[3][3], float eps, float M[9]) {
  if (DIM == 2) {
    const float det = L[0][0] * L[1][1] - L[0][1] * L[1][0];
    if (fabsf(det) > eps) {
      const float id = 1.0f / det;
      M[0] = L[1][1] * id;
      M[1] = -L[0][1] * id;
      M[2] = 0.0f;
      M[3] = -L[1][0] * id;
      M[4] = L[0][0] * id;
      M[5] = 0.0f;
      M[6] = 0.0f;
      M[7] = 0.0f;
      M[8] = 0.0f;
    }
    return;
  }
  const float c00 = L[1][1] * L[2][2] - L[1][2] * L[2][1];
  const float c01 = L[1][2] * L[2][0] - L[1][0] * L[2][2];
  const float c02 = L[1][0] * L[2][1] - L[1][1] * L[2][0];
  const float det = L[0][0] * c00 + L[0][1] * c01 + L[0][2] * c02;
  if (fabsf(det) > eps) {
    const float id = 1.0f / det;
    M[0] = c00 * id;
    M[1] = (L[0][2] * L[2][1] - L[0][1] * L[2][2]) * id;
    M[2] = (L[0][1] * L[1][2] - L[0][2] * L[1][1]) * id;
    M[3] = c01 * id;
    M[4] = (L[0][0] * L[2][2] - L[0][2] * L[2][0]) * id;
    M[5] = (L[0][2] * L[1][0] - L[0][0] * L[1][2]) * id;
    M[6] = c02 * id;
    M[7] = (L[0][1] * L[2][0] - L[0][0] * L[2][1]) * id;
    M[8] = (L[0][0] * L[1][1] - L[0][1] * L[1][0]) * id;
  }
}

// Repulsive-particle force calc_repulsive_force (solver_sph_base.py:676-690):
// F = fac * x_ij with fac = 0.01 c^2 chi(r) f(r / (0.75 h)) / r^2.
__device__ __forceinline__ float rep_fac(const SceneDev& S, float rn) {
  const float chi = (rn > 0.0f && rn < S.rep_d) ? 1.0f - rn / S.rep_d : 0.0f;
  const float gam = rn / S.rep_h;
  const float two3 = (float)(2.0 / 3.0);
  float f = 0.0f;
  if (gam > 0.0f && gam <= two3) {
    f = two3;
  } else if (gam > two3 && gam <= 1.0f) {
    f = 2.0f * gam - 1.5f * (gam * gam);
  } else if (gam > 1.0f && gam < 2.0f) {
    const float t = 2.0f - gam;
    f = 0.5f * (t * t);
  }
  return S.rep_k * chi * f / (rn * rn);
}

template <class T>
__device__ __forceinline__ T ipow_dev(T x, int n) {
  T r = T(1), b = x;
  int m = n < 0 ? -n : n;
  while (m) {
    if (m & 1) r = r * b;
    b = b * b;
    m >>= 1;
  }
  return n < 0 ? T(1) / r : r;
}

// Tait equation of state (solver_sph_wc.py:88).
__device__ __forceinline__ float wc_eos(const SceneDev& S, float rt) {
  float x = rt / S.rho0;
  float xp = S.iexp != INT32_MIN ? ipow_dev(x, S.iexp) : powf(x, S.exponent);
  float v = S.stiffness * (xp - 1.0f);
  return v > 0.0f ? v : 0.0f;
}

// Cell of an offset along one axis: floor((double)o/grid) with the
// offset renormalised into [0, grid) (same rule as the oracle).
__device__ __forceinline__ void renorm(int32_t& c, float& o, double grid) {
  double od = (double)o;
  if (od != od) return;  // NaN offset: keep the cell (the NaN is reported by the step)
  double k = floor(od / grid);
  double r = od - k * grid;
  if (r >= grid) {
    k += 1.0;
    r -= grid;
  }
  float on = (float)r;
  if (on < 0.0f) on = 0.0f;
  if ((double)on >= grid) {
    k += 1.0;
    on = 0.0f;
  }
  c += (int32_t)k;
  o = on;
}

__device__ __forceinline__ void decode_cell(const SceneDev& S, int32_t c, int& x, int& y, int& z) {
  int yz = S.gn[1] * S.gn[2];
  x = c / yz;
  int r = c - x * yz;
  y = r / S.gn[2];
  z = r - y * S.gn[2];
}

// The neighbour walk of for_all_neighbors (particle_system.py:259-269):
// the 3^dim stencil in ndrange((-1,2),...) order around the centre cell
// (scx,scy,scz), particles j ascending in each cell, j != i and
// |x_ij|^2 < r_s^2.  Cells outside the grid are skipped.  (cix,ciy,ciz) is
// the cell the offset `oi` is measured from (equal to the centre except
// after advect_pos, before the next hash).
// fn(j, x, y, z, r2, m_V_j, code) with code = (dx+1)<<4 | (dy+1)<<2 | (dz+1)
// the stencil cell of j.
//
// CULL (only with the centre = i's own cell and offsets in [0, g), i.e.
// right after the hash): skip stencil cells whose box lies farther than
// r_s from i.  A candidate there is at least the per-axis gap away
// (offsets are >= 0 and < g), so its r2 exceeds rs2 by more than the
// rounding of either sum; the threshold rs2c = 1.0001 rs2 keeps that
// margin.  Visited pairs and their order are unchanged.
template <int DIM, bool CULL = false, class Fn>
__device__ __forceinline__ void walk(const SceneDev& S, const int32_t* __restrict__ start,
                                     const float4* __restrict__ pos, int32_t shift, int i,
                                     int scx, int scy, int scz, int cix, int ciy, int ciz,
                                     float oix, float oiy, float oiz, Fn&& fn) {
  const int gy = S.gn[1], gz = S.gn[2];
#pragma unroll 1
  for (int dx = -1; dx <= 1; ++dx) {
    const int nx = scx + dx;
    if (nx < 0 || nx >= S.gn[0]) continue;
    const float bx = oix + (float)(cix - nx) * S.g;
    const float ax = dx < 0 ? oix : (dx > 0 ? S.g - oix : 0.0f);
#pragma unroll 1
    for (int dy = -1; dy <= 1; ++dy) {
      const int ny = scy + dy;
      if (ny < 0 || ny >= gy) continue;
      const float by = oiy + (float)(ciy - ny) * S.g;
      const float ay = dy < 0 ? oiy : (dy > 0 ? S.g - oiy : 0.0f);
      const int32_t rowkey = S.cbase + (nx * gy + ny) * gz;
#pragma unroll 1
      for (int dz = (DIM == 3 ? -1 : 0); dz <= (DIM == 3 ? 1 : 0); ++dz) {
        const int nz = scz + dz;
        if (DIM == 3 && (nz < 0 || nz >= gz)) continue;
        if (CULL) {
          const float az = DIM == 3 ? (dz < 0 ? oiz : (dz > 0 ? S.g - oiz : 0.0f)) : 0.0f;
          if (fmaf(az, az, fmaf(ay, ay, ax * ax)) > S.rs2c) continue;
        }
        const float bz = DIM == 3 ? oiz + (float)(ciz - nz) * S.g : 0.0f;
        const int32_t key = rowkey + nz;
        const int code = ((dx + 1) << 4) | ((dy + 1) << 2) | (dz + 1);
        const int32_t jb = start[key] + shift;
        const int32_t je = start[key + 1] + shift;
        auto cand = [&](int32_t j, const float4& pj) {
          const float x = bx - pj.x;
          const float y = by - pj.y;
          const float z = DIM == 3 ? bz - pj.z : 0.0f;
          const float r2 = fmaf(z, z, fmaf(y, y, x * x));
          if (r2 < S.rs2 && j != i) fn(j, x, y, z, r2, pj.w, code);
        };
        int32_t j = jb;
        // four candidates' loads in flight before the first test
        for (; j + 4 <= je; j += 4) {
          const float4 p0 = pos[j], p1 = pos[j + 1], p2 = pos[j + 2], p3 = pos[j + 3];
          cand(j, p0);
          cand(j + 1, p1);
          cand(j + 2, p2);
          cand(j + 3, p3);
        }
        for (; j < je; ++j) cand(j, pos[j]);
      }
    }
  }
}

// Neighbour-list entry: particle index << 6 | stencil code (2 bits per axis).
constexpr int kNlShift = 6;
__device__ __forceinline__ uint32_t nl_entry(int j, int code) {
  return ((uint32_t)j << kNlShift) | (uint32_t)code;
}
// Storage of the lists, blocked per 64-particle tile: entry k of particle p
// is at nl_base(p) + nl_at(k), the tile's piece of 64 nl_cap entries being
// rows of 256, four entries (16 bytes) of each particle.  A replay load (16
// particles, a quad of lanes each) is 256 contiguous bytes and a build store
// (64 particles, four entries each) a contiguous kilobyte; a tile's lists
// are one piece whatever the engine capacity.  nl_cap is a multiple of 4.
__host__ __device__ __forceinline__ size_t nl_base(int p, int nl_cap) {
  return (size_t)(p >> 6) * ((size_t)nl_cap << 6) + ((size_t)(p & 63) << 2);
}
__host__ __device__ __forceinline__ size_t nl_at(int k) {
  return ((size_t)(k >> 2) << 8) + (size_t)(k & 3);
}

// Lanes per particle of the list replay: L = 4 lanes of a quad share one
// particle (L = 1: the stencil walk).  Lane q forms the terms of the list
// entries k + q, and every lane then adds the four terms in list order, the
// other lanes' read through DPP quad permutations: the same additions in the
// same order as with one lane, so the sums have the same bits.
// Lists are padded to a multiple of kNlPad entries with the null particle,
// whose terms are replaced by +0 (which changes no sum, since a sum that
// starts at +0 is never -0 in round-to-nearest).  Bound by vector issue
// on large scenes, by latency on small ones.  Against a lane per particle:
// WC fluid pass 1090 -> 925 us at 4.5 M particles in 3D, step 365 -> 200 at
// 191 k in 3D and 94 -> 58 at 9 k in 2D (with the list build's part).
constexpr int kMaxBlock = 256;  // largest threads per block of a pair kernel
constexpr int kNlPad = 4;
constexpr int kLanes = 4;

// x of lane SRC of this lane's group of L.
template <int L, int SRC>
__device__ __forceinline__ float group_read(float x) {
  static_assert(L == 4, "a quad");
  constexpr int ctrl = SRC * 0x55;  // quad_perm [SRC, SRC, SRC, SRC]
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xf, 0xf, true));
}
// on ? x : +0 as a select (the guard keeps the compiler from forming x in a
// branch, which also keeps the quad's additions from reading it through
// their DPP operand).
__device__ __forceinline__ float term_if(bool on, float x) {
  asm("" : "+v"(x));
  return on ? x : 0.0f;
}
// acc += the terms of the group's lanes, lane 0 first.
template <int L, int NT>
__device__ __forceinline__ void ordered_add(float (&acc)[NT], const float (&t)[NT]) {
#pragma unroll
  for (int c = 0; c < NT; ++c) {
    if (L == 1) {
      acc[c] += t[c];
    } else {
      acc[c] += group_read<4, 0>(t[c]);
      acc[c] += group_read<4, 1>(t[c]);
      acc[c] += group_read<4, 2>(t[c]);
      acc[c] += group_read<4, 3>(t[c]);
    }
  }
}

// Tables of the list replay: one LDS array per kernel, shared by all its
// replays (an array inside the template below would be one per instance).
constexpr int kTabCols = kMaxBlock / 4;
__device__ __forceinline__ float2* xy_table() {
  __shared__ float2 tab[11 * kTabCols];
  return tab;
}
__device__ __forceinline__ float* z_table() {
  __shared__ float tab[3 * kTabCols];
  return tab;
}

// A record of six floats (and one more) per particle, padded to 32 bytes: a
// pair pass gathers a neighbour's in two loads, where six arrays took six.
constexpr int kRec = 8;
__device__ __forceinline__ void rec6_load(const float* __restrict__ r, int i, float (&s)[6]) {
  const float4 a = *reinterpret_cast<const float4*>(r + (size_t)i * kRec);
  const float2 b = *reinterpret_cast<const float2*>(r + (size_t)i * kRec + 4);
  s[0] = a.x;
  s[1] = a.y;
  s[2] = a.z;
  s[3] = a.w;
  s[4] = b.x;
  s[5] = b.y;
}
__device__ __forceinline__ float rec7_load(const float* __restrict__ r, int i, float (&s)[6]) {
  const float4 a = *reinterpret_cast<const float4*>(r + (size_t)i * kRec);
  const float4 b = *reinterpret_cast<const float4*>(r + (size_t)i * kRec + 4);
  s[0] = a.x;
  s[1] = a.y;
  s[2] = a.z;
  s[3] = a.w;
  s[4] = b.x;
  s[5] = b.y;
  return b.z;
}
__device__ __forceinline__ void rec6_store(float* __restrict__ r, int i, const float (&s)[6], float e = 0.0f) {
  float4* __restrict__ o = reinterpret_cast<float4*>(r + (size_t)i * kRec);
  o[0] = make_float4(s[0], s[1], s[2], s[3]);
  o[1] = make_float4(s[4], s[5], e, 0.0f);
}

// A particle with the start of its list.
struct Own {
  float4 P;
  int n;            // list length
  uint32_t e0, e1;  // this lane's entries of the first two quads
};

// acc[c] += term c of every neighbour of particle i, in list order.
// fn(j, x, y, z, r2, m_V_j, t) forms the terms t of one pair.
template <int DIM, int NT, class Fn>
__device__ __forceinline__ void sum_list(const SceneDev& S, const uint32_t* __restrict__ nl, int nl_cap,
                                         const float4* __restrict__ pos, int i, const Own& o,
                                         float (&acc)[NT], Fn&& fn) {
  const int n = o.n;
  const float oix = o.P.x, oiy = o.P.y, oiz = o.P.z;
  const uint32_t* __restrict__ li = nl + nl_base(i, nl_cap) + (threadIdx.x & 3);
  // shifted centres oi + (c_i - c_j) g for c_j - c_i = -1, 0, +1 (exact
  // products, rounded once: the same values the walk forms), kept in LDS
  // (one table per kernel, a wave only ever touches its own columns, one per
  // particle): x and y together in row (x digit, y digit) of the stencil
  // code, z in a table of its own, so a pair looks them up by address
  // instead of by compares and selects
  constexpr int kCols = kTabCols;
  float2* __restrict__ txy = xy_table();
  float* __restrict__ tz = DIM == 3 ? z_table() : nullptr;
  const int col = (int)threadIdx.x >> 2;
#pragma unroll
  for (int dx = 0; dx < 3; ++dx)
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
      txy[(dx * 4 + dy) * kCols + col] =
          make_float2(dx == 0 ? oix + S.g : (dx == 1 ? oix : oix + (-1.0f) * S.g),
                      dy == 0 ? oiy + S.g : (dy == 1 ? oiy : oiy + (-1.0f) * S.g));
  if (DIM == 3) {
    tz[0 * kCols + col] = oiz + S.g;
    tz[1 * kCols + col] = oiz;
    tz[2 * kCols + col] = oiz + (-1.0f) * S.g;
  }
  auto pair = [&](uint32_t e, const float4& pj, float (&tm)[NT]) {
    const int j = (int)(e >> kNlShift);
    const float2 c = txy[(int)((e >> 2) & 15u) * kCols + col];
    const float x = c.x - pj.x;
    const float y = c.y - pj.y;
    const float z = DIM == 3 ? tz[(int)(e & 3u) * kCols + col] - pj.z : 0.0f;
    const float r2 = DIM == 3 ? fmaf(z, z, fmaf(y, y, x * x)) : fmaf(y, y, x * x);
    fn(j, x, y, z, r2, pj.w, tm);
  };
  auto rec = [&](uint32_t e) {
    float4 v = pos[e >> kNlShift];
    // whole 16-byte record: in 2D z is unused, and the compiler would split
    // the load into two
    if (DIM == 2) asm volatile("" : "+v"(v.z));
    return v;
  };
  if (n <= 0) return;
  // Two quads of entries per turn, the next turn's loaded while this turn's
  // neighbours arrive (and none past the list's end: a line of list that no
  // pair needs cost the batched 2D pass 20 %).
  uint32_t e0 = o.e0, e1 = o.e1;
  float t[NT];
  int k = 0;
  for (; k + 8 <= n; k += 8) {
    const float4 p0 = rec(e0), p1 = rec(e1);
    uint32_t f0 = 0, f1 = 0;
    if (k + 8 < n) f0 = li[nl_at(k + 8)];
    if (k + 12 < n) f1 = li[nl_at(k + 12)];
    pair(e0, p0, t);
    ordered_add<4>(acc, t);
    pair(e1, p1, t);
    ordered_add<4>(acc, t);
    e0 = f0;
    e1 = f1;
  }
  if (k + 4 < n) {
    pair(e0, rec(e0), t);
    ordered_add<4>(acc, t);
    e0 = e1;
    k += 4;
  }
  if (k < n) {
    // the last quad: the padding's terms are left out, which an infinite state
    // of the particle itself would make 0 * infinity
    const bool in = k + (int)(threadIdx.x & 3) < n;
    pair(e0, rec(e0), t);
#pragma unroll
    for (int c = 0; c < NT; ++c) t[c] = term_if(in, t[c]);
    ordered_add<4>(acc, t);
  }
}

}  // namespace tsph
