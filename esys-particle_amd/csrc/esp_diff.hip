// esp_diff.hip - the differentiable, batched engine of include/esp_diff.h.
//
// Forward: the reference's time step for the calibration model class over one
// particle set holding any number of specimens (per-specimen parameters),
// with the main engine's neighbour-search kernels (cell binning, 27-cell pair
// search) and two launches a step:
//   k_bond_fwd_pairs  per bond: ARotBondedInteraction::calcForces + the break
//                 test (the bond leaves at the next step); per neighbour pair:
//                 RotFriction unless a live bond excludes it, shear history read
//                 from one buffer, written to the other
//   k_gather_fwd  per particle: walls, gravity, then its interactions in a
//                 fixed order (pairs by key, then bonds), the CParticle /
//                 CRotParticle update, the rebuild test
// plus a per-specimen, fixed-order sum of the measured wall's force at sample
// steps.  The neighbour lists ("epochs", one per rebuild) are immutable and kept
// for the whole run.
//
// Every step writes its state next to the one before, so a run whose states and
// shear histories fit the tape limit is its own tape.  A longer run keeps a checkpoint
// every K steps (state, shear histories), and the reverse sweep recomputes one
// segment's tape at a time (recorded epochs, no search).
//
// Backward, per step, three launches:
//   k_adj_bond      vector-Jacobian product of the bond law (16 inputs), by
//                   its hand-written reverse mode
//   k_adj_fric      vector-Jacobian product of the friction law (24 inputs,
//                   the history among them, on the recorded slip branch), by
//                   its hand-written reverse mode
//   k_adj_step      per particle, the interactions' adjoints in a fixed order
//                   and the parameter gradients credited to the first particle,
//                   then the integrator's adjoint (symplectic Euler, quaternion
//                   step and normalisation), the walls' and the loss's terms of
//                   the step before
// Every reduction has a fixed order (no atomics on doubles).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/esp_diff.h"
#include "esp_difflaw.h"
#include "esp_internal.h"
#include "esp_math.h"
#include "esp_wave.h"

namespace {

struct DiffError : std::runtime_error {
  int code;
  DiffError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

struct DiffMemory : DiffError {
  explicit DiffMemory(const std::string& m) : DiffError(ESP_ERR_DEVICE, m) {}
};

#define DCHK(expr)                                                                       \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess)                                                                \
      throw DiffError(ESP_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t cap = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf()
  {
    if (p) (void)hipFree(p);
  }
  void reserve(size_t n)
  {
    if (n <= cap && p) return;
    if (p) {
      DCHK(hipDeviceSynchronize());
      DCHK(hipFree(p));
    }
    p = nullptr;
    const size_t c = std::max<size_t>(n, 16);
    cap = 0;
    if (hipError_t e = hipMalloc(&p, c * sizeof(T)); e != hipSuccess) {
      p = nullptr;
      if (e != hipErrorOutOfMemory) DCHK(e);
      (void)hipGetLastError();
      throw DiffMemory(std::string("hipMalloc: ") + hipGetErrorString(e));
    }
    cap = c;
  }
  void release()
  {
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
  }
  void swap(DevBuf& o)
  {
    std::swap(p, o.p);
    std::swap(cap, o.cap);
  }
};

thread_local std::string g_diff_create_err;

// Branch digest of a step: each wave hashes (its first index, its lanes'
// branch bits) and adds the hash into the step's word; the sum is independent
// of the order the waves finish in.  Two runs with equal digests took the same
// contact, slip and wall-contact branches (pair and particle indices of the
// same neighbour-table epochs).
__device__ __forceinline__ unsigned long long dmix(unsigned long long z)
{
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ void wave_digest(unsigned long long* dig, unsigned long long tag,
                                            unsigned long long m0, unsigned long long m1)
{
  const int first = __ffsll((long long)__ballot(1)) - 1;
  if ((int)__lane_id() == first) atomicAdd(dig, dmix(dmix(tag) ^ m0) + dmix(m1 ^ ~tag));
}

// ---------------------------------------------------------------------------
// device views
// ---------------------------------------------------------------------------
struct DState {
  double4* x;  // position, radius
  double4* v;  // velocity, 1/mass
  double4* w;  // angular velocity, 1/inertia
  double4* q;  // orientation
  const int* spec;
  int n;
};

#define DIFF_MAX_WALLS 4
struct DWall {
  double o[3], n[3], k;
  int measure;
};
struct DStep {
  int nw;
  DWall wall[DIFF_MAX_WALLS];
  int has_g;
  double g[3];
  double dt;
  int step;
};

// Steps are queued without host decisions: a step whose displacement test asks
// for a neighbour search records itself in `halt`, and every later step of the
// queue returns at once.
struct DRun {
  int halt, pad;
};

__device__ __forceinline__ bool run_skip(const DRun* R, int step)
{
  const int h = R->halt;
  return h != 0 && h < step;
}

// Largest block of the per-step kernels.  The law kernels declare it as their
// launch bound, which gives them 256 VGPRs a lane (the default bound of 1024
// threads caps them at 128, and the bond law then spills to scratch memory).
#define DIFF_MAX_BS 512

__global__ void k_clear_run(DRun* R)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) R->halt = 0;
}

struct DBonds {
  int nb;
  const int2* ij;
  const double4* D0;   // initial p2 - p1, |D0|
  const double4* rel;  // relative break values (n, s, t, b)
  int* bstep;          // step whose criterion broke the bond (INT_MAX: intact)
  const double2* tkb;  // per specimen (kt, kb)
};

struct DCands {
  int nc;
  const int2* ij;
  const int* bond;  // bond between the two, or -1
};

__device__ __forceinline__ tv3<double> dx3(double4 a) { return tv3<double>{a.x, a.y, a.z}; }

// ---------------------------------------------------------------------------
// tangent-linear (forward-mode) kernels: the derivative of one forward run
// along a parameter direction, on the branch the run takes.  T holds the
// state's tangent (x, v, w, q), th the shear histories' tangents; the laws run
// on duals seeded with the state's tangents and the parameters' direction.
// ---------------------------------------------------------------------------
struct DTan {
  double4* x;
  double4* v;
  double4* w;
  double4* q;
};

__device__ __forceinline__ tv3<esp_dual> dd3(double4 a, double4 t)
{
  return tv3<esp_dual>{esp_dual(a.x, t.x), esp_dual(a.y, t.y), esp_dual(a.z, t.z)};
}
__device__ __forceinline__ tquat<esp_dual> ddq(double4 a, double4 t)
{
  return tquat<esp_dual>{esp_dual(a.x, t.x), {esp_dual(a.y, t.y), esp_dual(a.z, t.z), esp_dual(a.w, t.w)}};
}

__global__ __launch_bounds__(DIFF_MAX_BS) void k_bond_tan(DState S, DTan T, DBonds B, const double4* theta, const double4* dtheta,
                           const DRun* run, int step, double* bt)
{
  if (run_skip(run, step)) return;
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B.nb) return;
  double* o = bt + 9 * (size_t)b;
  if (B.bstep[b] < step) {
    for (int k = 0; k < 9; k++) o[k] = 0.0;
    return;
  }
  const int2 e = B.ij[b];
  const double4 D = B.D0[b];
  const int s = S.spec[e.x];
  const double4 th = theta[s], dth = dtheta[s];
  const double2 tk = B.tkb[s];
  const double4 P1 = S.x[e.x], P2 = S.x[e.y];
  esp_dual kr, ks;
  double kt, kb;
  tbond_k<esp_dual>(esp_dual(th.x, dth.x), esp_dual(th.y, dth.y), tk.x, tk.y, D.w, P1.w, P2.w, 1,
                    1, 0, kr, ks, kt, kb);
  TBondResult<esp_dual> r;
  tbond_law<esp_dual>(dd3(P1, T.x[e.x]), ddq(S.q[e.x], T.q[e.x]), P1.w, dd3(P2, T.x[e.y]),
                      ddq(S.q[e.y], T.q[e.y]), P2.w, kr, ks, esp_dual(kt), esp_dual(kb),
                      tv3<esp_dual>{esp_dual(D.x), esp_dual(D.y), esp_dual(D.z)}, r);
  o[0] = r.f1.x.d; o[1] = r.f1.y.d; o[2] = r.f1.z.d;
  o[3] = r.m1.x.d; o[4] = r.m1.y.d; o[5] = r.m1.z.d;
  o[6] = r.m2.x.d; o[7] = r.m2.y.d; o[8] = r.m2.z.d;
}

__global__ __launch_bounds__(DIFF_MAX_BS) void k_fric_tan(DState S, DTan T, DCands C, const int* bstep, const double4* theta,
                           const double4* dtheta, const double4* H0, const double4* H1,
                           double4* TH0, double4* TH1, const DRun* run, int step, double dt, double* ct)
{
  if (run_skip(run, step)) return;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C.nc) return;
  // step s reads the histories of buffer s & 1 and writes the other
  const double4* hin = (step & 1) ? H1 : H0;
  const double4* thin = (step & 1) ? TH1 : TH0;
  double4* thout = (step & 1) ? TH0 : TH1;
  double* o = ct + 9 * (size_t)c;
  const int bb = C.bond[c];
  if (bb >= 0 && bstep[bb] >= step) {
    for (int k = 0; k < 9; k++) o[k] = 0.0;
    thout[c] = make_double4(0.0, 0.0, 0.0, 0.0);
    return;
  }
  const int2 e = C.ij[c];
  const double4 P1 = S.x[e.x], P2 = S.x[e.y];
  const int s = S.spec[e.x];
  const double4 th = theta[s], dth = dtheta[s];
  esp_dual kk, kks;
  tfriction_k<esp_dual>(esp_dual(th.x, dth.x), esp_dual(th.y, dth.y), 1, 1, P1.w, P2.w, 0, kk, kks);
  const double4 h = hin[c], dh = thin[c];
  tv3<esp_dual> ffr{esp_dual(h.x, dh.x), esp_dual(h.y, dh.y), esp_dual(h.z, dh.z)}, f1, m1, m2;
  bool slipping = (((int)h.w) & 1) != 0;
  const esp_dual mu(th.w, dth.w);
  tfriction_law<esp_dual>(dd3(P1, T.x[e.x]), dd3(S.v[e.x], T.v[e.x]), dd3(S.w[e.x], T.w[e.x]), P1.w,
                          dd3(P2, T.x[e.y]), dd3(S.v[e.y], T.v[e.y]), dd3(S.w[e.y], T.w[e.y]), P2.w,
                          kk, kks, mu, mu, dt, ffr, slipping, f1, m1, m2);
  thout[c] = make_double4(ffr.x.d, ffr.y.d, ffr.z.d, 0.0);
  o[0] = f1.x.d; o[1] = f1.y.d; o[2] = f1.z.d;
  o[3] = m1.x.d; o[4] = m1.y.d; o[5] = m1.z.d;
  o[6] = m2.x.d; o[7] = m2.y.d; o[8] = m2.z.d;
}

// ---------------------------------------------------------------------------
// forward kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ void bond_fwd_item(const DState& S, const DBonds& B, const double4* theta,
                                              int step, int b, double* bout)
{
  if (b >= B.nb) return;
  double* o = bout + 9 * (size_t)b;
  const int bs = B.bstep[b];
  // removed after the step whose criterion broke it: the record is zero from then on
  if (bs < step) {
    if (bs == step - 1)
      for (int k = 0; k < 9; k++) o[k] = 0.0;
    return;
  }
  const int2 e = B.ij[b];
  const double4 P1 = S.x[e.x], P2 = S.x[e.y], Q1 = S.q[e.x], Q2 = S.q[e.y];
  const double4 D = B.D0[b];
  const int s = S.spec[e.x];
  const double4 th = theta[s];
  const double2 tk = B.tkb[s];
  double kr, ks, kt, kb;
  tbond_k<double>(th.x, th.y, tk.x, tk.y, D.w, P1.w, P2.w, 1, 1, 0, kr, ks, kt, kb);
  TBondResult<double> r;
  tbond_law<double>(dx3(P1), tquat<double>{Q1.x, {Q1.y, Q1.z, Q1.w}}, P1.w, dx3(P2),
                    tquat<double>{Q2.x, {Q2.y, Q2.z, Q2.w}}, P2.w, kr, ks, kt, kb,
                    tv3<double>{D.x, D.y, D.z}, r);
  o[0] = r.f1.x; o[1] = r.f1.y; o[2] = r.f1.z;
  o[3] = r.m1.x; o[4] = r.m1.y; o[5] = r.m1.z;
  o[6] = r.m2.x; o[7] = r.m2.y; o[8] = r.m2.z;
  if (bs != INT_MAX) return;
  // CRotBondedInteraction::broken on the size-scaled break values
  // (RotBondedInteraction.cpp:144-157, 175-219): cohesion times the relative
  // values, scaled like esp_bond_constants
  const double4 rl = B.rel[b];
  const double effR = 0.5 * D.w, effA = effR * effR;
  const double momentJ = 0.5 * effR * effR * effR * effR, momentI = 0.5 * momentJ;
  const double mx_n = (th.z * rl.x) * effA, mx_s = (th.z * rl.y) * effA;
  const double mx_b = (th.z * rl.w) * momentI / effR, mx_t = (th.z * rl.z) * momentJ / effR;
  if (esp_bond_broken(r.nForce, r.shForce, r.tMoment, r.bMoment, mx_n, mx_s, mx_t, mx_b, 1.0, 1.0,
                      1.0))
    B.bstep[b] = step;
}

// History flag bits (w of a history): 1 slipping, 2 touching, 4 zero in both
// buffers (the pair has been apart for at least the last step, so neither
// buffer needs writing until it touches).  act[c]: the record of pair c holds
// this step's (nonzero) force; the gathers read only such records.  htape
// (nullable): the histories touching pairs read, kept for the reverse sweep.
__device__ __forceinline__ void fric_fwd_item(const DState& S, const DCands& C, const int* bstep,
                                              const double4* theta, double4* H0, double4* H1,
                                              double4* htape, int step, double dt, int c,
                                              double* cout, unsigned char* act,
                                              unsigned long long* dig_base)
{
  if (c >= C.nc) return;
  // step s reads the histories of buffer s & 1 and writes the other
  double4* hin = (step & 1) ? H1 : H0;
  double4* hout = (step & 1) ? H0 : H1;
  unsigned long long* dig = dig_base ? dig_base + step : nullptr;
  const int bb = C.bond[c];
  if (bb >= 0 && bstep[bb] >= step) {
    // excluded while the bond lives (a break found by this launch's bonds sets
    // bstep to step: excluded still): no record.  Its history is the zero it
    // starts with, in both buffers.
    act[c] = 0;
    return;
  }
  const int2 e = C.ij[c];
  const double4 P1 = S.x[e.x], P2 = S.x[e.y];
  const double4 h = hin[c];
  // the law's contact test, before the velocities are loaded
  const tv3<double> Dq = tsub(dx3(P1), dx3(P2));
  const double eq = P1.w + P2.w;
  const bool touching = tdot(Dq, Dq) < (eq * eq);
  tv3<double> ffr{h.x, h.y, h.z}, f1, m1, m2;
  bool slipping = false;
  if (touching) {
    const double4 V1 = S.v[e.x], V2 = S.v[e.y], W1 = S.w[e.x], W2 = S.w[e.y];
    const double4 th = theta[S.spec[e.x]];
    double kk, kks;
    tfriction_k<double>(th.x, th.y, 1, 1, P1.w, P2.w, 0, kk, kks);
    slipping = (((int)h.w) & 1) != 0;
    tfriction_law<double>(dx3(P1), dx3(V1), dx3(W1), P1.w, dx3(P2), dx3(V2), dx3(W2), P2.w, kk, kks,
                          th.w, th.w, dt, ffr, slipping, f1, m1, m2);
  }
  if (dig) {
    const unsigned long long mt = __ballot(touching), ms = __ballot(touching && slipping);
    wave_digest(dig, (unsigned long long)(c & ~63), mt, ms);
  }
  if (!touching) {
    // apart: history cleared, no force
    act[c] = 0;
    const int fw = (int)h.w;
    if ((fw & 3) != 0 || h.x != 0.0 || h.y != 0.0 || h.z != 0.0) {
      hout[c] = make_double4(0.0, 0.0, 0.0, 0.0);
    } else if (!(fw & 4)) {
      hin[c] = make_double4(0.0, 0.0, 0.0, 4.0);
      hout[c] = make_double4(0.0, 0.0, 0.0, 4.0);
    }
    return;
  }
  double* o = cout + 9 * (size_t)c;
  if (htape) htape[c] = h;
  hout[c] = make_double4(ffr.x, ffr.y, ffr.z, (double)((slipping ? 1 : 0) | 2));
  o[0] = f1.x; o[1] = f1.y; o[2] = f1.z;
  o[3] = m1.x; o[4] = m1.y; o[5] = m1.z;
  o[6] = m2.x; o[7] = m2.y; o[8] = m2.z;
  act[c] = 1;
}

// The force laws of one step: blocks [0, nbb) take the bonds, the others the
// candidate pairs, so the two laws' latencies overlap in one launch.
__global__ __launch_bounds__(DIFF_MAX_BS) void k_bond_fwd_pairs(DState S, DBonds B, DCands C,
                                                            const double4* theta, double4* H0,
                                                            double4* H1, double4* htape,
                                                            const DRun* run, int step, double dt,
                                                            int nbb, double* bout, double* cout,
                                                            unsigned char* act,
                                                            unsigned long long* dig_base)
{
  if (run_skip(run, step)) return;
  if ((int)blockIdx.x < nbb)
    bond_fwd_item(S, B, theta, step, blockIdx.x * blockDim.x + threadIdx.x, bout);
  else
    fric_fwd_item(S, C, B.bstep, theta, H0, H1, htape, step, dt,
                  ((int)blockIdx.x - nbb) * (int)blockDim.x + (int)threadIdx.x, cout, act, dig_base);
}

// The wall contacts' part of a step's branch digest (tracked runs), of the state
// before it: one launch of its own, since what a wave of the gather integrates
// depends on the launch's shape and the digest must not.
__global__ void k_wall_digest(DState S, DStep sp, const DRun* run, unsigned long long* dig_base)
{
  if (run_skip(run, sp.step)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= S.n) return;
  const double4 P = S.x[i];
  for (int k = 0; k < sp.nw; k++) {
    const DWall& W = sp.wall[k];
    const double dist = dot3(sub3(mk3(P.x, P.y, P.z), mk3(W.o[0], W.o[1], W.o[2])),
                             mk3(W.n[0], W.n[1], W.n[2]));
    wave_digest(dig_base + sp.step,
                ((unsigned long long)(i & ~63) << 3) | (unsigned long long)(k + 1),
                __ballot(dist < P.w), 0ull);
  }
}

// per particle: the measured wall's normal force on it (sample steps), walls,
// gravity, interactions in CSR order, then the update from S into So (the same
// arrays, or the next step's of a tape).
// Bound by the chain entry -> activity -> record over a particle's run.  G lanes (a
// quad, or a row of 16) share a particle: each takes every G-th entry, with the next
// one's activity and the entry after that under way, and the shares are added in
// entry order by all of them; the block's first threads, one for each of its
// particles, integrate.  One lane a particle -> this (us a step): 2,000 particles
// 22.0 -> 6.9, 20,000 26.6 -> 11.1, 254,000 55.0 -> 41.4.  TAN: the state's tangent
// is carried along.
template <int G, bool TAN>
__global__ __launch_bounds__(DIFF_MAX_BS) void k_gather_fwd(
    DState S, DState So, const double4* mass_old, const int* inc_off, const int* inc_ent, int ncand,
    const double* cout, const double* bout, const unsigned char* cact, DStep sp,
    double* wfn, DRun* run, unsigned long long thresh, DTan T, const double* ct, const double* bt,
    double* wft)
{
  constexpr int NS = TAN ? 12 : 6;
  __shared__ double sum[NS * (DIFF_MAX_BS / G)];  // [particle][component]
  const int step = sp.step;
  const int t = threadIdx.x;
  const int PB = blockDim.x / G;  // particles per block
  const int p0 = blockIdx.x * PB;
  const int pi = p0 + t / G, sub = t % G;  // the particle whose entries it adds
  const int pc = pi < S.n ? pi : 0;
  const int i = p0 + t;  // the particle it integrates (t < PB)
  const bool own = t < PB && i < S.n;
  const int e0 = inc_off[pc];
  const int e1 = pi < S.n ? inc_off[pc + 1] : e0;
  if (run_skip(run, step)) return;  // the same for the whole block
  double4 P = make_double4(0.0, 0.0, 0.0, 0.0), Om = P, Vv = P, A = P, Q = P;
  if (own) {
    P = S.x[i];
    Om = mass_old[i];
    Vv = S.v[i];
    A = S.w[i];
    Q = S.q[i];
    const dv3 x0 = mk3(P.x, P.y, P.z);
    const double r = P.w;
    dv3 F = mk3(0.0, 0.0, 0.0), tF = F;
    double wn = 0.0, twn = 0.0;
    for (int k = 0; k < sp.nw; k++) {  // CElasticWallInteraction::calcForces
      const DWall& W = sp.wall[k];
      const dv3 n = mk3(W.n[0], W.n[1], W.n[2]);
      const double dist = dot3(sub3(x0, mk3(W.o[0], W.o[1], W.o[2])), n);
      if (dist < r) {
        double f = 1.0;
        f *= 3.141592654 * r;
        const dv3 force = mul3(n, (f * W.k) * (r - dist));
        F = add3(F, force);
        if (W.measure) wn = dot3(force, n);
        if (TAN) {  // d force = -k' n (n . dx)
          const double4 Tx = T.x[i];
          const dv3 tf = mul3(n, -((f * W.k) * dot3(n, mk3(Tx.x, Tx.y, Tx.z))));
          tF = add3(tF, tf);
          if (W.measure) twn = dot3(tf, n);
        }
      }
    }
    if (wfn) wfn[i] = wn;
    if (TAN && wft) wft[i] = twn;
    if (sp.has_g) F = add3(F, mul3(mk3(sp.g[0], sp.g[1], sp.g[2]), Om.w));
    double* o = sum + NS * t;
    o[0] = F.x; o[1] = F.y; o[2] = F.z;
    if (TAN) {
      o[6] = tF.x; o[7] = tF.y; o[8] = tF.z;
    }
  }
  __syncthreads();
  double acc[NS];
  {
    const double* o = sum + NS * (t / G);
    for (int c = 0; c < NS; c++) acc[c] = (c < 3 || (c >= 6 && c < 9)) ? o[c] : 0.0;
  }
  // The interactions in CSR order.  A record with no force this step (a pair
  // apart or excluded by its bond) adds zeros: a sum that starts at +0 is not
  // changed by a zero.
  auto entry = [&](int at) { return at < e1 ? inc_ent[at] : -1; };
  auto active = [&](int e) { return e >= 0 && ((e >> 1) >= ncand || cact[e >> 1] != 0); };
  int ent = entry(e0 + sub), nxt = entry(e0 + G + sub);
  bool on = active(ent);
  for (int b = e0; b < e1; b += G) {  // as often for the G lanes of a particle
    double v[NS];
    for (int c = 0; c < NS; c++) v[c] = 0.0;
    if (on) {
      const int rec = ent >> 1, side = ent & 1;
      const size_t at = 9 * (size_t)(rec < ncand ? rec : rec - ncand);
      const double* q = (rec < ncand ? cout : bout) + at;
      const double* qm = q + 3 + 3 * side;
      const double sg = side ? -1.0 : 1.0;  // the second particle's force is the opposite
      v[0] = sg * q[0]; v[1] = sg * q[1]; v[2] = sg * q[2];
      v[3] = qm[0]; v[4] = qm[1]; v[5] = qm[2];
      if (TAN) {
        const double* u = (rec < ncand ? ct : bt) + at;
        const double* um = u + 3 + 3 * side;
        v[6] = sg * u[0]; v[7] = sg * u[1]; v[8] = sg * u[2];
        v[9] = um[0]; v[10] = um[1]; v[11] = um[2];
      }
    }
    ent = nxt;
    on = active(ent);
    nxt = entry(b + 2 * G + sub);
    add_in_order<G>(acc, v);
  }
  __syncthreads();  // the walls' forces have been read
  if (sub == 0)
    for (int c = 0; c < NS; c++) sum[NS * (t / G) + c] = acc[c];
  __syncthreads();
  if (!own) return;
  for (int c = 0; c < NS; c++) acc[c] = sum[NS * t + c];
  const dv3 F = mk3(acc[0], acc[1], acc[2]), M = mk3(acc[3], acc[4], acc[5]);
  // CRotParticle::integrate + rescale, CParticle::integrate (RotParticle.cpp:
  // 277-321, Particle.cpp:257-274), the expression order of the plain engine
  const double dt = sp.dt;
  dv3 v = mk3(Vv.x, Vv.y, Vv.z), x = mk3(P.x, P.y, P.z);
  dv3 w = mk3(A.x, A.y, A.z);
  dquat qq = dquat{Q.x, mk3(Q.y, Q.z, Q.w)};
  w = add3(w, mul3(M, dt * A.w));
  const dquat dq = qmul4(dquat{0, w}, qq);
  const double h = dt / 2.0;
  qq.s += h * dq.s;
  qq.v = add3(qq.v, mul3(dq.v, h));
  v = add3(v, mul3(mul3(F, Vv.w), dt));
  x = add3(x, mul3(v, dt));
  const double module = sqrt(qq.s * qq.s + qq.v.x * qq.v.x + qq.v.y * qq.v.y + qq.v.z * qq.v.z);
  if (module != 0.0) {
    const double inverse = 1.0 / module;
    qq.s = inverse * qq.s;
    qq.v = mul3(qq.v, inverse);
  }
  if (TAN) {
    const dv3 tF = mk3(acc[6], acc[7], acc[8]), tM = mk3(acc[9], acc[10], acc[11]);
    // tangents of w1 = w + M dt/I, qt = q + h (0, w1) q, q1 = qt/|qt|,
    // v1 = v + F dt/m, x1 = x + v1 dt (q0, w: the state before the step)
    const double4 Tx = T.x[i], Tv = T.v[i], Tw = T.w[i], Tq = T.q[i];
    const dquat q0 = dquat{Q.x, mk3(Q.y, Q.z, Q.w)}, tq0 = dquat{Tq.x, mk3(Tq.y, Tq.z, Tq.w)};
    const dv3 tw1 = add3(mk3(Tw.x, Tw.y, Tw.z), mul3(tM, dt * A.w));
    const dquat a1 = qmul4(dquat{0, tw1}, q0), a2 = qmul4(dquat{0, w}, tq0);
    const dquat tqt = dquat{tq0.s + h * (a1.s + a2.s), add3(tq0.v, mul3(add3(a1.v, a2.v), h))};
    dquat tq1 = tqt;
    if (module != 0.0) {
      const double pr = qq.s * tqt.s + dot3(qq.v, tqt.v);
      tq1 = dquat{(tqt.s - qq.s * pr) / module, div3(sub3(tqt.v, mul3(qq.v, pr)), module)};
    }
    const dv3 tv1 = add3(mk3(Tv.x, Tv.y, Tv.z), mul3(mul3(tF, Vv.w), dt));
    const dv3 tx1 = add3(mk3(Tx.x, Tx.y, Tx.z), mul3(tv1, dt));
    T.x[i] = make_double4(tx1.x, tx1.y, tx1.z, 0.0);
    T.v[i] = make_double4(tv1.x, tv1.y, tv1.z, 0.0);
    T.w[i] = make_double4(tw1.x, tw1.y, tw1.z, 0.0);
    T.q[i] = make_double4(tq1.s, tq1.v.x, tq1.v.y, tq1.v.z);
  }
  So.x[i] = make_double4(x.x, x.y, x.z, P.w);
  So.v[i] = make_double4(v.x, v.y, v.z, Vv.w);
  So.w[i] = make_double4(w.x, w.y, w.z, A.w);
  So.q[i] = make_double4(qq.s, qq.v.x, qq.v.y, qq.v.z);
  const dv3 d = sub3(x, mk3(Om.x, Om.y, Om.z));
  const unsigned long long m = (unsigned long long)__double_as_longlong(dot3(d, d));
  if (m > thresh) atomicMax(&run->halt, step);  // a neighbour search before the next step
}

// per specimen: fixed-order sum of its particles' measured wall forces
__global__ __launch_bounds__(256) void k_spec_sum(const DRun* run, int step, const double* val,
                                                  const int* spec_start, double* out)
{
  __shared__ double red[4];
  if (run_skip(run, step)) return;
  const int s = blockIdx.x;
  const int a = spec_start[s], b = spec_start[s + 1];
  double acc = 0.0;
  // eight loads in flight a thread (20,000 particles: 20 us with one)
  for (int i = a + (int)threadIdx.x; i < b; i += 256 * 8) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = i + 256 * k < b ? val[i + 256 * k] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) acc = acc + v[k];
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[s] = ((red[0] + red[1]) + red[2]) + red[3];
}

// ---------------------------------------------------------------------------
// neighbour lists of an epoch
// ---------------------------------------------------------------------------
__device__ __forceinline__ int dbsearch(const long long* a, int n, long long key)
{
  int lo = 0, hi = n - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const long long v = a[mid];
    if (v == key) return mid;
    if (v < key) lo = mid + 1;
    else hi = mid - 1;
  }
  return -1;
}

// candidate pairs -> pair slots, their bond and the pair of the previous epoch
// with the same key (whose shear history it takes over)
__global__ void k_epoch_pairs(int nc, const int* cp, const int* cq, const long long* ckey,
                              const long long* bkey, int nb, const long long* pkey, int np,
                              int2* ij, int* bond, int* src)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  ij[c] = make_int2(cp[c], cq[c]);
  bond[c] = dbsearch(bkey, nb, ckey[c]);
  src[c] = pkey ? dbsearch(pkey, np, ckey[c]) : -1;
}

__global__ void k_carry_hist(int nc, const int* src, const double4* hold, double4* hnew)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const int s = src[c];
  hnew[c] = s >= 0 ? hold[s] : make_double4(0.0, 0.0, 0.0, 0.0);
}

__global__ void k_inc_count2(int nrec, const int2* ij, int* cnt)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nrec) return;
  const int2 e = ij[c];
  atomicAdd(&cnt[e.x], 1);
  atomicAdd(&cnt[e.y], 1);
}

__global__ void k_inc_fill2(int nrec, int rec0, const int2* ij, const int* off, int* fill, int* ent)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nrec) return;
  const int2 e = ij[c];
  const int rec = rec0 + c;
  ent[off[e.x] + atomicAdd(&fill[e.x], 1)] = rec << 1;
  ent[off[e.y] + atomicAdd(&fill[e.y], 1)] = (rec << 1) | 1;
}

// each particle's run in ascending entry order: pairs by key, then bonds
__global__ void k_inc_sort2(int n, const int* off, int* ent)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int a = off[i], b = off[i + 1];
  for (int s = a + 1; s < b; s++) {
    const int v = ent[s];
    int j = s - 1;
    while (j >= a && ent[j] > v) {
      ent[j + 1] = ent[j];
      j--;
    }
    ent[j + 1] = v;
  }
}


// ---------------------------------------------------------------------------
// adjoint kernels
// ---------------------------------------------------------------------------
// The adjoint of one particle's update in the step whose state before is Sn and
// after Sn1: L holds the adjoint of the state after the step (x, v, w, q) on
// entry and the partial adjoint of the state before it on exit; o: (lambda_F,
// lambda_M) for the interaction adjoints.  cf: d loss / d stress / area of the
// particle's specimen at a sample step (else 0).
__device__ __forceinline__ void adj_particle_item(const DState& Sn, const DState& Sn1, int i,
                                                  double4 (&L)[4], double* o, const DStep& sp,
                                                  double cf)
{
  const double4 Lx = L[0], Lv1 = L[1], Lw1 = L[2], Lq1 = L[3];
  const double dt = sp.dt, h = dt / 2.0;
  const double4 Vv = Sn.v[i], A = Sn.w[i], Q = Sn.q[i];
  const double4 A1 = Sn1.w[i], Q1 = Sn1.q[i];
  // x' = x + v' dt, v' = v + F invm dt
  const dv3 lv1 = add3(mk3(Lv1.x, Lv1.y, Lv1.z), mul3(mk3(Lx.x, Lx.y, Lx.z), dt));
  const dv3 lF = mul3(lv1, Vv.w * dt);
  dv3 lx = mk3(Lx.x, Lx.y, Lx.z);
  // q' = qt / |qt|, qt = q + h (0, w') q, w' = w + M invI dt
  const dv3 w1 = mk3(A1.x, A1.y, A1.z);
  const dquat q = dquat{Q.x, mk3(Q.y, Q.z, Q.w)};
  const dquat dq = qmul4(dquat{0, w1}, q);
  const dquat qt = dquat{q.s + h * dq.s, add3(q.v, mul3(dq.v, h))};
  const double mod = sqrt(qt.s * qt.s + qt.v.x * qt.v.x + qt.v.y * qt.v.y + qt.v.z * qt.v.z);
  const dquat qn = dquat{Q1.x, mk3(Q1.y, Q1.z, Q1.w)};
  const double pr = qn.s * Lq1.x + qn.v.x * Lq1.y + qn.v.y * Lq1.z + qn.v.z * Lq1.w;
  const dquat lqt = dquat{(Lq1.x - qn.s * pr) / mod,
                          div3(sub3(mk3(Lq1.y, Lq1.z, Lq1.w), mul3(qn.v, pr)), mod)};
  // d(dq)/dq^T lqt = (w1 . lqt.v, -w1 lqt.s - w1 x lqt.v)
  const dquat lq = dquat{lqt.s + h * dot3(w1, lqt.v),
                         add3(lqt.v, mul3(sub3(mul3(w1, -lqt.s), cross3(w1, lqt.v)), h))};
  // d(dq)/dw1^T lqt = -q.v lqt.s + q.s lqt.v + q.v x lqt.v
  const dv3 lw1 = add3(mk3(Lw1.x, Lw1.y, Lw1.z),
                       mul3(add3(add3(mul3(q.v, -lqt.s), mul3(lqt.v, q.s)), cross3(q.v, lqt.v)), h));
  const dv3 lM = mul3(lw1, dt * A.w);
  // walls: f = n k' (r - (x - o).n) while touching; the measured wall's normal
  // force also enters the stress
  const double4 P = Sn.x[i];
  const double r = P.w;
  for (int k = 0; k < sp.nw; k++) {
    const DWall& W = sp.wall[k];
    const dv3 n = mk3(W.n[0], W.n[1], W.n[2]);
    const double dist = dot3(sub3(mk3(P.x, P.y, P.z), mk3(W.o[0], W.o[1], W.o[2])), n);
    if (dist < r) {
      const double kk = (3.141592654 * r) * W.k;
      // d f / d x = -kk n n^T;  d (f . n) / d x = -kk n
      double s = dot3(n, lF);
      if (W.measure) s += cf;
      lx = sub3(lx, mul3(n, kk * s));
    }
  }
  L[0] = make_double4(lx.x, lx.y, lx.z, 0.0);
  L[1] = make_double4(lv1.x, lv1.y, lv1.z, 0.0);
  L[2] = make_double4(lw1.x, lw1.y, lw1.z, 0.0);
  L[3] = make_double4(lq.s, lq.v.x, lq.v.y, lq.v.z);
  o[0] = lF.x; o[1] = lF.y; o[2] = lF.z;
  o[3] = lM.x; o[4] = lM.y; o[5] = lM.z;
}

// Interaction adjoints, 32-byte vectors that one lane of k_adj_step loads whole:
// of a bond (x1, kn), (x2, ks), q1, q2 (its particles are of one specimen); of a
// pair (x1, kn), (x2, 0), (v1, mu), (v2, 0), (w1, ks), (w2, 0): the parameters, in
// the fourth component, are credited to the first particle's specimen.
#define NB_REC 4
#define NF_REC 6

// bond law VJP, one thread per bond, by the law's hand-written reverse mode
// (tbond_law_vjp) on the branch the forward step took: about 2,300 FP64
// instructions, 66 divisions among them, so a wave alone on its SIMD leaves the
// memory phases of its gathers and stores uncovered.  The law takes its two halves
// one after the other and parks what is used only at the ends in LDS: 223 VGPRs
// instead of 326, two waves a SIMD, 478,000 bonds 79.2 -> 52.9 us a step (2,000
// particles 9.8, one wave's time either way).
#define ADJ_BOND_BS 256
__global__ __launch_bounds__(ADJ_BOND_BS, 2) void k_adj_bond(DState S, DBonds B,
                                                           const double4* theta, int step,
                                                           const double* lfm, double4* ab)
{
  // volatile: the compiler would keep the values in registers instead
  typedef __attribute__((address_space(3))) volatile double* lds_park;
  __shared__ double park[BOND_VJP_PARK * ADJ_BOND_BS];
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B.nb) return;
  // broken earlier: the record is the zero the sweep, which goes back in time,
  // started with
  if (B.bstep[b] < step) return;
  double4* c = ab + NB_REC * (size_t)b;
  const int2 e = B.ij[b];
  const double4 P1 = S.x[e.x], P2 = S.x[e.y], Q1 = S.q[e.x], Q2 = S.q[e.y];
  const double4 D = B.D0[b];
  const int s = S.spec[e.x];
  const double4 th = theta[s];
  const double2 tk = B.tkb[s];
  const double* l1 = lfm + 6 * (size_t)e.x;
  const double* l2 = lfm + 6 * (size_t)e.y;
  double kr, ks, kt, kb, dkr, dks, dkt, dkb;
  tbond_k<double>(th.x, th.y, tk.x, tk.y, D.w, P1.w, P2.w, 1, 1, 0, kr, ks, kt, kb);
  // d kr / d theta_kn, d ks / d theta_ks (the constants are linear in them)
  tbond_k<double>(1.0, 1.0, tk.x, tk.y, D.w, P1.w, P2.w, 1, 1, 0, dkr, dks, dkt, dkb);
  tv3<double> g1, g2;
  tquat<double> gq1, gq2;
  double gkr, gks;
  // f2 = -f1: particle 2's force adjoint enters with the opposite sign
  tbond_law_vjp(dx3(P1), tquat<double>{Q1.x, {Q1.y, Q1.z, Q1.w}}, P1.w, dx3(P2),
                tquat<double>{Q2.x, {Q2.y, Q2.z, Q2.w}}, P2.w, kr, ks, kt, kb,
                tv3<double>{D.x, D.y, D.z}, tv3<double>{l1[0] - l2[0], l1[1] - l2[1], l1[2] - l2[2]},
                tv3<double>{l1[3], l1[4], l1[5]}, tv3<double>{l2[3], l2[4], l2[5]}, g1, g2, gq1, gq2,
                gkr, gks, (lds_park)(park + threadIdx.x), ADJ_BOND_BS);
  c[0] = make_double4(g1.x, g1.y, g1.z, gkr * dkr);
  c[1] = make_double4(g2.x, g2.y, g2.z, gks * dks);
  c[2] = make_double4(gq1.s, gq1.v.x, gq1.v.y, gq1.v.z);
  c[3] = make_double4(gq2.s, gq2.v.x, gq2.v.y, gq2.v.z);
}

// friction law VJP over the inputs (x1, x2, v1, v2, w1, w2, history,
// theta_kn, theta_ks, theta_mu), one thread per pair, by the law's hand-written
// reverse mode (tfriction_law_vjp) on the slip branch the forward step took;
// lh: adjoint of the history this step wrote; lh_prev: adjoint of the history
// it read
// act[c]: the record of pair c holds a (nonzero) Jacobian this step; the
// gather reads only such records.
__global__ void k_adj_fric(DState S, DCands C, const int* bstep, const double4* theta,
                           const double4* hin, int step, double dt, const double* lfm,
                           const double4* lh, double4* ac, unsigned char* act, double4* lh_prev)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C.nc) return;
  const int bb = C.bond[c];
  if (bb >= 0 && bstep[bb] >= step) {
    // excluded while bonded: zero Jacobian.  The history adjoint it would pass
    // back is not written: the pair was excluded in the step before too (a
    // bond that lives now lived then), so no step reads it.
    act[c] = 0;
    return;
  }
  const int2 e = C.ij[c];
  const double4 P1 = S.x[e.x], P2 = S.x[e.y];
  // apart (no force, history cleared): zero Jacobian
  const double dxx = P1.x - P2.x, dyy = P1.y - P2.y, dzz = P1.z - P2.z;
  const double eq = P1.w + P2.w;
  if (!((dxx * dxx + dyy * dyy + dzz * dzz) < eq * eq)) {
    act[c] = 0;
    lh_prev[c] = make_double4(0.0, 0.0, 0.0, 0.0);
    return;
  }
  act[c] = 1;
  const double4 V1 = S.v[e.x], V2 = S.v[e.y], W1 = S.w[e.x], W2 = S.w[e.y];
  const double4 th = theta[S.spec[e.x]];
  const double4 hh = hin[c];
  const double4 lo = lh[c];
  const double* l1 = lfm + 6 * (size_t)e.x;
  const double* l2 = lfm + 6 * (size_t)e.y;
  double kk, kks, dk, dks;
  tfriction_k<double>(th.x, th.y, 1, 1, P1.w, P2.w, 0, kk, kks);
  // d k / d theta_kn, d ks / d theta_ks (linear in them)
  tfriction_k<double>(1.0, 1.0, 1, 1, P1.w, P2.w, 0, dk, dks);
  tv3<double> g[8];
  // f2 = -f1: particle 2's force adjoint enters with the opposite sign
  tfriction_law_vjp(dx3(P1), dx3(V1), dx3(W1), P1.w, dx3(P2), dx3(V2), dx3(W2), P2.w, kk, kks, th.w,
                    dt, tv3<double>{hh.x, hh.y, hh.z}, (((int)hh.w) & 1) != 0,
                    tv3<double>{l1[0] - l2[0], l1[1] - l2[1], l1[2] - l2[2]},
                    tv3<double>{l1[3], l1[4], l1[5]}, tv3<double>{l2[3], l2[4], l2[5]},
                    tv3<double>{lo.x, lo.y, lo.z}, g);
  double4* o = ac + NF_REC * (size_t)c;
  const double par[6] = {g[7].x * dk, 0.0, g[7].z, 0.0, g[7].y * dks, 0.0};
  for (int t = 0; t < 6; t++) o[t] = make_double4(g[t].x, g[t].y, g[t].z, par[t]);
  lh_prev[c] = make_double4(g[6].x, g[6].y, g[6].z, 0.0);
}

// Per particle: the interactions' adjoints of step `step` are added to the state
// adjoint lam in CSR order (GATHER; parameter gradients of the interactions whose
// first particle this is go to gth: kn, ks, -, mu), then the particle's own update
// in the step before, sp.step, is taken back (PART: states Sn, Sn1, adjoints for
// its interactions to lfm).  One launch between two steps' laws instead of two,
// and lam passes through memory once.
// The lanes of a quad take one of lam's vectors each (x, v, w, q) and load the
// entry's record for that vector; the next entries' activity and the entries after
// those are under way meanwhile.  G: one quad a particle, or four that take the
// entries in turn and add them in entry order.  Records of pairs without a Jacobian
// this step (apart or excluded) are skipped; those of bonds broken earlier are
// zeros.  Two launches of one lane a particle, 13 components an entry -> this (us a
// step): 2,000 particles 25.4 -> 8.2, 20,000 30.8 -> 13.2, 254,000 83.8 -> 72.6.
template <bool GATHER, bool PART, int G>
__global__ __launch_bounds__(DIFF_MAX_BS) void k_adj_step(
    int n, const int* inc_off, const int* inc_ent, int ncand, const double4* ac, const double4* ab,
    const unsigned char* cact, double4* lam, double4* gth, DState Sn, DState Sn1, double* lfm,
    DStep sp, const double* coef)
{
  constexpr int NQ = G / 4;         // quads a particle
  constexpr int R = G == 4 ? 4 : 2;  // entries a quad has in flight
  __shared__ double4 sl[PART ? DIFF_MAX_BS / NQ : 1];
  const int t = threadIdx.x;
  const int PB = blockDim.x / G;
  const int p0 = blockIdx.x * PB;
  const int pi = p0 + t / G, sub = t % 4, quad = (t % G) / 4;
  const int pc = pi < n ? pi : 0;
  double4 L = lam[4 * (size_t)pc + sub];
  if (GATHER) {
    const int e0 = inc_off[pc], e1 = pi < n ? inc_off[pc + 1] : e0;
    // the vector's adjoint; parameters: in the lanes of x, v, w kn, mu, the pairs'
    // ks; the bonds' ks (in the first quad of a particle)
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto entry = [&](int at) { return at < e1 ? inc_ent[at] : -1; };
    auto active = [&](int ent) {
      return ent >= 0 && ((ent >> 1) >= ncand || cact[ent >> 1] != 0);
    };
    int ent[R], nxt[R];
    bool on[R];
#pragma unroll
    for (int r = 0; r < R; r++) ent[r] = entry(e0 + r * NQ + quad);
#pragma unroll
    for (int r = 0; r < R; r++) nxt[r] = entry(e0 + (R + r) * NQ + quad);
#pragma unroll
    for (int r = 0; r < R; r++) on[r] = active(ent[r]);
    for (int b = e0; b < e1; b += R * NQ) {
      double4 a[R];
      int side[R];
#pragma unroll
      for (int r = 0; r < R; r++) {
        a[r] = make_double4(0.0, 0.0, 0.0, 0.0);
        const int rec = ent[r] >> 1;
        side[r] = ent[r] & 1;
        if (!on[r]) continue;
        if (rec < ncand) {
          if (sub < 3) a[r] = ac[NF_REC * (size_t)rec + 2 * sub + side[r]];
        } else if (sub == 0 || sub == 3) {
          a[r] = ab[NB_REC * (size_t)(rec - ncand) + (sub ? 2 : 0) + side[r]];
        }
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        ent[r] = nxt[r];
        on[r] = active(ent[r]);
      }
#pragma unroll
      for (int r = 0; r < R; r++) nxt[r] = entry(b + (2 * R + r) * NQ + quad);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const bool p = sub != 3, s2 = side[r] != 0;
        const double v[6] = {a[r].x, a[r].y, a[r].z, p ? 0.0 : a[r].w, p && !s2 ? a[r].w : 0.0,
                             p && s2 ? a[r].w : 0.0};
        add_quads<NQ>(acc, v);
      }
    }
    L.x += acc[0];
    L.y += acc[1];
    L.z += acc[2];
    L.w += acc[3];
    const double g0 = acc[4], g1 = acc[5];
    const double gmu = group_value<4>(g0, 1), gks = group_value<4>(g0, 2);
    if (t % G == 0 && pi < n) {
      double4 g = gth[pi];
      g.x += g0;
      g.y += g1 + gks;
      g.w += gmu;
      gth[pi] = g;
    }
  }
  if (!PART) {
    if (quad == 0 && pi < n) lam[4 * (size_t)pi + sub] = L;
    return;
  }
  if (quad == 0) sl[4 * (t / G) + sub] = L;
  __syncthreads();
  const int i = p0 + t;
  if (t < PB && i < n) {
    double4 l4[4] = {sl[4 * t], sl[4 * t + 1], sl[4 * t + 2], sl[4 * t + 3]};
    adj_particle_item(Sn, Sn1, i, l4, lfm + 6 * (size_t)i, sp, coef ? coef[Sn.spec[i]] : 0.0);
    for (int k = 0; k < 4; k++) sl[4 * t + k] = l4[k];
  }
  __syncthreads();
  if (quad == 0 && pi < n) lam[4 * (size_t)pi + sub] = sl[4 * (t / G) + sub];
}

// adjoint of the history read at the first step of an epoch, to the pairs of
// the previous epoch it was taken from
__global__ void k_map_lh(int nc, const int* src, const double4* lnew, double4* lold)
{
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const int s = src[c];
  if (s >= 0) lold[s] = lnew[c];
}

__global__ __launch_bounds__(256) void k_spec_sum4(const double4* val, const int* spec_start, double4* out)
{
  __shared__ double4 red[4];
  const int s = blockIdx.x;
  const int a = spec_start[s], b = spec_start[s + 1];
  double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
  for (int i = a + (int)threadIdx.x; i < b; i += 256) {
    const double4 v = val[i];
    acc.x = acc.x + v.x; acc.y = acc.y + v.y; acc.z = acc.z + v.z; acc.w = acc.w + v.w;
  }
  acc = make_double4(wave_sum(acc.x), wave_sum(acc.y), wave_sum(acc.z), wave_sum(acc.w));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double4 t = red[0];
    for (int k = 1; k < 4; k++) {
      t.x = t.x + red[k].x; t.y = t.y + red[k].y; t.z = t.z + red[k].z; t.w = t.w + red[k].w;
    }
    out[s] = t;
  }
}

inline int nblocks(long long n, int bs) { return (int)std::max<long long>(1, (n + bs - 1) / bs); }

// one neighbour-table epoch: the pairs found at a rebuild and the CSR of every
// particle's interactions (pairs, then bonds)
struct Epoch {
  int start = 0;  // first step it serves
  int nc = 0;
  DevBuf<int2> ij;
  DevBuf<long long> key;
  DevBuf<int> bond, src;
  DevBuf<int> inc_off, inc_ent;
};

struct Checkpoint {
  int step = 0;
  int epoch = 0;
  DevBuf<double4> x, v, w, q, hist;
};

}  // namespace

struct esp_diff {
  esp_diff_config cfg;
  GridParams grid;
  int ncell = 0;
  hipStream_t stream = nullptr;
  int bs = 256;
  std::string err;
  // particles
  int n = 0, nspec = 0;
  std::vector<int> h_spec, h_spec_start;
  std::vector<double> h_pos, h_rad, h_mass, h_vel;
  DevBuf<double4> x, v, w, q, o;
  DevBuf<int> spec, spec_start, id;
  DevBuf<unsigned> flags;
  // bonds (sorted by key)
  int nb = 0;
  std::vector<int> h_bi, h_bj;
  std::vector<double> h_rel, h_tk, h_bk;
  DevBuf<int2> bij;
  DevBuf<long long> bkey;
  DevBuf<double4> bD0, brel;
  DevBuf<int> bstep;
  DevBuf<double2> tkb;
  // walls, gravity, run
  int nw = 0;
  DWall wall0[DIFF_MAX_WALLS];
  double wstep[DIFF_MAX_WALLS][3];
  std::vector<double> h_area;
  DevBuf<double> area;
  int has_g = 0;
  double g[3] = {0, 0, 0};
  int nsteps = 0, every = 1;
  // run state
  std::vector<std::unique_ptr<Epoch>> epochs;
  std::vector<std::unique_ptr<Checkpoint>> ckpts;
  std::vector<int> rebuild_steps;
  DevBuf<double4> H[2];  // shear histories: step s reads H[s & 1], writes the other
  DevBuf<DRun> run;
  std::vector<double> wo;  // wall origins per step of the run [step][wall][3]
  int run_nw = 0;          // its walls
  int run_has_g = 0;       // its gravity
  double run_g[3] = {0, 0, 0};
  // The states of the last forward run, step by step ([step][x, v, w, q][n]), and
  // the histories touching pairs read in each: kept by runs whose tape fits
  // tape_limit, so that the adjoint sweeps them without recomputing its segments.
  // Longer runs keep checkpoints, and the sweep one segment's tape at a time.
  bool full_tape = false;
  size_t tape_limit;
  DevBuf<double4> tape;
  std::vector<std::unique_ptr<DevBuf<double4>>> hchunk;  // room the histories are laid out in
  std::vector<double4*> htape;                           // [step]
  // the reverse sweep's arrays
  DevBuf<double4> lam, gth, lh, lh2;
  DevBuf<double> lfm;
  DevBuf<double4> ab, ac;
  DevBuf<unsigned char> aact;  // per pair: its record holds a Jacobian this step
  std::vector<std::unique_ptr<DevBuf<double4>>> hseg;
  DevBuf<double> bout, cout, wfn, stress_dev;
  DevBuf<unsigned char> cact;  // per pair of the epoch: its record holds this step's force
  DevBuf<double4> theta;
  std::vector<double> h_theta, h_target, h_stress;
  DevBuf<unsigned long long> md;
  DevBuf<unsigned long long> digest;  // per step: branch digest of the last forward run
  // branch digests are computed only when asked for (esp_diff_track_branches):
  // every wave of the contact and gather kernels adds to one counter per step
  bool track_digest = false;
  DState fin = {};  // the state the last forward run ended with, or had reached when it failed
  DevBuf<double4> x0, v0, w0, q0;  // the initial state
  // tangent-linear run (forward with a parameter direction)
  bool tan_on = false;
  DevBuf<double4> tx, tv, tw, tq, TH[2], dtheta;
  DevBuf<double> bt, ct, wft, stress_t;
  std::vector<double> h_stress_t;
  DTan tan() { return DTan{tx.p, tv.p, tw.p, tq.p}; }
  DevBuf<int> cell, cell_count, cell_start, cell_fill, cell_items, ccnt, coff, cp, cq, scan_tmp,
      inc_cnt, inc_fill;
  DevBuf<long long> ckey;
  bool have_forward = false;
  double t_fwd = 0, t_bwd = 0;

  DState state()
  {
    return DState{x.p, v.p, w.p, q.p, spec.p, n};
  }
  // a state of a tape laid out as [x][v][w][q]
  DState tape_state(double4* t)
  {
    const size_t c = (size_t)n;
    return DState{t, t + c, t + 2 * c, t + 3 * c, spec.p, n};
  }
  // wall origins of a step: moved by their step before every step (the
  // pre-time-step moveWallBy of the main engine's setWallStepMotion)
  DStep step_params(int step)
  {
    DStep s;
    memset(&s, 0, sizeof s);
    s.nw = run_nw;
    for (int k = 0; k < run_nw; k++) {
      s.wall[k] = wall0[k];
      for (int c = 0; c < 3; c++) s.wall[k].o[c] = wo[((size_t)step * run_nw + k) * 3 + c];
    }
    s.has_g = run_has_g;
    for (int c = 0; c < 3; c++) s.g[c] = run_g[c];
    s.dt = cfg.dt;
    s.step = step;
    return s;
  }
};

namespace {

// a run's tape (states and histories of every step) is kept up to this size unless
// the caller sets another
// (24 specimens of 2,000 to 30,000 particles take 70 MB a step); recomputing the
// segments and copying their states cost a third of a forward and backward pass
// (2,000 particles, 100 steps: 12.7 -> 5.8 ms with the launches below)
constexpr size_t kTapeLimit = (size_t)24 << 30;
// A row of 16 lanes a particle up to this many particles, a quad above (the sums
// are the same, bit by bit): the longest run of interactions sets the time while
// the chip is not full.  Quad / row, us a step: forward gather 2,000 particles
// 9.7 / 6.9, 20,000 11.1 / 12.1, 50,000 12.2 / 15.9; adjoint 2,000 14.5 / 8.2,
// 20,000 17.0 / 13.2, 254,000 72.6 / 108.2.
constexpr int kGatherRow = 8192, kAdjointRow = 32768;

void dsync(esp_diff* d) { DCHK(hipStreamSynchronize(d->stream)); }

int dscan(esp_diff* d, const int* in, int* out, int cnt)
{
  d->scan_tmp.reserve(scan_tmp_size(cnt));
  launch_exclusive_scan(d->stream, in, out, cnt, d->scan_tmp.p);
  DCHK(hipGetLastError());
  int total = 0;
  DCHK(hipMemcpyAsync(&total, out + cnt, sizeof(int), hipMemcpyDeviceToHost, d->stream));
  dsync(d);
  return total;
}

// neighbour search (NeighborTable::build + getFullList) -> a new epoch
void rebuild(esp_diff* d, const DState& S, int step)
{
  const int n = d->n;
  PView pv;
  memset(&pv, 0, sizeof pv);
  pv.pos = S.x; pv.vel = S.v; pv.ang = S.w; pv.quat = S.q; pv.old = d->o.p;
  pv.flags = d->flags.p; pv.id = d->id.p; pv.n = n;
  DCHK(hipMemsetAsync(d->cell_count.p, 0, sizeof(int) * (d->ncell + 1), d->stream));
  DCHK(hipMemsetAsync(d->md.p, 0, sizeof(unsigned long long) * 2, d->stream));
  int* nout = reinterpret_cast<int*>(d->md.p + 1);
  launch_cells_count(d->stream, pv, d->grid, d->cell.p, d->cell_count.p, nout);
  int hout = 0;
  DCHK(hipMemcpyAsync(&hout, nout, sizeof(int), hipMemcpyDeviceToHost, d->stream));
  dsync(d);
  if (hout > 0)
    throw DiffError(ESP_ERR_STATE, "particles left the neighbour-table domain (the differentiable "
                                   "engine keeps every particle)");
  dscan(d, d->cell_count.p, d->cell_start.p, d->ncell);
  DCHK(hipMemsetAsync(d->cell_fill.p, 0, sizeof(int) * d->ncell, d->stream));
  launch_cells_fill(d->stream, n, d->cell.p, d->cell_start.p, d->cell_fill.p, d->cell_items.p);
  launch_cells_sort(d->stream, d->ncell, d->cell_start.p, d->cell_items.p);
  launch_pairs(d->stream, 0, 0, pv, d->grid, d->cfg.verlet_dist, d->cell.p, d->cell_start.p,
               d->cell_items.p, d->ccnt.p, nullptr, 0, nullptr, nullptr, nullptr);
  const int nc = dscan(d, d->ccnt.p, d->coff.p, n);
  d->cp.reserve(std::max(nc, 1));
  d->cq.reserve(std::max(nc, 1));
  d->ckey.reserve(std::max(nc, 1));
  launch_pairs(d->stream, 1, 0, pv, d->grid, d->cfg.verlet_dist, d->cell.p, d->cell_start.p,
               d->cell_items.p, nullptr, d->coff.p, nc, d->cp.p, d->cq.p, d->ckey.p);
  DCHK(hipGetLastError());
  auto E = std::make_unique<Epoch>();
  E->start = step;
  E->nc = nc;
  const size_t c1 = std::max(nc, 1);
  E->ij.reserve(c1);
  E->key.reserve(c1);
  E->bond.reserve(c1);
  E->src.reserve(c1);
  DCHK(hipMemcpyAsync(E->key.p, d->ckey.p, sizeof(long long) * nc, hipMemcpyDeviceToDevice,
                      d->stream));
  const Epoch* P = d->epochs.empty() ? nullptr : d->epochs.back().get();
  const int bs = d->bs;
  if (nc > 0)
    hipLaunchKernelGGL(k_epoch_pairs, dim3(nblocks(nc, bs)), dim3(bs), 0, d->stream, nc, d->cp.p,
                       d->cq.p, d->ckey.p, d->bkey.p, d->nb, P ? P->key.p : nullptr, P ? P->nc : 0,
                       E->ij.p, E->bond.p, E->src.p);
  // CSR: pairs (records 0..nc-1), then bonds (nc..nc+nb-1)
  d->inc_cnt.reserve(n + 1);
  d->inc_fill.reserve(n + 1);
  DCHK(hipMemsetAsync(d->inc_cnt.p, 0, sizeof(int) * (n + 1), d->stream));
  if (nc > 0)
    hipLaunchKernelGGL(k_inc_count2, dim3(nblocks(nc, bs)), dim3(bs), 0, d->stream, nc, E->ij.p,
                       d->inc_cnt.p);
  if (d->nb > 0)
    hipLaunchKernelGGL(k_inc_count2, dim3(nblocks(d->nb, bs)), dim3(bs), 0, d->stream, d->nb,
                       d->bij.p, d->inc_cnt.p);
  E->inc_off.reserve(n + 1);
  const int tot = dscan(d, d->inc_cnt.p, E->inc_off.p, n);
  E->inc_ent.reserve(std::max(tot, 1));
  DCHK(hipMemsetAsync(d->inc_fill.p, 0, sizeof(int) * (n + 1), d->stream));
  if (nc > 0)
    hipLaunchKernelGGL(k_inc_fill2, dim3(nblocks(nc, bs)), dim3(bs), 0, d->stream, nc, 0, E->ij.p,
                       E->inc_off.p, d->inc_fill.p, E->inc_ent.p);
  if (d->nb > 0)
    hipLaunchKernelGGL(k_inc_fill2, dim3(nblocks(d->nb, bs)), dim3(bs), 0, d->stream, d->nb, nc,
                       d->bij.p, E->inc_off.p, d->inc_fill.p, E->inc_ent.p);
  hipLaunchKernelGGL(k_inc_sort2, dim3(nblocks(n, bs)), dim3(bs), 0, d->stream, n, E->inc_off.p,
                     E->inc_ent.p);
  // shear histories carried by key (PIS_ED::update: persistent pairs keep theirs;
  // a pair that is not is apart and holds zero anyway)
  // (the step reads buffer step & 1)
  const int cur = step & 1;
  DevBuf<double4> hn;
  hn.reserve(c1);
  if (nc > 0) {
    hipLaunchKernelGGL(k_carry_hist, dim3(nblocks(nc, bs)), dim3(bs), 0, d->stream, nc, E->src.p,
                       P ? d->H[cur].p : nullptr, hn.p);
    if (!P) DCHK(hipMemsetAsync(hn.p, 0, sizeof(double4) * nc, d->stream));
  }
  DevBuf<double4> tn;
  if (d->tan_on) {
    tn.reserve(c1);
    if (nc > 0) {
      hipLaunchKernelGGL(k_carry_hist, dim3(nblocks(nc, bs)), dim3(bs), 0, d->stream, nc, E->src.p,
                         P ? d->TH[cur].p : nullptr, tn.p);
      if (!P) DCHK(hipMemsetAsync(tn.p, 0, sizeof(double4) * nc, d->stream));
    }
    d->ct.reserve(c1 * 9);
  }
  DCHK(hipGetLastError());
  dsync(d);
  d->H[cur].swap(hn);
  d->H[cur ^ 1].reserve(c1);
  // both buffers equal: a pair flagged "zero in both buffers" writes neither
  if (nc > 0)
    DCHK(hipMemcpyAsync(d->H[cur ^ 1].p, d->H[cur].p, sizeof(double4) * nc,
                        hipMemcpyDeviceToDevice, d->stream));
  if (d->tan_on) {
    d->TH[cur].swap(tn);
    d->TH[cur ^ 1].reserve(c1);
  }
  d->epochs.push_back(std::move(E));
  d->rebuild_steps.push_back(step);
  d->bout.reserve((size_t)std::max(d->nb, 1) * 9);
  d->cout.reserve(c1 * 9);
  d->cact.reserve(c1);
  if (d->tan_on) d->bt.reserve((size_t)std::max(d->nb, 1) * 9);
}

template <class T>
void d2d(esp_diff* d, T* dst, const T* src, size_t cnt)
{
  if (cnt) DCHK(hipMemcpyAsync(dst, src, cnt * sizeof(T), hipMemcpyDeviceToDevice, d->stream));
}

void save_checkpoint(esp_diff* d, int step, const DState& S)
{
  auto C = std::make_unique<Checkpoint>();
  C->step = step;
  C->epoch = (int)d->epochs.size() - 1;
  const size_t n = std::max(d->n, 1);
  C->x.reserve(n); C->v.reserve(n); C->w.reserve(n); C->q.reserve(n);
  d2d(d, C->x.p, S.x, d->n); d2d(d, C->v.p, S.v, d->n); d2d(d, C->w.p, S.w, d->n);
  d2d(d, C->q.p, S.q, d->n);
  const int nc = d->epochs.back()->nc;
  C->hist.reserve(std::max(nc, 1));
  d2d(d, C->hist.p, d->H[step & 1].p, nc);
  d->ckpts.push_back(std::move(C));
}

// a checkpoint's state into the tape at T, its histories into the arrays a segment
// is recomputed with (the run's break steps hold for every step of it: a bond lives
// up to the step it breaks in)
void restore_checkpoint(esp_diff* d, const Checkpoint& C, double4* T)
{
  const DState S = d->tape_state(T);
  d2d(d, S.x, C.x.p, d->n); d2d(d, S.v, C.v.p, d->n); d2d(d, S.w, C.w.p, d->n);
  d2d(d, S.q, C.q.p, d->n);
  const int nc = d->epochs[C.epoch]->nc;
  d->H[0].reserve(std::max(nc, 1));
  d->H[1].reserve(std::max(nc, 1));
  // the history the checkpoint's step reads, in both buffers (a pair flagged
  // "zero in both buffers" writes neither)
  d2d(d, d->H[0].p, C.hist.p, nc);
  d2d(d, d->H[1].p, C.hist.p, nc);
  // bonds broken before the segment have zero records; what a sweep before this
  // one left is of other steps
  if (d->nb > 0) DCHK(hipMemsetAsync(d->bout.p, 0, sizeof(double) * 9 * (size_t)d->nb, d->stream));
}

// The launches of one forward step (no search) from S into So: tangents (tangent
// runs), the force laws, the update.  htape: where touching pairs leave the
// histories they read, or nullptr; record: branch digests and samples (forward
// runs); halting: the displacement test may stop the queue (not while recomputing
// a recorded segment).
void fwd_step(esp_diff* d, const Epoch& E, int step, const DState& S, const DState& So,
              double4* htape, bool record, bool halting)
{
  const int bs = d->bs;
  DBonds B{d->nb, d->bij.p, d->bD0.p, d->brel.p, d->bstep.p, d->tkb.p};
  DCands C{E.nc, E.ij.p, E.bond.p};
  DRun* R = d->run.p;
  const DTan T = d->tan_on ? d->tan() : DTan{nullptr, nullptr, nullptr, nullptr};
  if (d->tan_on) {  // tangents from the state before the step (before the forward kernels)
    if (d->nb > 0)
      hipLaunchKernelGGL(k_bond_tan, dim3(nblocks(d->nb, bs)), dim3(bs), 0, d->stream, S, T, B,
                         d->theta.p, d->dtheta.p, R, step, d->bt.p);
    if (E.nc > 0)
      hipLaunchKernelGGL(k_fric_tan, dim3(nblocks(E.nc, bs)), dim3(bs), 0, d->stream, S, T, C,
                         d->bstep.p, d->theta.p, d->dtheta.p, d->H[0].p, d->H[1].p, d->TH[0].p,
                         d->TH[1].p, R, step, d->cfg.dt, d->ct.p);
  }
  unsigned long long* dig = record && d->track_digest ? d->digest.p : nullptr;
  const int nbb = d->nb > 0 ? nblocks(d->nb, bs) : 0, ncb = E.nc > 0 ? nblocks(E.nc, bs) : 0;
  if (nbb + ncb > 0)
    hipLaunchKernelGGL(k_bond_fwd_pairs, dim3(nbb + ncb), dim3(bs), 0, d->stream, S, B, C, d->theta.p,
                       d->H[0].p, d->H[1].p, htape, R, step, d->cfg.dt, nbb, d->bout.p, d->cout.p,
                       d->cact.p, dig);
  unsigned long long thresh = ~0ull;
  if (halting) {
    const double a = 0.5 * d->cfg.verlet_dist;
    const double sr = a * a;
    memcpy(&thresh, &sr, 8);
  }
  const DStep sp = d->step_params(step);
  if (dig && sp.nw > 0)
    hipLaunchKernelGGL(k_wall_digest, dim3(nblocks(d->n, bs)), dim3(bs), 0, d->stream, S, sp, R, dig);
  const bool sample = record && step % d->every == 0;
  const bool wide = d->n <= kGatherRow;
  const auto gather = d->tan_on ? k_gather_fwd<4, true>
                      : wide    ? k_gather_fwd<16, false>
                                : k_gather_fwd<4, false>;
  hipLaunchKernelGGL(gather,
                     dim3(nblocks((wide && !d->tan_on ? 16ll : 4ll) * d->n, bs)), dim3(bs), 0, d->stream, S, So, d->o.p,
                     E.inc_off.p, E.inc_ent.p, E.nc, d->cout.p, d->bout.p, d->cact.p, sp,
                     sample ? d->wfn.p : nullptr, R, thresh, T, d->ct.p, d->bt.p,
                     sample && d->tan_on ? d->wft.p : nullptr);
  if (sample) {
    const size_t at = (size_t)(step / d->every - 1) * d->nspec;
    hipLaunchKernelGGL(k_spec_sum, dim3(d->nspec), dim3(256), 0, d->stream, R, step, d->wfn.p,
                       d->spec_start.p, d->stress_dev.p + at);
    if (d->tan_on)
      hipLaunchKernelGGL(k_spec_sum, dim3(d->nspec), dim3(256), 0, d->stream, R, step, d->wft.p,
                         d->spec_start.p, d->stress_t.p + at);
  }
  DCHK(hipGetLastError());
}

void clear_run(esp_diff* d)
{
  hipLaunchKernelGGL(k_clear_run, dim3(1), dim3(64), 0, d->stream, d->run.p);
  DCHK(hipGetLastError());
}

// device bytes kept for tapes
size_t tape_bytes(const esp_diff* d)
{
  size_t c = d->tape.cap;
  for (const auto& h : d->hchunk) c += h->cap;
  return c * sizeof(double4);
}

// Gives the tape back.  Queries keep their answer; a sweep of the run that was on
// it runs it again first.
void release_tape(esp_diff* d)
{
  const size_t n = d->n, b = n * sizeof(double4);
  // the state queries answer with moves by way of the host: there may be no room for
  // it beside the tape
  std::vector<double4> h;
  if (d->tape.p && d->fin.x >= d->tape.p && d->fin.x < d->tape.p + d->tape.cap) {
    h.resize(4 * n);
    const double4* src[4] = {d->fin.x, d->fin.v, d->fin.w, d->fin.q};
    for (int k = 0; k < 4; k++)
      DCHK(hipMemcpyAsync(h.data() + k * n, src[k], b, hipMemcpyDeviceToHost, d->stream));
    d->fin = DState{};
  }
  dsync(d);
  d->tape.release();
  d->hchunk.clear();
  d->htape.clear();
  d->full_tape = false;
  if (h.empty()) return;
  d->x.reserve(n); d->v.reserve(n); d->w.reserve(n); d->q.reserve(n);
  const DState S = d->state();
  double4* dst[4] = {S.x, S.v, S.w, S.q};
  for (int k = 0; k < 4; k++)
    DCHK(hipMemcpyAsync(dst[k], h.data() + k * n, b, hipMemcpyHostToDevice, d->stream));
  dsync(d);
  d->fin = S;
}

// where a step's touching pairs leave their histories: laid out one after the
// other in chunks that are kept for later runs; past the tape limit (searches may
// list more pairs than the first one did) the run keeps checkpoints instead
struct HistoryRoom {
  esp_diff* d;
  size_t chunk, at;
  double4* take(size_t n, int steps_left)
  {
    while (chunk < d->hchunk.size() && at + n > d->hchunk[chunk]->cap) {
      chunk++;
      at = 0;
    }
    if (chunk == d->hchunk.size()) {
      const size_t kept = tape_bytes(d);
      const size_t left = d->tape_limit > kept ? (d->tape_limit - kept) / sizeof(double4) : 0;
      if (n > left) throw DiffMemory("the run's tape is past its limit");
      d->hchunk.push_back(std::make_unique<DevBuf<double4>>());
      const size_t most = std::min(left, (size_t)1 << 25);  // 1 GiB
      d->hchunk.back()->reserve(std::max(n, std::min(most, n * (size_t)std::max(steps_left, 1))));
      at = 0;
    }
    double4* p = d->hchunk[chunk]->p + at;
    at += n;
    return p;
  }
};

int nsamples(const esp_diff* d) { return d->nsteps / d->every; }

// the steps of a forward run; tape: keep every step's state if that fits the limit
void run_forward(esp_diff* d, bool tape)
{
  if (d->tan_on)  // the start state is fixed
    for (DevBuf<double4>* b : {&d->tx, &d->tv, &d->tw, &d->tq})
      DCHK(hipMemsetAsync(b->p, 0, sizeof(double4) * std::max(d->n, 1), d->stream));
  d->epochs.clear();
  d->ckpts.clear();
  d->rebuild_steps.clear();
  d->full_tape = false;
  DCHK(hipMemsetAsync(d->digest.p, 0, sizeof(unsigned long long) * (d->nsteps + 1), d->stream));
  if (d->nb > 0) launch_fill_int(d->stream, d->nb, d->bstep.p, INT_MAX);
  // chunks of steps between checkpoints queued without host decisions; a step
  // whose displacement asks for a neighbour search halts the queue, the host
  // rebuilds the table before the next step and continues
  const int K = std::max(1, d->cfg.checkpoint_every);
  const size_t c4 = 4 * (size_t)d->n;
  DState S0{d->x0.p, d->v0.p, d->w0.p, d->q0.p, d->spec.p, d->n};
  d->fin = S0;
  rebuild(d, S0, 1);
  const size_t states = ((size_t)d->nsteps + 1) * c4;
  const size_t hists = (size_t)d->nsteps * std::max(d->epochs[0]->nc, 1);
  const size_t room_for = d->tape_limit / sizeof(double4);
  const bool fits = tape && !d->tan_on && states + hists <= room_for;
  // an earlier run's tape that this one cannot use within the limit is given back, as
  // is one beside a run of checkpoints (but for the room of a segment's states)
  const size_t kept = tape_bytes(d) / sizeof(double4) - d->tape.cap;
  if (fits ? std::max(d->tape.cap, states) + std::max(kept, hists) > room_for
           : !d->tan_on && (kept > 0 || d->tape.cap > ((size_t)std::min(K, d->nsteps) + 1) * c4))
    release_tape(d);
  d->full_tape = fits;
  DState cur;
  if (d->full_tape) {
    d->tape.reserve(states);
    cur = d->tape_state(d->tape.p);
    d->htape.assign((size_t)d->nsteps + 1, nullptr);
  } else {
    const size_t c = std::max(d->n, 1);
    d->x.reserve(c); d->v.reserve(c); d->w.reserve(c); d->q.reserve(c);
    cur = d->state();
  }
  d2d(d, cur.x, S0.x, d->n); d2d(d, cur.v, S0.v, d->n); d2d(d, cur.w, S0.w, d->n);
  d2d(d, cur.q, S0.q, d->n);
  d->fin = cur;
  HistoryRoom room{d, 0, 0};
  bool need = false;
  int step = 1;
  std::vector<HistoryRoom> mark;
  while (step <= d->nsteps) {
    if (need) {
      rebuild(d, d->fin, step);
      need = false;
    }
    if (!d->full_tape && (step - 1) % K == 0) save_checkpoint(d, step, cur);
    const int end = std::min(d->nsteps, d->full_tape ? step + 63 : ((step - 1) / K + 1) * K);
    const Epoch& E = *d->epochs.back();
    clear_run(d);
    mark.clear();
    for (int s = step; s <= end; s++) {
      if (d->full_tape) {
        mark.push_back(room);
        d->htape[s] = room.take(std::max(E.nc, 1), d->nsteps - s + 1);
        fwd_step(d, E, s, d->tape_state(d->tape.p + (size_t)(s - 1) * c4),
                 d->tape_state(d->tape.p + (size_t)s * c4), d->htape[s], true, true);
      } else {
        fwd_step(d, E, s, cur, cur, nullptr, true, true);
      }
    }
    DRun r;
    DCHK(hipMemcpyAsync(&r, d->run.p, sizeof r, hipMemcpyDeviceToHost, d->stream));
    dsync(d);
    if (r.halt != 0) {
      need = true;
      if (d->full_tape && r.halt < end) room = mark[r.halt + 1 - step];  // the rest did nothing
      step = r.halt + 1;
    } else {
      step = end + 1;
    }
    if (d->full_tape) d->fin = d->tape_state(d->tape.p + (size_t)(step - 1) * c4);
  }
}

// dtheta (nullable): a parameter direction per specimen; the run then also
// carries the state's tangent along it and dloss gets d loss / d epsilon at
// theta + epsilon dtheta
void forward(esp_diff* d, const double* theta, const double* target, double* stress, double* loss,
             const double* dtheta = nullptr, double* dloss = nullptr)
{
  if (d->n <= 0 || d->nsteps <= 0) throw DiffError(ESP_ERR_STATE, "particles and run not set");
  hipEvent_t e0, e1;
  DCHK(hipEventCreate(&e0));
  DCHK(hipEventCreate(&e1));
  DCHK(hipEventRecord(e0, d->stream));
  const int ns = nsamples(d);
  d->h_theta.assign(theta, theta + 4 * d->nspec);
  d->h_target.assign(target, target + (size_t)ns * d->nspec);
  d->theta.reserve(d->nspec);
  std::vector<double4> th(d->nspec);
  for (int s = 0; s < d->nspec; s++)
    th[s] = make_double4(theta[4 * s], theta[4 * s + 1], theta[4 * s + 2], theta[4 * s + 3]);
  DCHK(hipMemcpyAsync(d->theta.p, th.data(), sizeof(double4) * d->nspec, hipMemcpyHostToDevice,
                      d->stream));
  d->stress_dev.reserve((size_t)std::max(ns, 1) * d->nspec);
  d->digest.reserve((size_t)d->nsteps + 1);
  d->have_forward = false;
  d->tan_on = dtheta != nullptr;
  if (d->tan_on) {
    const size_t c = std::max(d->n, 1);
    d->tx.reserve(c); d->tv.reserve(c); d->tw.reserve(c); d->tq.reserve(c);
    d->wft.reserve(c);
    d->bt.reserve((size_t)std::max(d->nb, 1) * 9);
    d->stress_t.reserve((size_t)std::max(ns, 1) * d->nspec);
    d->dtheta.reserve(d->nspec);
    std::vector<double4> dt4(d->nspec);
    for (int s = 0; s < d->nspec; s++)
      dt4[s] = make_double4(dtheta[4 * s], dtheta[4 * s + 1], dtheta[4 * s + 2], dtheta[4 * s + 3]);
    DCHK(hipMemcpyAsync(d->dtheta.p, dt4.data(), sizeof(double4) * d->nspec, hipMemcpyHostToDevice,
                        d->stream));
    dsync(d);  // the copy reads dt4, which ends with this block
  }
  // wall origins of every step: moved by their step before every step (the
  // pre-time-step moveWallBy of the main engine's setWallStepMotion)
  {
    const int nw = d->run_nw = d->nw;
    d->run_has_g = d->has_g;
    for (int c = 0; c < 3; c++) d->run_g[c] = d->g[c];
    std::vector<double>& wo = d->wo;
    wo.assign((size_t)(d->nsteps + 2) * nw * 3, 0.0);
    double o[DIFF_MAX_WALLS][3];
    for (int k = 0; k < d->nw; k++)
      for (int c = 0; c < 3; c++) o[k][c] = d->wall0[k].o[c];
    for (int t = 0; t <= d->nsteps + 1; t++) {
      for (int k = 0; k < d->nw; k++)
        for (int c = 0; c < 3; c++) wo[((size_t)t * nw + k) * 3 + c] = o[k][c];
      for (int k = 0; k < d->nw; k++)
        for (int c = 0; c < 3; c++) o[k][c] = o[k][c] + d->wstep[k][c];
    }
  }
  d->run.reserve(1);
  d->wfn.reserve(std::max(d->n, 1));
  try {
    run_forward(d, true);
  } catch (const DiffMemory&) {
    // no room for the run's tape, or beside one kept: again with checkpoints
    if (tape_bytes(d) == 0 && !d->full_tape) throw;
    release_tape(d);
    run_forward(d, false);
  }
  d->h_stress.assign((size_t)ns * d->nspec, 0.0);
  DCHK(hipMemcpyAsync(d->h_stress.data(), d->stress_dev.p, sizeof(double) * ns * d->nspec,
                      hipMemcpyDeviceToHost, d->stream));
  if (d->tan_on) {
    d->h_stress_t.assign((size_t)ns * d->nspec, 0.0);
    DCHK(hipMemcpyAsync(d->h_stress_t.data(), d->stress_t.p, sizeof(double) * ns * d->nspec,
                        hipMemcpyDeviceToHost, d->stream));
  }
  DCHK(hipEventRecord(e1, d->stream));
  dsync(d);
  float ms = 0;
  DCHK(hipEventElapsedTime(&ms, e0, e1));
  d->t_fwd = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  for (int s = 0; s < d->nspec; s++) {
    double acc = 0.0;
    for (int k = 0; k < ns; k++) {
      const double st = d->h_stress[(size_t)k * d->nspec + s] / d->h_area[s];
      if (stress) stress[(size_t)s * ns + k] = st;
      const double df = st - d->h_target[(size_t)s * ns + k];
      acc = acc + df * df;
    }
    loss[s] = ns > 0 ? acc / ns : 0.0;
    if (d->tan_on && dloss) {
      double dacc = 0.0;
      for (int k = 0; k < ns; k++) {
        const double st = d->h_stress[(size_t)k * d->nspec + s] / d->h_area[s];
        const double dst = d->h_stress_t[(size_t)k * d->nspec + s] / d->h_area[s];
        dacc = dacc + 2.0 * (st - d->h_target[(size_t)s * ns + k]) * dst;
      }
      dloss[s] = ns > 0 ? dacc / ns : 0.0;
    }
  }
  d->tan_on = false;
  d->have_forward = true;
}

// the reverse sweep over the last forward run; done is recorded at its end
void sweep(esp_diff* d, double* grad, hipEvent_t done)
{
  const int n = d->n, bs = d->bs, ns = nsamples(d);
  const int K = std::max(1, d->cfg.checkpoint_every);
  const size_t c = std::max(n, 1);
  // d loss / d stress_s at each sample, divided by the area (the stress is the
  // specimen's wall force over its area)
  std::vector<double> coef((size_t)std::max(ns, 1) * d->nspec, 0.0);
  for (int s = 0; s < d->nspec; s++)
    for (int k = 0; k < ns; k++) {
      const double st = d->h_stress[(size_t)k * d->nspec + s] / d->h_area[s];
      coef[(size_t)k * d->nspec + s] = 2.0 * (st - d->h_target[(size_t)s * ns + k]) / ns / d->h_area[s];
    }
  DevBuf<double> coef_d;
  coef_d.reserve(coef.size());
  DCHK(hipMemcpyAsync(coef_d.p, coef.data(), sizeof(double) * coef.size(), hipMemcpyHostToDevice,
                      d->stream));
  auto &lam = d->lam, &gth = d->gth, &lh = d->lh, &lh2 = d->lh2;
  auto& lfm = d->lfm;
  auto &ab = d->ab, &ac = d->ac;
  auto& aact = d->aact;
  lam.reserve(4 * c);
  gth.reserve(c);
  lfm.reserve(6 * c);
  ab.reserve((size_t)std::max(d->nb, 1) * NB_REC);
  DCHK(hipMemsetAsync(ab.p, 0, sizeof(double4) * NB_REC * std::max(d->nb, 1), d->stream));
  DCHK(hipMemsetAsync(lam.p, 0, sizeof(double4) * 4 * c, d->stream));
  DCHK(hipMemsetAsync(gth.p, 0, sizeof(double4) * c, d->stream));
  const size_t c4 = 4 * (size_t)n;
  // without the run's tape: that of one segment, the states of steps s0..s1 and
  // the histories read at s0..s1-1
  if (!d->full_tape) d->tape.reserve((size_t)(std::min(K, d->nsteps) + 1) * c4);
  int lh_epoch = -1;  // epoch whose pairs lh is indexed by
  DBonds B{d->nb, d->bij.p, d->bD0.p, d->brel.p, d->bstep.p, d->tkb.p};
  auto epoch_of = [&](int step) {
    int e = 0;
    while (e + 1 < (int)d->epochs.size() && d->epochs[e + 1]->start <= step) e++;
    return e;
  };
  clear_run(d);
  const int nseg = d->full_tape ? 1 : (int)d->ckpts.size();
  for (int seg = nseg - 1; seg >= 0; seg--) {
    const int s0 = d->full_tape ? 1 : d->ckpts[seg]->step;
    const int s1 = d->full_tape ? d->nsteps + 1 : std::min(s0 + K, d->nsteps + 1);
    auto state_before = [&](int step) { return d->tape_state(d->tape.p + (size_t)(step - s0) * c4); };
    if (!d->full_tape) {
      const Checkpoint& C = *d->ckpts[seg];
      restore_checkpoint(d, C, d->tape.p);
      // recompute the segment forward, recording the states and histories
      if ((int)d->hseg.size() < K) d->hseg.resize(K);
      int cur = C.epoch;
      for (int step = s0; step < s1; step++) {
        const int e = epoch_of(step);
        if (e != cur) {  // the rebuild of this step: histories carried by key
          const Epoch& E = *d->epochs[e];
          DevBuf<double4> hn;
          hn.reserve(std::max(E.nc, 1));
          if (E.nc > 0)
            hipLaunchKernelGGL(k_carry_hist, dim3(nblocks(E.nc, bs)), dim3(bs), 0, d->stream, E.nc,
                               E.src.p, d->H[step & 1].p, hn.p);
          d->H[step & 1].swap(hn);
          d->H[(step + 1) & 1].reserve(std::max(E.nc, 1));
          d2d(d, d->H[(step + 1) & 1].p, d->H[step & 1].p, E.nc);
          d->cout.reserve((size_t)std::max(E.nc, 1) * 9);
          d->cact.reserve((size_t)std::max(E.nc, 1));
          dsync(d);  // hn now holds the old histories, freed with this block
          cur = e;
        }
        const int t = step - s0;
        if (!d->hseg[t]) d->hseg[t] = std::make_unique<DevBuf<double4>>();
        d->hseg[t]->reserve(std::max(d->epochs[cur]->nc, 1));
        fwd_step(d, *d->epochs[cur], step, state_before(step), state_before(step + 1),
                 d->hseg[t]->p, false, false);
      }
    }
    // reverse sweep: a step's particle updates, its laws, then its gather with
    // the particle updates of the step before it
    auto coef_of = [&](int step) {
      return step % d->every == 0 ? coef_d.p + (size_t)(step / d->every - 1) * d->nspec : nullptr;
    };
    const bool wide = n <= kAdjointRow;
    auto adj_step = [&](auto kern, const Epoch* E, const DState& Sn, const DState& Sn1, int part) {
      hipLaunchKernelGGL(kern, dim3(nblocks((wide ? 16ll : 4ll) * n, bs)), dim3(bs), 0, d->stream, n,
                         E ? E->inc_off.p : nullptr, E ? E->inc_ent.p : nullptr, E ? E->nc : 0, ac.p,
                         ab.p, aact.p, lam.p, gth.p, Sn, Sn1, lfm.p,
                         d->step_params(part), part > 0 ? coef_of(part) : nullptr);
    };
    adj_step(wide ? k_adj_step<false, true, 16> : k_adj_step<false, true, 4>, nullptr,
             state_before(s1 - 1), state_before(s1), s1 - 1);
    for (int step = s1 - 1; step >= s0; step--) {
      const int e = epoch_of(step);
      const Epoch& E = *d->epochs[e];
      if (lh_epoch != e) {
        // the history adjoint of the next step's pairs, taken back to this
        // step's pairs (the next step started an epoch) or started at zero
        lh2.reserve(std::max(E.nc, 1));
        DCHK(hipMemsetAsync(lh2.p, 0, sizeof(double4) * std::max(E.nc, 1), d->stream));
        if (lh_epoch >= 0) {
          const Epoch& N = *d->epochs[lh_epoch];
          if (N.nc > 0)
            hipLaunchKernelGGL(k_map_lh, dim3(nblocks(N.nc, bs)), dim3(bs), 0, d->stream, N.nc,
                               N.src.p, lh.p, lh2.p);
        }
        lh.swap(lh2);
        lh_epoch = e;
        lh2.reserve(std::max(E.nc, 1));
        ac.reserve((size_t)std::max(E.nc, 1) * NF_REC);
        aact.reserve((size_t)std::max(E.nc, 1));
      }
      const DState Sn = state_before(step);
      if (d->nb > 0)
        hipLaunchKernelGGL(k_adj_bond, dim3(nblocks(d->nb, ADJ_BOND_BS)), dim3(ADJ_BOND_BS), 0,
                           d->stream, Sn, B, d->theta.p, step, lfm.p, ab.p);
      DCands Cd{E.nc, E.ij.p, E.bond.p};
      if (E.nc > 0)
        hipLaunchKernelGGL(k_adj_fric, dim3(nblocks(E.nc, bs)), dim3(bs), 0, d->stream, Sn, Cd,
                           d->bstep.p, d->theta.p, d->full_tape ? d->htape[step] : d->hseg[step - s0]->p,
                           step, d->cfg.dt, lfm.p, lh.p, ac.p, aact.p, lh2.p);
      if (step > s0)
        adj_step(wide ? k_adj_step<true, true, 16> : k_adj_step<true, true, 4>, &E,
                 state_before(step - 1), Sn, step - 1);
      else
        adj_step(wide ? k_adj_step<true, false, 16> : k_adj_step<true, false, 4>, &E, Sn, Sn, 0);
      DCHK(hipGetLastError());
      lh.swap(lh2);
    }
    if (!d->full_tape) dsync(d);
  }
  DevBuf<double4> gs;
  gs.reserve(std::max(d->nspec, 1));
  hipLaunchKernelGGL(k_spec_sum4, dim3(d->nspec), dim3(256), 0, d->stream, gth.p, d->spec_start.p,
                     gs.p);
  std::vector<double4> hg(d->nspec);
  DCHK(hipMemcpyAsync(hg.data(), gs.p, sizeof(double4) * d->nspec, hipMemcpyDeviceToHost,
                      d->stream));
  DCHK(hipEventRecord(done, d->stream));
  dsync(d);
  for (int s = 0; s < d->nspec; s++) {
    grad[4 * s] = hg[s].x;
    grad[4 * s + 1] = hg[s].y;
    grad[4 * s + 2] = 0.0;  // cohesion moves only the break events
    grad[4 * s + 3] = hg[s].w;
  }
}

// the last run again (its walls, gravity and parameters), with checkpoints: every
// step gives the bits it gave
void rerun(esp_diff* d)
{
  d->have_forward = false;
  run_forward(d, false);
  d->have_forward = true;
}

void backward(esp_diff* d, double* grad)
{
  if (!d->have_forward) throw DiffError(ESP_ERR_STATE, "backward needs a forward run first");
  hipEvent_t e0, e1;
  DCHK(hipEventCreate(&e0));
  DCHK(hipEventCreate(&e1));
  DCHK(hipEventRecord(e0, d->stream));
  if (!d->full_tape && d->ckpts.empty()) rerun(d);  // its tape was given back
  try {
    sweep(d, grad, e1);
  } catch (const DiffMemory&) {
    // no room for the adjoint beside the tape
    if (!d->full_tape) throw;
    release_tape(d);
    rerun(d);
    sweep(d, grad, e1);
  }
  float ms = 0;
  DCHK(hipEventElapsedTime(&ms, e0, e1));
  d->t_bwd = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
}

}  // namespace

// ===========================================================================
// C-ABI
// ===========================================================================
#define DAPI_BEGIN try {
#define DAPI_END                     \
  }                                  \
  catch (const DiffError& ex)        \
  {                                  \
    d->err = ex.what();              \
    return ex.code;                  \
  }                                  \
  catch (const std::exception& ex)   \
  {                                  \
    d->err = ex.what();              \
    return ESP_ERR_STATE;            \
  }

extern "C" {

const char* esp_diff_create_error(void) { return g_diff_create_err.c_str(); }
const char* esp_diff_last_error(const esp_diff* d) { return d ? d->err.c_str() : ""; }

int esp_diff_create(const esp_diff_config* cfg, esp_diff** out)
{
  g_diff_create_err.clear();
  if (!cfg || !out) {
    g_diff_create_err = "null argument";
    return ESP_ERR_ARG;
  }
  if (!(cfg->grid_spacing > 0) || !(cfg->verlet_dist >= 0) || !(cfg->dt > 0)) {
    g_diff_create_err = "gridSpacing, dt must be > 0 and verletDist >= 0";
    return ESP_ERR_ARG;
  }
  const int bsz = cfg->block > 0 ? cfg->block : 256;
  if (bsz < 64 || bsz > DIFF_MAX_BS || bsz % 64) {
    g_diff_create_err = "block must be a multiple of 64 in [64, 512]";
    return ESP_ERR_ARG;
  }
  // the neighbour table of TSubLattice::initNeighborTable (SubLattice.hpp:455-478)
  const double nr = cfg->grid_spacing;
  double nmin[3], nmax[3];
  long ng[3];
  for (int c = 0; c < 3; c++) {
    const double mn = cfg->domain_min[c], mx = cfg->domain_max[c];
    const double sz = nr * std::ceil((mx - mn) / nr);
    const double grow = sz - (mx - mn);
    nmin[c] = mn - grow * 0.5;
    nmax[c] = mx + grow * 0.5;
    ng[c] = lrint((nmax[c] - nmin[c]) / nr);
    if (std::fabs((double)ng[c] - (nmax[c] - nmin[c]) / nr) > 1e-6 || ng[c] < 1) {
      g_diff_create_err = "size doesn't fit range";
      return ESP_ERR_ARG;
    }
  }
  if ((double)(ng[0] + 2) * (double)(ng[1] + 2) * (double)(ng[2] + 2) > 2.0e8) {
    g_diff_create_err = "neighbour table too large";
    return ESP_ERR_CAPACITY;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
    g_diff_create_err = "no HIP device available";
    return ESP_ERR_DEVICE;
  }
  if (cfg->device < 0 || cfg->device >= ndev || hipSetDevice(cfg->device) != hipSuccess) {
    g_diff_create_err = "bad device";
    return ESP_ERR_DEVICE;
  }
  esp_diff* d = new esp_diff();
  d->cfg = *cfg;
  d->tape_limit = kTapeLimit;
  d->bs = bsz;
  memset(&d->grid, 0, sizeof d->grid);
  d->grid.x0 = nmin[0]; d->grid.y0 = nmin[1]; d->grid.z0 = nmin[2];
  d->grid.dim = nr;
  d->grid.gx = d->grid.gy = d->grid.gz = -1;
  d->grid.nx = (int)ng[0] + 2; d->grid.ny = (int)ng[1] + 2; d->grid.nz = (int)ng[2] + 2;
  d->ncell = d->grid.nx * d->grid.ny * d->grid.nz;
  if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
    delete d;
    g_diff_create_err = "hipStreamCreate failed";
    return ESP_ERR_DEVICE;
  }
  try {
    d->md.reserve(2);
    d->cell_count.reserve(d->ncell + 1);
    d->cell_start.reserve(d->ncell + 1);
    d->cell_fill.reserve(d->ncell + 1);
  } catch (const DiffError& ex) {
    g_diff_create_err = ex.what();
    delete d;
    return ex.code;
  }
  *out = d;
  return ESP_OK;
}

void esp_diff_destroy(esp_diff* d)
{
  if (!d) return;
  if (d->stream) (void)hipStreamSynchronize(d->stream);
  d->epochs.clear();
  d->ckpts.clear();
  hipStream_t s = d->stream;
  delete d;
  if (s) (void)hipStreamDestroy(s);
}

int esp_diff_set_particles(esp_diff* d, int n, int nspec, const int* spec, const double* pos,
                           const double* rad, const double* mass, const double* vel)
{
  DAPI_BEGIN
  if (n <= 0 || nspec <= 0 || !spec || !pos || !rad || !mass)
    throw DiffError(ESP_ERR_ARG, "bad particle arrays");
  std::vector<int> start(nspec + 1, 0);
  for (int i = 0; i < n; i++) {
    if (spec[i] < 0 || spec[i] >= nspec || (i > 0 && spec[i] < spec[i - 1]))
      throw DiffError(ESP_ERR_ARG, "specimen ids must be non-decreasing in [0, nspec)");
    start[spec[i] + 1]++;
  }
  for (int s = 0; s < nspec; s++) start[s + 1] += start[s];
  d->n = n;
  d->nspec = nspec;
  d->fin = DState{};
  d->have_forward = false;
  d->h_spec.assign(spec, spec + n);
  d->h_spec_start = start;
  d->h_pos.assign(pos, pos + 3 * n);
  d->h_rad.assign(rad, rad + n);
  d->h_mass.assign(mass, mass + n);
  d->h_vel.assign(vel ? vel : pos, (vel ? vel : pos) + 3 * n);
  if (!vel) std::fill(d->h_vel.begin(), d->h_vel.end(), 0.0);
  d->spec.reserve(n);
  d->spec_start.reserve(nspec + 1);
  d->id.reserve(n);
  d->flags.reserve(n);
  d->cell.reserve(n);
  d->cell_items.reserve(n);
  d->ccnt.reserve(n + 1);
  d->coff.reserve(n + 1);
  d->wfn.reserve(n);
  std::vector<double4> X(n), V(n), W(n), Q(n), O(n);
  for (int i = 0; i < n; i++) {
    const double m = d->h_mass[i], r = d->h_rad[i];
    X[i] = make_double4(d->h_pos[3 * i], d->h_pos[3 * i + 1], d->h_pos[3 * i + 2], r);
    V[i] = make_double4(d->h_vel[3 * i], d->h_vel[3 * i + 1], d->h_vel[3 * i + 2],
                        m != 0.0 ? 1.0 / m : 0.0);
    const double I = 0.4 * m * r * r;  // CRotParticle, 3-D (RotParticle.cpp:80-124)
    W[i] = make_double4(0.0, 0.0, 0.0, 1.0 / I);
    Q[i] = make_double4(1.0, 0.0, 0.0, 0.0);
    O[i] = make_double4(X[i].x, X[i].y, X[i].z, m);
  }
  d->x0.reserve(n); d->v0.reserve(n); d->w0.reserve(n); d->q0.reserve(n); d->o.reserve(n);
  DCHK(hipMemcpyAsync(d->x0.p, X.data(), sizeof(double4) * n, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->v0.p, V.data(), sizeof(double4) * n, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->w0.p, W.data(), sizeof(double4) * n, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->q0.p, Q.data(), sizeof(double4) * n, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->o.p, O.data(), sizeof(double4) * n, hipMemcpyHostToDevice, d->stream));
  std::vector<int> ids(n);
  std::vector<unsigned> fl(n, PF_DYN | PF_ROT);
  for (int i = 0; i < n; i++) ids[i] = i;
  DCHK(hipMemcpyAsync(d->spec.p, spec, sizeof(int) * n, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->spec_start.p, start.data(), sizeof(int) * (nspec + 1),
                      hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->id.p, ids.data(), sizeof(int) * n, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->flags.p, fl.data(), sizeof(unsigned) * n, hipMemcpyHostToDevice,
                      d->stream));
  dsync(d);
  return ESP_OK;
  DAPI_END
}

int esp_diff_set_bonds(esp_diff* d, int nb, const int* bi, const int* bj, const double* rel,
                       const double* tk, const double* bk)
{
  DAPI_BEGIN
  if (d->n <= 0) throw DiffError(ESP_ERR_STATE, "set the particles first");
  if (nb < 0 || (nb > 0 && (!bi || !bj || !rel)) || !tk || !bk)
    throw DiffError(ESP_ERR_ARG, "bad bond arrays");
  std::vector<int> order(nb);
  for (int k = 0; k < nb; k++) {
    if (bi[k] < 0 || bj[k] >= d->n || bi[k] >= bj[k] || d->h_spec[bi[k]] != d->h_spec[bj[k]])
      throw DiffError(ESP_ERR_ARG, "a bond needs i < j within one specimen");
    order[k] = k;
  }
  auto key = [&](int k) { return ((long long)bi[k] << 32) | (long long)bj[k]; };
  std::sort(order.begin(), order.end(), [&](int a, int b) { return key(a) < key(b); });
  for (int k = 1; k < nb; k++)
    if (key(order[k]) == key(order[k - 1])) throw DiffError(ESP_ERR_ARG, "repeated bond");
  std::vector<int2> ij(nb);
  std::vector<long long> kk(nb);
  std::vector<double4> D0(nb), R(nb);
  for (int t = 0; t < nb; t++) {
    const int k = order[t], a = bi[k], b = bj[k];
    ij[t] = make_int2(a, b);
    kk[t] = key(k);
    const double dx = d->h_pos[3 * b] - d->h_pos[3 * a], dy = d->h_pos[3 * b + 1] - d->h_pos[3 * a + 1],
                 dz = d->h_pos[3 * b + 2] - d->h_pos[3 * a + 2];
    // ARotBondedInteraction / CRotBondedInteraction: D = p2 - p1, dist = |D|
    D0[t] = make_double4(dx, dy, dz, std::sqrt(dx * dx + dy * dy + dz * dz));
    R[t] = make_double4(rel[4 * k], rel[4 * k + 1], rel[4 * k + 2], rel[4 * k + 3]);
  }
  std::vector<double2> tkb(d->nspec);
  for (int s = 0; s < d->nspec; s++) tkb[s] = make_double2(tk[s], bk[s]);
  d->nb = nb;
  const size_t c = std::max(nb, 1);
  d->bij.reserve(c); d->bkey.reserve(c); d->bD0.reserve(c); d->brel.reserve(c); d->bstep.reserve(c);
  d->tkb.reserve(std::max(d->nspec, 1));
  DCHK(hipMemcpyAsync(d->bij.p, ij.data(), sizeof(int2) * nb, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->bkey.p, kk.data(), sizeof(long long) * nb, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->bD0.p, D0.data(), sizeof(double4) * nb, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->brel.p, R.data(), sizeof(double4) * nb, hipMemcpyHostToDevice, d->stream));
  DCHK(hipMemcpyAsync(d->tkb.p, tkb.data(), sizeof(double2) * d->nspec, hipMemcpyHostToDevice,
                      d->stream));
  d->h_bi.resize(nb);
  d->h_bj.resize(nb);
  for (int t = 0; t < nb; t++) { d->h_bi[t] = ij[t].x; d->h_bj[t] = ij[t].y; }
  dsync(d);
  d->have_forward = false;
  return ESP_OK;
  DAPI_END
}

int esp_diff_add_wall(esp_diff* d, const double origin[3], const double normal[3], double k,
                      const double step[3], int measure, const double* area)
{
  DAPI_BEGIN
  if (d->nw >= DIFF_MAX_WALLS) throw DiffError(ESP_ERR_CAPACITY, "more than 4 walls");
  if (!origin || !normal || !step) throw DiffError(ESP_ERR_ARG, "bad wall");
  DWall& W = d->wall0[d->nw];
  for (int c = 0; c < 3; c++) {
    W.o[c] = origin[c];
    W.n[c] = normal[c];
    d->wstep[d->nw][c] = step[c];
  }
  W.k = k;
  W.measure = measure ? 1 : 0;
  if (measure) {
    if (!area || d->nspec <= 0) throw DiffError(ESP_ERR_ARG, "the measured wall needs the areas");
    for (int w = 0; w < d->nw; w++)
      if (d->wall0[w].measure) throw DiffError(ESP_ERR_ARG, "one measured wall");
    d->h_area.assign(area, area + d->nspec);
  }
  d->nw++;
  return ESP_OK;
  DAPI_END
}

int esp_diff_set_gravity(esp_diff* d, const double g[3])
{
  DAPI_BEGIN
  d->has_g = 1;
  for (int c = 0; c < 3; c++) d->g[c] = g[c];
  return ESP_OK;
  DAPI_END
}

int esp_diff_set_run(esp_diff* d, int nsteps, int sample_every)
{
  DAPI_BEGIN
  if (nsteps <= 0 || sample_every <= 0) throw DiffError(ESP_ERR_ARG, "bad run");
  if (nsteps != d->nsteps || sample_every != d->every) d->have_forward = false;
  d->nsteps = nsteps;
  d->every = sample_every;
  return ESP_OK;
  DAPI_END
}

int esp_diff_set_tape_limit(esp_diff* d, unsigned long long bytes)
{
  DAPI_BEGIN
  d->tape_limit = (size_t)bytes;
  if (tape_bytes(d) > d->tape_limit) release_tape(d);
  return ESP_OK;
  DAPI_END
}

int esp_diff_get_tape_bytes(esp_diff* d, unsigned long long* out)
{
  DAPI_BEGIN
  if (!out) throw DiffError(ESP_ERR_ARG, "null argument");
  *out = d->full_tape ? tape_bytes(d) : 0;
  return ESP_OK;
  DAPI_END
}

int esp_diff_forward(esp_diff* d, const double* theta, const double* target, double* stress,
                     double* loss)
{
  DAPI_BEGIN
  if (!theta || !target || !loss) throw DiffError(ESP_ERR_ARG, "null argument");
  if (d->h_area.empty()) throw DiffError(ESP_ERR_STATE, "no measured wall");
  forward(d, theta, target, stress, loss);
  return ESP_OK;
  DAPI_END
}

int esp_diff_forward_tangent(esp_diff* d, const double* theta, const double* dtheta,
                             const double* target, double* stress, double* loss, double* dloss)
{
  DAPI_BEGIN
  if (!theta || !dtheta || !target || !loss || !dloss) throw DiffError(ESP_ERR_ARG, "null argument");
  if (d->h_area.empty()) throw DiffError(ESP_ERR_STATE, "no measured wall");
  forward(d, theta, target, stress, loss, dtheta, dloss);
  return ESP_OK;
  DAPI_END
}

int esp_diff_backward(esp_diff* d, double* grad)
{
  DAPI_BEGIN
  if (!grad) throw DiffError(ESP_ERR_ARG, "null argument");
  backward(d, grad);
  return ESP_OK;
  DAPI_END
}

int esp_diff_get_particle_data(esp_diff* d, int field, double* out)
{
  DAPI_BEGIN
  const int n = d->n;
  std::vector<double4> a(n);
  const double4* src = field == ESP_FIELD_POS ? d->fin.x : field == ESP_FIELD_VEL ? d->fin.v
                     : field == ESP_FIELD_ANGVEL ? d->fin.w : field == ESP_FIELD_QUAT ? d->fin.q
                                                                                     : nullptr;
  if (!src) throw DiffError(ESP_ERR_ARG, "unknown field");
  DCHK(hipMemcpyAsync(a.data(), src, sizeof(double4) * n, hipMemcpyDeviceToHost, d->stream));
  dsync(d);
  for (int i = 0; i < n; i++) {
    if (field == ESP_FIELD_QUAT) {
      out[4 * i] = a[i].x; out[4 * i + 1] = a[i].y; out[4 * i + 2] = a[i].z; out[4 * i + 3] = a[i].w;
    } else {
      out[3 * i] = a[i].x; out[3 * i + 1] = a[i].y; out[3 * i + 2] = a[i].z;
    }
  }
  return ESP_OK;
  DAPI_END
}

int esp_diff_get_bond_breaks(esp_diff* d, int* step, int* bi, int* bj)
{
  DAPI_BEGIN
  std::vector<int> bs(std::max(d->nb, 1));
  DCHK(hipMemcpyAsync(bs.data(), d->bstep.p, sizeof(int) * d->nb, hipMemcpyDeviceToHost, d->stream));
  dsync(d);
  std::vector<int> idx;
  for (int b = 0; b < d->nb; b++)
    if (bs[b] != INT_MAX && bs[b] < d->nsteps) idx.push_back(b);  // left the group at bs + 1
  std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) { return bs[a] < bs[b]; });
  if (step)
    for (size_t k = 0; k < idx.size(); k++) {
      step[k] = bs[idx[k]] + 1;
      bi[k] = d->h_bi[idx[k]];
      bj[k] = d->h_bj[idx[k]];
    }
  return (int)idx.size();
  DAPI_END
}

int esp_diff_get_rebuild_steps(esp_diff* d, int* steps)
{
  DAPI_BEGIN
  if (steps)
    for (size_t k = 0; k < d->rebuild_steps.size(); k++) steps[k] = d->rebuild_steps[k];
  return (int)d->rebuild_steps.size();
  DAPI_END
}

int esp_diff_track_branches(esp_diff* d, int enable)
{
  DAPI_BEGIN
  d->track_digest = enable != 0;
  return ESP_OK;
  DAPI_END
}

int esp_diff_get_branch_digest(esp_diff* d, unsigned long long* out)
{
  DAPI_BEGIN
  if (!d->track_digest)
    throw DiffError(ESP_ERR_STATE, "branch digests are not tracked (esp_diff_track_branches)");
  if (!d->have_forward) throw DiffError(ESP_ERR_STATE, "no forward run");
  if (out) {
    DCHK(hipMemcpyAsync(out, d->digest.p + 1, sizeof(unsigned long long) * d->nsteps,
                        hipMemcpyDeviceToHost, d->stream));
    dsync(d);
  }
  return d->nsteps;
  DAPI_END
}

int esp_diff_get_times(esp_diff* d, double* fwd, double* bwd)
{
  DAPI_BEGIN
  if (fwd) *fwd = d->t_fwd;
  if (bwd) *bwd = d->t_bwd;
  return ESP_OK;
  DAPI_END
}

}  // extern "C"
