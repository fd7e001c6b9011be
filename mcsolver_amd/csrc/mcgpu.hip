// libmcgpu — MI355X (gfx950) Monte Carlo sweep engine for Ising / XY /
// Heisenberg spins on arbitrary bond graphs.  See include/mcgpu.h for the ABI.
//
// Kernels
//   k_lds<NC,ST,MODE,FULL,PERSIST>
//                     LDS sweep: each workgroup owns R replicas of one
//                     lattice (or one part of a replica split over 2-4
//                     workgroups), stages their spins in LDS once, runs many
//                     graph-coloured Metropolis sweeps with in-kernel fused
//                     measurement, writes spins back once.  PERSIST: every
//                     workgroup resident; tempering and part exchange inside
//                     the kernel.  HBM traffic per sweep ~1 MB of bookkeeping;
//                     bound by VALU issue and the per-sweep exchanges.
//   k_pass<NC,ST,..>  streaming colour pass over all replicas (spins in HBM /
//                     L2), for lattices too large for LDS; also the "plain"
//                     one-launch-per-replica-per-colour baseline.
//   k_measure<NC,ST>  one workgroup per replica: FP64 full-Hamiltonian
//                     recomputation and/or one measured frame.
//   k_wolff<NC,ST,..> one workgroup per replica: level-synchronous frontier
//                     BFS Wolff clusters (embedded-spin for O(n)).
//   k_pt              parallel-tempering swaps of temperature rows.
//
// Every single-site update is the same deterministic function of
// (spins, site, sweep index, replica key), with a counter-based Philox
// stream, so all kernels produce the same trajectory bit for bit.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <queue>
#include <tuple>
#include <vector>

#include "../../include/mcgpu.h"
#include "mc_math.h"

using namespace mcg;

// ---------------------------------------------------------------------------
// error reporting
// ---------------------------------------------------------------------------
static thread_local std::string g_err;

static int fail(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return -1;
}

#define HIPCHK(x)                                                                        \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) return fail("%s failed: %s", #x, hipGetErrorString(e_));       \
  } while (0)

extern "C" const char* mcg_last_error(void) { return g_err.c_str(); }
extern "C" int mcg_version(void) { return 1; }

// ---------------------------------------------------------------------------
// spin storage
// ---------------------------------------------------------------------------
// pointers into HBM with their address space spelled out, so that the
// compiler emits global (not flat) memory instructions
#define GAS __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ GAS T* gas(T* p) {
  return (GAS T*)p;
}
template <typename T>
__device__ __forceinline__ const GAS T* gas(const T* p) {
  return (const GAS T*)p;
}

template <typename ST>
struct SIO;
template <>
struct SIO<float> {
  template <class P>
  static __device__ __forceinline__ float ld(P p) { return *p; }
  template <class P>
  static __device__ __forceinline__ void st(P p, float v) { *p = v; }
};
template <>
struct SIO<__half> {
  static __device__ __forceinline__ float ld(const __half* p) { return __half2float(*p); }
  static __device__ __forceinline__ void st(__half* p, float v) { *p = __float2half_rn(v); }
  // HBM: move the 16-bit pattern as a scalar
  static __device__ __forceinline__ float ld(const GAS __half* p) {
    return __half2float(__ushort_as_half(*(const GAS unsigned short*)p));
  }
  static __device__ __forceinline__ void st(GAS __half* p, float v) {
    *(GAS unsigned short*)p = __half_as_ushort(__float2half_rn(v));
  }
};
template <>
struct SIO<int8_t> {
  template <class P>
  static __device__ __forceinline__ float ld(P p) { return (float)*p; }
  template <class P>
  static __device__ __forceinline__ void st(P p, float v) { *p = (int8_t)v; }
};

// one replica's spins; PT is ST* (LDS, inferred) or GAS ST* (HBM)
template <typename ST, typename PT = ST*>
struct Spins {
  typedef ST value_type;
  PT p;
  int n;
  __device__ __forceinline__ float get(int i, int c) const { return SIO<ST>::ld(p + (size_t)c * n + i); }
  __device__ __forceinline__ void set(int i, int c, float v) const { SIO<ST>::st(p + (size_t)c * n + i, v); }
};
template <typename ST>
using GSpins = Spins<ST, GAS ST*>;

// neighbour accessor of graphs without link patterns: the global link table
struct GlobalLinks {
  const GAS uint32_t* lk;
  const GAS int32_t* lc;  // per-link coupling indices (wide graphs) or nullptr
  __device__ __forceinline__ int nbr(int l) const { return (int)(lk[l] & 0xFFFFFFu); }
  __device__ __forceinline__ uint32_t cid(int l) const { return lc ? (uint32_t)lc[l] : lk[l] >> 24; }
};
// Pattern rows in LDS: zmax link words, then the site class, padded to a
// multiple of four words so that four links come in one 128-bit read.  Graphs
// of one coupling: each link word is the byte offset from the site's spin to
// the neighbour's (same component).  Others: position delta << 8 | coupling.
__host__ __device__ constexpr int pat_stride(int zmax) { return (zmax + 4) & ~3; }
// couplings in LDS: 12 floats each, the 3x3 tensor in three 128-bit reads
static constexpr int COUP_LDS = 12;
template <bool UNI>
__device__ __forceinline__ int32_t row_word(int32_t w, int ssize) {  // w: a link word of mcg_graph.pattab
  const int32_t d = (int32_t)((uint32_t)w << 8) >> 8;
  return UNI ? d * ssize : (int32_t)(((uint32_t)d << 8) | ((uint32_t)w >> 24));
}

static constexpr double REF_PI = 3.1415926535;  // heisenbergLib.c:6

// a value that is the same in every active lane, as a scalar
__device__ __forceinline__ int wave_uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float wave_uniform(float x) { return __int_as_float(wave_uniform(__float_as_int(x))); }
__device__ __forceinline__ double wave_uniform(double x) {
  return __hiloint2double(wave_uniform(__double2hiint(x)), wave_uniform(__double2loint(x)));
}
// a wave-uniform value kept in a vector register: FP32 adds, products and
// FMAs whose operands are all vector registers issue at 2.8-3.2 cycles per
// SIMD on gfx950, those with a scalar operand at 4.4 (measured, 4 waves)
__device__ __forceinline__ float in_vgpr(float x) {
  asm("" : "+v"(x));
  return x;
}

// The acceptance of a row: beta, and for exact Ising the row's threshold
// table thr[k] = floor(2^32 exp(-beta k u)) for dE = k u (u = 1 / inv_unit, a
// power of two; thr0 / nthr: the whole table, for replicas of other rows).
// A float converts to an Acc without a table (the FP32 exp path).
struct Acc {
  float beta;
  const uint32_t* thr;
  float inv_unit;
  const uint32_t* thr0;
  int nthr;
  const uint32_t* lds;  // the table's copy in LDS, or nullptr; lds0: every group's, lstride words apart
  const uint32_t* lds0;
  int lstride;
  __device__ __forceinline__ Acc(float b)
      : beta(b), thr(nullptr), inv_unit(0.0f), thr0(nullptr), nthr(0), lds(nullptr), lds0(nullptr), lstride(0) {}
  __device__ __forceinline__ Acc(float b, const uint32_t* t, float iu, const uint32_t* t0, int n)
      : beta(b), thr(t), inv_unit(iu), thr0(t0), nthr(n), lds(nullptr), lds0(nullptr), lstride(0) {}
  // the same table at another row (beta b), of group g
  __device__ __forceinline__ Acc at(float b, int row, int g) const {
    Acc x(b, thr0 ? thr0 + (size_t)row * nthr : nullptr, inv_unit, thr0, nthr);
    if (lds0) x.lds = lds0 + g * lstride;
    return x;
  }
};
// the acceptance of row `row` of the batch
__device__ __forceinline__ Acc acc_of(const mcg_batch& B, float beta, int row) {
  return B.ithr ? Acc(beta, B.ithr + (size_t)row * B.nthr, B.e_unit_inv, B.ithr, B.nthr) : Acc(beta);
}

// ---------------------------------------------------------------------------
// the single-site Metropolis update
// ---------------------------------------------------------------------------
// Energy: E = sum_i [ 1/2 sum_l s_i^T J_il s_j(i,l) + sum_a D_a s_ia^2 - h s_i,axis ]
// (axis z for Heisenberg, x for XY; Ising s = sigma*S).  Proposal: reflection
// s' = s - 2 (s.r) r with r uniform on the sphere / circle
// (heisenbergLib.c:441-473, xyLib.c:382-409); Ising: flip (isingLib.c:238-254).
// Accept if beta*dE <= 0 or u < exp(-beta*dE).  Accepted O(n) spins are
// renormalised to |S|.
// Random words: w_a = r_z (Heisenberg), w_b = phi (XY, Heisenberg),
// w_c = acceptance.
// UNI: every link of the graph carries the tensor at coup (a uniform
// graph); the field is that tensor times the sum of the neighbour spins.
// aniso = false: no site class has an on-site term (D = 0), so the D terms,
// each an exact +0 to dE, are skipped.
// the field: H = J . S of a uniform graph's neighbour sum, or one link's
// J . t added to H (row-major J, the same operations in every kernel)
template <int NC, typename CP>
__device__ __forceinline__ void uniform_field(CP J, const float* S, float* H) {
  H[0] = J[0] * S[0]; H[0] = fmaf(J[1], S[1], H[0]);
  H[1] = J[3] * S[0]; H[1] = fmaf(J[4], S[1], H[1]);
  if constexpr (NC == 3) {
    H[0] = fmaf(J[2], S[2], H[0]);
    H[1] = fmaf(J[5], S[2], H[1]);
    H[2] = J[6] * S[0]; H[2] = fmaf(J[7], S[1], H[2]); H[2] = fmaf(J[8], S[2], H[2]);
  }
}
template <int NC, typename CP>
__device__ __forceinline__ void add_field(CP J, const float* t, float* H) {
  H[0] = fmaf(J[0], t[0], H[0]); H[0] = fmaf(J[1], t[1], H[0]);
  if constexpr (NC == 3) H[0] = fmaf(J[2], t[2], H[0]);
  H[1] = fmaf(J[3], t[0], H[1]); H[1] = fmaf(J[4], t[1], H[1]);
  if constexpr (NC == 3) {
    H[1] = fmaf(J[5], t[2], H[1]);
    H[2] = fmaf(J[6], t[0], H[2]); H[2] = fmaf(J[7], t[1], H[2]); H[2] = fmaf(J[8], t[2], H[2]);
  }
}

// An update in its pieces, so that the sites of one draw can go through them
// together: the field (site and neighbour spins), then the proposal and its
// decision, then the store.
//
// the proposed axis of an O(n) reflection
template <int NC>
__device__ __forceinline__ void metro_axis(uint32_t w_a, uint32_t w_b, float* r) {
  if constexpr (NC == 3) {
    r[2] = fmaf((float)(w_a >> 8), 0x1p-23f, -1.0f);
    const float rho = unit_rho(r[2]);
    float c, sn;
    sincos_turn(w_b, &c, &sn);
    r[0] = rho * c;
    r[1] = rho * sn;
  } else {
    sincos_turn(w_b, r, r + 1);
    r[2] = 0.0f;
  }
}

// the O(n) decision: s the site's spin, H its field, r the axis; n gets the
// reflected spin (not renormalised), dE the energy change.  D: on-site terms
// (aniso = false: none).
template <int NC>
__device__ __forceinline__ bool metro_decide(const float* s, const float* H, const float* r, float beta, float h,
                                             bool aniso, const float* D, uint32_t w_c, float* n, float& dE) {
  float p = s[0] * r[0];
  p = fmaf(s[1], r[1], p);
  if constexpr (NC == 3) p = fmaf(s[2], r[2], p);
  const float a = -2.0f * p;
  const float d0 = a * r[0], d1 = a * r[1], d2 = NC == 3 ? a * r[2] : 0.0f;
  dE = d0 * H[0];
  dE = fmaf(d1, H[1], dE);
  if constexpr (NC == 3) dE = fmaf(d2, H[2], dE);
  n[0] = s[0] + d0;
  n[1] = s[1] + d1;
  if constexpr (NC == 3) n[2] = s[2] + d2;
  if (aniso) {
    const float a0 = n[0] * n[0], b0 = s[0] * s[0], q0 = a0 - b0;
    const float a1 = n[1] * n[1], b1 = s[1] * s[1], q1 = a1 - b1;
    dE = fmaf(D[0], q0, dE);
    dE = fmaf(D[1], q1, dE);
    if constexpr (NC == 3) {
      const float a2 = n[2] * n[2], b2 = s[2] * s[2], q2 = a2 - b2;
      dE = fmaf(D[2], q2, dE);
    }
  }
  dE = fmaf(-h, NC == 3 ? d2 : d0, dE);  // h = 0 adds an exact 0
  const float db = dE * beta;
  return (db <= 0.0f) | below_exp(w_c, -db);  // no branch: some lane of a wave needs the exponential
}

// the accepted spin, renormalised, as stored; its change goes to dM
template <int NC, typename ST>
__device__ __forceinline__ void metro_commit(const float* s, float* n, float is2, float* dMacc) {
  float nn = n[0] * n[0];
  nn = fmaf(n[1], n[1], nn);
  if constexpr (NC == 3) nn = fmaf(n[2], n[2], nn);
  const float f = renorm_factor(nn, is2);
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    n[k] *= f;
    // FP32 storage keeps the value as computed; FP16 rounds it
    if constexpr (std::is_same<ST, __half>::value)
      dMacc[k] += __half2float(__float2half_rn(n[k])) - s[k];
    else
      dMacc[k] += n[k] - s[k];
  }
}

// Ising: the decision for sigma = sg, spin s = sg*S and field f
__device__ __forceinline__ bool ising_decide(float s, float f, float h, const Acc& ac, uint32_t w_c, float& dE) {
  const float t = f - h;
  dE = (-2.0f * s) * t;
  if (ac.lds) {  // as below; downhill flips read entry 0 and ignore it
    const uint32_t x = ac.lds[max((int)(dE * ac.inv_unit), 0)];
    return (dE <= 0.0f) | (w_c < x);
  }
  if (ac.thr)
    // exact: couplings, fields and spin lengths are multiples of powers of
    // two small enough that every operation above is exact, dE = k u with
    // 0 < k < nthr, and thr[k] = floor(2^32 exp(-beta k u))
    return dE <= 0.0f || w_c < ac.thr[(int)(dE * ac.inv_unit)];
  const float db = dE * ac.beta;
  return (db <= 0.0f) | below_exp(w_c, -db);
}

// One Philox draw (128 bits) serves G sites of a colour class: 4 Ising
// updates (one acceptance word each), 2 XY updates (angle + acceptance), or
// 1 Heisenberg update (r_z, angle, acceptance).  Group q of colour c covers
// colour-list positions q*G .. q*G+G-1; counter (q, sweep, c<<8 | TAG).
template <int NC>
struct SitesPerDraw {
  static constexpr int G = NC == 1 ? 4 : NC == 2 ? 2 : 1;
};

// One replica's spins, in LDS or in HBM: a site's place, and loads and stores
// at a byte offset from it.  In LDS a place is one address per component (a
// vector add to reach a neighbour's).  In HBM it is a 32-bit offset from
// scalar bases, so that a neighbour's components share one add; 64-bit
// addresses per lane took 6.5 instructions a link.
template <int NC, typename ST>
struct LdsView {
  typedef ST value_type;
  ST* p;
  int n;
  struct Site {
    char* a[NC];
  };
  __device__ __forceinline__ Site at(int i) const {
    Site s;
#pragma unroll
    for (int k = 0; k < NC; ++k) s.a[k] = (char*)(p + i) + k * n * (int)sizeof(ST);
    return s;
  }
  __device__ __forceinline__ Site base() const { return at(0); }
  static __device__ __forceinline__ float ld(const Site& s, int k, int off) { return SIO<ST>::ld((const ST*)(s.a[k] + off)); }
  static __device__ __forceinline__ void st(const Site& s, int k, float v) { SIO<ST>::st((ST*)s.a[k], v); }
};
template <int NC, typename ST>
struct HbmView {
  typedef ST value_type;
  GAS ST* p[NC];
  typedef uint32_t Site;
  __device__ __forceinline__ HbmView(GAS ST* p0, int n) {
    // separate scalar bases: the compiler would fold the component stride
    // into each lane's address
    for (int c = 0; c < NC; ++c) {
      p[c] = p0 + (size_t)c * n;
      asm("" : "+s"(p[c]));
    }
  }
  __device__ __forceinline__ Site at(int i) const { return (uint32_t)i * (uint32_t)sizeof(ST); }
  __device__ __forceinline__ Site base() const { return 0; }
  __device__ __forceinline__ float ld(const Site& s, int k, int off) const {
    return SIO<ST>::ld((const GAS ST*)((const GAS char*)p[k] + (s + (uint32_t)off)));
  }
  __device__ __forceinline__ void st(const Site& s, int k, float v) const { SIO<ST>::st((GAS ST*)((GAS char*)p[k] + s), v); }
};
// spins in HBM read by site: the same 32-bit offsets from scalar bases
template <int NC, typename ST>
struct HbmSpins {
  typedef ST value_type;
  HbmView<NC, ST> v;
  __device__ __forceinline__ HbmSpins(ST* p, int n) : v(gas(p), n) {}
  __device__ __forceinline__ float get(int i, int c) const { return v.ld(v.at(i), c, 0); }
};

// What the updates of a sweep read besides spins and draws.  Neighbours come
// from link patterns (rows in LDS, pat: the row of each position) or from the
// global link table (link, lcid).  coup (cst floats a tensor), clsdat: LDS or
// HBM.  With one coupling or one site class their values are kept in
// registers: read where they are used, each update would wait for them.
template <int NC, typename PP, typename KP, typename CP>
struct SweepTab {
  const int32_t* rows;
  int stride;  // bytes per row
  PP pat;
  const GAS uint32_t* link;
  const GAS int32_t *lcid, *cls;
  KP coup;
  int cst;
  CP clsdat;
  int zmax;
  bool aniso, one;  // any on-site term; one site class
  float J[9];       // the coupling of a uniform graph
  float cls0[5];    // the one class: S, D, 1/S^2
};
template <int NC, bool UNI, typename PP, typename KP, typename CP, typename JP>
__device__ __forceinline__ SweepTab<NC, PP, KP, CP> sweep_tab(const mcg_graph& G, const int32_t* rows, PP pat, KP coup,
                                                              int cst, JP ucoup, CP clsdat, bool aniso) {
  SweepTab<NC, PP, KP, CP> T;
  T.rows = rows;
  T.stride = pat_stride(G.zmax) * 4;
  T.pat = pat;
  T.link = gas(G.link);
  T.lcid = G.lcid ? gas(G.lcid) : nullptr;
  T.cls = gas(G.cls);
  T.coup = coup;
  T.cst = cst;
  T.clsdat = clsdat;
  T.zmax = G.zmax;
  T.aniso = aniso;
  T.one = G.ncls == 1;
  if constexpr (UNI)
    for (int k = 0; k < 9; ++k) T.J[k] = in_vgpr(ucoup[k]);
  for (int k = 0; k < 5; ++k) T.cls0[k] = in_vgpr(clsdat[k]);
  return T;
}

// four words of a pattern row
__device__ __forceinline__ void read_row(const int32_t* row, int32_t* x) {
  const int4 a = *(const int4*)row;
  x[0] = a.x;
  x[1] = a.y;
  x[2] = a.z;
  x[3] = a.w;
}
// the field of a uniform graph from the sum of the neighbour spins
template <int NC, typename T>
__device__ __forceinline__ void sum_field(const T& tab, const float* S, float* H) {
  if constexpr (NC == 1)
    H[0] = tab.J[0] * S[0];
  else
    uniform_field<NC>(tab.J, S, H);
}

// one coupling of a graph of several: 128-bit reads from LDS
template <int NC>
__device__ __forceinline__ void read_coup(const float* c, float* J) {
  if constexpr (NC == 1) {
    J[0] = c[0];
  } else {
    const float4 a = *(const float4*)c, b = *(const float4*)(c + 4);
    J[0] = a.x; J[1] = a.y; J[2] = a.z; J[3] = a.w; J[4] = b.x;
    if constexpr (NC == 3) {
      J[5] = b.y; J[6] = b.z; J[7] = b.w; J[8] = c[8];
    }
  }
}
template <int NC>
__device__ __forceinline__ void read_coup(const GAS float* c, float* J) {
#pragma unroll
  for (int k = 0; k < (NC == 1 ? 1 : NC == 2 ? 5 : 9); ++k) J[k] = c[k];
}

// the next B link words of a site from link l on: pattern row words, or the
// link table's (neighbour | coupling << 24)
template <bool PAT, int B, typename T>
__device__ __forceinline__ void link_words(const T& tab, const int32_t* row, const GAS uint32_t* lk, int l, int zmax,
                                           int32_t* w) {
  if constexpr (PAT) {
#pragma unroll
    for (int u = 0; u < B; u += 4) read_row(row + l + u, w + u);
  } else {
#pragma unroll
    for (int u = 0; u < B; ++u) w[u] = (int32_t)lk[l + u < zmax ? l + u : zmax - 1];
  }
}
// the neighbour of a link word
template <bool PAT, bool UNI, typename V>
__device__ __forceinline__ float link_spin(const V& v, const typename V::Site& own, int32_t w, int k) {
  typedef typename V::value_type ST;
  if constexpr (PAT)
    return v.ld(own, k, UNI ? w : (w >> 8) * (int)sizeof(ST));
  else
    return v.ld(v.base(), k, (int)(((uint32_t)w & 0xFFFFFFu) * (uint32_t)sizeof(ST)));
}

// Field of the site at `own` (its pattern row, or its link table row lk and
// coupling row lc): every neighbour is read before the first is used.  Z: the
// number of links, or 0 where it is only known at run time (then four links
// at a time).
template <int NC, bool PAT, bool UNI, int Z, typename V, typename T>
__device__ __forceinline__ void site_field(const V& v, const typename V::Site& own, const int32_t* row,
                                           const GAS uint32_t* lk, const GAS int32_t* lc, const T& tab, float* H) {
  constexpr int B = Z == 0 ? 4 : Z == 9 ? 3 : Z;  // links per batch
  const int zmax = Z > 0 ? Z : tab.zmax;
  float S[3] = {0.0f, 0.0f, 0.0f};
  H[0] = H[1] = H[2] = 0.0f;
  int32_t rw[Z > 0 ? (Z + 3) / 4 * 4 : 4];
  if constexpr (Z > 0) link_words<PAT, Z>(tab, row, lk, 0, Z, rw);
  for (int l0 = 0; l0 < zmax; l0 += B) {
    int32_t w[B];
    if constexpr (Z == 0) link_words<PAT, 4>(tab, row, lk, l0, zmax, rw);
    uint32_t c[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      w[u] = rw[Z > 0 ? l0 + u : u];
      if (PAT && Z == 0 && l0 + u >= zmax) w[u] = 0;  // past the last link: the site itself, not used
      if constexpr (!UNI)
        c[u] = PAT ? (uint32_t)w[u] & 0xFFu
                   : lc ? (uint32_t)lc[l0 + u < zmax ? l0 + u : zmax - 1] : (uint32_t)w[u] >> 24;
    }
    float t[B][NC];
#pragma unroll
    for (int u = 0; u < B; ++u)
#pragma unroll
      for (int k = 0; k < NC; ++k) t[u][k] = link_spin<PAT, UNI>(v, own, w[u], k);
    if constexpr (UNI) {
#pragma unroll
      for (int u = 0; u < B; ++u) {
        if (Z == 0 && l0 + u >= zmax) break;
#pragma unroll
        for (int k = 0; k < NC; ++k) S[k] += t[u][k];
      }
    } else {
      // each link's tensor is read while the one before it is used (all at
      // once would take 9 registers a link)
      float J[2][9];
      read_coup<NC>(tab.coup + c[0] * tab.cst, J[0]);
#pragma unroll
      for (int u = 0; u < B; ++u) {
        if (u + 1 < B && (Z > 0 || l0 + u + 1 < zmax)) read_coup<NC>(tab.coup + c[u + 1] * tab.cst, J[(u + 1) & 1]);
        if (Z == 0 && l0 + u >= zmax) break;
        if constexpr (NC == 1)
          H[0] = fmaf(J[u & 1][0], t[u][0], H[0]);
        else
          add_field<NC>(J[u & 1], t[u], H);
        // keep the sum here: sunk to where H is used, it would hold every
        // link's tensor and spin in registers until then
        asm volatile("" : "+v"(H[0]), "+v"(H[1]), "+v"(H[2]));
      }
    }
  }
  if constexpr (UNI) sum_field<NC>(tab, S, H);
}

// The sites of one draw: group q of a colour class of cnt positions from b
// on.  They share a colour, so none is another's neighbour: all fields are
// read, then all decisions taken, then the accepted spins stored, and the
// sites' loads overlap instead of each site waiting for its own chain.
// Changes are added in site order.  PAT: neighbours from link patterns,
// otherwise from the link table.
template <int NC, bool PAT, bool UNI, int Z, typename V, typename T>
__device__ __forceinline__ void metro_sites(const V& v, int b, int cnt, int q, int colour, const T& tab, const Acc& ac,
                                            float h, uint64_t sweep, uint32_t key0, uint32_t key1, float& dEacc,
                                            float* dMacc) {
  typedef typename V::value_type ST;
  constexpr int G = SitesPerDraw<NC>::G;
  typename V::Site own[G];
  float s[G][3], H[G][3];
  const int32_t* row[G];
  const GAS uint32_t* lk[G];
  const GAS int32_t* lc[G];
  int cl[G];
  bool live[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int lp = q * G + g;
    live[g] = lp < cnt;  // the last group may be short: its missing sites read the last one
    const int p = b + (G == 1 || live[g] ? lp : cnt - 1);
    cl[g] = 0;
    if constexpr (PAT) {
      row[g] = (const int32_t*)((const char*)tab.rows + __umul24((uint32_t)tab.pat[p], (uint32_t)tab.stride));
      lk[g] = nullptr;
      lc[g] = nullptr;
    } else {
      const int z = Z > 0 ? Z : tab.zmax;
      row[g] = nullptr;
      lk[g] = tab.link + (uint32_t)p * (uint32_t)z;
      lc[g] = tab.lcid ? tab.lcid + (uint32_t)p * (uint32_t)z : nullptr;
      if (Z == 0 && !tab.one) cl[g] = tab.cls[p] * 8;
    }
    own[g] = v.at(p);
#pragma unroll
    for (int k = 0; k < NC; ++k) s[g][k] = v.ld(own[g], k, 0);
  }
  if constexpr (UNI && Z > 0) {
    // every site's links, then every neighbour, then the sums
    int32_t w[G][(Z + 3) / 4 * 4];
    float t[G][Z][NC];
#pragma unroll
    for (int g = 0; g < G; ++g) link_words<PAT, Z>(tab, row[g], lk[g], 0, Z, w[g]);
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int u = 0; u < Z; ++u)
#pragma unroll
        for (int k = 0; k < NC; ++k) t[g][u][k] = link_spin<PAT, true>(v, own[g], w[g][u], k);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float S[3] = {t[g][0][0], NC > 1 ? t[g][0][NC > 1 ? 1 : 0] : 0.0f, NC > 2 ? t[g][0][NC > 2 ? 2 : 0] : 0.0f};
#pragma unroll
      for (int u = 1; u < Z; ++u)
#pragma unroll
        for (int k = 0; k < NC; ++k) S[k] += t[g][u][k];
      sum_field<NC>(tab, S, H[g]);
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (PAT && Z == 0 && !tab.one) cl[g] = row[g][tab.zmax] * 8;
      site_field<NC, PAT, UNI, Z>(v, own[g], row[g], lk[g], lc[g], tab, H[g]);
    }
  }
  const u32x4 x = philox4x32_10(
      u32x4{(uint32_t)q, (uint32_t)sweep, (uint32_t)(sweep >> 32), TAG_METRO | ((uint32_t)colour << 8)}, key0, key1);
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
  float n[G][3], dE[G], is2[G];
  bool acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float c[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) c[k] = tab.cls0[k];
    if (Z == 0 && !tab.one)
#pragma unroll
      for (int k = 0; k < 5; ++k) c[k] = tab.clsdat[cl[g] + k];
    if constexpr (NC == 1) {
      n[g][0] = s[g][0] * c[0];  // the spin sigma*S
      acc[g] = ising_decide(n[g][0], H[g][0], h, ac, w[g], dE[g]) & live[g];
    } else {
      float r[3];
      metro_axis<NC>(NC == 3 ? w[0] : 0u, NC == 3 ? w[1] : w[2 * g], r);
      acc[g] = metro_decide<NC>(s[g], H[g], r, ac.beta, h, tab.aniso, c + 1, NC == 3 ? w[2] : w[2 * g + 1], n[g],
                                dE[g]) & live[g];
      is2[g] = c[4];
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g)
    if (acc[g]) {
      dEacc += dE[g];
      if constexpr (NC == 1) {
        v.st(own[g], 0, -s[g][0]);
        dMacc[0] += -2.0f * n[g][0];
      } else {
        metro_commit<NC, ST>(s[g], n[g], is2[g], dMacc);
#pragma unroll
        for (int k = 0; k < NC; ++k) v.st(own[g], k, n[g][k]);
      }
    }
}

// f(Z) with the link count a compile-time constant for graphs of one site
// class with a common count: square (4), triangular and cubic (6) lattices,
// honeycomb with second neighbours (9); f(0) for any other
template <bool PAT, bool UNI, typename T, typename F>
__device__ __forceinline__ void with_links(const T& t, F&& f) {
  if (UNI && t.one && t.zmax == 4)
    f(std::integral_constant<int, 4>());
  else if ((PAT || UNI) && t.one && t.zmax == 6)
    f(std::integral_constant<int, 6>());
  else if (PAT && !UNI && t.one && t.zmax == 9)
    f(std::integral_constant<int, 9>());
  else
    f(std::integral_constant<int, 0>());
}

// spin vector of site i (Ising: sigma*S)
template <int NC, typename SV>
__device__ __forceinline__ void spin_vec(const SV& sp, int i, const int32_t* __restrict__ cls, const float* clsdat,
                                         float* v) {
  if constexpr (NC == 1) {
    v[0] = sp.get(i, 0) * clsdat[cls ? cls[i] * 8 : 0];  // no cls: one class
    v[1] = v[2] = 0.0f;
  } else {
    v[0] = sp.get(i, 0);
    v[1] = sp.get(i, 1);
    v[2] = NC == 3 ? sp.get(i, 2) : 0.0f;
  }
}

// per-site energy e_i (FP32): 1/2 s_i.H_i + onsite - h s_axis
template <int NC, typename SV>
__device__ __forceinline__ float site_energy(const SV& sp, int i, const uint32_t* __restrict__ link,
                                             const int32_t* __restrict__ lcid, int zmax, const float* coup, int cst,
                                             const int32_t* __restrict__ cls, const float* clsdat, float h) {
  const int ci = cls[i];
  const GlobalLinks lk{gas(link) + (size_t)i * zmax, lcid ? gas(lcid) + (size_t)i * zmax : nullptr};
  if constexpr (NC == 1) {
    float f = 0.0f;
    for (int l = 0; l < zmax; ++l) f = fmaf(coup[lk.cid(l) * cst], sp.get(lk.nbr(l), 0), f);
    const float s = sp.get(i, 0) * clsdat[ci * 8];
    return fmaf(0.5f * s, f, -h * s);
  } else {
    const float s0 = sp.get(i, 0), s1 = sp.get(i, 1), s2 = NC == 3 ? sp.get(i, 2) : 0.0f;
    float H0 = 0.0f, H1 = 0.0f, H2 = 0.0f;
    for (int l = 0; l < zmax; ++l) {
      const int j = lk.nbr(l);
      const float* J = coup + lk.cid(l) * cst;
      const float t0 = sp.get(j, 0), t1 = sp.get(j, 1), t2 = NC == 3 ? sp.get(j, 2) : 0.0f;
      H0 = fmaf(J[0], t0, H0); H0 = fmaf(J[1], t1, H0); H0 = fmaf(J[2], t2, H0);
      H1 = fmaf(J[3], t0, H1); H1 = fmaf(J[4], t1, H1); H1 = fmaf(J[5], t2, H1);
      H2 = fmaf(J[6], t0, H2); H2 = fmaf(J[7], t1, H2); H2 = fmaf(J[8], t2, H2);
    }
    float e = s0 * H0;
    e = fmaf(s1, H1, e);
    e = fmaf(s2, H2, e);
    e = 0.5f * e;
    e = fmaf(clsdat[ci * 8 + 1] * s0, s0, e);
    e = fmaf(clsdat[ci * 8 + 2] * s1, s1, e);
    if constexpr (NC == 3) e = fmaf(clsdat[ci * 8 + 3] * s2, s2, e);
    e = fmaf(-h, NC == 3 ? s2 : s0, e);
    return e;
  }
}

// ---------------------------------------------------------------------------
// group reductions (a group = TPR consecutive threads, TPR a multiple of 64)
// ---------------------------------------------------------------------------
// accesses at the device coherence point (device-scope atomics): visible to
// every workgroup of the launch whatever XCD it runs on
template <typename T>
__device__ __forceinline__ void dev_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T dev_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void dev_add(double* p, double v) { unsafeAtomicAdd(p, v); }

static constexpr int RK = 12;  // most values per reduction call
static constexpr int FRM_ACC = 96;       // frame scratch: accumulator staging starts here
static constexpr int FRM = FRM_ACC + 48;  // frame scratch doubles per group: scalars, then accumulator staging

// FP64 value moved across lanes by DPP (two 32-bit halves); lanes of rows
// outside ROWMASK get 0.  With every row enabled (the quad permutes and row
// mirrors used here, where each lane reads a lane of its own row) there is
// no old value to keep, so the destination is not zeroed first: those two
// moves per step were a third of the instructions of a wave's FP64 sum,
// which all waves of a workgroup run at once at the end of every sweep.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_f64(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  int l2, h2;
  if constexpr (ROWMASK == 0xF) {
    l2 = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, true);
    h2 = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, true);
  } else {
    l2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWMASK, 0xF, false);
    h2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROWMASK, 0xF, false);
  }
  return __hiloint2double(h2, l2);
}

// sum over the 64 lanes of a wave (every lane active); the total lands in
// lane 63.  Quad swaps, half-row and row mirrors give every lane its 16-lane
// row sum; row broadcasts 15 and 31 then add the rows up.  DPP moves are
// VALU operations: no LDS traffic, unlike a shuffle butterfly.
__device__ __forceinline__ double wave_sum_f64(double x) {
  x += dpp_f64<0xB1, 0xF>(x);   // quad_perm [1,0,3,2]
  x += dpp_f64<0x4E, 0xF>(x);   // quad_perm [2,3,0,1]
  x += dpp_f64<0x141, 0xF>(x);  // row_half_mirror
  x += dpp_f64<0x140, 0xF>(x);  // row_mirror
  x += dpp_f64<0x142, 0xA>(x);  // row_bcast:15 into rows 1, 3
  x += dpp_f64<0x143, 0xC>(x);  // row_bcast:31 into rows 2, 3
  return x;
}

// The thread's index, read anew: the reductions and frames sit inside the
// sweep loop, and what the compiler derives from the plain index (addresses,
// masks) it computes before the loop and keeps, spilled, across the sweeps.
__device__ __forceinline__ int tid() {
  int x = (int)threadIdx.x;
  asm volatile("" : "+v"(x));
  return x;
}

// x summed over lanes l and l ^ 16, or l and l ^ 32
__device__ __forceinline__ double add_lane16(double x) {
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(x), (uint32_t)__double2loint(x), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(x), (uint32_t)__double2hiint(x), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double add_lane32(double x) {
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(x), (uint32_t)__double2loint(x), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(x), (uint32_t)__double2hiint(x), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// Totals of N values over the 64 lanes (every lane active): lane l gets in
// r[j] the total of value 4 j + (l & 3).  The first two steps halve the
// number of values with the number of lanes each still has to cover (a lane
// keeps one of two values and sends the other), so that four values take 7
// FP64 additions a lane instead of 24.
template <int N>
__device__ __forceinline__ void wave_totals(const double* v, double* r) {
  const int tx = tid();
  const bool b0 = (tx & 1) != 0, b1 = (tx & 2) != 0;
#pragma unroll
  for (int j = 0; 4 * j < N; ++j) {
    const double a = v[4 * j], b = 4 * j + 1 < N ? v[4 * j + 1] : 0.0;
    const double c = 4 * j + 2 < N ? v[4 * j + 2] : 0.0, d = 4 * j + 3 < N ? v[4 * j + 3] : 0.0;
    const double x = (b0 ? b : a) + dpp_f64<0xB1, 0xF>(b0 ? a : b);  // quad_perm [1,0,3,2]
    const double y = (b0 ? d : c) + dpp_f64<0xB1, 0xF>(b0 ? c : d);
    double t = (b1 ? y : x) + dpp_f64<0x4E, 0xF>(b1 ? x : y);  // quad_perm [2,3,0,1]
    t += dpp_f64<0x124, 0xF>(t);                               // row_ror:4
    t += dpp_f64<0x128, 0xF>(t);                               // row_ror:8
    r[j] = add_lane32(add_lane16(t));
  }
}

// lane src's value (src the same in every lane), in every lane of the wave
__device__ __forceinline__ double lane_f64(double x, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), src);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane63(double x) { return lane_f64(x, 63); }

// LDS written by a wave's lanes is read by other lanes of it after this
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Totals of N (<= RK) values over the TPR threads of group g (TPR a multiple
// of 64): sink(k, total of v[k]) is called once per value, by lane k of the
// group's first wave, then post() by that whole wave.  All threads call it;
// it ends with a workgroup barrier.  Each wave's totals go through LDS (lanes
// 16 p + k of the first wave add value k of waves p, p + 4, ...).
template <int N, typename F, typename P>
__device__ __forceinline__ void group_add(const double* v, double* s_red, int g, int TPR, F&& sink, P&& post) {
  constexpr int M = (N + 3) / 4;
  double r[M];
  wave_totals<N>(v, r);
  const int tx = tid(), lane = tx & 63, wave = tx >> 6;
  const int nw = TPR >> 6;
  if (nw == 1) {  // the same for every group of the workgroup
#pragma unroll
    for (int j = 0; j < M; ++j)
      if (lane < 4 && 4 * j + lane < N) sink(4 * j + lane, r[j]);
    wave_lds_fence();
    post();
    __syncthreads();
    return;
  }
  if (lane < 4)
#pragma unroll
    for (int j = 0; j < M; ++j) s_red[wave * RK + 4 * j + lane] = r[j];
  __syncthreads();
  const int w0 = g * nw;
  if (wave == w0) {
    const int k = lane & 15;
    double x = 0.0;
    if (k < N)
      for (int w = lane >> 4; w < nw; w += 4) x += s_red[(w0 + w) * RK + k];
    x = add_lane32(add_lane16(x));
    if (lane < N) sink(lane, x);
    wave_lds_fence();
    post();
  }
  __syncthreads();
}
template <int N, typename F>
__device__ __forceinline__ void group_add(const double* v, double* s_red, int g, int TPR, F&& sink) {
  group_add<N>(v, s_red, g, TPR, sink, [] {});
}

// ---------------------------------------------------------------------------
// measurement of one frame (all flagged observables) for one replica
// ---------------------------------------------------------------------------
struct FrameCtx {
  const mcg_graph* G;  // in device memory
  const float* coup;
  int cst;         // floats per coupling
  const float* clsdat;
  double* s_red;   // reduction scratch (nwaves*RK)
  double* s_frm;   // per-group frame values (>= 64 doubles per group)
  int g, lt, TPR;
  double inv_n, inv_nlat, inv_nf;  // 1 / sites, 1 / correlation pairs (or sites), 1 / planned frames
  int last;                        // position of the last site
  float* blk;                      // the group's block spins (LDS, nr x NC), or nullptr
};
template <int NC>
__device__ __forceinline__ void frame_consts(FrameCtx& C, const mcg_graph& G, const mcg_batch& B) {
  // (scalars: they live across the sweeps)
  C.inv_n = wave_uniform(1.0 / (double)G.n);
  C.inv_nlat = wave_uniform(1.0 / (double)(G.nlat > 0 ? G.nlat : G.n));
  C.inv_nf = wave_uniform(1.0 / (double)(B.nframes > 0 ? B.nframes : 1));
  C.last = G.pos[G.n - 1];
  C.blk = nullptr;
}
// a frame's spin-derived sums need no pass over the spins: nothing but self
// pairs, whose sums follow from the tracked state
__device__ __forceinline__ bool frame_light(const mcg_graph& G, int flags) {
  return !(flags & (MCG_MEAS_Q | MCG_MEAS_RNORM | MCG_MEAS_GROUPS)) &&
         (!(flags & MCG_MEAS_PAIRS) || G.nlat <= 0 || G.self_pairs);
}

// Frames and recomputes sit inside the sweep loop.  Left to itself the
// compiler keeps everything they read (some 60 words of the graph, an address
// per loop and thread) in registers across the sweeps, and spills what the
// sweeps need.  fresh reads the graph again where it is needed (scalar loads);
// opaque hides a thread index, so that nothing computed from it is moved out
// of the loop.
__device__ __forceinline__ mcg_graph fresh(const mcg_graph* G) {
  const uint64_t x = (uint64_t)G;
  uint32_t lo = (uint32_t)wave_uniform((int)x), hi = (uint32_t)wave_uniform((int)(x >> 32));
  asm volatile("" : "+s"(lo), "+s"(hi));
  const uint64_t a = (uint64_t)hi << 32 | lo;
  return *(const mcg_graph*)(const __attribute__((address_space(4))) mcg_graph*)a;
}
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// majority spin of block-spin site `site`, whose cluster is row ri of rclu
// (heisenbergLib.c:255-267, isingLib.c:133-150); cls: nullptr with one class
template <int NC, typename SV>
__device__ __forceinline__ void majority(const SV& sp, const mcg_graph& G, const int32_t* cls, const float* clsdat,
                                         int ri, int site, uint64_t frame, uint32_t key0, uint32_t key1, float* v) {
  float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
  for (int k0 = 0; k0 < G.nclu; k0 += 4) {
    // four cluster sites at a time, all read before they are added
    float t[4][3];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      spin_vec<NC>(sp, G.rclu[ri * G.nclu + (k0 + u < G.nclu ? k0 + u : G.nclu - 1)], cls, clsdat, t[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (k0 + u >= G.nclu) break;
      a0 += t[u][0];
      a1 += t[u][1];
      a2 += t[u][2];
    }
  }
  const float S = clsdat[cls ? cls[site] * 8 : 0];
  if constexpr (NC == 1) {
    float sg;
    if (a0 > 0.0f)
      sg = 1.0f;
    else if (a0 < 0.0f)
      sg = -1.0f;
    else {
      const u32x4 x = philox4x32_10(u32x4{(uint32_t)site, (uint32_t)frame, (uint32_t)(frame >> 32), TAG_MAJORITY},
                                    key0, key1);
      sg = u24(x.x) > 0.5f ? 1.0f : -1.0f;
    }
    v[0] = sg * fabsf(S);
    v[1] = v[2] = 0.0f;
  } else {
    const float l = sqrtf(a0 * a0 + a1 * a1 + a2 * a2);
    if (l >= 1e-5f) {
      a0 /= l;
      a1 /= l;
      a2 /= l;
    }
    v[0] = a0 * S;
    v[1] = a1 * S;
    v[2] = a2 * S;
  }
}
// the block spin of index ri computed earlier in this frame
template <int NC>
__device__ __forceinline__ void block_spin(const float* blk, int ri, float* v) {
  v[0] = blk[ri * NC];
  v[1] = NC > 1 ? blk[ri * NC + (NC > 1 ? 1 : 0)] : 0.0f;
  v[2] = NC > 2 ? blk[ri * NC + (NC > 2 ? 2 : 0)] : 0.0f;
}

// solid angle of a spin triangle, heisenbergLib.c:114-127 (atan, +-pi branch)
// (ia, ib, ic: 1/|S| of the three sites).  An observable, compared within
// statistics: products with reciprocal lengths and one fast division stand
// in for the reference's seven divisions.
__device__ __forceinline__ float signed_area(const float* a, const float* b, const float* c, float ia, float ib,
                                             float ic) {
  const float ab = (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]) * (ia * ib);
  const float bc = (b[0] * c[0] + b[1] * c[1] + b[2] * c[2]) * (ib * ic);
  const float ca = (c[0] * a[0] + c[1] * a[1] + c[2] * a[2]) * (ic * ia);
  const float x0 = b[1] * c[2] - b[2] * c[1], x1 = b[2] * c[0] - b[0] * c[2], x2 = b[0] * c[1] - b[1] * c[0];
  const float re = 1.0f + ab + bc + ca;
  const float im = (a[0] * x0 + a[1] * x1 + a[2] * x2) * (ia * ib * ic);
  if (fabsf(re) < 1e-6f) return im > 0.0f ? (float)REF_PI : -(float)REF_PI;
  return 2.0f * atanf(__fdividef(im, re));
}

// 1/|S| of a site class: sqrt of the stored 1/S^2
__device__ __forceinline__ float inv_len(const float* clsdat, const int32_t* cls, int i) {
  return sqrtf(clsdat[cls[i] * 8 + 4]);
}

// Measures one frame.  Tracked E and M (FP64) of the replica are passed in
// st[]; everything else is computed from the spins.  Only the group leader
// (lt == 0) writes the accumulators.
// Observables taken from the spins themselves (pairs, Q, block spins,
// groups); a kernel compiled without them (FULL = false) is much smaller.
static constexpr int MEAS_SPIN_OBS = MCG_MEAS_PAIRS | MCG_MEAS_Q | MCG_MEAS_RNORM | MCG_MEAS_GROUPS;

template <int NC>
__device__ __forceinline__ int frame_groups(const mcg_graph& G, int flags) {
  return (NC > 1 && (flags & MCG_MEAS_GROUPS)) ? G.ngroup : 0;
}

// apply a frame staged by measure_frame to the accumulators of its row: one
// device-scope FP64 atomic per non-zero term, spread over the group's
// threads.  Fire-and-forget: nothing here waits for the atomics.
template <int NC>
__device__ __forceinline__ void flush_frame(const FrameCtx& C, const mcg_batch& B, int row, int flags) {
  const mcg_graph G = fresh(C.G);
  const int lt = opaque(C.lt), TPR = C.TPR;
  const double* F = C.s_frm;
  const double* Cn = F + FRM_ACC;
  const int ngq = frame_groups<NC>(G, flags);
  double* A = B.acc + (size_t)row * MCG_NACC;
  const int nge = ngq > 0 ? (ngq + 1) * (ngq + 1) : 0;
  // from the group's last thread down: a wave's later loads wait for its
  // atomics, and the last wave has the least of a sweep's work
  for (int q = TPR - 1 - lt; q < MCG_NACC + MCG_NBINQ + nge; q += TPR) {
    if (q < MCG_NACC) {
      if (q != MCG_A_MPREV && Cn[q] != 0.0) dev_add(A + q, Cn[q]);  // adding 0 changes nothing
    } else if (q < MCG_NACC + MCG_NBINQ) {
      const int64_t bin = (int64_t)Cn[MCG_NACC + MCG_NBINQ];
      if (Cn[q] != 0.0) dev_add(B.bins + ((size_t)row * B.nbins + bin) * MCG_NBINQ + (q - MCG_NACC), Cn[q]);
    } else {
      // orbital groups (heisenbergLib.c:805-830): <g_a . g_b> and <(g_a . g_a)^2>
      const int j = q - MCG_NACC - MCG_NBINQ, ga = j / (ngq + 1), gb = j % (ngq + 1);
      double* GA = B.gacc + (size_t)row * ((ngq + 2) * (ngq + 1));
      const double* va = F + 32 + 3 * ga;
      const double* vb = F + 32 + 3 * gb;
      const double d = va[0] * vb[0] + va[1] * vb[1] + va[2] * vb[2];
      dev_add(GA + j, d);
      if (ga == gb) dev_add(GA + (ngq + 1) * (ngq + 1) + ga, d * d);
    }
  }
}

// the previous frame's M of a row (for <M M'>)
__device__ __forceinline__ double frame_mprev(const mcg_batch& B, int row) {
  return dev_load(B.acc + (size_t)row * MCG_NACC + MCG_A_MPREV);
}

// One frame's contribution to every FP64 accumulator of a row
// (isingLib.c:388-431, heisenbergLib.c:677-830 / xyLib.c:605-757), staged in
// Cn for flush_frame: [0, NACC) accumulators ([MM] holds M itself until the
// frame's M' product replaces it), [NACC, +NBINQ) the bin terms, then the bin
// index.  st: the replica's state; F: the frame's spin-derived values.  One
// thread per replica; Cn is zero before (zero_terms).
static constexpr int NTERMS = MCG_NACC + MCG_NBINQ + 1;
__device__ __forceinline__ void zero_terms(double* s_frm, int R) {  // by one wave, for R groups
  const int lane = tid() & 63;
  for (int r = 0; r < R; ++r)
    if (lane < NTERMS) s_frm[r * FRM + FRM_ACC + lane] = 0.0;
  wave_lds_fence();
}
template <int NC>
__device__ __forceinline__ void frame_terms(const FrameCtx& C, const mcg_graph& G, const mcg_batch& B, const double* st,
                                            double* F, int flags, int64_t frame, double* Cn) {
  const int ngq = frame_groups<NC>(G, flags);
  const double inv_nLat = C.inv_nlat;
  const bool pairs = (flags & MCG_MEAS_PAIRS) && G.nlat > 0;
  const bool charge = (flags & MCG_MEAS_Q) && NC == 3 && G.ncirc > 0;
  const bool blocks = (flags & MCG_MEAS_RNORM) && G.nr > 0;
  // everything is read before the first term is stored: reads and stores of
  // the same memory stay in order, and one lane would wait for each in turn
  double E = st[MCG_S_E];
  const double Eref = st[MCG_S_EREF];
  const double M0 = st[MCG_S_M], M1 = st[MCG_S_M + 1], M2 = st[MCG_S_M + 2];
  double P[8];  // the pairs' sums
#pragma unroll
  for (int k = 0; k < 8; ++k) P[k] = pairs ? F[k] : 0.0;
  const double q8 = charge ? F[8] : 0.0;
  if (flags & MCG_ISING_RELE) E -= Eref;
  const double e = E * C.inv_n;
  if (pairs && G.self_pairs) {
    // pairs (i, i) over every site: sum s_i is the tracked magnetisation,
    // sum s_i.s_i the sum of the squared spin lengths
    P[0] = P[3] = M0;
    P[1] = P[4] = M1;
    P[2] = P[5] = M2;
    P[6] = G.pair_s2;
  }
  double Mf;
  constexpr int ax = NC == 3 ? 2 : 0;
  if constexpr (NC == 1) {
    Mf = (pairs ? P[0] : M0) * inv_nLat;
    if (pairs) {
      Cn[MCG_A_SI] = fabs(P[0]) * inv_nLat;
      Cn[MCG_A_SJ] = fabs(P[3]) * inv_nLat;
      Cn[MCG_A_SIJ] = P[6] * inv_nLat;
      Cn[MCG_A_LAST] = P[7];
    }
    Cn[MCG_A_TOT] = M0;
  } else {
    const double Mv[3] = {M0, M1, NC == 3 ? M2 : 0.0};
    double dir[3] = {Mv[0], Mv[1], Mv[2]};
    const double ml = sqrt(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2]);
    if (ml >= 1e-5) {
      const double il = 1.0 / ml;
#pragma unroll
      for (int k = 0; k < NC; ++k) dir[k] *= il;
    }
    if (NC == 3 || !pairs)
      Mf = ml * inv_nLat;
    else
      Mf = sqrt(P[0] * P[0] + P[1] * P[1]) * inv_nLat;
    if (pairs) {
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        Cn[MCG_A_SI + k] = fabs(P[k] * inv_nLat);
        Cn[MCG_A_SJ + k] = fabs(P[3 + k] * inv_nLat);
      }
      Cn[MCG_A_SIJ] = P[6] * inv_nLat;
      Cn[MCG_A_ZI] = (dir[0] * P[0] + dir[1] * P[1] + dir[2] * P[2]) * inv_nLat;
      Cn[MCG_A_ZJ] = (dir[0] * P[3] + dir[1] * P[4] + dir[2] * P[5]) * inv_nLat;
      Cn[MCG_A_HI] = P[ax] * inv_nLat;
      Cn[MCG_A_HJ] = P[3 + ax] * inv_nLat;
    }
    Cn[MCG_A_ZT] = (dir[0] * Mv[0] + dir[1] * Mv[1] + dir[2] * Mv[2]) * inv_nLat;
    Cn[MCG_A_HT] = Mv[ax] * inv_nLat;
    if (charge) Cn[MCG_A_Q] = q8 / REF_PI / 4;
    if (blocks) {
      double R[11];
#pragma unroll
      for (int k = 0; k < 11; ++k) R[k] = F[16 + k];
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        Cn[MCG_A_SIR + k] = fabs(R[k] / R[8]);
        Cn[MCG_A_SJR + k] = fabs(R[3 + k] / R[9]);
      }
      Cn[MCG_A_SIJR] = R[6] / R[10];
    }
    // groups: the total (all sites / nLat) is group ng
    if (ngq > 0)
      for (int k = 0; k < 3; ++k) F[32 + 3 * ngq + k] = Mv[k] * inv_nLat;
  }
  if (blocks) {
    const double er = (F[27] / 2 + F[28]) / G.nr;
    Cn[MCG_A_ER] = er;
    Cn[MCG_A_ER2] = er * er;
  }
  Cn[MCG_A_E] = e;
  Cn[MCG_A_E2] = e * e;
  Cn[MCG_A_M] = Mf;
  Cn[MCG_A_M2] = Mf * Mf;
  Cn[MCG_A_M4] = Mf * Mf * Mf * Mf;
  Cn[MCG_A_MM] = Mf;  // applied as A[MM] += A[MPREV] * Mf; A[MPREV] = Mf
  Cn[MCG_A_COUNT] = 1.0;
  Cn[MCG_A_ABSM] = fabs(Mf);
  // bins for error bars: bin = floor(frame * nbins / nframes), from an FP64
  // quotient corrected to the exact integer floor
  const int64_t nf = B.nframes > 0 ? B.nframes : 1;
  const int64_t num = frame * (int64_t)B.nbins;
  int64_t bin = (int64_t)floor((double)num * C.inv_nf);  // corrected to the exact floor below
  if (bin * nf > num) --bin;
  if ((bin + 1) * nf <= num) ++bin;
  if (bin >= B.nbins) bin = B.nbins - 1;
  if (bin < 0) bin = 0;
  Cn[MCG_NACC + 0] = e;
  Cn[MCG_NACC + 1] = e * e;
  Cn[MCG_NACC + 2] = Mf;
  Cn[MCG_NACC + 3] = Mf * Mf;
  Cn[MCG_NACC + 4] = Mf * Mf * Mf * Mf;
  Cn[MCG_NACC + MCG_NBINQ] = (double)bin;
}

// One measured frame of the group's replica at `row`: the observables are
// computed and staged in the group's frame area, <M M'> and M' are brought
// up to date at once (thread MCG_A_MM; mprev, if have_prev, is M' read ahead
// by that thread), and the rest is applied to the accumulators now or, with
// defer, left staged for the caller's flush_frame.
// [lo, hi): share `part` of `np` of a loop over cnt items
__device__ __forceinline__ void slice(int cnt, int part, int np, int& lo, int& hi) {
  lo = (int)((int64_t)cnt * part / np);
  hi = (int)((int64_t)cnt * (part + 1) / np);
}

// The frame's share of one part of a split replica: the correlation pairs
// and circuits whose first site the part owns (indices into G.pairs and
// G.circ, from the split tables), and whether it owns the last site.
struct PartFrame {
  const int32_t* pairs;
  const int32_t* circs;
  int npairs, ncircs;
  bool last;
};

// The spin-derived sums of one frame over share `part` of `np` of every
// loop (pairs, circuits, block spins, groups), left in F (valid in the
// group's first thread): F[0..8) pairs, F[8] solid angles, F[16..29) block
// spins, F[32..) groups.  np = 1: the whole frame.  With `own`, the share
// is instead own's pairs and circuits (their other sites being current in
// the part's copy), and block spins and groups are not measured.
static constexpr int FRAME_TRI = 2;  // triangles in flight per thread
static constexpr int FSUMS = 88;     // frame sums per replica (F[0, 88))
static constexpr int FSUMS_PQ = 9;   // of which pairs and circuits (F[0, 9))
// Inlined wherever it is used: as a call it takes the batch, the graph and the
// replica by address, which keeps them in scratch memory for the whole kernel.
template <int NC, typename SV, bool FULL = true>
__device__ __forceinline__ void frame_sums(const SV& sp, const FrameCtx& C, const mcg_batch& B, int64_t frame, uint32_t key0,
                           uint32_t key1, float h, int part, int np, const PartFrame* own = nullptr) {
  const mcg_graph G = fresh(C.G);
  const int lt = opaque(C.lt), TPR = C.TPR;
  double* F = C.s_frm;
  double v[RK];
  const int32_t* cls = G.ncls == 1 ? nullptr : G.cls;
  const int flags = FULL ? B.meas : (B.meas & ~MEAS_SPIN_OBS);
  int lo, hi;
  // --- correlation pairs: S_i, S_j, sum s_i.s_j, last-site spin
  if ((flags & MCG_MEAS_PAIRS) && G.nlat > 0) {
    for (int k = 0; k < RK; ++k) v[k] = 0.0;
    slice(G.nlat, part, np, lo, hi);
    if (own) lo = 0, hi = own->npairs;
    if (G.self_pairs) hi = lo;  // the sums follow from the state (frame_terms)
    for (int q = lo + lt; q < hi; q += TPR) {
      const int p = own ? own->pairs[q] : q;
      float a[3], b[3];
      spin_vec<NC>(sp, G.pairs[2 * p], cls, C.clsdat, a);
      spin_vec<NC>(sp, G.pairs[2 * p + 1], cls, C.clsdat, b);
      v[0] += a[0]; v[1] += a[1]; v[2] += a[2];
      v[3] += b[0]; v[4] += b[1]; v[5] += b[2];
      v[6] += (double)(a[0] * b[0] + a[1] * b[1] + a[2] * b[2]);
    }
    if (lt == 0 && (own ? own->last : part == 0)) {
      float t[3];
      spin_vec<NC>(sp, C.last, cls, C.clsdat, t);
      v[7] = t[0];
    }
    // self pairs: every other lane holds zeros, so the group reduction (a
    // microsecond of FP64 DPP steps and barriers per frame) is not needed
    if (!G.self_pairs) {
      group_add<8>(v, C.s_red, C.g, TPR, [&](int k, double x) { F[k] = x; });
    } else if (lt == 0) {
      for (int k = 0; k < 8; ++k) F[k] = v[k];
    }
  }
  // --- topological charge
  if ((flags & MCG_MEAS_Q) && NC == 3 && G.ncirc > 0) {
    for (int k = 0; k < RK; ++k) v[k] = 0.0;
    slice(G.ncirc, part, np, lo, hi);
    if (own) lo = 0, hi = own->ncircs;
    // one spin length for every class: no per-site class lookups
    float il = sqrtf(C.clsdat[4]);
    bool one_len = G.ncls <= 64;
    for (int q = 1; q < G.ncls && one_len; ++q) one_len = C.clsdat[q * 8 + 4] == C.clsdat[4];
    auto triangles = [&](auto one, auto uc) {
      // U at a time: their indices, then their spins are in flight together
      // (triangular 128^2 x 1024, 5 sweeps: one 1365 us, two 1304, three 1309)
      constexpr int U = decltype(uc)::value;
      for (int q = lo + lt; q < hi; q += U * TPR) {
        int id[U][3];
        float x[U][3][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int qu = min(q + u * TPR, hi - 1), p = own ? own->circs[qu] : qu;
          const GAS int32_t* t = (const GAS int32_t*)((const GAS char*)gas(G.circ) + (uint32_t)p * 12u);
#pragma unroll
          for (int k = 0; k < 3; ++k) id[u][k] = t[k];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < 3; ++k) spin_vec<NC>(sp, id[u][k], nullptr, C.clsdat, x[u][k]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (u > 0 && q + u * TPR >= hi) break;
          if constexpr (decltype(one)::value)
            v[0] += (double)signed_area(x[u][0], x[u][1], x[u][2], il, il, il);
          else
            v[0] += (double)signed_area(x[u][0], x[u][1], x[u][2], inv_len(C.clsdat, G.cls, id[u][0]),
                                        inv_len(C.clsdat, G.cls, id[u][1]), inv_len(C.clsdat, G.cls, id[u][2]));
        }
      }
    };
    if (one_len)
      triangles(std::true_type(), std::integral_constant<int, FRAME_TRI>());
    else
      triangles(std::false_type(), std::integral_constant<int, 1>());
    group_add<1>(v, C.s_red, C.g, TPR, [&](int, double x) { F[8] = x; });
  }
  // --- block-spin observables
  if ((flags & MCG_MEAS_RNORM) && G.nr > 0 && !own) {
    for (int k = 0; k < RK; ++k) v[k] = 0.0;
    // Every block spin is used by its own pairs and links and by its
    // neighbours' links.  Where LDS has room each is computed once, here, and
    // looked up below; otherwise at every use (each use waits for its rank,
    // its cluster's sites and their spins one after another).
    const float* blk = C.blk;
    if (blk) {
      for (int ri = lt; ri < G.nr; ri += TPR) {
        float m[3];
        majority<NC>(sp, G, cls, C.clsdat, ri, G.rorb[ri], frame, key0, key1, m);
#pragma unroll
        for (int k = 0; k < NC; ++k) C.blk[ri * NC + k] = m[k];
      }
      __syncthreads();
    }
    auto block = [&](int ri, int site, float* m) {
      if (blk)
        block_spin<NC>(blk, ri, m);
      else
        majority<NC>(sp, G, cls, C.clsdat, ri, site, frame, key0, key1, m);
    };
    slice(G.nlat, part, np, lo, hi);
    for (int p = lo + lt; p < hi; p += TPR) {
      const int ia = G.pairs[2 * p], ib = G.pairs[2 * p + 1];
      const int ra = G.rrank[ia], rb = G.rrank[ib];
      const bool ca = ra >= 0, cb = rb >= 0;
      float ma[3] = {0, 0, 0}, mb[3] = {0, 0, 0};
      if (ca) {
        block(ra, ia, ma);
        v[0] += ma[0]; v[1] += ma[1]; v[2] += ma[2];
        v[7] += 1.0;
      }
      if (cb) {
        block(rb, ib, mb);
        v[3] += mb[0]; v[4] += mb[1]; v[5] += mb[2];
        v[8] += 1.0;
      }
      if (ca && cb) {
        v[6] += (double)(ma[0] * mb[0] + ma[1] * mb[1] + ma[2] * mb[2]);
        v[9] += 1.0;
      }
    }
    slice(G.nr, part, np, lo, hi);
    for (int ri = lo + lt; ri < hi; ri += TPR) {
      const int j = G.rorb[ri];
      float m[3];
      block(G.rrank[j], j, m);
      float cc = 0.0f;
      for (int l0 = 0; l0 < G.zmax; l0 += 4) {
        // four links at a time: their words, then their ranks, then their
        // block spins (link order in the sum)
        uint32_t wd[4];
        int rt[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) wd[u] = G.rlink[(size_t)ri * G.zmax + (l0 + u < G.zmax ? l0 + u : G.zmax - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) rt[u] = G.rrank[wd[u] & 0xFFFFFFu];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (l0 + u >= G.zmax) break;
          // wide graphs: the block-spin link takes the coupling of the site's
          // link l; a set high byte marks an absent link
          if (G.lcid && (wd[u] >> 24)) continue;
          const float* J =
              C.coup + (G.lcid ? G.lcid[(size_t)j * G.zmax + l0 + u] : (int)(wd[u] >> 24)) * C.cst;
          float mt[3];
          block(rt[u], (int)(wd[u] & 0xFFFFFFu), mt);
          if constexpr (NC == 1) {
            cc += J[1] * m[0] * mt[0];
          } else {
            float H0 = J[0] * mt[0] + J[1] * mt[1] + J[2] * mt[2];
            float H1 = J[3] * mt[0] + J[4] * mt[1] + J[5] * mt[2];
            float H2 = J[6] * mt[0] + J[7] * mt[1] + J[8] * mt[2];
            cc += m[0] * H0 + m[1] * H1 + m[2] * H2;
          }
        }
      }
      v[10] += (double)cc;
      // on-site part with the site's actual spin (heisenbergLib.c:798-800,
      // isingLib.c:390)
      float s[3];
      spin_vec<NC>(sp, j, cls, C.clsdat, s);
      const int ci = cls ? cls[j] : 0;
      float eo;
      if constexpr (NC == 1)
        eo = -h * s[0];
      else
        eo = C.clsdat[ci * 8 + 1] * s[0] * s[0] + C.clsdat[ci * 8 + 2] * s[1] * s[1] +
             C.clsdat[ci * 8 + 3] * s[2] * s[2] - h * (NC == 3 ? s[2] : s[0]);
      v[11] += (double)eo;
    }
    group_add<12>(v, C.s_red, C.g, TPR, [&](int k, double x) { F[k < 7 ? 16 + k : 17 + k] = x; });
  }
  // --- orbital groups (heisenbergLib.c:805-830): 2 groups per reduction
  const int ng = (flags & MCG_MEAS_GROUPS) && !own ? G.ngroup : 0;
  for (int g0 = 0; g0 < ng; g0 += 2) {
    for (int k = 0; k < RK; ++k) v[k] = 0.0;
    slice(G.gmax, part, np, lo, hi);
    for (int q = 0; q < 2 && g0 + q < ng; ++q) {
      for (int k = lo + lt; k < hi; k += TPR) {
        const int o = G.groups[(g0 + q) * G.gmax + k];
        if (o < 0) continue;
        float s[3];
        spin_vec<NC>(sp, o, cls, C.clsdat, s);
        v[3 * q] += s[0]; v[3 * q + 1] += s[1]; v[3 * q + 2] += s[2];
      }
    }
    group_add<6>(v, C.s_red, C.g, TPR, [&](int k, double x) { F[32 + 3 * g0 + k] = x; });
  }
}

// The frame's terms, by the group's first wave: Cn zeroed, lane 0's
// frame_terms, <M M'> from the row's previous M in *mp (LDS), which gets this
// frame's M.  Self pairs: the last site's spin is read here.
template <int NC, typename SV>
__device__ __forceinline__ void first_wave_terms(const SV& sp, const FrameCtx& C, const mcg_batch& B, const double* st,
                                                 int64_t frame, int flags, double* mp) {
  double* F = C.s_frm;
  double* Cn = F + FRM_ACC;
  zero_terms(F, 1);
  if ((tid() & 63) == 0) {
    const mcg_graph G = fresh(C.G);
    if (NC == 1 && (flags & MCG_MEAS_PAIRS) && G.self_pairs) {
      float t[3];
      spin_vec<NC>(sp, C.last, G.ncls == 1 ? nullptr : G.cls, C.clsdat, t);
      F[7] = t[0];
    }
    frame_terms<NC>(C, G, B, st, F, flags, frame, Cn);
    const double Mf = Cn[MCG_A_MM];
    Cn[MCG_A_MM] = *mp * Mf;
    *mp = Mf;
  }
}
// One measured frame of the group's replica at `row`, from the tracked state
// st and the spins; *mp as above.  All threads call it; the accumulators'
// atomics are queued, not waited for.
template <int NC, typename SV, bool FULL = true>
__device__ __forceinline__ void measure_frame(const SV& sp, const FrameCtx& C, const mcg_batch& B, const double* st, int row,
                                              int64_t frame, uint32_t key0, uint32_t key1, float h, double* mp) {
  const int flags = FULL ? B.meas : (B.meas & ~MEAS_SPIN_OBS);
  if (FULL) frame_sums<NC, SV, FULL>(sp, C, B, frame, key0, key1, h, 0, 1);
  if (C.lt < 64) {
    wave_lds_fence();
    first_wave_terms<NC>(sp, C, B, st, frame, flags, mp);
  }
  __syncthreads();
  flush_frame<NC>(C, B, row, flags);
}

// full FP64 recomputation of one replica (group-parallel): out[0] E (out:
// LDS, complete at return), out[1..3] M, out[4] the summed relative
// spin-length deviation sum_i | |s_i|^2 / S_i^2 - 1 | (0 for Ising)
static constexpr int NREC = 5;
template <int NC, typename SV>
__device__ __forceinline__ void recompute(const SV& sp, const mcg_graph* Gd, const float* coup, int cst, const float* clsdat, float h,
                          double* s_red, int g, int lt, int TPR, double* out, int part = 0, int np = 1) {
  const mcg_graph G = fresh(Gd);
  lt = opaque(lt);
  double v[RK];
  for (int k = 0; k < RK; ++k) v[k] = 0.0;
  int lo, hi;
  slice(G.n, part, np, lo, hi);
  for (int i = lo + lt; i < hi; i += TPR) {
    v[0] += (double)site_energy<NC>(sp, i, G.link, G.lcid, G.zmax, coup, cst, G.cls, clsdat, h);
    float s[3];
    spin_vec<NC>(sp, i, G.cls, clsdat, s);
    v[1] += s[0];
    v[2] += s[1];
    v[3] += s[2];
    if constexpr (NC > 1) {
      const double l2 = (double)s[0] * s[0] + (double)s[1] * s[1] + (double)s[2] * s[2];
      v[4] += fabs(fma(l2, (double)clsdat[G.cls[i] * 8 + 4], -1.0));
    }
  }
  group_add<NREC>(v, s_red, g, TPR, [&](int k, double x) { out[k] = x; });
}

// Health checks on a recompute (called by the thread holding its result;
// drift = |E_tracked - E_full|): NaN / Inf in the spins makes E or M
// non-finite; spin lengths whose mean relative deviation exceeds the
// storage's tolerance (FP32 keeps |s|^2 to ~1e-7 by the renormalisation,
// FP16 rounds each component to 11 bits) mean the renormalisation no longer
// holds; a drift above the storage's tolerance per site (FP32 tracking
// wanders by ~1e-9 per site per sweep, FP16 by the untracked rounding of
// stored spins) means the spins changed behind the sweep's back.  Each
// raises a bit of the device error flag.
template <typename ST>
__device__ __forceinline__ void recompute_checks(const mcg_batch& B, const mcg_graph& G, const double* r,
                                                 double drift) {
  const bool f16 = sizeof(ST) == 2;
  if (!isfinite(r[0] + r[1] + r[2] + r[3] + r[4])) {
    atomicOr(B.err, MCG_ERR_NONFINITE);
    return;
  }
  if (r[4] > (f16 ? 1e-2 : 1e-4) * G.n) atomicOr(B.err, MCG_ERR_LENGTH);
  if (drift > (f16 ? 1e-2 : 1e-4) * G.n) atomicOr(B.err, MCG_ERR_DRIFT);
}

// ---------------------------------------------------------------------------
// k_lds: persistent LDS-resident sweeps
// ---------------------------------------------------------------------------
// One workgroup of the LDS kernel: nrep replicas of one graph, or one part
// of a replica split over nparts workgroups (part, nparts, slot of its
// counter and partial sums, offset of its extra-group table).
struct WorkItem {
  int32_t graph, nrep, off;
  uint8_t part, nparts;
  uint16_t slot;
  int32_t hoff;
};

// what a workgroup needs of each of its replicas, resolved on the host so
// that staging starts one dependent load after the work item
struct ItemRep {
  int64_t spin_off;
  int32_t rep, serial, row0, nrung, ladder, pad;  // nrung 0: no tempering ladder
};

static constexpr int MAX_PARTS = 4;
static constexpr int SYNC_STRIDE = 16;  // uint32 per replica counter (one 64-byte line)

__host__ __device__ inline size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

struct SweepArgs {
  int64_t k_begin;      // run-relative index of the first sweep of this launch
  int64_t philox_base;  // added to k for the Philox counter
  int32_t nsweeps;      // 1 whenever the launch has split replicas
  int32_t nthermal;     // run-relative: sweeps < nthermal are thermal
  int32_t spf;          // sweeps per frame
  int32_t frame0;       // index of the first frame of the run
  uint32_t* sync;       // split replicas: arrival counters, zero at run start
  double* xpart;        // split replicas: per-part (dE, dM) partial sums
  const int32_t* halo;  // split replicas: extra-group tables
  // persistent launches (many sweeps, tempering inside the kernel)
  int32_t sync_base;         // exchanges (of parts or ladders) before this launch in the run
  int32_t pt_every;          // tempering period in sweeps (0: none)
  int32_t has_split;         // the launch holds split replicas
  int32_t nrow_parts;        // parts a row has words for in rowslot: the most of any replica
  uint64_t* rowslot;         // [4][nrow][nrow_parts][2] energies published for tempering (tagged words)
  uint64_t* pslot;           // [2][nslots][MAX_PARTS][2] energies of a split replica's parts (tagged words)
  double* mslot;             // [2][nslots][MAX_PARTS-1][3] published magnetisation changes of parts 1, ...
  void* xbuf;                // [2][nslots][MAX_PARTS][max_export][NC] exported sites
  uint64_t* mprev;           // [2][nrow][2] M' of each row's last frames (tagged words, by the tag's parity)
  double* fpart;             // [2][nslots][MAX_PARTS-1][FSUMS] split replicas' partial frame sums
                             // (spin-derived observables); their arrival count is sync[slot]
  void* fspin;               // [2][nslots][NC][fspin_n] split replicas' sites as published for a
                             // frame, by sweep parity: the next sweep's publication must not
                             // overwrite sites a slower part still reads
  int32_t fspin_n;
  int32_t max_export;
  int32_t nslots;
  int32_t thr;               // LDS bytes per group for its row's Ising thresholds, after those (0: none)
  int32_t blk;               // LDS bytes per group for a frame's block spins, after the spins (0: none)
  int32_t rec_host;          // the full recompute is the host's (a launch ends at each
                             // recompute sweep, then k_measure recomputes every replica)
};

// The schedules of the full recompute and of tempering follow the global
// sweep index (Philox counter), not the index within a call, so that a run
// split into calls (frames, checkpoints) does the same thing at the same
// sweeps as one call.
__host__ __device__ inline bool recompute_due(const mcg_batch& B, int64_t global_sweep) {
  return B.recompute_every > 0 && ((global_sweep + 1) % B.recompute_every) == 0;
}

// LDS of the tempering state a persistent launch keeps in every workgroup:
// beta and h per row; per group its row, and its ladder's first row and rungs;
// the flag of a wait that timed out
static constexpr int MAX_GROUPS = 16;  // replicas per workgroup (1024 threads, a wave each)
__host__ __device__ inline size_t persist_lds_bytes(int nrow) {
  return align16((size_t)2 * nrow * 4) + (size_t)MAX_GROUPS * 12 + 16;
}

typedef unsigned int v4u32 __attribute__((ext_vector_type(4)));
// copy one replica between HBM (16-byte aligned) and LDS in 16-byte vectors,
// four in flight per thread

template <typename ST, bool IN>
__device__ __forceinline__ void stage(ST* lds, ST* g, int count, int lt, int TPR) {
  const int nbytes = count * (int)sizeof(ST);
  const int nvec = nbytes >> 4;
  v4u32* lv = (v4u32*)lds;
  GAS v4u32* gv = (GAS v4u32*)gas(g);
  int t = lt;
  for (; t + 3 * TPR < nvec; t += 4 * TPR) {
    if constexpr (IN) {
      const v4u32 a0 = gv[t], a1 = gv[t + TPR], a2 = gv[t + 2 * TPR], a3 = gv[t + 3 * TPR];
      lv[t] = a0; lv[t + TPR] = a1; lv[t + 2 * TPR] = a2; lv[t + 3 * TPR] = a3;
    } else {
      const v4u32 a0 = lv[t], a1 = lv[t + TPR], a2 = lv[t + 2 * TPR], a3 = lv[t + 3 * TPR];
      gv[t] = a0; gv[t + TPR] = a1; gv[t + 2 * TPR] = a2; gv[t + 3 * TPR] = a3;
    }
  }
  for (; t < nvec; t += TPR) {
    if constexpr (IN) lv[t] = gv[t];
    else gv[t] = lv[t];
  }
  unsigned char* lb = (unsigned char*)lds;
  GAS unsigned char* gb = (GAS unsigned char*)gas(g);
  for (int e = (nvec << 4) + lt; e < nbytes; e += TPR) {
    if constexpr (IN) lb[e] = gb[e];
    else gb[e] = lb[e];
  }
}

__host__ __device__ inline size_t lds_fixed_bytes(int ncoup, int ncls, int ncol, int npat, int zmax, int n,
                                                  int nwaves, int R) {
  size_t b = align16((size_t)(ncoup * COUP_LDS + ncls * 8) * 4) + align16((size_t)(ncol + 1) * 4);
  if (npat > 0) b += align16((size_t)npat * pat_stride(zmax) * 4) + align16((size_t)n);
  return b + align16((size_t)nwaves * RK * 8) + align16((size_t)R * (MCG_NSTATE + FRM + 1) * 8) + align16((size_t)R * 16);
}

__host__ __device__ inline size_t lds_replica_bytes(int nc, int n, int ssize) {
  return align16((size_t)nc * n * ssize);
}

// Split replicas.  A replica too large for one CU's share of a sweep runs as
// P workgroups (parts), each holding the whole replica in LDS.  Part p owns
// the Philox groups [ngrp*p/P, ngrp*(p+1)/P) of every colour class.  Its own
// sites need, when they are updated, the current values of their neighbours;
// those of lower colour that another part owns are recomputed here too: the
// host lists, per part and colour, the extra groups that close the own
// sites under "neighbour of lower colour".  Every part starts the sweep from
// the same spins and draws the same Philox words, so the recomputed sites
// come out bit for bit as their owner computes them, and no data moves
// between parts during a sweep.  A launch with split replicas does one
// sweep.  At its end each part publishes its own sites and its partial
// sums (dE, dM) at the device coherence point and counts itself on the
// replica's counter; the part that arrives last reads the other parts' sites
// back, combines the sums and does the measurement.  Nothing waits.
//
// Device coherence: the parts may sit on different XCDs, whose L2 caches are
// not coherent with each other for ordinary accesses.  Published data goes
// through device-scope (agent) atomic stores and loads, which the compiler
// emits at the device coherence point (sc1), and each wave waits for its
// stores to be acknowledged (s_waitcnt 0) before the workgroup barrier that
// precedes the counter increment.
__device__ __forceinline__ void part_range(int b, int cnt, int ngrp, int gd, int p, int np, int& e0, int& e1) {
  const int qa = (int)((int64_t)ngrp * p / np), qb = (int)((int64_t)ngrp * (p + 1) / np);
  e0 = b + qa * gd;
  e1 = b + min(qb * gd, cnt);
}

// every store this wave issued has been acknowledged
__device__ __forceinline__ void stores_done() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A published FP64 value: two words, each with half of its bits and the tag
// of the event it belongs to, in device-coherent stores.  A reader that sees
// its tag in both words has the value: the store needs no acknowledgement, no
// counter and no release word, and the reader no second trip for the data.
// Tags only grow during a run, and every run starts with zeroed words.
__device__ __forceinline__ void tag_store(uint64_t* w, uint32_t tag, double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x), t = (uint64_t)tag << 32;
  dev_store(w, t | (u & 0xFFFFFFFFu));
  dev_store(w + 1, t | (u >> 32));
}
struct Tagged {
  uint64_t a = 0, b = 0;
  // both words in one 16-byte load (with the wait: its registers are not free
  // before), half the requests of two loads
  __device__ __forceinline__ void load(const uint64_t* w) {
    v4u32 u;
    asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(u) : "v"(w) : "memory");
    a = (uint64_t)u.y << 32 | u.x;
    b = (uint64_t)u.w << 32 | u.z;
  }
  __device__ __forceinline__ void load_ahead(const uint64_t* w) {  // not waited for here
    a = dev_load(w);
    b = dev_load(w + 1);
  }
  // the tag, but for the bits in `any`
  __device__ __forceinline__ bool has(uint32_t tag, uint32_t any = 0u) const {
    return ((((uint32_t)(a >> 32) ^ tag) | ((uint32_t)(b >> 32) ^ tag)) & ~any) == 0u;
  }
  __device__ __forceinline__ double value() const {
    return __hiloint2double((int)(uint32_t)b, (int)(uint32_t)a);
  }
};
// Waits are bounded: on time-out bit 16 of the error flag is raised and the
// workgroup's flag cleared, and the workgroup leaves the kernel.
static constexpr uint32_t WAIT_POLLS = 1u << 22;
__device__ __forceinline__ void wait_failed(int32_t* err, int* s_flag) {
  atomicOr(err, MCG_ERR_BARRIER);
  *s_flag = 0;
}
// the value of tag `tag` at w (t: words read ahead)
__device__ __forceinline__ double tag_wait(const uint64_t* w, Tagged t, uint32_t tag, int32_t* err, int* s_flag) {
  uint32_t it = 0;
  while (!t.has(tag)) {
    t.load(w);
    if (++it > WAIT_POLLS) {
      wait_failed(err, s_flag);
      break;
    }
  }
  return t.value();
}

template <int S>
struct RawBits;
template <>
struct RawBits<1> {
  typedef uint8_t T;
};
template <>
struct RawBits<2> {
  typedef uint16_t T;
};
template <>
struct RawBits<4> {
  typedef uint32_t T;
};

// copy the sites of part p (every colour) between LDS and global memory, as
// raw bit patterns of the storage type (ordinary accesses; the caller
// orders them with fences where another workgroup reads them)
template <typename ST, bool OUT>
__device__ __forceinline__ void part_copy(ST* lds_s, ST* gsp, int n, int nc, const int32_t* colptr, int ncol, int gd, int p, int np,
                          int lt, int TPR) {
  typedef typename RawBits<sizeof(ST)>::T U;
  U* lds = (U*)lds_s;
  GAS U* g = (GAS U*)gas((U*)gsp);
  for (int c = 0; c < ncol; ++c) {
    const int b = colptr[c], cnt = colptr[c + 1] - b;
    const int ngrp = (cnt + gd - 1) / gd;
    int e0, e1;
    part_range(b, cnt, ngrp, gd, p, np, e0, e1);
    for (int k = 0; k < nc; ++k) {
      U* l = lds + (size_t)k * n;
      GAS U* q = g + (size_t)k * n;
      for (int e = e0 + lt; e < e1; e += TPR) {
        if constexpr (OUT) q[e] = l[e];
        else l[e] = q[e];
      }
    }
  }
}

// the sites of part p (every colour) from LDS (component stride n) to a
// copy of the replica in global memory (component stride dn) with
// device-scope stores, so that any workgroup of the launch can read them
// (DevSpins) after the parts' next exchange.  The copy is not the replica's
// spin array: other parts still stage from that at the launch start.
template <typename ST>
__device__ __forceinline__ void part_publish(const ST* lds_s, typename RawBits<sizeof(ST)>::T* dst, int n, int dn, int nc,
                             const int32_t* colptr, int ncol, int gd, int p, int np, int lt, int TPR) {
  typedef typename RawBits<sizeof(ST)>::T U;
  const U* lds = (const U*)lds_s;
  for (int c = 0; c < ncol; ++c) {
    const int b = colptr[c], cnt = colptr[c + 1] - b;
    const int ngrp = (cnt + gd - 1) / gd;
    int e0, e1;
    part_range(b, cnt, ngrp, gd, p, np, e0, e1);
    for (int k = 0; k < nc; ++k)
      for (int e = e0 + lt; e < e1; e += TPR) dev_store(dst + (size_t)k * dn + e, lds[(size_t)k * n + e]);
  }
}

// one replica's spins in global memory read with device-scope loads: the
// sites other workgroups of the same launch published with part_publish
template <typename ST>
__device__ __forceinline__ float raw_spin(typename RawBits<sizeof(ST)>::T u);
template <>
__device__ __forceinline__ float raw_spin<float>(uint32_t u) { return __uint_as_float(u); }
template <>
__device__ __forceinline__ float raw_spin<__half>(uint16_t u) { return __half2float(__ushort_as_half(u)); }
template <>
__device__ __forceinline__ float raw_spin<int8_t>(uint8_t u) { return (float)(int8_t)u; }
template <typename ST>
struct DevSpins {
  typedef ST value_type;
  typedef typename RawBits<sizeof(ST)>::T U;
  const U* p;
  int n;
  __device__ __forceinline__ float get(int i, int c) const { return raw_spin<ST>(dev_load(p + (size_t)c * n + i)); }
};

// ints per part in the split tables: (start, count) of the extra groups per
// colour, (start, count) of the export list, of the correlation pairs and
// of the circuits whose first site the part owns, 1 if the part owns the
// last site, then 1 if no pair or circuit of the replica has sites of two
// parts (the frame then needs only each part's own sites)
__host__ __device__ inline int halo_desc_ints(int ncol) { return 2 * ncol + 8; }

// The leftover groups of a workgroup whose replicas each have one wave
// (64 threads per replica, R replicas, every colour with the same number of
// Philox groups): each replica's last, partial round of rem groups goes to
// a pool of R*rem groups dealt over the workgroup's first threads, so that
// it costs ceil(R*rem/64) wave-rounds instead of R.  Thread t takes group
// ngrp-rem + t%rem of replica t/rem (pr; -1: no pool group).  A group's
// result does not depend on the thread that takes it; the ΔE, ΔM of the
// pool groups are summed per replica in a fixed order (pool_sums).
template <typename ST>
struct PoolInfo {
  int rem = 0;             // 0: no pool
  int pr = -1, pq = 0;     // this thread's pool group: replica pr (group index), group ngrp-rem+pq
  const float4* par = nullptr;  // per group: beta, h, key1 bits
  ST* spin0 = nullptr;     // the workgroup's replicas in LDS, stride sstride
  int sstride = 0;
  double* pp = nullptr;    // pool partials [NC+1][nr], nr = R*rem
  int nr = 0;
};

struct PartInfo {
  int part = 0, np = 1;            // this workgroup's part of the replica
  const int32_t* hx = nullptr;     // extra groups: [2c] start, [2c+1] count per colour, into halo
  const int32_t* halo = nullptr;
};

// End-of-sweep work of an unsplit replica (or of the last part of a split
// one) outside a persistent launch: the state takes the sweeps' changes dE,
// dM (and the pool's), then full recompute (drift check), energy reference at
// the end of thermalisation, measured frame.  With no recompute and no pass
// over the spins the first wave does all of it between two barriers.
template <int NC, typename ST, bool FULL, typename SV>
__device__ __forceinline__ void lds_sweep_tail(const SV& sv, const mcg_graph& G, const mcg_batch& B, double* st,
                                               FrameCtx& C, int row, float h, int64_t k, const SweepArgs& a, bool meas,
                                               bool therm_end, bool rec, double& dE, double* dM, uint32_t key0,
                                               uint32_t key1, double* mp, const PoolInfo<ST>& pl) {
  const double v[4] = {dE, dM[0], dM[1], dM[2]};
  const int flags = FULL ? B.meas : (B.meas & ~MEAS_SPIN_OBS);
  const bool light = !rec && (!FULL || frame_light(G, B.meas));
  const int64_t frame = meas ? (k - a.nthermal + 1) / a.spf - 1 + a.frame0 : 0;
  group_add<4>(
      v, C.s_red, C.g, C.TPR,
      [&](int q, double x) {
        if (pl.rem > 0 && q <= NC) {
          double ps = 0.0;
          for (int i = 0; i < pl.rem; ++i) ps += pl.pp[q * pl.nr + C.g * pl.rem + i];
          x += ps;
        }
        st[MCG_S_E + q] += x;
      },
      [&] {
        if (!light) return;
        if (therm_end && C.lt == 0) st[MCG_S_EREF] = st[MCG_S_E];
        if (pl.rem > 0 || !meas) return;  // with a pool, other groups' partials are in the frame area until all are read
        first_wave_terms<NC>(sv, C, B, st, frame, flags, mp);
      });
  dE = 0.0;
  dM[0] = dM[1] = dM[2] = 0.0;
  if (light && pl.rem == 0) {
    if (meas) flush_frame<NC>(C, B, row, flags);
    return;
  }
  if (rec) {
    double* r4 = C.s_frm;  // the frame area
    recompute<NC>(sv, C.G, C.coup, C.cst, C.clsdat, h, C.s_red, C.g, C.lt, C.TPR, r4);
    if (C.lt == 0) {
      const double d = fabs(st[MCG_S_E] - r4[0]);
      if (d > st[MCG_S_DRIFT]) st[MCG_S_DRIFT] = d;
      for (int q = 0; q < 4; ++q) st[MCG_S_E + q] = r4[q];
      recompute_checks<ST>(B, G, r4, d);
    }
  }
  if (therm_end && !light && C.lt == 0) st[MCG_S_EREF] = st[MCG_S_E];
  __syncthreads();
  if (meas) measure_frame<NC, SV, FULL>(sv, C, B, st, row, frame, key0, key1, h, mp);
  __syncthreads();
}

// One exported site of a split replica: its NC components (raw bits, SoA in
// LDS) as one device-scope store when they fill 4 or 8 bytes, else one per
// component.
template <int NC, typename U>
__device__ __forceinline__ void export_site(U* dst, const U* lraw, int n, int site) {
  constexpr int W = NC * (int)sizeof(U);
  if constexpr (W == 8 || W == 4) {
    typedef typename std::conditional<W == 8, uint64_t, uint32_t>::type P;
    P w = 0;
#pragma unroll
    for (int q = 0; q < NC; ++q) w |= (P)lraw[(size_t)q * n + site] << (q * 8 * sizeof(U));
    dev_store((P*)dst, w);
  } else {
#pragma unroll
    for (int q = 0; q < NC; ++q) dev_store(dst + q, lraw[(size_t)q * n + site]);
  }
}
// The other parts' exported sites, into this part's LDS copy (replicas
// split into three or more parts).  The parts' lists form one round-robin:
// thread lt takes flat indices lt, lt + TPR, ... over the lists of parts
// 0..np-1 (its own list has no entries here), so that it imports about
// (sites of all lists) / TPR sites in all instead of working through every
// part's list in turn, one device-scope round trip per list.  K sites are
// loaded before any is stored (honeycomb 64^2 x 64, 50 sweeps: one 916 us,
// two 906).  xs: part 0's export area of this replica and sweep
// parity; parts are max_export * NC words apart.  dsc: this part's
// descriptor; part p's is (p - part) * ds ints away.
template <int NC, typename U>
__device__ __forceinline__ void import_parts(const U* xs, int max_export, const int32_t* halo, const int32_t* dsc,
                                             int ds, int ncol, int part, int np, U* lraw, int n, int lt, int TPR) {
  constexpr int W = NC * (int)sizeof(U);
  constexpr bool PACKED = W == 8 || W == 4;
  typedef typename std::conditional<W == 8, uint64_t, uint32_t>::type P;
  constexpr int K = 2;
  int ofs[MAX_PARTS], lst[MAX_PARTS], tot = 0;
#pragma unroll
  for (int p = 0; p < MAX_PARTS; ++p) {
    const int32_t* d = dsc + (p - part) * ds;
    const bool other = p < np && p != part;
    ofs[p] = tot;
    lst[p] = other ? d[2 * ncol] : 0;
    tot += other ? d[2 * ncol + 1] : 0;
  }
  for (int j0 = lt; j0 < tot; j0 += K * TPR) {
    P w[K];
    U v[K][NC];
    int site[K];
#pragma unroll
    for (int u = 0; u < K; ++u) {
      const int j = j0 + u * TPR;
      site[u] = -1;
      if (j < tot) {
        // the part of flat index j: the last one whose list starts at or
        // before j (a part with an empty list starts where the next one does)
        int p = 0;
#pragma unroll
        for (int q = 1; q < MAX_PARTS; ++q)
          if (ofs[q] <= j) p = q;
        const int i = j - ofs[p];
        const U* src = xs + ((size_t)p * max_export + i) * NC;
        site[u] = halo[lst[p] + i];
        if constexpr (PACKED) {
          w[u] = dev_load((const P*)src);
        } else {
#pragma unroll
          for (int q = 0; q < NC; ++q) v[u][q] = dev_load(src + q);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < K; ++u) {
      if (site[u] < 0) continue;
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        if constexpr (PACKED)
          lraw[(size_t)q * n + site[u]] = (U)(w[u] >> (q * 8 * sizeof(U)));
        else
          lraw[(size_t)q * n + site[u]] = v[u][q];
      }
    }
  }
}

// Split replica, measured frame with spin-derived observables: each part's
// share F[0, FSUMS) of the sums (frame_sums) goes to a.fpart and counts in
// on the replica's counter a.sync[slot]; part 0 waits for the other parts of
// this frame (the counter counts from the run's first frame, a.frame0), then
// adds their sums to its own in part order, so the result does not depend on
// arrival order.  Called by every thread of the part's workgroup; false:
// time-out (the caller leaves the kernel).  A part overwrites its slot only
// after the parts' next exchange, which part 0 joins after reading it.
__device__ __forceinline__ bool gather_frame_sums(const SweepArgs& a, const mcg_batch& B, double* F, int slot, int part, int np,
                                  int64_t frame, int* s_flag) {
  double* fp = a.fpart + (size_t)slot * (MAX_PARTS - 1) * FSUMS;  // part p at p - 1
  uint32_t* cnt = a.sync + (size_t)slot * SYNC_STRIDE;
  const int tx = tid();
  __syncthreads();  // F is written by the first thread
  if (part != 0) {
    if (tx < 64)
      for (int q = tx; q < FSUMS; q += 64) dev_store(fp + (size_t)(part - 1) * FSUMS + q, F[q]);
    stores_done();
    __syncthreads();
    if (tx == 0) __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  if (tx == 0) {
    const uint32_t want = (uint32_t)((frame - a.frame0 + 1) * (int64_t)(np - 1));
    uint32_t it = 0;
    while ((int32_t)(dev_load(cnt) - want) < 0) {
      if (++it > WAIT_POLLS) {
        wait_failed(B.err, s_flag);
        break;
      }
    }
  }
  __syncthreads();
  if (!*s_flag) return false;
  if (tx < 64)
    for (int q = tx; q < FSUMS; q += 64) {
      // the parts' values loaded together, then added in part order
      double y[MAX_PARTS];
#pragma unroll
      for (int p = 1; p < MAX_PARTS; ++p) y[p] = p < np ? dev_load(fp + (size_t)(p - 1) * FSUMS + q) : 0.0;
      double x = F[q];
#pragma unroll
      for (int p = 1; p < MAX_PARTS; ++p)
        if (p < np) x += y[p];
      F[q] = x;
    }
  __syncthreads();
  return true;
}

// Totals of every group's changes v[0..NC] (E, M) over its waves, in the
// workgroup's first wave and in wave `also`, each for itself: sink(g, k, total)
// by lane group_lane(g) + k.  Called by every thread; s_red is free again only
// after the caller's next workgroup barrier.
__device__ __forceinline__ int group_lane_stride(int TPR) {
  const int nw = TPR >> 6;
  return nw == 8 || nw == 16 ? 4 * nw : 4;
}
template <int NC, typename F>
__device__ __forceinline__ void wave0_add(double* s_red, int TPR, const double* v, int also, F&& sink) {
  double r[1];
  wave_totals<NC + 1>(v, r);
  const int tx = tid(), lane = tx & 63, wave = tx >> 6;
  if (lane < 4) s_red[wave * RK + lane] = r[0];
  __syncthreads();
  if (wave == 0 || wave == also) {
    const int nw = TPR >> 6, nwaves = (int)blockDim.x >> 6;
    const int k = lane & 3;
    double x = 0.0;
    if (nw == 8 || nw == 16) {
      // lane 4 w + k holds wave w's value k
      x = (lane >> 2) < nwaves ? s_red[(lane >> 2) * RK + k] : 0.0;
      x += dpp_f64<0x124, 0xF>(x);  // row_ror:4
      x += dpp_f64<0x128, 0xF>(x);  // row_ror:8
      x = add_lane16(x);
      if (nw == 16) x = add_lane32(x);
      const int g = (lane >> 2) / nw;
      if ((lane >> 2) == g * nw && g * nw < nwaves && k <= NC) sink(g, k, x);
    } else {
      const int g = lane >> 2;  // at most 16 groups
      if (g * nw < nwaves && k <= NC) {
        for (int w = 0; w < nw; ++w) x += s_red[(g * nw + w) * RK + k];
        sink(g, k, x);
      }
    }
  }
}

// End of a persistent sweep for a workgroup of unsplit replicas: the state
// update (and published energy) of every replica is done by the workgroup's
// first wave, so that this serial per-replica work runs once per workgroup
// instead of once in every group.  es_l: lane g's words to publish its energy
// in, with tag `tag`, or nullptr.  Called by every thread; the state and s_red
// are the first wave's until the caller's next workgroup barrier.  Pool
// partials (PoolInfo): thread t's changes are kept in pp[k*nr + t] (nr =
// R*rem, k < NC+1; pp is the frame area, free between a sweep's frames and the
// next tail); replica g adds its rem entries in thread order.  Wave pw, which
// decides the swaps, keeps the energies for itself (e_pw, of the lane's group).
template <int NC>
__device__ __forceinline__ void tail_wave0(double* s_red, double* s_st, int R, int TPR, const double* v, bool therm_end,
                                           uint64_t* es_l, uint32_t tag, const double* pp, int prem, int pw,
                                           double& e_pw) {
  const int tx = tid();
  wave0_add<NC>(s_red, TPR, v, pw, [&](int g, int k, double x) {
    if (prem > 0) {
      double ps = 0.0;
      for (int i = 0; i < prem; ++i) ps += pp[k * R * prem + g * prem + i];
      x += ps;
    }
    if (k == 0) e_pw += x;
    if (tx < 64) s_st[g * MCG_NSTATE + MCG_S_E + k] += x;
  });
  if (tx < 64) {
    wave_lds_fence();
    const int lane = tx;
    if (lane < R) {
      double* st = s_st + lane * MCG_NSTATE;
      if (es_l) tag_store(es_l, tag, st[MCG_S_E]);
      if (therm_end) st[MCG_S_EREF] = st[MCG_S_E];
    }
  }
}

// one sweep of a workgroup's replica group: every colour class in turn,
// own Philox groups (changes counted in fE, fM) and, for a split replica,
// the other parts' groups this part depends on (changes not counted)
template <int NC, typename ST, int MODE>
__device__ __forceinline__ void sweep_colours(const mcg_graph& G, const Spins<ST>& sp, const float* coup,
                                              const float* clsdat, const int32_t* s_colptr, const uint8_t* s_pid,
                                              const int32_t* s_pat, int lt, int TPR, Acc beta, float h, uint64_t kk,
                                              uint32_t key0, uint32_t key1, const PartInfo& pi, float& fE, float* fM,
                                              bool aniso, const PoolInfo<ST>& pl, bool pfresh) {
  constexpr int GD = SitesPerDraw<NC>::G;
  const bool split = pi.np > 1;
  beta.beta = in_vgpr(beta.beta);
  h = in_vgpr(h);
  // A colour's groups are dealt out in rounds of TPR; the last, partial
  // round falls to the first lanes of the deal.  The deal starts at wave r
  // of the group, chosen so that the groups' partial rounds land on
  // different SIMDs (wave w of a workgroup runs on SIMD w % 4).  Which
  // thread takes a Philox group does not change its result.
  {
    const int nw = TPR >> 6, g = (int)threadIdx.x / TPR;
    const int r = nw >= 4 ? g & 3 : nw == 2 ? (g >> 1) & 1 : 0;
    lt = lt - 64 * r;
    if (lt < 0) lt += TPR;
  }
  const LdsView<NC, ST> v{sp.p, sp.n};
  auto colours = [&](auto pc, auto uc, const auto& T) {
    constexpr bool PAT = decltype(pc)::value, UNI = decltype(uc)::value;
    with_links<PAT, UNI>(T, [&](auto zc) {
      constexpr int Z = decltype(zc)::value;
      for (int c = 0; c < G.ncol; ++c) {
        const int b = s_colptr[c], cnt = s_colptr[c + 1] - b;
        const int ngrp = (cnt + GD - 1) / GD;
        const int q0 = split ? (int)((int64_t)ngrp * pi.part / pi.np) : 0;
        const int q1 = split ? (int)((int64_t)ngrp * (pi.part + 1) / pi.np) : ngrp;
        const int qm = q1 - pl.rem;  // the pool takes the last rem groups (unsplit replicas only)
        int q = q0 + lt;
        for (; q < qm; q += TPR) metro_sites<NC, PAT, UNI, Z>(v, b, cnt, q, c, T, beta, h, kk, key0, key1, fE, fM);
        if constexpr (PAT) {
          if (pl.pr >= 0) {
            const float4 pv = pl.par[pl.pr];
            float pe = 0.0f, pm[3] = {0.0f, 0.0f, 0.0f};
            const LdsView<NC, ST> pv_s{pl.spin0 + pl.sstride * pl.pr, G.n};
            metro_sites<NC, PAT, UNI, Z>(pv_s, b, cnt, qm + pl.pq, c, T, beta.at(pv.x, __float_as_int(pv.w), pl.pr), pv.y, kk,
                                         key0, __float_as_uint(pv.z), pe, pm);
            // the first pool group after a tail stores, later ones add
            double* pp = pl.pp + threadIdx.x;
            const bool first = pfresh && c == 0;
            pp[0] = first ? (double)pe : pp[0] + (double)pe;
#pragma unroll
            for (int k = 1; k <= NC; ++k) pp[k * pl.nr] = first ? (double)pm[k - 1] : pp[k * pl.nr] + (double)pm[k - 1];
          }
        }
        if (split) {
          // A split part's recomputed groups continue the round-robin of its
          // own groups: a thread whose own loop ends at q (the first q >= q1
          // of its deal) takes xl[q - q1], xl[q - q1 + TPR], ...  They fill
          // the part's last own round: a round of them alone would cost about
          // as much as a full one (one wave's dependent chain).
          const int nx = pi.hx[2 * c + 1];
          const int32_t* xl = pi.halo + pi.hx[2 * c];
          float xE = 0.0f, xM[3] = {0.0f, 0.0f, 0.0f};
          for (int j = q - qm; j < nx; j += TPR)
            metro_sites<NC, PAT, UNI, Z>(v, b, cnt, xl[j], c, T, beta, h, kk, key0, key1, xE, xM);
        }
        __syncthreads();
      }
    });
  };
  typedef std::true_type Y;
  typedef std::false_type N;
  if constexpr (MODE == 0 || MODE == 3) {
    constexpr bool UNI = MODE == 3;
    colours(Y(), std::integral_constant<bool, UNI>(),
            sweep_tab<NC, UNI>(G, s_pat, s_pid, coup, COUP_LDS, coup + (UNI ? G.ucid : 0) * COUP_LDS, clsdat, aniso));
  } else if constexpr (MODE == 1) {
    if (G.ucid >= 0)
      colours(N(), Y(), sweep_tab<NC, true>(G, s_pat, s_pid, coup, COUP_LDS, coup + G.ucid * COUP_LDS, clsdat, aniso));
    else
      colours(N(), N(), sweep_tab<NC, false>(G, s_pat, s_pid, coup, COUP_LDS, coup, clsdat, aniso));
  } else {
    const GAS float* gc = gas(coup);
    if (G.ucid >= 0)
      colours(N(), Y(), sweep_tab<NC, true>(G, s_pat, s_pid, gc, 9, gc + G.ucid * 9, gas(clsdat), aniso));
    else
      colours(N(), N(), sweep_tab<NC, false>(G, s_pat, s_pid, gc, 9, gc, gas(clsdat), aniso));
  }
}

// sweep loop of one LDS block; MODE 0: pattern links (colour-permuted
// replica), 1: global link table with LDS-staged couplings/classes, 2:
// global link table with couplings/classes read from HBM (> 256 tensors or
// classes).  Each mode is its own instantiation so that every table pointer
// has one address space.
template <int NC, typename ST, int MODE, bool FULL>
__device__ __forceinline__ void lds_sweeps(const mcg_graph& G, const mcg_batch& B, const SweepArgs& a,
                                           const Spins<ST>& sp, const float* coup,
                                           const float* clsdat, const int32_t* s_colptr, const uint8_t* s_pid,
                                           const int32_t* s_pat, double* st, FrameCtx& C, int lt, int TPR, int row,
                                           const Acc& beta, float h, uint32_t key0, uint32_t key1, const PartInfo& pi,
                                           double& dE, double* dM, bool aniso, const PoolInfo<ST>& pl, double* mp) {
  const bool split = pi.np > 1;
  dE = 0.0;
  dM[0] = dM[1] = dM[2] = 0.0;
  bool pfresh = true;  // the next pool group starts the pool partials
  for (int s = 0; s < a.nsweeps; ++s) {
    const int64_t k = a.k_begin + s;
    const uint64_t kk = (uint64_t)(a.philox_base + k);
    const bool meas = k >= a.nthermal && ((k - a.nthermal + 1) % a.spf) == 0;
    float fE = 0.0f, fM[3] = {0.0f, 0.0f, 0.0f};  // this sweep's accepted changes
    sweep_colours<NC, ST, MODE>(G, sp, coup, clsdat, s_colptr, s_pid, s_pat, lt, TPR, beta, h, kk, key0, key1, pi, fE,
                                fM, aniso, pl, pfresh);
    pfresh = false;
    dE += (double)fE;
    dM[0] += (double)fM[0];
    dM[1] += (double)fM[1];
    dM[2] += (double)fM[2];
    if (split) continue;  // one sweep per launch; the last part to finish runs the tail
    const bool therm_end = (k + 1 == a.nthermal);
    const bool rec = recompute_due(B, a.philox_base + k);
    if (meas || therm_end || rec || s == a.nsweeps - 1) {
      lds_sweep_tail<NC, ST, FULL>(sp, G, B, st, C, row, h, k, a, meas, therm_end, rec, dE, dM, key0, key1, mp, pl);
      pfresh = true;
    }
  }
}

// The kernel's arguments, and the same read again from the kernel's argument
// memory: the persistent loop's parts read what they use where they use it (a
// few scalar loads), so that some 60 words of arguments do not live, spilled,
// across the sweeps.
struct LdsArgs {
  mcg_batch B;
  const WorkItem* items;
  const ItemRep* recs;
  SweepArgs a;
};
__device__ __forceinline__ const LdsArgs& args_again() {
  uint64_t x = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(x));
  return *(const LdsArgs*)(const __attribute__((address_space(4))) LdsArgs*)x;
}

// MODE: link mode of every graph of the launch (0 pattern, 1 global links
// with LDS tables, 2 wide); FULL: spin-derived observables are measured.
// Both are compile-time so that each instantiation carries only the code it
// runs (instruction-cache misses dominate the per-launch cost otherwise).
// PERSIST: a persistent launch (every workgroup resident, see below).
template <int NC, typename ST, int MODE, bool FULL, bool PERSIST>
__global__ __launch_bounds__(1024) void k_lds(LdsArgs A) {
  const mcg_batch& B = A.B;
  const SweepArgs& a = A.a;
  const WorkItem* __restrict__ items = A.items;
  const ItemRep* __restrict__ recs = A.recs;
  const WorkItem w = items[blockIdx.x];
  const mcg_graph G = B.graphs[w.graph];
  const int R = w.nrep;
  const int TPR = blockDim.x / R;
  // a group is whole waves, so its index, and with it the replica's record,
  // row, keys, couplings and LDS base, are scalars
  const int g = wave_uniform((int)threadIdx.x / TPR);
  const int lt = threadIdx.x - g * TPR;
  const ItemRep ir = recs[w.off + g];
  const int rep = ir.rep;
  const int row = ir.row0 + B.rung[rep];
  const float beta = B.row_beta[row], h = B.row_h[row];
  const int nwaves = blockDim.x / 64;
  const bool perm = MODE == 0 || MODE == 3;
  const int n = G.n, zmax = G.zmax;
  const bool wide = MODE == 2;
  const int ncl = wide ? 0 : G.ncoup;  // couplings staged in LDS
  const int ncs = wide ? 0 : G.ncls;   // site classes staged in LDS

  extern __shared__ __align__(16) unsigned char smem[];
  size_t off = 0;
  float* s_coup = (float*)smem;
  float* s_clsl = s_coup + ncl * COUP_LDS;
  off += align16((size_t)(ncl * COUP_LDS + ncs * 8) * 4);
  int32_t* s_colptr = (int32_t*)(smem + off);
  off += align16((size_t)(G.ncol + 1) * 4);
  int32_t* s_pat = (int32_t*)(smem + off);
  if (perm) off += align16((size_t)G.npat * pat_stride(zmax) * 4);
  uint8_t* s_pid = (uint8_t*)(smem + off);
  if (perm) off += align16((size_t)n);
  double* s_red = (double*)(smem + off);
  off += align16((size_t)nwaves * RK * 8);
  double* s_st = (double*)(smem + off);  // R * NSTATE
  double* s_frm = s_st + R * MCG_NSTATE;  // R * FRM
  double* s_mp = s_frm + R * FRM;         // the rows' previous M
  off += align16((size_t)R * (MCG_NSTATE + FRM + 1) * 8);
  float4* s_par = (float4*)(smem + off);  // per group: beta, h, key1 bits (the pool's parameters)
  off += align16((size_t)R * 16);
  unsigned char* s_pers = smem + off;  // tempering state of a persistent launch
  if (PERSIST) off += persist_lds_bytes(B.nrow);
  ST* s_spin = (ST*)(smem + off);

  for (int t = threadIdx.x; t < ncl * 9; t += blockDim.x) s_coup[t / 9 * COUP_LDS + t % 9] = G.coup[t];
  for (int t = threadIdx.x; t < ncs * 8; t += blockDim.x) s_clsl[t] = G.clsdat[t];
  // does any site class carry an on-site term? (the D terms are skipped if not)
  int anz = 0;
  for (int t = threadIdx.x; t < G.ncls; t += blockDim.x)
    anz |= (G.clsdat[t * 8 + 1] != 0.0f) | (G.clsdat[t * 8 + 2] != 0.0f) | (G.clsdat[t * 8 + 3] != 0.0f);
  const bool aniso = __syncthreads_or(anz) != 0;
  for (int t = threadIdx.x; t <= G.ncol; t += blockDim.x) s_colptr[t] = G.col_ptr[t];
  if (perm) {
    for (int t = threadIdx.x; t < G.npat * (zmax + 1); t += blockDim.x) {
      const int l = t % (zmax + 1);
      const int32_t v = G.pattab[t];
      s_pat[(t / (zmax + 1)) * pat_stride(zmax) + l] = l < zmax ? row_word<MODE == 3>(v, sizeof(ST)) : v;
    }
    for (int t = threadIdx.x; t < n; t += blockDim.x) s_pid[t] = G.pat[t];
  }

  ST* gsp = (ST*)B.spins + ir.spin_off;
  ST* my = s_spin + lds_replica_bytes(NC, n, sizeof(ST)) / sizeof(ST) * g;
  stage<ST, true>(my, gsp, NC * n, lt, TPR);
  double* st = s_st + g * MCG_NSTATE;
  if (lt < MCG_NSTATE) st[lt] = B.state[(size_t)rep * MCG_NSTATE + lt];
  if (lt == 0) s_par[g] = make_float4(beta, h, __uint_as_float(B.seed_hi ^ (uint32_t)ir.serial), __int_as_float(row));
  __syncthreads();

  const uint32_t key0 = B.seed_lo, key1 = B.seed_hi ^ (uint32_t)ir.serial;
  const Spins<ST> sp{my, n};
  // pool of the replicas' partial last rounds (PoolInfo)
  PoolInfo<ST> pl;
  if (perm && TPR == 64 && R > 1 && w.nparts <= 1) {
    constexpr int GDp = SitesPerDraw<NC>::G;
    int rem = -1;
    for (int c = 0; c < G.ncol; ++c) {
      const int rc = ((s_colptr[c + 1] - s_colptr[c] + GDp - 1) / GDp) % 64;
      rem = rem < 0 ? rc : rem == rc ? rem : 0;
    }
    if (rem > 0 && rem * 4 <= FRM) pl.rem = rem;  // partials fit the frame area
  }
  if (pl.rem > 0) {
    pl.par = s_par;
    pl.spin0 = s_spin;
    pl.sstride = (int)(lds_replica_bytes(NC, n, sizeof(ST)) / sizeof(ST));
    pl.pp = s_frm;
    pl.nr = R * pl.rem;
    if ((int)threadIdx.x < R * pl.rem) {
      pl.pr = (int)threadIdx.x / pl.rem;
      pl.pq = (int)threadIdx.x - pl.pr * pl.rem;
    }
  }
  PartInfo pi;
  if (w.nparts > 1) {
    pi.part = w.part;
    pi.np = w.nparts;
    pi.hx = a.halo + w.hoff;
    pi.halo = a.halo;
  }
  FrameCtx C{B.graphs + w.graph, wide ? G.coup : s_coup, wide ? 9 : COUP_LDS, wide ? G.clsdat : s_clsl, s_red, s_frm + g * FRM, g, lt, TPR};
  frame_consts<NC>(C, G, B);
  if (FULL && a.blk && w.nparts <= 1) C.blk = (float*)((unsigned char*)s_spin + R * lds_replica_bytes(NC, n, sizeof(ST)) + g * a.blk);
  if constexpr (PERSIST) {
    // Persistent launch: many sweeps with the replicas in LDS.  Nothing waits
    // for the whole grid, or for a whole ladder: where tempering is due a
    // replica's energy is published under its row (tagged words), and the
    // workgroup reads the energy published under the partner row and decides
    // the swap itself, as the partner's workgroup does (same energies, same
    // Philox word).  A row's words are written in turn to four slots: a slot
    // is written again four events later, by a workgroup that has got there
    // through the event two before, which has the same pairs, and so after the
    // reader of the slot had gone on (pairs alternate, or never change).
    // The parts of a split replica exchange sites after every sweep: a part
    // publishes its sums and the sites another part reads (export lists), waits
    // for these stores, then publishes its energy, whose tag the other parts
    // wait for; a part is at most one sweep ahead of the others, and the
    // parity buffers keep what the slower ones still read.
    // Measured against one barrier of all workgroups per event (two-level
    // counters, after the stores' acknowledgement and before the loads of every
    // energy of the ladder), with the end of a sweep on two waves and no
    // scratch: XY 48^2 x 48 rungs 8.2 -> 6.0 us a sweep, 96^2 x 256 rungs
    // 12.2 -> 9.8, 16^2 x 1024 rungs 9.1 -> 5.4; honeycomb 64^2 x 64 in four
    // parts each 20 -> 18.
    typedef typename RawBits<sizeof(ST)>::T U;
    constexpr int GD = SitesPerDraw<NC>::G;
    const int nrow = B.nrow;
    float* s_beta = (float*)s_pers;
    float* s_h = s_beta + nrow;
    int32_t* s_row = (int32_t*)(s_pers + align16((size_t)2 * nrow * 4));
    int2* s_lad = (int2*)(s_row + MAX_GROUPS);  // first row, rungs (0: no ladder)
    int* s_flag = (int*)(s_lad + MAX_GROUPS);
    for (int t = threadIdx.x; t < nrow; t += blockDim.x) {
      s_beta[t] = B.row_beta[t];
      s_h[t] = B.row_h[t];
    }
    if (lt == 0) {
      s_row[g] = row;
      s_lad[g] = make_int2(ir.row0, ir.nrung);
    }
    if (threadIdx.x == 0) *s_flag = 1;  // cleared by a wait that times out
    __syncthreads();
    U* lraw = (U*)my;
    U* xb = (U*)a.xbuf;
    const int DS = halo_desc_ints(G.ncol);
    uint32_t epoch = (uint32_t)a.sync_base;
    // Lane g of the first wave stands for group g (unsplit replicas) or for
    // the replica (part 0 of a split one) in the end-of-sweep work.  M' of a
    // row (for <M M'>) passes from frame to frame, and from workgroup to
    // workgroup where the row moves, in tagged words: a frame reads the words
    // of the last one's tag, then writes its own to the other slot, whose
    // reader wrote the words it has just read.  A[MPREV] seeds the words of the
    // rows held at the start and takes the last frame's M'.
    const int lane = threadIdx.x & 63;
    const int nfr = pi.np == 1 ? R : pi.part == 0 ? 1 : 0;  // groups whose frames this workgroup takes
    const bool l_grp = threadIdx.x < 64 && lane < nfr;
    // Swaps are the second wave's, so that the first wave's sums and frame and
    // the second's draw, wait and decision run side by side (each is a chain of
    // dependent instructions of one wave: 2,300 and 3,400 cycles).
    const int pw = blockDim.x >= 128 ? 1 : 0;
    const int gl = lane / group_lane_stride(TPR);
    const bool l_lad = (int)threadIdx.x >> 6 == pw && lane % group_lane_stride(TPR) == 0 && gl < R;
    double e_pw = 0.0;  // energy of the lane's replica (unsplit)
    if (l_lad) e_pw = s_st[gl * MCG_NSTATE + MCG_S_E];
    const int fflags = FULL ? B.meas : (B.meas & ~MEAS_SPIN_OBS);  // what a frame measures
    // A split part measures the pairs and circuits whose first site it owns
    // from its own copy before the parts' exchange, when none of them has
    // sites of two parts and no block spins or orbital groups are measured;
    // its sums reach part 0 through the exchange (a.fpart, by sweep parity).
    // Otherwise every part publishes its sites and, after the exchange, sums
    // its share over the published copy; part 0 waits for the others' sums.
    const bool own_frame = FULL && pi.np > 1 && !(B.meas & (MCG_MEAS_RNORM | MCG_MEAS_GROUPS)) &&
                           pi.hx[2 * G.ncol + 7] != 0;
    int64_t fcur = a.k_begin > a.nthermal ? (a.k_begin - a.nthermal) / a.spf + a.frame0 : a.frame0;  // next frame
    uint32_t ftag = (uint32_t)(fcur - a.frame0) + 1u;  // tag of the last frame's M'
    auto mprev_at = [&](uint32_t tag, int r) { return a.mprev + ((size_t)(tag & 1u) * nrow + r) * 2; };
    const int ladder_l = l_lad ? recs[w.off + gl].ladder : 0;
    int frow_l = -1;  // the row of the lane's last frame, whose M is in s_mp
    if (l_grp) {
      const int r = s_row[lane];
      tag_store(mprev_at(ftag, r), ftag, B.acc[(size_t)r * MCG_NACC + MCG_A_MPREV]);
    }
    uint32_t ev = 0;  // tempering events of this launch
    // the thread's first exported site, and (two parts) its first imported one
    int ex0 = 0, im0 = 0;
    if (pi.np > 1 && lt < pi.hx[2 * G.ncol + 1]) ex0 = a.halo[pi.hx[2 * G.ncol] + lt];
    if (pi.np == 2) {
      const int32_t* hq = pi.hx + (1 - 2 * pi.part) * DS;
      if (lt < hq[2 * G.ncol + 1]) im0 = a.halo[hq[2 * G.ncol] + lt];
    }
    // The sweeps' changes are added up (FP64, per thread) until a sweep needs
    // the energies: a frame, a swap pass, a recompute, the end.  Sweeps in
    // between end without the reduction over the workgroup.
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    bool vfresh = true;
    auto stage_frame = [&](const mcg_batch& B, const SweepArgs& a, int64_t f, uint32_t tag, int row_l, int lane) {
      const bool l_grp = lane < nfr;
      // frame f, by the first wave; tag: of the frame before; M' is read ahead
      Tagged mpw;
      const uint64_t* w = a.mprev + ((size_t)(tag & 1u) * nrow + row_l) * 2;
      if (l_grp) mpw.load_ahead(w);
      zero_terms(s_frm, nfr);
      if (l_grp) {
        double* F = s_frm + lane * FRM;
        frame_terms<NC>(C, fresh(C.G), B, s_st + lane * MCG_NSTATE, F, fflags, f, F + FRM_ACC);
        double* mm = F + FRM_ACC + MCG_A_MM;  // holds the frame's M
        const double m = *mm;
        s_mp[lane] = m;
        frow_l = row_l;
        tag_store(a.mprev + ((size_t)((tag + 1u) & 1u) * nrow + row_l) * 2, tag + 1u, m);
        *mm = tag_wait(w, mpw, tag, B.err, s_flag) * m;
      }
    };
    // sweeps until the next frame, swap pass and recompute (each event's
    // period, 0: never), so that no sweep divides 64-bit indices
    const int64_t gs0 = a.philox_base + a.k_begin;
    const int rec_every = a.rec_host ? 0 : B.recompute_every;
    auto until = [&](int every) {  // sweeps from gs0 on until one with (index + 1) % every == 0
      if (every <= 0) return 0;
      const int m = (int)(gs0 % every);
      return m < 0 ? -m : every - m;
    };
    int to_pt = until(a.pt_every), to_rec = until(rec_every);
    int64_t to_frame = a.k_begin > a.nthermal ? a.spf - (a.k_begin - a.nthermal) % a.spf
                                              : (int64_t)a.nthermal - a.k_begin + a.spf;
    const int nsweeps = a.nsweeps;
    const int64_t k_begin = a.k_begin;
    const uint64_t philox_base = (uint64_t)a.philox_base;
    const int spf = a.spf, pt_every = a.pt_every;
    const int64_t nthermal = a.nthermal;
    const bool has_split = a.has_split != 0;
    for (int s = 0; s < nsweeps; ++s) {
      const int64_t k = k_begin + s;
      const uint64_t kk = philox_base + (uint64_t)k;
      const int rowg = wave_uniform(s_row[g]);
      const float bg = wave_uniform(s_beta[rowg]), hg = wave_uniform(s_h[rowg]);
      const bool meas = --to_frame == 0;
      const bool therm_end = (k + 1 == nthermal);
      const bool rec = --to_rec == 0;
      const bool pt_now = --to_pt == 0;
      if (meas) to_frame = spf;
      if (rec) to_rec = rec_every;
      if (pt_now) to_pt = pt_every;
      const bool need = meas || therm_end || rec || pt_now || s == nsweeps - 1;
      if (pt_now || has_split) ++epoch;
      const int par = (int)(epoch & 1u);
      if (pl.rem > 0) {  // the pool's parameters of this sweep (rows move with tempering)
        if (lt == 0) s_par[g] = make_float4(bg, hg, __uint_as_float(key1), __int_as_float(rowg));
        __syncthreads();
      }
      float fE = 0.0f, fM[3] = {0.0f, 0.0f, 0.0f};
      sweep_colours<NC, ST, MODE>(G, sp, C.coup, C.clsdat, s_colptr, s_pid, s_pat, lt, TPR, acc_of(B, bg, rowg), hg, kk,
                                  key0, key1, pi,
                                  fE, fM, aniso, pl, vfresh);
      vfresh = false;
      v[0] += (double)fE;
      v[1] += (double)fM[0];
      v[2] += (double)fM[1];
      v[3] += (double)fM[2];
      const LdsArgs& A = args_again();
      const mcg_batch& B = A.B;
      const SweepArgs& a = A.a;
      const int tx = tid(), lane = tx & 63, lt = tx - g * TPR;
      const bool wave0 = tx < 64, l_grp = wave0 && lane < nfr;
      const int gl = lane / group_lane_stride(TPR);
      const bool l_lad = tx >> 6 == pw && lane == gl * group_lane_stride(TPR) && gl < R;
      // words of the row's energy (part `part`) in this event; the tag also
      // says how many parts the row's replica has
      auto row_words = [&](int r, int part) {
        return a.rowslot + ((((size_t)(ev & 3u) * nrow + r) * a.nrow_parts) + part) * 2;
      };
      const uint32_t rtag = epoch << 2;
      double e_l = 0.0;  // the lane's replica's energy
      // The swap of the lane's replica: first the draw, which does not depend
      // on the energies, then the partner's words, then the decision
      const int row_l = wave0 && lane < R ? s_row[lane] : 0;  // the frame's
      const int row_p = l_lad ? s_row[gl] : 0;
      int rb = -1;     // the partner row, if the lane's replica has one
      int t0 = 0;      // row of the pair's lower rung
      float pu = 0.0f;
      Tagged ew;
      auto swap_draw = [&] {
        if (!pt_now || !l_lad) return;
        const int2 ld = s_lad[gl];
        const int pp = (int)(kk & 1), t = row_p - ld.x;
        const bool low = ((t - pp) & 1) == 0;  // the lower rung of its pair
        const int tl = low ? t : t - 1;
        if (tl < pp || tl + 1 >= ld.y) return;
        const u32x4 x = philox4x32_10(u32x4{(uint32_t)tl, (uint32_t)kk, (uint32_t)(kk >> 32), TAG_PT}, B.seed_lo,
                                      B.seed_hi ^ (0x80000000u | (uint32_t)ladder_l));
        pu = u24(x.x);
        t0 = ld.x + tl;
        rb = low ? row_p + 1 : row_p - 1;
      };
      auto swap_read = [&] {
        if (rb >= 0) ew.load_ahead(row_words(rb, 0));
      };
      if (pi.np == 1) {
        // state update and published energy (with a full recompute due, the
        // recomputed state is published instead)
        if (need) {
          tail_wave0<NC>(s_red, s_st, R, TPR, v, therm_end && !rec,
                         pt_now && !rec && wave0 && lane < R && s_lad[lane].y > 0 ? row_words(row_l, 0) : nullptr,
                         rtag, s_frm, pl.rem, pw, e_pw);
          vfresh = true;
          v[0] = v[1] = v[2] = v[3] = 0.0;
        }
        if (rec) {
          __syncthreads();
          double* r4 = C.s_frm;
          recompute<NC>(sp, C.G, C.coup, C.cst, C.clsdat, hg, s_red, g, lt, TPR, r4);
          if (lt == 0) {
            const double d = fabs(st[MCG_S_E] - r4[0]);
            if (d > st[MCG_S_DRIFT]) st[MCG_S_DRIFT] = d;
            recompute_checks<ST>(B, G, r4, d);
            for (int q = 0; q < 4; ++q) st[MCG_S_E + q] = r4[q];
            if (therm_end) st[MCG_S_EREF] = st[MCG_S_E];
            if (pt_now && ir.nrung > 0) tag_store(row_words(rowg, 0), rtag, st[MCG_S_E]);
          }
          __syncthreads();
          if (l_lad) e_pw = s_st[gl * MCG_NSTATE + MCG_S_E];
        }
        if constexpr (FULL) {
          // the spin-derived sums of every group's frame, from its LDS
          // replica (the frame area is free after the tail); the first wave
          // takes every group's frame
          if (meas) {
            __syncthreads();
            frame_sums<NC, Spins<ST>, true>(sp, C, B, fcur, key0, key1, hg, 0, 1);
            __syncthreads();
          }
        }
        swap_draw();
        swap_read();
      } else {
        // one replica: the part's sums, published and kept in LDS
        double* ms = a.mslot + ((size_t)par * a.nslots + w.slot) * (MAX_PARTS - 1) * 3;
        if (need) {
          wave0_add<NC>(s_red, TPR, v, 0, [&](int, int q, double x) {
            if (q > 0 && pi.part > 0) dev_store(ms + (pi.part - 1) * 3 + (q - 1), x);
            if (q == 0 && pi.part == 0) x += st[MCG_S_E];
            if (q == 0 && pt_now && ir.nrung > 0)
              tag_store(row_words(rowg, pi.part), rtag | (uint32_t)(pi.np - 1), x);
            s_frm[FRM - 4 + q] = x;
          });
          v[0] = v[1] = v[2] = v[3] = 0.0;
        }
        const int32_t* ex = a.halo + pi.hx[2 * G.ncol];
        const int nex = pi.hx[2 * G.ncol + 1];
        U* xo = xb + (((size_t)par * a.nslots + w.slot) * MAX_PARTS + pi.part) * (size_t)a.max_export * NC;
        if (lt < nex) export_site<NC>(xo + (size_t)lt * NC, lraw, n, ex0);
        for (int i = lt + TPR; i < nex; i += TPR) export_site<NC>(xo + (size_t)i * NC, lraw, n, ex[i]);
        if constexpr (FULL) {
          if (meas && own_frame) {
            __syncthreads();  // s_red
            const int32_t* d = pi.hx + 2 * G.ncol;
            const PartFrame pf{a.halo + d[2], a.halo + d[4], d[3], d[5], d[6] != 0};
            frame_sums<NC, Spins<ST>, true>(sp, C, B, fcur, key0, key1, hg, pi.part, pi.np, &pf);
            if (pi.part != 0) {
              __syncthreads();  // F is written by the first thread
              double* fp = a.fpart + (((size_t)par * a.nslots + w.slot) * (MAX_PARTS - 1) + pi.part - 1) * FSUMS;
              if (tx < FSUMS_PQ) dev_store(fp + tx, s_frm[tx]);
            }
          }
          // the frame reads every part's sites: publish this part's own
          if (meas && !own_frame)
            part_publish<ST>(my, (U*)a.fspin + ((size_t)par * a.nslots + w.slot) * NC * a.fspin_n, n, a.fspin_n,
                             NC, s_colptr, G.ncol, GD, pi.part, pi.np, lt, TPR);
        }
        // the energy last: its tag says that everything above has arrived
        stores_done();
        __syncthreads();
        uint64_t* ps = a.pslot + ((size_t)par * a.nslots + w.slot) * MAX_PARTS * 2;
        const double own_e = need ? s_frm[FRM - 4] : 0.0;  // part 0: with the replica's energy before
        if (tx == 0) tag_store(ps + pi.part * 2, epoch, own_e);
        swap_draw();
        // the other parts' tags, lane p for part p, by the waves that need their
        // energies (every wave for itself: 3 % slower on honeycomb 64^2 x 64)
        Tagged pw;
        {
          uint32_t it = 0;
          bool ok = !(tx < 128 && lane < pi.np && lane != pi.part);
          while (!ok) {
            pw.load(ps + lane * 2);
            ok = pw.has(epoch);
            if (!ok && ++it > WAIT_POLLS) {
              wait_failed(B.err, s_flag);
              break;
            }
          }
        }
        __syncthreads();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        // part 0 reads part p's sums in lane p, overlapping the import
        const bool w0 = need && pi.part == 0 && wave0;
        const double pe = lane == pi.part ? own_e : pw.value();
        double pm[3] = {0.0, 0.0, 0.0};
        if (w0 && lane >= 1 && lane < pi.np) {
          for (int q = 0; q < NC; ++q) pm[q] = dev_load(ms + (lane - 1) * 3 + q);
        }
        swap_read();
        double Esum = lane_f64(pe, 0);  // the replica's energy: its parts', in part order
        for (int p = 1; p < pi.np; ++p) Esum += lane_f64(pe, p);
        if (pi.np == 2) {
          // the other part's list directly (measured faster than the flat
          // round-robin on the XY scan's two-part replicas)
          for (int p = 0; p < pi.np; ++p) {
            if (p == pi.part) continue;
            const int32_t* hq = pi.hx + (p - pi.part) * DS;
            const int32_t* ex = a.halo + hq[2 * G.ncol];
            const int nex = hq[2 * G.ncol + 1];
            const U* xi = xb + (((size_t)par * a.nslots + w.slot) * MAX_PARTS + p) * (size_t)a.max_export * NC;
            for (int i = lt; i < nex; i += TPR) {
              const U* src = xi + (size_t)i * NC;
              const int site = i < TPR ? im0 : ex[i];
              constexpr int W = NC * (int)sizeof(U);
              if constexpr (W == 8 || W == 4) {
                typedef typename std::conditional<W == 8, uint64_t, uint32_t>::type P;
                const P w = dev_load((const P*)src);
#pragma unroll
                for (int q = 0; q < NC; ++q) lraw[(size_t)q * n + site] = (U)(w >> (q * 8 * sizeof(U)));
              } else {
#pragma unroll
                for (int q = 0; q < NC; ++q) lraw[(size_t)q * n + site] = dev_load(src + q);
              }
            }
          }
        } else {
          import_parts<NC>(xb + ((size_t)par * a.nslots + w.slot) * MAX_PARTS * (size_t)a.max_export * NC,
                           a.max_export, a.halo, pi.hx, DS, G.ncol, pi.part, pi.np, lraw, n, lt, TPR);
        }
        e_l = Esum;
        if (w0) {
          const double* own = s_frm + FRM - 4;  // this part's sums
          double dm[3] = {own[1], NC > 1 ? own[2] : 0.0, NC > 2 ? own[3] : 0.0};
          for (int p = 1; p < pi.np; ++p)
            for (int q = 0; q < 3; ++q) dm[q] += lane_f64(pm[q], p);
          if (lane == 0) {
            st[MCG_S_E] = Esum;
            for (int q = 0; q < 3; ++q) st[MCG_S_M + q] += dm[q];
            if (therm_end) st[MCG_S_EREF] = st[MCG_S_E];
          }
        }
        // the imported sites are read by other threads: by the frame's sums
        // over the spins, and by the next sweep's first colour
        if (FULL && meas) {
          __syncthreads();
          if (*s_flag == 0) return;
        }
      }
      if constexpr (FULL) {
        if (meas && pi.np > 1) {
          // this part's share of the spin-derived sums: from its own copy, or
          // over every part's published sites; part 0 gathers the others'
          if (own_frame) {
            // the other parts' sums, stored before the exchange, added in
            // part order
            if (pi.part == 0 && tx < FSUMS_PQ) {
              const double* fp = a.fpart + ((size_t)par * a.nslots + w.slot) * (MAX_PARTS - 1) * FSUMS + tx;
              double y[MAX_PARTS];
#pragma unroll
              for (int p = 1; p < MAX_PARTS; ++p) y[p] = p < pi.np ? dev_load(fp + (size_t)(p - 1) * FSUMS) : 0.0;
              double x = s_frm[tx];
#pragma unroll
              for (int p = 1; p < MAX_PARTS; ++p)
                if (p < pi.np) x += y[p];
              s_frm[tx] = x;
            }
            __syncthreads();
          } else {
            const DevSpins<ST> dsp{(const U*)a.fspin + ((size_t)par * a.nslots + w.slot) * NC * a.fspin_n,
                                   a.fspin_n};
            frame_sums<NC, DevSpins<ST>, true>(dsp, C, B, fcur, key0, key1, hg, pi.part, pi.np);
            if (!gather_frame_sums(a, B, s_frm, w.slot, pi.part, pi.np, fcur, s_flag)) return;
          }
        }
      }
      // the frame of every replica (first wave, lane g)
      if (meas) {
        if (wave0 && nfr > 0) stage_frame(B, a, fcur, ftag, row_l, lane);
        ++ftag;
        ++fcur;
      }
      if (pt_now) {
        // the swaps of the workgroup's replicas
        if (rb >= 0) {
          double eb = 0.0;
          uint32_t it = 0;
          for (int q = 0, np = 1; q < np;) {
            if (ew.has(rtag, 3u)) {
              np = (int)((uint32_t)(ew.a >> 32) & 3u) + 1;
              eb = q ? eb + ew.value() : ew.value();  // in part order
              if (++q == np) break;
            } else if (++it > WAIT_POLLS) {
              wait_failed(B.err, s_flag);
              break;
            }
            ew.load(row_words(rb, q));
          }
          const bool low = rb > row_p;
          const double ea = pi.np == 1 ? e_pw : e_l;
          const double ba = s_beta[t0], bb = s_beta[t0 + 1];
          const double d = (ba - bb) * (low ? ea - eb : eb - ea);
          if (d >= 0.0 || pu < exp_neg((float)d)) {
            if (low && pi.part == 0) atomicAdd(B.pt_acc + t0, 1);
            s_row[gl] = rb;
          }
        }
        ++ev;
      }
      if (pt_now || meas || pi.np > 1) {
        __syncthreads();
        if (*s_flag == 0) return;
      }
      if (meas && g < nfr) flush_frame<NC>(C, B, rowg, fflags);
    }
    __syncthreads();
    if (frow_l >= 0) B.acc[(size_t)frow_l * MCG_NACC + MCG_A_MPREV] = s_mp[lane];
    if (pi.np == 1)
      stage<ST, false>(my, gsp, NC * n, lt, TPR);
    else
      part_copy<ST, true>(my, gsp, n, NC, s_colptr, G.ncol, GD, pi.part, pi.np, lt, TPR);
    if (pi.part == 0 && lt < MCG_NSTATE) B.state[(size_t)rep * MCG_NSTATE + lt] = st[lt];
    if (l_grp && s_lad[lane].y > 0) {  // every row is held by one replica
      const int r = s_row[lane], q = recs[w.off + lane].rep;
      B.who[r] = q;
      B.rung[q] = r - s_lad[lane].x;
    }
    return;
  } else {
  double dE, dM[3];
  double* mp = s_mp + g;
  Acc acc = acc_of(B, beta, row);
  if constexpr (NC == 1) {
    // the rows' thresholds into LDS: a flip's decision is the last link of the
    // chain of a colour's round, and waited for L2 there.
    // Ising 32^2 x 16, 200 sweeps with frames: 964 -> 905 us.
    if (a.thr) {
      uint32_t* s_thr = (uint32_t*)((unsigned char*)s_spin + R * (lds_replica_bytes(NC, n, sizeof(ST)) + a.blk));
      acc.lstride = a.thr / 4;
      acc.lds0 = s_thr;
      acc.lds = s_thr + g * acc.lstride;
      for (int t = lt; t < B.nthr; t += TPR) s_thr[g * acc.lstride + t] = acc.thr[t];
      __syncthreads();
    }
  }
  if (lt == 0) *mp = B.acc[(size_t)row * MCG_NACC + MCG_A_MPREV];  // read by the same thread
  lds_sweeps<NC, ST, MODE, FULL>(G, B, a, sp, C.coup, C.clsdat, s_colptr, s_pid, s_pat, st, C, lt, TPR, row, acc, h,
                                 key0, key1, pi, dE, dM, aniso, pl, mp);
  __syncthreads();
  if (pi.np == 1) {
    stage<ST, false>(my, gsp, NC * n, lt, TPR);
    if (lt < MCG_NSTATE) B.state[(size_t)rep * MCG_NSTATE + lt] = st[lt];
    if (lt == 0 && a.k_begin + a.nsweeps > a.nthermal) B.acc[(size_t)row * MCG_NACC + MCG_A_MPREV] = *mp;
    return;
  }
  // split replica (one workgroup per part, R = 1): write back own sites,
  // publish the partial sums, count in; the last part to arrive finishes
  // the sweep.  It needs the other parts' sites only when this sweep is
  // measured with observables taken from the spins, or recomputed; then the
  // parts make their sites visible device-wide (one L2 write-back per
  // workgroup) and the last part reads them after an acquire.
  constexpr int GD = SitesPerDraw<NC>::G;
  const int64_t k = a.k_begin;
  const bool meas = k >= a.nthermal && ((k - a.nthermal + 1) % a.spf) == 0;
  const bool therm_end = (k + 1 == a.nthermal);
  const bool rec = recompute_due(B, a.philox_base + k);
  const bool need_all = rec || (FULL && meas && (B.meas & MEAS_SPIN_OBS));
  uint32_t* ctr = a.sync + (size_t)w.slot * SYNC_STRIDE;
  double* xp = a.xpart + (size_t)w.slot * MAX_PARTS * 4;
  part_copy<ST, true>(my, gsp, n, NC, s_colptr, G.ncol, GD, pi.part, pi.np, lt, TPR);
  const double v[4] = {dE, dM[0], dM[1], dM[2]};
  double* tot = s_frm;  // this part's sums (the frame area)
  group_add<4>(v, s_red, g, TPR, [&](int q, double x) {
    tot[q] = x;
    dev_store(xp + pi.part * 4 + q, x);
  });
  stores_done();
  __syncthreads();
  int* s_last = (int*)s_red;
  if (lt == 0) {
    if (need_all) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    *s_last = (__hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) % pi.np) ==
              (uint32_t)(pi.np - 1);
  }
  __syncthreads();
  if (!*s_last) return;
  if (need_all) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    for (int p = 0; p < pi.np; ++p)
      if (p != pi.part) part_copy<ST, false>(my, gsp, n, NC, s_colptr, G.ncol, GD, p, pi.np, lt, TPR);
  }
  double tE = 0.0, tM[3] = {0.0, 0.0, 0.0};
  if (lt == 0)
    for (int p = 0; p < pi.np; ++p) {
      tE += p == pi.part ? tot[0] : dev_load(xp + p * 4);
      for (int q = 0; q < 3; ++q) tM[q] += p == pi.part ? tot[1 + q] : dev_load(xp + p * 4 + 1 + q);
    }
  if (lt == 0) *mp = frame_mprev(B, row);  // an earlier launch's last part stored it
  __syncthreads();
  lds_sweep_tail<NC, ST, FULL>(sp, G, B, st, C, row, h, k, a, meas, therm_end, rec, tE, tM, key0, key1, mp,
                               PoolInfo<ST>{});
  if (meas && lt == 0) dev_store(B.acc + (size_t)row * MCG_NACC + MCG_A_MPREV, *mp);
  if (lt < MCG_NSTATE) B.state[(size_t)rep * MCG_NSTATE + lt] = st[lt];
  }
}

// ---------------------------------------------------------------------------
// k_pass: one colour class of every listed replica, spins in HBM / L2.
// grid = (chunks, nrep) of 256 threads; thread t of chunk x takes the Philox
// groups (x * PASS_GPT + u) * 256 + t of the colour, u < PASS_GPT, so that
// a wave touches consecutive positions and each thread's reduction is shared
// by PASS_GPT groups.  Graphs with link patterns read their neighbours as
// position deltas from pattern rows staged in LDS (no link-table traffic); the
// others read the global link table.  Bound: HBM traffic and the round trips
// of one update (pattern, spins, store).  Measured on cubic 64^3 x 128 T
// (16.8M updates, 615 MB a pass): 241 -> 160 us when the links came to be read
// together through 32-bit offsets (2.6 -> 3.8 TB/s; a copy reaches 5.3), and
// 61 us for each 64 replicas (5.0 TB/s) since they come in groups that the
// last-level cache holds.
// Changes of E and M: FP32 per thread, FP64 DPP wave sums, one device
// atomic per value per block.
// ---------------------------------------------------------------------------
// Philox groups per thread and the unrolling of that loop (measured on the
// cubic 64^3 and triangular 128^2 streaming sets: 8 groups, not unrolled,
// is 7 % faster than 4 unrolled and 22 % faster than 2)
#ifndef MCG_PASS_GPT
#define MCG_PASS_GPT 8
#endif
#ifndef MCG_PASS_UNROLL
#define MCG_PASS_UNROLL 1
#endif
static constexpr int PASS_GPT = MCG_PASS_GPT;
static constexpr int PASS_PAT_INTS = 4096;  // most LDS for pattern rows (16 KB)
// the pass uses link patterns, and its LDS for them: rows, and the couplings
// of graphs that have several
__host__ __device__ inline bool pass_patterns(const mcg_graph& G) {
  return G.npat > 0 && G.lcid == nullptr && G.npat * pat_stride(G.zmax) <= PASS_PAT_INTS;
}
// the pass's link mode of a graph (a compile-time argument of k_pass, so that
// each instantiation has only its own loads in registers: together they
// exceed the 64 that 8 waves per SIMD leave)
enum { PASS_LINKS = 0, PASS_LINKS_UNI = 1, PASS_PAT = 2, PASS_PAT_UNI = 3, PASS_MODES = 4 };
__host__ __device__ inline int pass_mode(const mcg_graph& G) { return (pass_patterns(G) ? 2 : 0) + (G.ucid >= 0 ? 1 : 0); }
__host__ __device__ inline size_t pass_lds_bytes(const mcg_graph& G) {
  return pass_patterns(G) ? (size_t)G.npat * pat_stride(G.zmax) * 4 + (G.ucid >= 0 ? 0 : (size_t)G.ncoup * COUP_LDS * 4)
                          : 0;
}
// Workgroups are dealt to the 8 XCDs in turn (workgroup b to XCD b % 8),
// and each XCD has its own L2.  xcd_item maps workgroup b to a work item so
// that every XCD takes one contiguous run of the `total` items: the items of
// a run are neighbouring chunks of a replica, whose neighbour sites then
// come from that XCD's L2 instead of being fetched again by another XCD.
// The grid has 8 * ceil(total / 8) workgroups; -1: no item.
static constexpr int NXCD = 8;
__device__ __forceinline__ int xcd_item(int b, int total) {
  const int per = (total + NXCD - 1) / NXCD;
  const int w = (b % NXCD) * per + b / NXCD;
  return w < total ? w : -1;
}
__host__ __device__ inline int xcd_grid(int total) { return (total + NXCD - 1) / NXCD * NXCD; }

// 6 waves per SIMD (80 VGPRs): with a site's links all in flight at once, more
// waves gain nothing and 64 VGPRs spill the tensors of graphs with several
// couplings.  Passes with 8, 6 and 5 waves: triangular 128^2 x 1024 (with its
// frames) 1.85, 1.68, 1.68 ms; cubic 64^3 x 128 2.59, 2.55, 2.59 ms.
#ifndef MCG_PASS_MIN_WAVES
#define MCG_PASS_MIN_WAVES 6
#endif
template <int NC, typename ST, int MODE>
__global__ __launch_bounds__(256, MCG_PASS_MIN_WAVES) void k_pass(mcg_batch B, const int32_t* __restrict__ rep_list, int colour,
                                              int64_t sweep, int nchunk, int nitems) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double s_red[4 * 4];
  const int item = xcd_item(blockIdx.x, nitems);
  if (item < 0) return;  // the whole workgroup
  const int chunk = item % nchunk;
  const int rep = rep_list[item / nchunk];
  const mcg_replica rp = B.reps[rep];
  const mcg_graph G = B.graphs[rp.graph];
  const int zmax = G.zmax;
  constexpr bool pats = MODE >= PASS_PAT, uni = (MODE & 1) != 0;
  int32_t* s_pat = (int32_t*)smem;
  float* s_coup = (float*)(s_pat + G.npat * pat_stride(zmax));
  int anz = 0;
  if (pats) {
    for (int t = threadIdx.x; t < G.npat * (zmax + 1); t += blockDim.x) {
      const int l = t % (zmax + 1);
      const int32_t w = G.pattab[t];
      s_pat[t / (zmax + 1) * pat_stride(zmax) + l] = l == zmax ? w : row_word<uni>(w, sizeof(ST));
    }
    if (!uni)
      for (int t = threadIdx.x; t < G.ncoup * 9; t += blockDim.x) s_coup[t / 9 * COUP_LDS + t % 9] = G.coup[t];
  }
  // does any site class carry an on-site term? (the D terms are skipped if not)
  for (int t = threadIdx.x; t < G.ncls; t += blockDim.x)
    anz |= (G.clsdat[t * 8 + 1] != 0.0f) | (G.clsdat[t * 8 + 2] != 0.0f) | (G.clsdat[t * 8 + 3] != 0.0f);
  const bool aniso = __syncthreads_or(anz) != 0;
  float dE = 0.0f, dM[3] = {0.0f, 0.0f, 0.0f};
  if (colour < G.ncol) {
    const int b = G.col_ptr[colour], cnt = G.col_ptr[colour + 1] - b;
    const int ngrp = (cnt + SitesPerDraw<NC>::G - 1) / SitesPerDraw<NC>::G;
    const int row = rp.row0 + B.rung[rep];
    const float h = in_vgpr(B.row_h[row]);
    const Acc beta = acc_of(B, in_vgpr(B.row_beta[row]), row);
    const uint32_t key1 = B.seed_hi ^ rp.serial;
    GAS ST* spins = gas((ST*)B.spins + rp.spin_off);
    const HbmView<NC, ST> v(spins, G.n);
    auto pass = [&](const auto& T) {
      with_links<pats, uni>(T, [&](auto zc) {
#pragma unroll MCG_PASS_UNROLL
        for (int u = 0; u < PASS_GPT; ++u) {
          const int q = (chunk * PASS_GPT + u) * (int)blockDim.x + (int)threadIdx.x;
          if (q >= ngrp) break;
          metro_sites<NC, pats, uni, decltype(zc)::value>(v, b, cnt, q, colour, T, beta, h, (uint64_t)sweep, B.seed_lo,
                                                          key1, dE, dM);
        }
      });
    };
    const GAS float *gc = gas(G.coup), *uc = gc + (uni ? G.ucid * 9 : 0);
    if constexpr (pats)
      pass(sweep_tab<NC, uni>(G, s_pat, gas(G.pat), s_coup, COUP_LDS, uc, gas(G.clsdat), aniso));
    else
      pass(sweep_tab<NC, uni>(G, s_pat, gas(G.pat), gc, 9, uc, gas(G.clsdat), aniso));
  }
  // every lane reaches here: DPP sums per wave, the waves' totals through LDS
  double v[4] = {(double)dE, (double)dM[0], (double)dM[1], (double)dM[2]};
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = wave_sum_f64(v[k]);
  const int tx = tid(), lane = tx & 63, wave = tx >> 6;
  if (lane == 63)
#pragma unroll
    for (int k = 0; k < 4; ++k) s_red[wave * 4 + k] = v[k];
  __syncthreads();
  if (threadIdx.x < 4) {
    double t = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += s_red[w * 4 + threadIdx.x];
    if (t != 0.0) atomicAdd(B.state + (size_t)rep * MCG_NSTATE + MCG_S_E + threadIdx.x, t);
  }
}

// ---------------------------------------------------------------------------
// k_measure: one block per replica.  mode bits: 1 recompute, 2 set E_ref,
// 4 measure frame, 8 reset drift
// ---------------------------------------------------------------------------
template <int NC, typename ST>
__global__ __launch_bounds__(1024) void k_measure(mcg_batch B, const int32_t* __restrict__ rep_list, int mode,
                                                  int64_t frame) {
  const int rep = rep_list[blockIdx.x];
  const mcg_replica rp = B.reps[rep];
  const mcg_graph G = B.graphs[rp.graph];
  __shared__ double s_red[16 * RK];
  __shared__ double s_frm[FRM];
  __shared__ double st[MCG_NSTATE];
  const Spins<ST> sp{(ST*)B.spins + rp.spin_off, G.n};
  const int row = rp.row0 + B.rung[rep];
  const float h = B.row_h[row];
  if (threadIdx.x < MCG_NSTATE) st[threadIdx.x] = B.state[(size_t)rep * MCG_NSTATE + threadIdx.x];
  __syncthreads();
  if (mode & 1) {
    double* r4 = s_frm;
    recompute<NC>(sp, B.graphs + rp.graph, G.coup, 9, G.clsdat, h, s_red, 0, threadIdx.x, blockDim.x, r4);
    if (threadIdx.x == 0) {
      double d = 0.0;
      if (!(mode & 8)) {
        d = fabs(st[MCG_S_E] - r4[0]);
        if (d > st[MCG_S_DRIFT]) st[MCG_S_DRIFT] = d;
      }
      recompute_checks<ST>(B, G, r4, d);
      st[MCG_S_E] = r4[0];
      st[MCG_S_M] = r4[1];
      st[MCG_S_M + 1] = r4[2];
      st[MCG_S_M + 2] = r4[3];
    }
  }
  if ((mode & 2) && threadIdx.x == 0) st[MCG_S_EREF] = st[MCG_S_E];
  __syncthreads();
  if (mode & 4) {
    FrameCtx C{B.graphs + rp.graph, G.coup, 9, G.clsdat, s_red, s_frm, 0, (int)threadIdx.x, (int)blockDim.x};
    frame_consts<NC>(C, G, B);
    __shared__ double mp;
    if (threadIdx.x == 0) mp = frame_mprev(B, row);
    measure_frame<NC>(sp, C, B, st, row, frame, B.seed_lo, B.seed_hi ^ rp.serial, h, &mp);
    if (threadIdx.x == 0) B.acc[(size_t)row * MCG_NACC + MCG_A_MPREV] = mp;
  }
  __syncthreads();
  if (threadIdx.x < MCG_NSTATE) B.state[(size_t)rep * MCG_NSTATE + threadIdx.x] = st[threadIdx.x];
}

// ---------------------------------------------------------------------------
// Split measurement (streaming and Wolff paths): k_frame_part gives np
// workgroups to each replica, each reducing its share of the frame sums and
// of the full recompute and adding them into the replica's row of fsum;
// k_frame_end (one wave per replica) turns a row into the recompute
// bookkeeping and the frame's accumulator terms, and clears it.  mode bits
// as k_measure: 1 recompute, 2 set E_ref, 4 measure frame, 8 reset drift.
// ---------------------------------------------------------------------------
static constexpr int FSLOTS = FSUMS + 8;  // per replica: frame sums, then NREC recompute sums
template <int NC, typename ST>
__global__ __launch_bounds__(256) void k_frame_part(mcg_batch B, const int32_t* __restrict__ rep_list, int mode,
                                                    int64_t frame, double* __restrict__ fsum, int np, int nitems) {
  const int item = xcd_item(blockIdx.x, nitems);
  if (item < 0) return;  // the whole workgroup
  const int rep = rep_list[item / np];
  const mcg_replica rp = B.reps[rep];
  const mcg_graph G = B.graphs[rp.graph];
  __shared__ double s_red[4 * RK];
  __shared__ double s_frm[FSUMS];
  const HbmSpins<NC, ST> sp((ST*)B.spins + rp.spin_off, G.n);
  const int row = rp.row0 + B.rung[rep];
  const float h = B.row_h[row];
  const int part = item % np;
  double* out = fsum + (size_t)rep * FSLOTS;
  if (mode & 1) {
    double* r = s_frm;
    recompute<NC>(sp, B.graphs + rp.graph, G.coup, 9, G.clsdat, h, s_red, 0, threadIdx.x, blockDim.x, r, part, np);
    if (threadIdx.x < NREC && r[threadIdx.x] != 0.0) atomicAdd(out + FSUMS + threadIdx.x, r[threadIdx.x]);
    __syncthreads();
  }
  if (mode & 4) {
    for (int t = threadIdx.x; t < FSUMS; t += blockDim.x) s_frm[t] = 0.0;
    __syncthreads();
    FrameCtx C{B.graphs + rp.graph, G.coup, 9, G.clsdat, s_red, s_frm, 0, (int)threadIdx.x, (int)blockDim.x};
    frame_consts<NC>(C, G, B);
    frame_sums<NC>(sp, C, B, frame, B.seed_lo, B.seed_hi ^ rp.serial, h, part, np);
    __syncthreads();  // F is written by the first wave (or thread)
    for (int k = threadIdx.x; k < FSUMS; k += blockDim.x)
      if (s_frm[k] != 0.0) atomicAdd(out + k, s_frm[k]);
  }
}

template <int NC, typename ST>
__global__ __launch_bounds__(64) void k_frame_end(mcg_batch B, const int32_t* __restrict__ rep_list, int mode,
                                                  int64_t frame, double* __restrict__ fsum) {
  const int rep = rep_list[blockIdx.x];
  const mcg_replica rp = B.reps[rep];
  const mcg_graph G = B.graphs[rp.graph];
  __shared__ double s_red[RK];
  __shared__ double s_frm[FRM];
  __shared__ double st[MCG_NSTATE];
  const int lt = threadIdx.x;
  const int row = rp.row0 + B.rung[rep];
  double* in = fsum + (size_t)rep * FSLOTS;
  if (lt < MCG_NSTATE) st[lt] = B.state[(size_t)rep * MCG_NSTATE + lt];
  for (int t = lt; t < FSUMS; t += blockDim.x) s_frm[t] = in[t];
  __syncthreads();
  if ((mode & 1) && lt == 0) {
    double r[NREC];
    for (int k = 0; k < NREC; ++k) r[k] = in[FSUMS + k];
    double d = 0.0;
    if (!(mode & 8)) {
      d = fabs(st[MCG_S_E] - r[0]);
      if (d > st[MCG_S_DRIFT]) st[MCG_S_DRIFT] = d;
    }
    recompute_checks<ST>(B, G, r, d);
    for (int k = 0; k < 4; ++k) st[MCG_S_E + k] = r[k];
  }
  if ((mode & 2) && lt == 0) st[MCG_S_EREF] = st[MCG_S_E];
  __syncthreads();
  if (mode & 4) {
    FrameCtx C{B.graphs + rp.graph, G.coup, 9, G.clsdat, s_red, s_frm, 0, lt, (int)blockDim.x};
    frame_consts<NC>(C, G, B);
    zero_terms(s_frm, 1);
    if (lt == 0) {
      double* Cn = s_frm + FRM_ACC;
      frame_terms<NC>(C, G, B, st, s_frm, B.meas, frame, Cn);
      double* mprev = B.acc + (size_t)row * MCG_NACC + MCG_A_MPREV;
      const double Mf = Cn[MCG_A_MM];
      Cn[MCG_A_MM] = *mprev * Mf;
      *mprev = Mf;
    }
    __syncthreads();
    flush_frame<NC>(C, B, row, B.meas);
  }
  __syncthreads();
  for (int t = lt; t < FSLOTS; t += blockDim.x) in[t] = 0.0;
  if (lt < MCG_NSTATE) B.state[(size_t)rep * MCG_NSTATE + lt] = st[lt];
}

// ---------------------------------------------------------------------------
// k_pt: tempering swaps, one thread per ladder.  Pairs (t, t+1) with
// t = parity, parity+2, ...; parity alternates with the swap count.
// ---------------------------------------------------------------------------
// Replica-exchange swaps of one ladder (rows r0 .. r0+nr-1): pairs of one
// parity, alternating with the swap index; threads tid, tid+nthreads, ...
// take disjoint pairs.  Accept with min(1, exp((b_a - b_b)(E_a - E_b))).
__device__ void pt_ladder(const mcg_batch& B, int L, int r0, int nr, int64_t swap_index, int tid, int nthreads) {
  const int parity = (int)(swap_index & 1);
  for (int t = parity + 2 * tid; t + 1 < nr; t += 2 * nthreads) {
    const int ra = B.who[r0 + t], rb = B.who[r0 + t + 1];
    const double Ea = B.state[(size_t)ra * MCG_NSTATE + MCG_S_E], Eb = B.state[(size_t)rb * MCG_NSTATE + MCG_S_E];
    const double ba = B.row_beta[r0 + t], bb = B.row_beta[r0 + t + 1];
    const double d = (ba - bb) * (Ea - Eb);
    bool acc = d >= 0.0;
    if (!acc) {
      const u32x4 x = philox4x32_10(
          u32x4{(uint32_t)t, (uint32_t)swap_index, (uint32_t)((uint64_t)swap_index >> 32), TAG_PT}, B.seed_lo,
          B.seed_hi ^ (0x80000000u | (uint32_t)L));
      acc = u24(x.x) < exp_neg((float)d);
    }
    if (acc) {
      B.who[r0 + t] = rb;
      B.who[r0 + t + 1] = ra;
      B.rung[ra] = t + 1;
      B.rung[rb] = t;
      B.pt_acc[r0 + t] += 1;
    }
  }
}

__global__ void k_pt(mcg_batch B, const int32_t* __restrict__ ladder_row0, const int32_t* __restrict__ ladder_n,
                     int nladder, int64_t swap_index) {
  const int L = blockIdx.x;
  if (L >= nladder) return;
  pt_ladder(B, L, ladder_row0[L], ladder_n[L], swap_index, (int)threadIdx.x, (int)blockDim.x);
}

// ---------------------------------------------------------------------------
// k_wolff: one 1024-thread block per replica, ncl clusters, level-synchronous
// frontier BFS with one work item per (frontier site, link)
// (heisenbergLib.c:310-439, xyLib.c:256-380, isingLib.c:165-236)
//
// A cluster is a chain of levels, each of which waits for its slowest item.
// Everything an item needs but the neighbour's spin is therefore in LDS: the
// frontier (site, pattern and projection, computed when the site was added),
// the pattern rows, r.J.r per coupling, and the members as one bit per site
// (BITS; graphs too large for that use stamps in global memory, as before).
// An item then makes one round trip to L2, and the draw runs while it waits;
// reading frontier entry, link word, stamp, both spins and exchanging the
// stamp in global memory made five.  Cubic 64^3 at T_c, 16 replicas (clusters
// of 6,000 spins on average): 447 -> 270 us a cluster; smaller lattices gain 1.5x
// to 1.66x, clusters of a few spins 1.2x to 1.3x.  What is left is one CU's
// gathers (a cache line per lane) and draws per replica.
// ---------------------------------------------------------------------------
static constexpr int WOLFF_FRONT = 2048;  // frontier entries in LDS (a level's others are read from the member list)
static constexpr int WOLFF_RJR = 256;     // couplings whose r.J.r is kept
__host__ __device__ inline size_t wolff_lds_bytes(const mcg_graph& G, bool bits) {
  return (size_t)2 * WOLFF_FRONT * 8 + WOLFF_RJR * 4 +
         (pass_patterns(G) ? (size_t)G.npat * pat_stride(G.zmax) * 4 : 0) + (bits ? ((size_t)G.n + 127) / 128 * 16 : 0);
}
// accesses to a workgroup's private scratch in global memory (Wolff stamps
// and cluster lists): ordered among the workgroup's threads only
template <typename T>
__device__ __forceinline__ T wg_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename T>
__device__ __forceinline__ void wg_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int NC, typename ST, bool BITS>
__global__ __launch_bounds__(1024) void k_wolff(mcg_batch B, const int32_t* __restrict__ rep_list, int64_t cl0,
                                                int ncl) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint2* s_front = (uint2*)smem;  // [2][WOLFF_FRONT]: site | pattern << 24, projection (Ising: spin)
  float* s_rjr = (float*)(s_front + 2 * WOLFF_FRONT);
  int32_t* s_rows = (int32_t*)(s_rjr + WOLFF_RJR);
  const int rep = rep_list[blockIdx.x];
  const mcg_replica rp = B.reps[rep];
  const mcg_graph G = B.graphs[rp.graph];
  const GSpins<ST> sp{gas((ST*)B.spins + rp.spin_off), G.n};
  uint32_t* stamp = B.wstamp + rp.site_off;
  int32_t* mem = B.wlist + rp.site_off;
  const int row = rp.row0 + B.rung[rep];
  const float beta = B.row_beta[row], h = B.row_h[row];
  const uint32_t key0 = B.seed_lo, key1 = B.seed_hi ^ rp.serial;
  __shared__ int s_nc[3];
  __shared__ double s_red[16];
  __shared__ int s_acc;
  const int tid = threadIdx.x;
  const bool pats = pass_patterns(G), wide = G.lcid != nullptr;
  const int pstride = pat_stride(G.zmax);
  uint32_t* s_bits = (uint32_t*)(s_rows + (pats ? G.npat * pstride : 0));
  if (pats)
    for (int t = tid; t < G.npat * (G.zmax + 1); t += blockDim.x) {
      const int l = t % (G.zmax + 1);
      const int32_t w = G.pattab[t];
      s_rows[t / (G.zmax + 1) * pstride + l] = l == G.zmax ? w : row_word<false>(w, sizeof(ST));
    }
  // isotropic exchange (every tensor c*I on the spin components) and no
  // single-ion term: with h = 0 the cluster's acceptance energy
  // (heisenbergLib.c:403-423) is zero in exact arithmetic, so the cluster is
  // accepted without evaluating it (Ising: zero whenever h = 0)
  bool iso_ok = true;
  if constexpr (NC > 1) {
    for (int c = tid; c < G.ncoup; c += blockDim.x) {
      const float* J = G.coup + c * 9;
      iso_ok = iso_ok && J[1] == 0.0f && J[3] == 0.0f && J[0] == J[4];
      if (NC == 3) iso_ok = iso_ok && J[2] == 0.0f && J[5] == 0.0f && J[6] == 0.0f && J[7] == 0.0f && J[8] == J[0];
    }
    for (int c = tid; c < G.ncls; c += blockDim.x)
      for (int k = 0; k < NC; ++k) iso_ok = iso_ok && G.clsdat[c * 8 + 1 + k] == 0.0f;
  }
  const bool skip_acc = __syncthreads_and(iso_ok ? 1 : 0) != 0 && h == 0.0f;
  const uint32_t zl = (uint32_t)G.zmax, zmagic = zl > 0 ? 0xFFFFFFFFu / zl : 0u;
  double grown = 0.0, flipped = 0.0;  // sites grown and flipped (first thread)
  auto clear_bits = [&] {
    if (BITS)
      for (int w = tid; w < (G.n + 127) / 128; w += blockDim.x) ((uint4*)s_bits)[w] = make_uint4(0u, 0u, 0u, 0u);
  };
  clear_bits();
  __syncthreads();

  for (int c = 0; c < ncl; ++c) {
    const uint64_t cl = (uint64_t)(cl0 + c);
    const uint32_t cur = (uint32_t)(cl & 0x7FFFFFFFu) * 2u + 1u;  // odd: never 0
    // every thread draws the seed and the direction: no broadcast to wait for
    const u32x4 x0 = philox4x32_10(u32x4{0u, (uint32_t)cl, (uint32_t)(cl >> 32), TAG_WOLFF}, key0, key1);
    const int seed = (int)(((uint64_t)x0.x * (uint64_t)G.n) >> 32);
    float r0 = 0.0f, r1 = 0.0f, r2 = 0.0f;
    if constexpr (NC == 3) {
      r2 = fmaf(u24(x0.y), 2.0f, -1.0f);
      const float rho = unit_rho(r2);
      float cc, sn;
      sincos_turn(x0.z, &cc, &sn);
      r0 = rho * cc;
      r1 = rho * sn;
    } else if constexpr (NC == 2) {
      sincos_turn(x0.y, &r0, &r1);
    }
    auto rjr = [&](const float* J) {
      return r0 * (J[0] * r0 + J[1] * r1 + J[2] * r2) + r1 * (J[3] * r0 + J[4] * r1 + J[5] * r2) +
             r2 * (J[6] * r0 + J[7] * r1 + J[8] * r2);
    };
    // the projection of a site (Ising: its spin), as used by its links
    auto project = [&](int i) {
      float v[3];
      spin_vec<NC>(sp, i, G.cls, G.clsdat, v);
      return NC == 1 ? v[0] : -(v[0] * r0 + v[1] * r1 + v[2] * r2);
    };
    auto entry = [&](int i, float pj) {
      return make_uint2((uint32_t)i | (pats ? (uint32_t)gas(G.pat)[i] << 24 : 0u), __float_as_uint(pj));
    };
    if (!wide)
      for (int q = tid; q < G.ncoup; q += blockDim.x) s_rjr[q] = NC == 1 ? G.coup[q * 9] : rjr(G.coup + q * 9);
    if (tid == 0) {
      const uint2 e0 = entry(seed, project(seed));
      if (BITS)
        s_bits[seed >> 5] = 1u << (seed & 31);
      else
        wg_store(stamp + seed, cur);
      s_front[0] = e0;
      wg_store(mem, seed);
      s_nc[0] = s_nc[1] = s_nc[2] = 0;
    }
    __syncthreads();
    // Level-synchronous growth, one workgroup barrier per level: the sites
    // level k adds go to entry s_nc[k % 3]++ of the next frontier and to the
    // member list behind it.  During level k the first thread clears the
    // counter of level k+1, last read (level k-2's) before the barrier that
    // ended level k-1.
    int lo = 0, hi = 1, cnt = 1;
    for (int k = 0;; ++k) {
      const uint2* front = s_front + (k & 1) * WOLFF_FRONT;
      uint2* next = s_front + ((k + 1) & 1) * WOLFF_FRONT;
      const uint32_t nitem = (uint32_t)(hi - lo) * zl;
      for (uint32_t it = tid; it < nitem; it += blockDim.x) {
        uint32_t fq = __umulhi(it, zmagic);  // it / zl, or a little less
        while (it - fq * zl >= zl) ++fq;
        const int l = (int)(it - fq * zl);
        uint2 e;
        if (fq < (uint32_t)WOLFF_FRONT) {
          e = front[fq];
        } else {
          const int o = wg_load(mem + lo + (int)fq);
          e = entry(o, project(o));
        }
        const int o = (int)(e.x & 0xFFFFFFu);
        const float pjo = __uint_as_float(e.y);
        int t;
        uint32_t cw;
        if (pats) {
          const int32_t wd = s_rows[(e.x >> 24) * pstride + l];
          t = o + (wd >> 8);
          cw = (uint32_t)wd & 0xFFu;
        } else {
          const uint32_t wd = gas(G.link)[(size_t)o * G.zmax + l];
          t = (int)(wd & 0xFFFFFFu);
          cw = wide ? (uint32_t)gas(G.lcid)[(size_t)o * G.zmax + l] : (wd >> 24);
        }
        bool add = false;
        uint2 en = make_uint2(0u, 0u);
        const bool member = t == o || (BITS ? (s_bits[t >> 5] >> (t & 31) & 1u) != 0u : wg_load(stamp + t) == cur);
        if (!member) {
          const float pjt = project(t);
          en = entry(t, pjt);
          const float rj = !wide ? s_rjr[cw] : NC == 1 ? G.coup[cw * 9] : rjr(G.coup + cw * 9);
          const u32x4 x = philox4x32_10(
              u32x4{(uint32_t)(o * G.zmax + l), (uint32_t)cl, (uint32_t)(cl >> 32), TAG_BOND}, key0, key1);
          float corr;
          if constexpr (NC == 1) {
            corr = (rj * sp.get(t, 0)) * pjo * beta;  // J*S_t*sigma_t * s_o
            corr = 2.0f * corr;                        // add if J s s < 0, p = 1-exp(2 corr)
          } else {
            corr = 2.0f * pjo * pjt * rj * beta;
          }
          if (corr < 0.0f && 1.0f - exp_neg(corr) > u24(x.x)) {
            if (BITS) {
              const uint32_t bit = 1u << (t & 31);
              add = (atomicOr(s_bits + (t >> 5), bit) & bit) == 0u;
            } else {
              add = __hip_atomic_exchange(stamp + t, cur, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != cur;
            }
          }
        }
        // one counter update per wave for its new members
        const uint64_t who = __ballot(add);
        if (who) {
          int base = 0;
          const int first = __ffsll((unsigned long long)who) - 1, lane = tid & 63;
          if (lane == first) base = atomicAdd(&s_nc[k % 3], __popcll(who));
          base = __builtin_amdgcn_readlane(base, first);
          if (add) {
            const int pos = base + __popcll(who & ((1ull << lane) - 1ull));
            if (pos < WOLFF_FRONT) next[pos] = en;
            wg_store(mem + hi + pos, t);
          }
        }
      }
      if (tid == 0) s_nc[(k + 1) % 3] = 0;
      __syncthreads();
      const int add = s_nc[k % 3];
      if (add == 0) {
        cnt = hi;
        break;
      }
      lo = hi;
      hi += add;
    }
    // cluster acceptance energy (field / anisotropy correction)
    // O(n): one work item per (cluster site, link) plus one per site for the
    // single-ion and field terms
    double d = 0.0;
    const uint32_t zi = NC == 1 ? 1u : (uint32_t)G.zmax + 1u;
    const uint32_t nacc = skip_acc ? 0u : (uint32_t)cnt * zi;
    for (uint32_t it = tid; it < nacc; it += blockDim.x) {
      const uint32_t fq = it / zi;
      const int l = (int)(it - fq * zi);
      const int b = wg_load(mem + (int)fq);
      float sb[3];
      spin_vec<NC>(sp, b, G.cls, G.clsdat, sb);
      if constexpr (NC == 1) {
        d += (double)(2.0f * h * sb[0]);
      } else {
        const float sdb = -(sb[0] * r0 + sb[1] * r1 + sb[2] * r2);
        const float pb[3] = {sb[0] + sdb * r0, sb[1] + sdb * r1, sb[2] + sdb * r2};
        if (l < G.zmax) {
          const uint32_t wd = G.link[(size_t)b * G.zmax + l];
          const int t = (int)(wd & 0xFFFFFFu);
          const uint32_t cw = G.lcid ? (uint32_t)G.lcid[(size_t)b * G.zmax + l] : (wd >> 24);
          const float* J = G.coup + cw * 9;
          if (cw == 0u) continue;
          float stt[3];
          spin_vec<NC>(sp, t, G.cls, G.clsdat, stt);
          const float sdt = -(stt[0] * r0 + stt[1] * r1 + stt[2] * r2);
          const float pt[3] = {stt[0] + sdt * r0, stt[1] + sdt * r1, stt[2] + sdt * r2};
          // r^T J p_t
          const float src = sdb * (r0 * (J[0] * pt[0] + J[1] * pt[1] + J[2] * pt[2]) +
                                   r1 * (J[3] * pt[0] + J[4] * pt[1] + J[5] * pt[2]) +
                                   r2 * (J[6] * pt[0] + J[7] * pt[1] + J[8] * pt[2]));
          d += (double)src;
          if (BITS ? (s_bits[t >> 5] >> (t & 31) & 1u) != 0u : wg_load(stamp + t) == cur)
            d += (double)(sdt * (pb[0] * (J[0] * r0 + J[1] * r1 + J[2] * r2) +
                                 pb[1] * (J[3] * r0 + J[4] * r1 + J[5] * r2) +
                                 pb[2] * (J[6] * r0 + J[7] * r1 + J[8] * r2)));
          else
            d += (double)src;
        } else {
          // single-ion term with the half step s + sdn*r (heisenbergLib.c:418)
          const int ci = G.cls[b];
          const float* Dd = G.clsdat + ci * 8 + 1;
          const float tr[3] = {sdb * r0, sdb * r1, sdb * r2};
          float o = 0.0f;
          for (int k = 0; k < NC; ++k) {
            const float q = sb[k] + tr[k];
            o += Dd[k] * (q * q - sb[k] * sb[k]);
          }
          o -= h * tr[NC == 3 ? 2 : 0];
          d += (double)o;
        }
      }
    }
    bool flip = true;
    if (!skip_acc) {
      for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o, 64);
      if ((tid & 63) == 0) s_red[tid >> 6] = d;
      __syncthreads();
      if (tid == 0) {
        double t = 0.0;
        for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += s_red[q];
        const float db = (float)(t * (double)beta);
        s_acc = (db <= 0.0f || u24(x0.w) < exp_neg(-db)) ? 1 : 0;  // x0.w: the cluster's acceptance draw
      }
      __syncthreads();
      flip = s_acc != 0;
    }
    clear_bits();  // for the next cluster
    // cluster statistics: sites flipped and sites grown
    if (flip) flipped += (double)cnt;
    grown += (double)cnt;
    if (flip) {
      for (int f = tid; f < cnt; f += blockDim.x) {
        const int b = wg_load(mem + f);
        if constexpr (NC == 1) {
          sp.set(b, 0, -sp.get(b, 0));
        } else {
          float sb[3];
          spin_vec<NC>(sp, b, G.cls, G.clsdat, sb);
          const float a2 = -2.0f * (sb[0] * r0 + sb[1] * r1 + sb[2] * r2);
          float n0 = sb[0] + a2 * r0, n1 = sb[1] + a2 * r1, n2 = sb[2] + a2 * r2;
          float nn = n0 * n0 + n1 * n1 + n2 * n2;
          const float fct = fabsf(G.clsdat[G.cls[b] * 8]) / sqrtf(nn);
          sp.set(b, 0, n0 * fct);
          sp.set(b, 1, n1 * fct);
          if constexpr (NC == 3) sp.set(b, 2, n2 * fct);
        }
      }
    }
    __syncthreads();
  }
  if (tid == 0) {
    double* st = B.state + (size_t)rep * MCG_NSTATE;
    st[MCG_S_ACC] += flipped;
    st[MCG_S_TRY] += grown;
  }
}

// ---------------------------------------------------------------------------
// small utility kernels
// ---------------------------------------------------------------------------
__global__ void k_fill_f64(double* p, size_t n, double v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_i32(int32_t* p, size_t n, int32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// ===========================================================================
// host side
// ===========================================================================
namespace {

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  int upload(const void* src, size_t n, hipStream_t s) {
    if (n == 0) return 0;
    if (!p || bytes < n) {
      if (p) (void)hipFree(p);
      p = nullptr;
      if (hipMalloc(&p, n) != hipSuccess) return fail("hipMalloc(%zu) failed", n);
      bytes = n;
    }
    if (hipMemcpyAsync(p, src, n, hipMemcpyHostToDevice, s) != hipSuccess) return fail("hipMemcpyAsync failed");
    return 0;
  }
};

int store_size(int store) { return store == MCG_STORE_F32 ? 4 : store == MCG_STORE_F16 ? 2 : 1; }

int check_batch(const mcg_batch* B) {
  if (!B) return fail("null batch");
  if (B->nc < 1 || B->nc > 3) return fail("nc must be 1, 2 or 3 (got %d)", B->nc);
  if (B->nc == 1 && B->store != MCG_STORE_I8) return fail("Ising batches use int8 storage");
  if (B->nc > 1 && B->store == MCG_STORE_I8) return fail("int8 storage is for Ising only");
  if (!B->graphs_host || !B->reps_host) return fail("batch lacks host mirrors of graphs/reps");
  if (B->nbins < 1) return fail("nbins must be >= 1");
  for (int gi = 0; gi < B->ngraph; ++gi) {
    const mcg_graph& G = B->graphs_host[gi];
    if (G.n <= 0 || G.n > (1 << 24)) return fail("graph %d: n=%d outside 1..2^24", gi, G.n);
    if (G.ncoup < 1 || (G.ncoup > 256 && !G.lcid))
      return fail("graph %d: ncoup=%d needs per-link coupling indices (lcid) above 256", gi, G.ncoup);
    if (G.ncls < 1 || G.ncls > G.n) return fail("graph %d: ncls=%d outside 1..n", gi, G.ncls);
    if (G.ncol < 1) return fail("graph %d: no colours", gi);
    if ((B->meas & MCG_MEAS_GROUPS) && G.ngroup > 16) return fail("graph %d: more than 16 orbital groups", gi);
  }
  for (int r = 0; r < B->nrep; ++r) {
    const mcg_replica& R = B->reps_host[r];
    if (R.graph < 0 || R.graph >= B->ngraph) return fail("replica %d: bad graph index", r);
    if (R.row0 < 0 || R.row0 + R.nrung > B->nrow) return fail("replica %d: rows outside the batch", r);
  }
  return 0;
}

// A prepared run: the launch plan (host), and the device scratch the
// launches use beyond the batch's own arrays, carved from one region in
// 256-byte aligned pieces:
//   tables  work items, their replicas, replica lists, ladders, split and
//           workgroup-ladder tables; written once when the run is prepared
//   state   arrival counters, barrier words, published energies and M',
//           exported sites; every run starts them from zero (one fill kernel)
// Preparing plans and uploads; running only launches kernels, so repeated
// runs of one batch pay no planning, allocation or host copy.
struct RunCtx {
  // plan (host)
  std::vector<WorkItem> hitems;
  std::vector<int32_t> hitem_reps, hstream, hall, hhalo;
  std::vector<int32_t> hl_row0, hl_n;
  int block = 0;
  int ncu = 0;
  int nslots = 0;  // split replicas (arrival counters)
  int max_export = 0;  // longest export list of a part
  int blk = 0;  // LDS bytes per replica for a frame's block spins (0: looked up at every use)
  int thr = 0;  // and for its row's Ising thresholds (0: read from global memory)
  bool persist = false;  // persistent launches (barrier + tempering inside)
  int mode_begin[5] = {0, 0, 0, 0, 0};  // work items of link mode m: [mode_begin[m], mode_begin[m+1])
  size_t lds_max = 0;
  double lds_updates_per_sweep = 0;
  int device = 0;
  int stream_ncol = 0, stream_maxcnt = 0;  // colours and largest colour class of the streamed graphs
  uint32_t stream_lds = 0;                 // LDS of the streaming pass (pattern rows, couplings)
  int frame_np_stream = 1, frame_np_all = 1;  // workgroups per replica of the split measurement
  bool frame_spins = true;  // a measured frame reads spins (launch_frame)
  // what the plan was made for: a run whose plan or batch differs in any of
  // these is refused
  int32_t k_kernel = 0, k_block = 0, k_rpb = 0, k_parts = 0, k_nopersist = 0, k_pt = 0;
  int32_t k_nc = 0, k_store = 0, k_ngraph = 0, k_nrep = 0, k_nrow = 0, k_meas = 0, k_rec = 0;
  const void *k_graphs = nullptr, *k_reps = nullptr, *k_graphs_host = nullptr, *k_reps_host = nullptr;
  // device region: [0, tab_bytes) tables, [reset_off, reset_off + reset_bytes) state
  unsigned char* dev = nullptr;
  size_t dev_bytes = 0, tab_bytes = 0, reset_off = 0, reset_bytes = 0;
  std::vector<unsigned char> hstage;  // the tables as uploaded
  // offsets of the pieces, then their device addresses
  size_t o_items = 0, o_item_reps = 0, o_stream = 0, o_all = 0, o_lrow0 = 0, o_ln = 0, o_halo = 0,
         o_sync = 0, o_xpart = 0, o_rowslot = 0, o_pslot = 0, o_mslot = 0, o_xbuf = 0, o_mprev = 0,
         o_fsum = 0, o_fpart = 0, o_fspin = 0;
  int fspin_n = 0;  // component stride of the published-site copies
  int max_np = 1;   // most parts of a replica
  const WorkItem* items = nullptr;
  const ItemRep* item_reps = nullptr;
  const int32_t *stream_reps = nullptr, *all_reps = nullptr, *lad_row0 = nullptr, *lad_n = nullptr,
                *halo = nullptr;
  uint32_t* sync = nullptr;
  uint64_t *rowslot = nullptr, *pslot = nullptr, *mprev = nullptr;
  double *xpart = nullptr, *mslot = nullptr;
  double* fsum = nullptr;  // split measurement: FSLOTS per replica, zero between frames
  double* fpart = nullptr;  // persistent split replicas: partial frame sums of each part
  void* fspin = nullptr;    // persistent split replicas: sites published for a frame
  void* xbuf = nullptr;
};

// HIP-event bracketing of the sweep-kernel launches (plan->timing)
// Per-launch kernel timing: a start/stop event pair per timed launch,
// stamped by the kernel's own dispatch (hipExtLaunchKernelGGL), so the
// measured span is the kernel's execution and not the queue around it.
struct LaunchTimer {
  bool on = false;
  std::vector<hipEvent_t> ev;
  double launches = 0, sweeps = 0, updates = 0;
  ~LaunchTimer() {
    for (hipEvent_t e : ev) (void)hipEventDestroy(e);
  }
  // two fresh events when timing is on, null otherwise
  int pair(hipEvent_t* a, hipEvent_t* b) {
    *a = *b = nullptr;
    if (!on) return 0;
    HIPCHK(hipEventCreate(a));
    ev.push_back(*a);
    HIPCHK(hipEventCreate(b));
    ev.push_back(*b);
    return 0;
  }
  int finish(double* out) {
    if (!on || !out) return 0;
    double ms = 0;
    for (size_t i = 0; i + 1 < ev.size(); i += 2) {
      HIPCHK(hipEventSynchronize(ev[i + 1]));
      float t = 0;
      HIPCHK(hipEventElapsedTime(&t, ev[i], ev[i + 1]));
      ms += t;
    }
    out[0] = ms;
    out[1] = launches;
    out[2] = sweeps;
    out[3] = updates;
    return 0;
  }
};

int device_lds_max(size_t* out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  int v = 0;
  HIPCHK(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  *out = (size_t)v;
  return 0;
}

// link mode of a graph on the LDS path (the MODE of k_lds)
int lds_mode(const mcg_graph& G) {
  const bool wide = G.lcid != nullptr || G.ncls > 256;
  return wide ? 2 : G.npat > 0 ? (G.ucid >= 0 ? 3 : 0) : 1;
}

template <int NC, typename ST, int MODE, bool FULL, bool PERSIST>
int set_lds_attr(size_t bytes) {
  hipError_t e = hipFuncSetAttribute((const void*)k_lds<NC, ST, MODE, FULL, PERSIST>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  (void)e;
  (void)hipGetLastError();
  return 0;
}

// Tables of a replica split into np parts (see the comment on split
// replicas at the LDS kernel).  For each part p:
//   * extra groups: the other parts' groups of each colour that p's own
//     sites depend on, closed under "neighbour of lower colour";
//   * export list: p's own sites that another part reads during a sweep
//     (a recomputed site or a neighbour of one) or in a frame (the second
//     site of a correlation pair, a vertex of a circuit, whose first site
//     that part owns), which the persistent kernel hands over between
//     sweeps.
// The np descriptors are contiguous, DESC(ncol) ints each: per colour
// (start, count) of the extra groups, then (start, count) of the export
// list, all indices into `halo`.  Returns the offset of the first
// descriptor, or -1 when `limit` is set and a part would recompute more
// than a quarter of its own groups (then the replica is not worth
// splitting), or -2 when the link table cannot be read.  *max_export gets
// the longest export list.
int halo_tables(const mcg_graph& G, int gd, int np, bool limit, std::vector<int32_t>& halo, int* max_export) {
  const int n = G.n, zmax = G.zmax, ncol = G.ncol;
  std::vector<uint32_t> link((size_t)n * zmax);
  std::vector<int32_t> colptr(ncol + 1);
  if (zmax > 0 && hipMemcpy(link.data(), G.link, link.size() * 4, hipMemcpyDeviceToHost) != hipSuccess) return -2;
  if (hipMemcpy(colptr.data(), G.col_ptr, colptr.size() * 4, hipMemcpyDeviceToHost) != hipSuccess) return -2;
  std::vector<int32_t> col(n), grp(n), own(n);
  for (int c = 0; c < ncol; ++c) {
    const int b = colptr[c], cnt = colptr[c + 1] - b, ngrp = (cnt + gd - 1) / gd;
    for (int q = 0, part = 0; q < ngrp; ++q) {
      while (part + 1 < np && q >= (int)((int64_t)ngrp * (part + 1) / np)) ++part;
      for (int e = b + q * gd; e < std::min(b + (q + 1) * gd, b + cnt); ++e) {
        col[e] = c;
        grp[e] = q;
        own[e] = part;
      }
    }
  }
  auto nbr = [&](int e, int l) { return (int)(link[(size_t)e * zmax + l] & 0xFFFFFFu); };
  const int DS = halo_desc_ints(ncol);
  const size_t base = halo.size();
  halo.resize(base + (size_t)np * DS);
  std::vector<char> wanted(n, 0);  // read by a part that does not own it
  for (int part = 0; part < np; ++part) {
    std::vector<char> need(n);
    for (int e = 0; e < n; ++e) need[e] = own[e] == part;
    for (int c = ncol - 1; c >= 0; --c)
      for (int e = colptr[c]; e < colptr[c + 1]; ++e) {
        if (!need[e]) continue;
        for (int l = 0; l < zmax; ++l) {
          const int y = nbr(e, l);
          if (y != e && col[y] < c) need[y] = 1;
        }
      }
    for (int e = 0; e < n; ++e) {
      if (!need[e]) continue;
      if (own[e] != part) wanted[e] = 1;
      for (int l = 0; l < zmax; ++l) {
        const int y = nbr(e, l);
        if (own[y] != part) wanted[y] = 1;
      }
    }
    const size_t d = base + (size_t)part * DS;
    int64_t own_groups = 0, extra = 0;
    for (int c = 0; c < ncol; ++c) {
      const int b = colptr[c], cnt = colptr[c + 1] - b, ngrp = (cnt + gd - 1) / gd;
      own_groups += (int64_t)(ngrp * (part + 1) / np) - (int64_t)ngrp * part / np;
      const size_t start = halo.size();
      int last = -1;
      for (int e = b; e < b + cnt; ++e)
        if (need[e] && own[e] != part && grp[e] != last) {
          last = grp[e];
          halo.push_back(last);
        }
      halo[d + 2 * c] = (int32_t)start;
      halo[d + 2 * c + 1] = (int32_t)(halo.size() - start);
      extra += (int64_t)(halo.size() - start);
    }
    if (limit && extra * 4 > own_groups) return -1;
  }
  // the frame's pairs and circuits: local when none has sites of two parts
  std::vector<int32_t> pr((size_t)2 * G.nlat), cr((size_t)3 * G.ncirc);
  int32_t last = 0;  // position of the last site
  if (G.nlat > 0 && hipMemcpy(pr.data(), G.pairs, pr.size() * 4, hipMemcpyDeviceToHost) != hipSuccess) return -2;
  if (G.ncirc > 0 && hipMemcpy(cr.data(), G.circ, cr.size() * 4, hipMemcpyDeviceToHost) != hipSuccess) return -2;
  if (n > 0 && hipMemcpy(&last, G.pos + (n - 1), 4, hipMemcpyDeviceToHost) != hipSuccess) return -2;
  bool local = true;
  for (int k = 0; k < G.nlat; ++k) local = local && own[pr[2 * k + 1]] == own[pr[2 * k]];
  for (int k = 0; k < G.ncirc; ++k)
    for (int v = 1; v < 3; ++v) local = local && own[cr[3 * k + v]] == own[cr[3 * k]];
  int mx = 0;
  for (int part = 0; part < np; ++part) {
    const size_t d = base + (size_t)part * DS;
    const size_t start = halo.size();
    for (int e = 0; e < n; ++e)
      if (wanted[e] && own[e] == part) halo.push_back(e);
    halo[d + 2 * ncol] = (int32_t)start;
    halo[d + 2 * ncol + 1] = (int32_t)(halo.size() - start);
    mx = std::max(mx, (int)(halo.size() - start));
    // the part's share of the frame
    const size_t ps = halo.size();
    for (int k = 0; k < G.nlat; ++k)
      if (own[pr[2 * k]] == part) halo.push_back(k);
    halo[d + 2 * ncol + 2] = (int32_t)ps;
    halo[d + 2 * ncol + 3] = (int32_t)(halo.size() - ps);
    const size_t cs = halo.size();
    for (int k = 0; k < G.ncirc; ++k)
      if (own[cr[3 * k]] == part) halo.push_back(k);
    halo[d + 2 * ncol + 4] = (int32_t)cs;
    halo[d + 2 * ncol + 5] = (int32_t)(halo.size() - cs);
    halo[d + 2 * ncol + 6] = n > 0 && own[last] == part;
    halo[d + 2 * ncol + 7] = local;
  }
  *max_export = std::max(*max_export, mx);
  return (int)base;
}

// Plan the LDS work items.
//
// Replicas of one graph are packed R to a workgroup (R divides the wave
// count, so each replica gets whole waves).  R is bounded by the LDS budget
// and by a work target t (site updates per workgroup per sweep): t starts at
// the batch's updates per sweep over the CU count, so that the slowest
// workgroup carries about one CU's share.  A replica of n >= 8192 sites
// larger than t is split over P = min(4, ceil(n/t), n/2048) workgroups
// (parts); a launch with parts does one sweep.  The plan keeps at most one
// workgroup per CU (t grows by 5 % until it does), because the LDS the
// largest item asks for is given to every workgroup.  P->parts = 1 disables
// splitting, 2..4 splits every LDS replica into that many parts.  Parts of a
// replica are placed eight workgroup indices apart: workgroups are dealt to
// the eight XCDs in turn, so the parts share an XCD and its L2.
int plan_lds(const mcg_batch* B, const mcg_plan* P, RunCtx& X, bool force_stream) {
  const int ss = store_size(B->store);
  const int gd = B->nc == 1 ? 4 : B->nc == 2 ? 2 : 1;  // sites per Philox draw
  X.hitems.clear();
  X.hitem_reps.clear();
  X.hstream.clear();
  X.hall.clear();
  X.hhalo.clear();
  X.nslots = 0;
  for (int r = 0; r < B->nrep; ++r) X.hall.push_back(r);
  if (P->parts < 0 || P->parts > MAX_PARTS) return fail("parts must be in 0..%d", MAX_PARTS);
  int block = P->block;
  if (block <= 0) {
    int maxcol = 0;
    for (int gi = 0; gi < B->ngraph; ++gi) {
      const mcg_graph& G = B->graphs_host[gi];
      maxcol = std::max(maxcol, (G.n + G.ncol - 1) / std::max(G.ncol, 1));
    }
    block = maxcol >= 1024 ? 1024 : 256;
  }
  if (block % 64 || block < 64 || block > 1024) return fail("block must be a multiple of 64 in [64,1024]");
  X.block = block;
  const int nwaves = block / 64;
  // group replicas by graph, preserving order; Rmax from the LDS budget
  std::vector<std::vector<int>> by(B->ngraph);
  for (int r = 0; r < B->nrep; ++r) by[B->reps_host[r].graph].push_back(r);
  std::vector<int> rmax(B->ngraph, 0);
  double work = 0;
  for (int gi = 0; gi < B->ngraph; ++gi) {
    const mcg_graph& G = B->graphs_host[gi];
    if (by[gi].empty()) continue;
    const size_t per = lds_replica_bytes(B->nc, G.n, ss);
    if (!force_stream) {
      for (int R = nwaves; R >= 1; --R) {
        if (nwaves % R) continue;
        if (P->reps_per_block > 0 && R > P->reps_per_block) continue;
        const bool wide = G.lcid != nullptr || G.ncls > 256;
        if (lds_fixed_bytes(wide ? 0 : G.ncoup, wide ? 0 : G.ncls, G.ncol, G.npat, G.zmax, G.n, nwaves, R) + R * per <=
            X.lds_max) {
          rmax[gi] = R;
          break;
        }
      }
    }
    if (rmax[gi] == 0)
      for (int r : by[gi]) X.hstream.push_back(r);
    else
      work += (double)G.n * by[gi].size();
  }
  if (work == 0) return 0;
  const int ncu = std::max(1, X.ncu);
  std::vector<char> nosplit(B->ngraph, 0);
  // automatic splits only where the launch can be persistent: otherwise a
  // launch with split replicas runs one sweep and restages them every sweep,
  // which costs more than the imbalance it removes.  With spin-derived
  // observables a persistent launch needs pattern links (modes 0 and 3).
  // A part recomputes every group its own sites depend on through lower
  // colours, a cone that widens by a link per colour; halo_tables refuses
  // the split when that is more than a quarter of the part's own groups.
  // Parts keep at least 2048 sites.
  const bool auto_split = !P->no_persist;
  const bool spin_obs = (B->meas & MEAS_SPIN_OBS) != 0;
  struct Split {
    int gi, rep, np;
  };
  for (int attempt = 0; attempt <= B->ngraph; ++attempt) {
    double t = std::max(1.0, std::ceil(work / ncu));
    std::vector<WorkItem> items;
    std::vector<int32_t> ireps;
    std::vector<Split> splits;
    std::vector<int> gnp(B->ngraph, 1);
    for (int iter = 0; iter < 400; ++iter) {
      items.clear();
      ireps.clear();
      splits.clear();
      size_t nsplit_blocks = 0;
      for (int gi = 0; gi < B->ngraph; ++gi) {
        gnp[gi] = 1;
        if (rmax[gi] == 0) continue;
        const mcg_graph& G = B->graphs_host[gi];
        const std::vector<int>& rs = by[gi];
        int np = 1;
        if (P->parts >= 2)
          np = P->parts;
        else if (P->parts == 0 && auto_split && !nosplit[gi] && G.n >= 8192 && G.n > t &&
                 (!spin_obs || lds_mode(G) == 0 || lds_mode(G) == 3))
          np = std::min({MAX_PARTS, (int)std::ceil(G.n / t), G.n / 2048});
        if (np >= 2) {
          gnp[gi] = np;
          for (int r : rs) splits.push_back(Split{gi, r, np});
          nsplit_blocks += (size_t)np * rs.size();
          continue;
        }
        int R = rmax[gi];
        if (P->reps_per_block <= 0) R = std::min(R, std::max(1, (int)(t / G.n)));
        while (nwaves % R) --R;
        for (size_t i = 0; i < rs.size(); i += R) {
          const int cnt = (int)std::min<size_t>(R, rs.size() - i);
          // the tail item takes the largest divisor of nwaves that fits, repeatedly
          for (int q = 0; q < cnt;) {
            int Rq = cnt - q;
            while (nwaves % Rq) --Rq;
            items.push_back(WorkItem{gi, Rq, 0, 0, 1, 0, 0});
            for (int k = 0; k < Rq; ++k) ireps.push_back(rs[i + q + k]);
            q += Rq;
          }
        }
      }
      if (P->parts == 0 && !splits.empty() && items.size() + nsplit_blocks > (size_t)ncu) {
        t = t * 1.05 + 1.0;
        continue;
      }
      break;
    }
    if (splits.size() > 65535) return fail("too many split replicas");
    // split tables, one set per split graph
    std::vector<int> hbase(B->ngraph, -1);
    bool redo = false;
    X.hhalo.clear();
    X.max_export = 0;
    for (int gi = 0; gi < B->ngraph; ++gi) {
      if (gnp[gi] < 2) continue;
      hbase[gi] = halo_tables(B->graphs_host[gi], gd, gnp[gi], P->parts == 0, X.hhalo, &X.max_export);
      if (hbase[gi] == -2) return fail("graph %d: reading the link table for the split failed", gi);
      if (hbase[gi] < 0) {
        nosplit[gi] = 1;
        redo = true;
      }
    }
    if (redo) continue;
    // place parts: in each run of up to 8 split replicas with np parts,
    // part p of the run's replica j goes to index base + j + 8 p
    std::vector<WorkItem> out;
    std::vector<int32_t> oreps;
    X.nslots = 0;
    for (size_t j = 0; j < splits.size();) {
      const int np = splits[j].np;
      size_t e = j;
      while (e < splits.size() && e - j < 8 && splits[e].np == np) ++e;
      std::vector<WorkItem> run((size_t)8 * np, WorkItem{-1, 0, 0, 0, 0, 0, 0});
      std::vector<int32_t> run_rep((size_t)8 * np, -1);
      for (size_t q = j; q < e; ++q) {
        const uint16_t slot = (uint16_t)X.nslots++;
        const int gi = splits[q].gi;
        for (int p = 0; p < np; ++p) {
          run[(q - j) + (size_t)8 * p] =
              WorkItem{gi, 1, 0, (uint8_t)p, (uint8_t)np, slot,
                       hbase[gi] + p * halo_desc_ints(B->graphs_host[gi].ncol)};
          run_rep[(q - j) + (size_t)8 * p] = splits[q].rep;
        }
      }
      for (size_t q = 0; q < run.size(); ++q) {
        if (run[q].graph < 0) continue;  // holes of a short run
        run[q].off = (int)oreps.size();
        oreps.push_back(run_rep[q]);
        out.push_back(run[q]);
      }
      j = e;
    }
    size_t ir = 0;
    for (WorkItem w : items) {
      w.off = (int)oreps.size();
      for (int k = 0; k < w.nrep; ++k) oreps.push_back(ireps[ir + k]);
      ir += w.nrep;
      out.push_back(w);
    }
    // one kernel per link mode: sort the items by mode (stable, so the
    // parts of a split replica stay eight indices apart)
    std::stable_sort(out.begin(), out.end(), [&](const WorkItem& x, const WorkItem& y) {
      return lds_mode(B->graphs_host[x.graph]) < lds_mode(B->graphs_host[y.graph]);
    });
    for (int m = 0; m <= 4; ++m) X.mode_begin[m] = 0;
    for (const WorkItem& w : out) X.mode_begin[lds_mode(B->graphs_host[w.graph]) + 1]++;
    for (int m = 1; m <= 4; ++m) X.mode_begin[m] += X.mode_begin[m - 1];
    X.hitems = out;
    X.hitem_reps = oreps;
    return 0;
  }
  return fail("internal: LDS plan did not converge");
}

template <int NC, typename ST>
size_t lds_bytes_for(const mcg_batch* B, const RunCtx& X, int i0, int i1) {
  size_t mx = 0;
  const int nwaves = X.block / 64;
  for (int i = i0; i < i1; ++i) {
    const WorkItem& w = X.hitems[i];
    const mcg_graph& G = B->graphs_host[w.graph];
    const bool wide = G.lcid != nullptr || G.ncls > 256;
    const size_t b = lds_fixed_bytes(wide ? 0 : G.ncoup, wide ? 0 : G.ncls, G.ncol, G.npat, G.zmax, G.n, nwaves,
                                     w.nrep) +
                     w.nrep * (lds_replica_bytes(NC, G.n, sizeof(ST)) + (w.nparts > 1 ? 0 : (size_t)(X.blk + X.thr)));
    mx = std::max(mx, b);
  }
  return mx;
}

template <int NC, typename ST, int MODE, bool FULL, bool PERSIST>
int launch_lds_range(const mcg_batch* B, RunCtx& X, const SweepArgs& a, hipStream_t s, int i0, int i1, hipEvent_t e0,
                     hipEvent_t e1) {
  size_t bytes = lds_bytes_for<NC, ST>(B, X, i0, i1);
  if (PERSIST) bytes += persist_lds_bytes(B->nrow);
  set_lds_attr<NC, ST, MODE, FULL, PERSIST>(bytes);
  hipExtLaunchKernelGGL((k_lds<NC, ST, MODE, FULL, PERSIST>), dim3((unsigned)(i1 - i0)), dim3(X.block),
                        (uint32_t)bytes, s, e0, e1, 0, LdsArgs{*B, X.items + i0, X.item_reps, a});
  HIPCHK(hipGetLastError());
  return 0;
}

// one launch per link mode present (work items are sorted by mode)
template <int NC, typename ST>
int launch_lds(const mcg_batch* B, RunCtx& X, const SweepArgs& a, hipStream_t s, LaunchTimer& T) {
  const bool full = (B->meas & MEAS_SPIN_OBS) != 0;
  for (int m = 0; m < 4; ++m) {
    const int i0 = X.mode_begin[m], i1 = X.mode_begin[m + 1];
    if (i1 <= i0) continue;
    hipEvent_t e0, e1;
    if (T.pair(&e0, &e1)) return -1;
    int r;
    if (X.persist && full)  // single pattern mode (checked when planned)
      r = m == 0 ? launch_lds_range<NC, ST, 0, true, true>(B, X, a, s, i0, i1, e0, e1)
                 : launch_lds_range<NC, ST, 3, true, true>(B, X, a, s, i0, i1, e0, e1);
    else if (X.persist)  // single mode (checked when planned)
      r = m == 0   ? launch_lds_range<NC, ST, 0, false, true>(B, X, a, s, i0, i1, e0, e1)
          : m == 1 ? launch_lds_range<NC, ST, 1, false, true>(B, X, a, s, i0, i1, e0, e1)
          : m == 2 ? launch_lds_range<NC, ST, 2, false, true>(B, X, a, s, i0, i1, e0, e1)
                   : launch_lds_range<NC, ST, 3, false, true>(B, X, a, s, i0, i1, e0, e1);
    else if (m == 0)
      r = full ? launch_lds_range<NC, ST, 0, true, false>(B, X, a, s, i0, i1, e0, e1)
               : launch_lds_range<NC, ST, 0, false, false>(B, X, a, s, i0, i1, e0, e1);
    else if (m == 1)
      r = full ? launch_lds_range<NC, ST, 1, true, false>(B, X, a, s, i0, i1, e0, e1)
               : launch_lds_range<NC, ST, 1, false, false>(B, X, a, s, i0, i1, e0, e1);
    else if (m == 2)
      r = full ? launch_lds_range<NC, ST, 2, true, false>(B, X, a, s, i0, i1, e0, e1)
               : launch_lds_range<NC, ST, 2, false, false>(B, X, a, s, i0, i1, e0, e1);
    else
      r = full ? launch_lds_range<NC, ST, 3, true, false>(B, X, a, s, i0, i1, e0, e1)
               : launch_lds_range<NC, ST, 3, false, false>(B, X, a, s, i0, i1, e0, e1);
    if (r) return -1;
    T.launches += 1;
  }
  return 0;
}

// Room in LDS for a frame's block spins (X.blk) and for the rows' Ising
// thresholds (X.thr): taken when the workgroups still fit, and as many of them
// per CU as without it.
template <int NC, typename ST>
void plan_block_spins(const mcg_batch* B, RunCtx& X) {
  X.blk = X.thr = 0;
  if (X.hitems.empty()) return;
  const int ni = (int)X.hitems.size();
  const size_t pers = persist_lds_bytes(B->nrow);
  const size_t without = lds_bytes_for<NC, ST>(B, X, 0, ni) + pers;
  auto fits = [&] {
    const size_t with = lds_bytes_for<NC, ST>(B, X, 0, ni) + pers;
    return with <= X.lds_max && (ni <= X.ncu || X.lds_max / with == X.lds_max / without);
  };
  if (B->meas & MCG_MEAS_RNORM) {
    for (const WorkItem& w : X.hitems)
      X.blk = std::max(X.blk, (int)align16((size_t)B->graphs_host[w.graph].nr * NC * 4));
    if (!fits()) X.blk = 0;
  }
  if (NC == 1 && B->ithr && B->nthr <= 1024) {
    X.thr = (int)align16((size_t)B->nthr * 4);
    if (!fits()) X.thr = 0;
  }
}

// Can this run use a persistent launch?  All replicas on the LDS path, one
// link mode (a pattern mode when spin-derived observables are measured),
// tempering or split replicas to synchronise (otherwise a plain multi-sweep
// launch already is persistent), the tempering state fits in LDS, and every
// workgroup resident at once.
template <int NC, typename ST>
int check_persist(const mcg_batch* B, const mcg_plan* P, RunCtx& X, bool* ok) {
  *ok = false;
  if (X.hitems.empty() || !X.hstream.empty()) return 0;
  int modes = 0, m = -1;
  for (int q = 0; q < 4; ++q)
    if (X.mode_begin[q + 1] > X.mode_begin[q]) ++modes, m = q;
  if (modes != 1) return 0;
  const bool full = (B->meas & MEAS_SPIN_OBS) != 0;
  if (full && m != 0 && m != 3) return 0;
  const bool pt = P->pt_every > 0 && !X.hl_row0.empty();
  if (!pt && X.nslots == 0) return 0;
  const size_t bytes = lds_bytes_for<NC, ST>(B, X, 0, (int)X.hitems.size()) + persist_lds_bytes(B->nrow);
  if (bytes > X.lds_max) return 0;
  const void* f = full ? (m == 0 ? (const void*)k_lds<NC, ST, 0, true, true> : (const void*)k_lds<NC, ST, 3, true, true>)
                  : m == 0 ? (const void*)k_lds<NC, ST, 0, false, true>
                  : m == 1 ? (const void*)k_lds<NC, ST, 1, false, true>
                  : m == 2 ? (const void*)k_lds<NC, ST, 2, false, true>
                           : (const void*)k_lds<NC, ST, 3, false, true>;
  if (full && m == 0) set_lds_attr<NC, ST, 0, true, true>(bytes);
  else if (full) set_lds_attr<NC, ST, 3, true, true>(bytes);
  else if (m == 0) set_lds_attr<NC, ST, 0, false, true>(bytes);
  else if (m == 1) set_lds_attr<NC, ST, 1, false, true>(bytes);
  else if (m == 2) set_lds_attr<NC, ST, 2, false, true>(bytes);
  else set_lds_attr<NC, ST, 3, false, true>(bytes);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, X.block, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  *ok = (int64_t)per_cu * X.ncu >= (int64_t)X.hitems.size();
  return 0;
}


// one colour of nreps replicas (all of link mode `mode`)
template <int NC, typename ST>
int launch_pass(const mcg_batch* B, const int32_t* dreps, int nreps, int mode, int maxcnt, uint32_t lds, int colour,
                int64_t sweep, hipStream_t s, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr) {
  if (nreps == 0) return 0;
  const int ngrp = (maxcnt + SitesPerDraw<NC>::G - 1) / SitesPerDraw<NC>::G;
  const int chunks = std::max(1, (ngrp + 256 * PASS_GPT - 1) / (256 * PASS_GPT));
  const int64_t items = (int64_t)chunks * nreps;
  if (items > (1 << 30)) return fail("streaming pass: %lld work items", (long long)items);
  auto launch = [&](auto kernel) {
    hipExtLaunchKernelGGL(kernel, dim3((unsigned)xcd_grid((int)items)), dim3(256), lds, s, e0, e1, 0, *B, dreps, colour,
                          sweep, chunks, (int)items);
  };
  if (mode == PASS_PAT_UNI)
    launch(k_pass<NC, ST, PASS_PAT_UNI>);
  else if (mode == PASS_PAT)
    launch(k_pass<NC, ST, PASS_PAT>);
  else if (mode == PASS_LINKS_UNI)
    launch(k_pass<NC, ST, PASS_LINKS_UNI>);
  else
    launch(k_pass<NC, ST, PASS_LINKS>);
  HIPCHK(hipGetLastError());
  return 0;
}

template <int NC, typename ST>
int launch_measure(const mcg_batch* B, const int32_t* dreps, int nreps, int mode, int64_t frame, hipStream_t s) {
  if (nreps == 0) return 0;
  hipLaunchKernelGGL((k_measure<NC, ST>), dim3((unsigned)nreps), dim3(1024), 0, s, *B, dreps, mode, frame);
  HIPCHK(hipGetLastError());
  return 0;
}

// workgroups per replica of the split measurement: about MCG_FRAME_WG_PER_CU
// per CU over the batch, at least 1024 sites each
#ifndef MCG_FRAME_WG_PER_CU
#define MCG_FRAME_WG_PER_CU 16
#endif
int frame_parts(int nreps, int nmax, int ncu) {
  if (nreps <= 0) return 1;
  const int want = (MCG_FRAME_WG_PER_CU * std::max(ncu, 1) + nreps - 1) / nreps;
  return std::max(1, std::min({want, std::max(1, nmax / 1024), 65535}));
}

template <int NC, typename ST>
// spins: a measured frame reads spins (a spin-derived observable other than
// self pairs of an O(n) model); the recompute (mode bit 1) always does
int launch_frame(const mcg_batch* B, const int32_t* dreps, int nreps, int mode, int64_t frame, double* fsum, int np,
                 bool spins, hipStream_t s) {
  if (nreps == 0) return 0;
  if ((mode & 1) || ((mode & 4) && spins)) {
    const int64_t items = (int64_t)np * nreps;
    if (items > (1 << 30)) return fail("split measurement: %lld work items", (long long)items);
    hipLaunchKernelGGL((k_frame_part<NC, ST>), dim3((unsigned)xcd_grid((int)items)), dim3(256), 0, s, *B, dreps,
                       mode, frame, fsum, np, (int)items);
    HIPCHK(hipGetLastError());
  }
  hipLaunchKernelGGL((k_frame_end<NC, ST>), dim3((unsigned)nreps), dim3(64), 0, s, *B, dreps, mode, frame, fsum);
  HIPCHK(hipGetLastError());
  return 0;
}

int launch_fill_f64(double* p, size_t n, double v, hipStream_t s) {
  if (!p || n == 0) return 0;
  const unsigned g = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_f64, dim3(g), dim3(256), 0, s, p, n, v);
  HIPCHK(hipGetLastError());
  return 0;
}
int launch_fill_i32(int32_t* p, size_t n, int32_t v, hipStream_t s) {
  if (!p || n == 0) return 0;
  const unsigned g = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_i32, dim3(g), dim3(256), 0, s, p, n, v);
  HIPCHK(hipGetLastError());
  return 0;
}

// Spins that the chip's last-level cache (256 MB) keeps from one pass to the
// next.  Replicas do not meet between two swap passes, so a larger batch is
// taken in groups of about equal size, each through all the sweeps of the call
// before the next: its passes after the first read from that cache.
// Cubic 64^3 (3 MiB a replica), ns per 1,000 updates, one group and in groups:
// 64 replicas 8.1 either way, 80 8.0 and 8.5 (two groups of 40 leave the last
// wave of workgroups half empty, so a batch that just fits stays whole), 88 9.3
// and 8.4, 128 9.7 and 7.8, 200 9.0 and 7.8; groups of at most 156 MiB: 8.8 for
// 128.
#ifndef MCG_STREAM_GROUP_BYTES
#define MCG_STREAM_GROUP_BYTES ((int64_t)248 << 20)
#endif

// planned sweep schedule for the streaming / plain paths
template <int NC, typename ST>
int stream_sweeps(const mcg_batch* B, const mcg_plan* P, RunCtx& X, int64_t k0, int64_t nsw, int64_t nthermal,
                  int spf, bool plain, hipStream_t s, LaunchTimer& T) {
  if (X.hstream.empty()) return 0;
  const int ncolmax = X.stream_ncol;
  const int maxn = X.stream_maxcnt;  // largest colour class of the streamed graphs
  const int32_t* dreps = X.stream_reps;
  const int nrs = (int)X.hstream.size();
  auto graph_of = [&](int i) -> const mcg_graph& { return B->graphs_host[B->reps_host[X.hstream[i]].graph]; };
  auto mode_of = [&](int i) { return pass_mode(graph_of(i)); };
  auto bytes_of = [&](int i) { return (int64_t)NC * graph_of(i).n * (int64_t)sizeof(ST); };
  int64_t total = 0;
  for (int i = 0; i < nrs; ++i) total += bytes_of(i);
  const int64_t ngroups = plain ? 1 : (total + MCG_STREAM_GROUP_BYTES - 1) / MCG_STREAM_GROUP_BYTES;
  const int64_t share = (total + ngroups - 1) / ngroups;
  for (int g0 = 0, g1; g0 < nrs; g0 = g1) {
    int64_t bytes = bytes_of(g0);
    for (g1 = g0 + 1; g1 < nrs && (ngroups == 1 || bytes + bytes_of(g1) <= share); ++g1) bytes += bytes_of(g1);
    for (int64_t q = 0; q < nsw; ++q) {
      const int64_t k = k0 + q;
      const int64_t kk = P->sweep0 + k;
      for (int c = 0; c < ncolmax; ++c) {
        // one launch per run of replicas of one link mode (hstream is sorted by
        // it), or, plain, per replica
        for (int i = g0, e; i < g1; i = e) {
          const int mode = mode_of(i);
          for (e = i + 1; !plain && e < g1 && mode_of(e) == mode;) ++e;
          hipEvent_t e0, e1;
          if (T.pair(&e0, &e1) ||
              launch_pass<NC, ST>(B, dreps + i, e - i, mode, maxn, X.stream_lds, c, kk, s, e0, e1))
            return -1;
          T.launches += 1;
        }
      }
      if (T.on) {
        if (g0 == 0) T.sweeps += 1;
        for (int i = g0; i < g1; ++i) T.updates += graph_of(i).n;
      }
      const bool meas = k >= nthermal && ((k - nthermal + 1) % spf) == 0;
      const bool therm_end = (k + 1 == nthermal);
      const bool rec = recompute_due(*B, P->sweep0 + k);
      int mode = (rec ? 1 : 0) | (therm_end ? 2 : 0) | (meas ? 4 : 0);
      if (mode) {
        const int64_t frame = meas ? (k - nthermal + 1) / spf - 1 + P->frame0 : -1;
        if (plain) {
          for (int i = g0; i < g1; ++i)
            if (launch_measure<NC, ST>(B, dreps + i, 1, mode, frame, s)) return -1;
        } else if (launch_frame<NC, ST>(B, dreps + g0, g1 - g0, mode, frame, X.fsum, X.frame_np_stream, X.frame_spins,
                                        s)) {
          return -1;
        }
      }
    }
  }
  return 0;
}

// piece of the device region, 256-byte aligned
size_t take(size_t* off, size_t bytes) {
  const size_t o = *off;
  *off += (bytes + 255) & ~(size_t)255;
  return o;
}

// Plan the run of B under P and lay out its device region: fills everything
// in X but the device addresses (bind_region).  X.dev_bytes is the size of
// the region the run needs.
template <int NC, typename ST>
int prepare_typed(const mcg_batch* B, const mcg_plan* P, RunCtx& X) {
  HIPCHK(hipGetDevice(&X.device));
  if (device_lds_max(&X.lds_max)) return -1;
  HIPCHK(hipDeviceGetAttribute(&X.ncu, hipDeviceAttributeMultiprocessorCount, X.device));
  const bool force_stream = P->kernel == 2 || P->kernel == 3;
  if (plan_lds(B, P, X, force_stream)) return -1;
  std::stable_sort(X.hstream.begin(), X.hstream.end(), [&](int a, int b) {
    return pass_mode(B->graphs_host[B->reps_host[a].graph]) < pass_mode(B->graphs_host[B->reps_host[b].graph]);
  });
  if (P->kernel == 1 && !X.hstream.empty())
    return fail("LDS-resident kernel requested but %zu replica(s) do not fit in LDS", X.hstream.size());
  // tempering ladders (row0, rungs), each of one lattice
  X.hl_row0.clear();
  X.hl_n.clear();
  {
    std::vector<int32_t> seen(B->nrow, 0), lgraph(B->nrow, -1);
    for (int r = 0; r < B->nrep; ++r) {
      const mcg_replica& R = B->reps_host[r];
      if (R.ladder < 0 || R.nrung < 2) continue;
      if (lgraph[R.row0] >= 0 && lgraph[R.row0] != R.graph)
        return fail("replica %d: a tempering ladder holds replicas of one lattice", r);
      lgraph[R.row0] = R.graph;
      if (seen[R.row0]) continue;
      seen[R.row0] = 1;
      X.hl_row0.push_back(R.row0);
      X.hl_n.push_back(R.nrung);
    }
  }
  // colour classes of the streamed graphs (the streaming grid covers the largest)
  X.stream_ncol = X.stream_maxcnt = 0;
  X.stream_lds = 0;
  {
    std::vector<char> seen(B->ngraph, 0);
    for (int r : X.hstream) {
      const int gi = B->reps_host[r].graph;
      if (seen[gi]) continue;
      seen[gi] = 1;
      const mcg_graph& G = B->graphs_host[gi];
      std::vector<int32_t> cp(G.ncol + 1);
      HIPCHK(hipMemcpy(cp.data(), G.col_ptr, cp.size() * 4, hipMemcpyDeviceToHost));
      X.stream_ncol = std::max(X.stream_ncol, G.ncol);
      X.stream_lds = std::max(X.stream_lds, (uint32_t)pass_lds_bytes(G));
      for (int c = 0; c < G.ncol; ++c) X.stream_maxcnt = std::max(X.stream_maxcnt, cp[c + 1] - cp[c]);
    }
  }
  {
    int nmax = 1;
    for (int gi = 0; gi < B->ngraph; ++gi) nmax = std::max(nmax, B->graphs_host[gi].n);
    X.frame_np_stream = frame_parts((int)X.hstream.size(), nmax, X.ncu);
    // the frame reads spins unless its only spin-derived observable is the
    // self pairs of an O(n) model
    X.frame_spins = (B->meas & (MCG_MEAS_Q | MCG_MEAS_RNORM | MCG_MEAS_GROUPS)) != 0;
    if (B->meas & MCG_MEAS_PAIRS)
      for (int gi = 0; gi < B->ngraph; ++gi)
        X.frame_spins = X.frame_spins || B->nc == 1 || !B->graphs_host[gi].self_pairs;
    X.frame_np_all = frame_parts(B->nrep, nmax, X.ncu);
  }
  X.lds_updates_per_sweep = 0;
  for (const WorkItem& w : X.hitems)
    if (w.part == 0) X.lds_updates_per_sweep += (double)w.nrep * B->graphs_host[w.graph].n;
  plan_block_spins<NC, ST>(B, X);
  // persistent launches when possible (P->no_persist turns them off)
  X.persist = false;
  if (P->algorithm == MCG_METROPOLIS && !P->no_persist && !force_stream && check_persist<NC, ST>(B, P, X, &X.persist))
    return -1;
  std::vector<int32_t> lad_of_row(B->nrow, -1);
  for (size_t L = 0; L < X.hl_row0.size(); ++L) lad_of_row[X.hl_row0[L]] = (int32_t)L;
  X.max_np = 1;
  for (const WorkItem& w : X.hitems) X.max_np = std::max(X.max_np, (int)w.nparts);
  std::vector<ItemRep> recs(X.hitem_reps.size());
  for (size_t i = 0; i < recs.size(); ++i) {
    const mcg_replica& R = B->reps_host[X.hitem_reps[i]];
    const bool lad = R.ladder >= 0 && R.nrung >= 2;
    recs[i] = ItemRep{R.spin_off, X.hitem_reps[i], (int32_t)R.serial, R.row0, lad ? R.nrung : 0,
                      lad ? lad_of_row[R.row0] : -1, 0};
  }
  // layout: tables first, then the state every run clears
  size_t off = 0;
  X.o_items = take(&off, X.hitems.size() * sizeof(WorkItem));
  X.o_item_reps = take(&off, recs.size() * sizeof(ItemRep));
  X.o_stream = take(&off, X.hstream.size() * 4);
  X.o_all = take(&off, X.hall.size() * 4);
  X.o_lrow0 = take(&off, X.hl_row0.size() * 4);
  X.o_ln = take(&off, X.hl_n.size() * 4);
  X.o_halo = take(&off, X.hhalo.size() * 4);
  X.tab_bytes = off;
  X.reset_off = off;
  X.o_fsum = take(&off, (size_t)B->nrep * FSLOTS * 8);
  X.o_sync = take(&off, (size_t)X.nslots * SYNC_STRIDE * 4);
  X.o_xpart = take(&off, (size_t)X.nslots * MAX_PARTS * 4 * 8);
  if (X.persist) {
    X.o_rowslot = take(&off, (size_t)4 * B->nrow * X.max_np * 16);
    X.o_pslot = take(&off, (size_t)2 * X.nslots * MAX_PARTS * 16);
    X.o_mslot = take(&off, (size_t)2 * X.nslots * (MAX_PARTS - 1) * 3 * 8);
    X.o_xbuf = take(&off, (size_t)2 * std::max(X.nslots, 1) * MAX_PARTS * std::max(X.max_export, 1) * NC * sizeof(ST));
    X.o_mprev = take(&off, (size_t)2 * B->nrow * 16);
    X.o_fpart = take(&off, (size_t)2 * std::max(X.nslots, 1) * (MAX_PARTS - 1) * FSUMS * 8);
  }
  X.reset_bytes = off - X.reset_off;
  if (X.persist && X.nslots > 0 && (B->meas & MEAS_SPIN_OBS)) {
    // written in full before every read: outside the reset region
    int nmax = 0;
    for (int gi = 0; gi < B->ngraph; ++gi) nmax = std::max(nmax, B->graphs_host[gi].n);
    X.fspin_n = (int)((nmax + 63) / 64 * 64);
    X.o_fspin = take(&off, (size_t)2 * X.nslots * NC * X.fspin_n * sizeof(ST));
  }
  X.dev_bytes = off;
  X.hstage.assign(X.tab_bytes, 0);
  auto put = [&](size_t o, const void* src, size_t n) {
    if (n) std::memcpy(X.hstage.data() + o, src, n);
  };
  put(X.o_items, X.hitems.data(), X.hitems.size() * sizeof(WorkItem));
  put(X.o_item_reps, recs.data(), recs.size() * sizeof(ItemRep));
  put(X.o_stream, X.hstream.data(), X.hstream.size() * 4);
  put(X.o_all, X.hall.data(), X.hall.size() * 4);
  put(X.o_lrow0, X.hl_row0.data(), X.hl_row0.size() * 4);
  put(X.o_ln, X.hl_n.data(), X.hl_n.size() * 4);
  put(X.o_halo, X.hhalo.data(), X.hhalo.size() * 4);
  // the key
  X.k_kernel = P->kernel;
  X.k_block = P->block;
  X.k_rpb = P->reps_per_block;
  X.k_parts = P->parts;
  X.k_nopersist = P->no_persist;
  X.k_pt = P->pt_every > 0;
  X.k_nc = B->nc;
  X.k_store = B->store;
  X.k_ngraph = B->ngraph;
  X.k_nrep = B->nrep;
  X.k_nrow = B->nrow;
  X.k_meas = B->meas;
  X.k_rec = B->recompute_every;
  X.k_graphs = B->graphs;
  X.k_reps = B->reps;
  X.k_graphs_host = B->graphs_host;
  X.k_reps_host = B->reps_host;
  return 0;
}

// Give X its device region (X.dev_bytes at dev) and copy the tables there,
// on stream s.  The caller keeps X.hstage alive until the copy is done.
int bind_region(RunCtx& X, unsigned char* dev, hipStream_t s) {
  X.dev = dev;
  auto at = [&](size_t o) { return (void*)(dev + o); };
  X.items = (const WorkItem*)at(X.o_items);
  X.item_reps = (const ItemRep*)at(X.o_item_reps);
  X.stream_reps = (const int32_t*)at(X.o_stream);
  X.all_reps = (const int32_t*)at(X.o_all);
  X.lad_row0 = (const int32_t*)at(X.o_lrow0);
  X.lad_n = (const int32_t*)at(X.o_ln);
  X.halo = (const int32_t*)at(X.o_halo);
  X.sync = (uint32_t*)at(X.o_sync);
  X.xpart = (double*)at(X.o_xpart);
  X.rowslot = (uint64_t*)at(X.o_rowslot);
  X.pslot = (uint64_t*)at(X.o_pslot);
  X.mslot = (double*)at(X.o_mslot);
  X.xbuf = at(X.o_xbuf);
  X.mprev = (uint64_t*)at(X.o_mprev);
  X.fsum = (double*)at(X.o_fsum);
  X.fpart = (double*)at(X.o_fpart);
  X.fspin = at(X.o_fspin);
  if (X.tab_bytes && hipMemcpyAsync(dev, X.hstage.data(), X.tab_bytes, hipMemcpyHostToDevice, s) != hipSuccess)
    return fail("hipMemcpyAsync of the run tables failed");
  return 0;
}

// Is X the plan of this batch and plan?
int check_key(const mcg_batch* B, const mcg_plan* P, const RunCtx& X) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev != X.device) return fail("run prepared on device %d, called on device %d", X.device, dev);
  if (P->kernel != X.k_kernel || P->block != X.k_block || P->reps_per_block != X.k_rpb || P->parts != X.k_parts ||
      P->no_persist != X.k_nopersist || (P->pt_every > 0) != (X.k_pt != 0))
    return fail("plan differs from the prepared one in kernel, block, reps_per_block, parts, no_persist or "
                "tempering on/off; prepare a new run for it");
  if (B->nc != X.k_nc || B->store != X.k_store || B->ngraph != X.k_ngraph || B->nrep != X.k_nrep ||
      B->nrow != X.k_nrow || B->meas != X.k_meas || B->recompute_every != X.k_rec || B->graphs != X.k_graphs ||
      B->reps != X.k_reps || B->graphs_host != X.k_graphs_host || B->reps_host != X.k_reps_host)
    return fail("batch differs from the one the run was prepared for");
  return 0;
}

// The launches of one run of a prepared context (no allocation, no host
// copy): clear the run state, then the sweep / cluster / tempering launches.
template <int NC, typename ST>
int exec_typed(const mcg_batch* B, const mcg_plan* P, hipStream_t s, RunCtx& X) {
  const bool plain = P->kernel == 3;
  const int spf = P->sweeps_per_frame > 0 ? P->sweeps_per_frame : 1;
  const int64_t nth = P->nthermal;
  const int64_t total = nth + (int64_t)P->nsweep * spf;
  const int nall = B->nrep;
  if (X.nslots > 0 && total * MAX_PARTS >= ((int64_t)1 << 32))
    return fail("too many sweeps in one call for split replicas (%lld); split the call", (long long)total);
  if (X.reset_bytes) {
    const size_t nw = X.reset_bytes / 4;
    const unsigned g = (unsigned)std::min<size_t>((nw + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill_u32, dim3(g), dim3(256), 0, s, (uint32_t*)(X.dev + X.reset_off), nw, 0u);
    HIPCHK(hipGetLastError());
  }
  const bool pt_on = P->pt_every > 0 && !X.hl_row0.empty();

  if (P->algorithm == MCG_WOLFF) {
    if (!B->wstamp || !B->wlist) return fail("Wolff needs wstamp/wlist scratch");
    int64_t nmax = 0, wmax = 0;
    for (int gi = 0; gi < B->ngraph; ++gi) {
      nmax = std::max<int64_t>(nmax, B->graphs_host[gi].n);
      wmax = std::max<int64_t>(wmax, (int64_t)B->graphs_host[gi].n * (B->graphs_host[gi].zmax + 1));
    }
    if (wmax >= ((int64_t)1 << 32)) return fail("Wolff: sites x (links + 1) must stay below 2^32");
    // members as bits in LDS where every graph's fit
    bool bits = true;
    size_t wolff_lds = 0;
    for (int pass = 0; pass < 2; ++pass) {
      wolff_lds = 0;
      for (int gi = 0; gi < B->ngraph; ++gi) wolff_lds = std::max(wolff_lds, wolff_lds_bytes(B->graphs_host[gi], bits));
      if (wolff_lds + 1024 <= X.lds_max) break;  // 1024: the kernel's other LDS
      bits = false;
    }
    (void)hipFuncSetAttribute(bits ? (const void*)k_wolff<NC, ST, true> : (const void*)k_wolff<NC, ST, false>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)wolff_lds);
    (void)hipGetLastError();
    for (int64_t k = 0; k < total; ++k) {
      const int64_t kk = P->sweep0 + k;
      // clusters per sweep: plan value or n of the replica's graph (use max n)
      const int ncl = P->clusters_per_sweep > 0 ? P->clusters_per_sweep : (int)nmax;
      auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nall), dim3(1024), (uint32_t)wolff_lds, s, *B, X.all_reps,
                           kk * (int64_t)ncl, ncl);
      };
      if (bits)
        launch(k_wolff<NC, ST, true>);
      else
        launch(k_wolff<NC, ST, false>);
      HIPCHK(hipGetLastError());
      const bool meas = k >= nth && ((k - nth + 1) % spf) == 0;
      const bool therm_end = (k + 1 == nth);
      const int mode = 1 | 8 | (therm_end ? 2 : 0) | (meas ? 4 : 0);
      if (meas || therm_end || k + 1 == total) {
        const int64_t frame = meas ? (k - nth + 1) / spf - 1 + P->frame0 : -1;
        if (launch_frame<NC, ST>(B, X.all_reps, nall, mode, frame, X.fsum, X.frame_np_all, X.frame_spins, s)) return -1;
      }
      if (pt_on && ((P->sweep0 + k + 1) % P->pt_every) == 0) {
        if (launch_frame<NC, ST>(B, X.all_reps, nall, 1 | 8, -1, X.fsum, X.frame_np_all, X.frame_spins, s)) return -1;
        hipLaunchKernelGGL(k_pt, dim3((unsigned)X.hl_row0.size()), dim3(64), 0, s, *B, X.lad_row0, X.lad_n,
                           (int)X.hl_row0.size(), P->sweep0 + k);
        HIPCHK(hipGetLastError());
      }
    }
    return 0;
  }

  LaunchTimer T;
  T.on = P->timing != nullptr;
  // a persistent launch runs up to 4096 sweeps; otherwise split replicas
  // finish every launch (one sweep per launch) and tempering needs a launch
  // boundary every pt_every sweeps
  const int64_t chunk = X.persist ? 4096 : X.nslots > 0 ? 1 : P->pt_every > 0 ? P->pt_every : total;
  int64_t sync_base = 0;  // exchanges of parts and ladders before a launch
  for (int64_t k = 0; k < total;) {
    int64_t ns = std::min<int64_t>(chunk, total - k);
    if (!X.persist && X.nslots == 0 && P->pt_every > 0)  // launches end where swaps are due
      ns = std::min<int64_t>(ns, P->pt_every - (P->sweep0 + k) % P->pt_every);
    // split replicas in a persistent launch: launches end where a full
    // recompute is due, and the host recomputes every replica after them
    const bool rec_host = X.persist && X.nslots > 0 && B->recompute_every > 0;
    if (rec_host) ns = std::min<int64_t>(ns, B->recompute_every - (P->sweep0 + k) % B->recompute_every);
    SweepArgs a{k, P->sweep0, (int32_t)ns, (int32_t)nth, spf, P->frame0, X.sync, X.xpart, X.halo};
    a.blk = X.blk;
    a.thr = B->ithr && (int64_t)B->nthr * 4 <= X.thr ? X.thr : 0;
    if (X.persist) {
      a.sync_base = (int32_t)sync_base;
      a.pt_every = pt_on ? P->pt_every : 0;
      a.has_split = X.nslots > 0;
      a.nrow_parts = X.max_np;
      a.rowslot = X.rowslot;
      a.pslot = X.pslot;
      a.mslot = X.mslot;
      a.xbuf = X.xbuf;
      a.mprev = X.mprev;
      a.fpart = X.fpart;
      a.fspin = X.fspin;
      a.fspin_n = X.fspin_n;
      a.max_export = std::max(X.max_export, 1);
      a.nslots = std::max(X.nslots, 1);
      a.rec_host = rec_host ? 1 : 0;
      for (int64_t q = k; q < k + ns; ++q)
        if (X.nslots > 0 || (pt_on && ((P->sweep0 + q + 1) % P->pt_every) == 0)) ++sync_base;
      if (sync_base * (int64_t)std::max<size_t>(X.hitems.size(), 16) >= ((int64_t)1 << 31))
        return fail("too many barriers in one call (%lld); split the call", (long long)sync_base);
    }
    if (!X.hitems.empty()) {
      if (launch_lds<NC, ST>(B, X, a, s, T)) return -1;
      T.sweeps += (double)ns;
      T.updates += X.lds_updates_per_sweep * (double)ns;
    }
    if (stream_sweeps<NC, ST>(B, P, X, k, ns, nth, spf, plain, s, T)) return -1;
    if (rec_host && recompute_due(*B, P->sweep0 + k + ns - 1)) {
      const int mode = 1 | (k + ns == nth ? 2 : 0);  // recompute (+ energy reference at thermalisation end)
      if (launch_frame<NC, ST>(B, X.all_reps, nall, mode, -1, X.fsum, X.frame_np_all, X.frame_spins, s)) return -1;
    }
    k += ns;
    if (!X.persist && pt_on && ((P->sweep0 + k) % P->pt_every) == 0) {
      hipLaunchKernelGGL(k_pt, dim3((unsigned)X.hl_row0.size()), dim3(64), 0, s, *B, X.lad_row0, X.lad_n,
                         (int)X.hl_row0.size(), P->sweep0 + k - 1);
      HIPCHK(hipGetLastError());
    }
  }
  return T.finish(P->timing);
}

// mcg_run: prepare into a region of its own, run, wait, release
template <int NC, typename ST>
int run_typed(const mcg_batch* B, const mcg_plan* P, hipStream_t s) {
  RunCtx X;
  if (prepare_typed<NC, ST>(B, P, X)) return -1;
  void* dev = nullptr;
  if (X.dev_bytes && hipMalloc(&dev, X.dev_bytes) != hipSuccess) return fail("hipMalloc(%zu) failed", X.dev_bytes);
  int rc = bind_region(X, (unsigned char*)dev, s);
  if (!rc) rc = exec_typed<NC, ST>(B, P, s, X);
  // the region and the staged tables must outlive the launches
  const hipError_t e = hipStreamSynchronize(s);
  if (dev) (void)hipFree(dev);
  if (!rc && e != hipSuccess) rc = fail("hipStreamSynchronize: %s", hipGetErrorString(e));
  return rc;
}

// ---------------------------------------------------------------------------
// mcg_run_noalloc: mcg_run's launches with their device scratch in a
// file-scope array (allocated with the code object on every device that
// loads the library, held until the process ends), for callers that cannot
// allocate.  Host code never passes `scratch` itself to a kernel (in host
// code the name stands for a host-side shadow): each device's address is
// looked up once with hipGetSymbolAddress and kept in g_scratch_dev.
// ---------------------------------------------------------------------------
static constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)4 << 20;
static_assert(NOALLOC_SCRATCH_BYTES == (size_t)MCG_NOALLOC_SCRATCH_BYTES, "header and library disagree");
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

static constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static unsigned char* g_scratch_dev[MAX_DEVICES];

// the current device's copy of `scratch` (looked up on its first use)
int scratch_region(unsigned char** out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= MAX_DEVICES) return fail("device %d outside 0..%d", dev, MAX_DEVICES - 1);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail("hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_dev[dev] = (unsigned char*)p;
  }
  *out = g_scratch_dev[dev];
  return 0;
}

template <int NC, typename ST>
int run_noalloc_typed(const mcg_batch* B, const mcg_plan* P, hipStream_t s) {
  if (P->timing) return fail("mcg_run_noalloc does not time launches: plan->timing must be NULL");
  RunCtx X;
  if (prepare_typed<NC, ST>(B, P, X)) return -1;
  if (X.dev_bytes > NOALLOC_SCRATCH_BYTES)
    return fail("this run needs %zu bytes of device scratch; mcg_run_noalloc has %zu (use mcg_run or a runner)",
                X.dev_bytes, NOALLOC_SCRATCH_BYTES);
  unsigned char* dev = nullptr;
  if (scratch_region(&dev)) return -1;
  if (bind_region(X, dev, s)) return -1;
  // the tables are staged in X, which ends with this call: wait for their copy
  HIPCHK(hipStreamSynchronize(s));
  return exec_typed<NC, ST>(B, P, s, X);
}

template <int NC, typename ST>
int prepare_runner(const mcg_batch* B, const mcg_plan* P, hipStream_t s, RunCtx& X) {
  if (prepare_typed<NC, ST>(B, P, X)) return -1;
  void* dev = nullptr;
  if (X.dev_bytes && hipMalloc(&dev, X.dev_bytes) != hipSuccess) return fail("hipMalloc(%zu) failed", X.dev_bytes);
  X.dev = (unsigned char*)dev;
  if (bind_region(X, (unsigned char*)dev, s)) return -1;
  HIPCHK(hipStreamSynchronize(s));
  return 0;
}

template <int NC, typename ST>
int init_typed(const mcg_batch* B, hipStream_t s) {
  std::vector<int32_t> all(B->nrep);
  for (int r = 0; r < B->nrep; ++r) all[r] = r;
  DevBuf d;
  if (d.upload(all.data(), all.size() * 4, s)) return -1;
  if (launch_fill_f64(B->state, (size_t)B->nrep * MCG_NSTATE, 0.0, s)) return -1;
  if (launch_fill_f64(B->acc, (size_t)B->nrow * MCG_NACC, 0.0, s)) return -1;
  if (launch_fill_f64(B->bins, (size_t)B->nrow * B->nbins * MCG_NBINQ, 0.0, s)) return -1;
  if (B->gacc) {
    int ng = 0;
    for (int gi = 0; gi < B->ngraph; ++gi) ng = std::max(ng, B->graphs_host[gi].ngroup);
    if (launch_fill_f64(B->gacc, (size_t)B->nrow * (ng + 2) * (ng + 1), 0.0, s)) return -1;
  }
  if (launch_fill_i32(B->pt_acc, (size_t)B->nrow, 0, s)) return -1;
  if (launch_fill_i32(B->err, 1, 0, s)) return -1;
  if (B->wstamp) {
    size_t tot = 0;
    for (int r = 0; r < B->nrep; ++r)
      tot = std::max<size_t>(tot, (size_t)B->reps_host[r].site_off + B->graphs_host[B->reps_host[r].graph].n);
    const unsigned g = (unsigned)std::min<size_t>((tot + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill_u32, dim3(g), dim3(256), 0, s, B->wstamp, tot, 0u);
    HIPCHK(hipGetLastError());
  }
  if (launch_measure<NC, ST>(B, (const int32_t*)d.p, B->nrep, 1 | 2 | 8, -1, s)) return -1;
  HIPCHK(hipStreamSynchronize(s));
  return 0;
}

template <int NC, typename ST>
int measure_typed(const mcg_batch* B, int64_t frame, hipStream_t s) {
  std::vector<int32_t> all(B->nrep);
  for (int r = 0; r < B->nrep; ++r) all[r] = r;
  DevBuf d;
  if (d.upload(all.data(), all.size() * 4, s)) return -1;
  if (launch_measure<NC, ST>(B, (const int32_t*)d.p, B->nrep, 1 | 4, frame, s)) return -1;
  HIPCHK(hipStreamSynchronize(s));
  return 0;
}

}  // namespace

#define DISPATCH(fn, ...)                                                                    \
  do {                                                                                       \
    if (B->nc == 1) return fn<1, int8_t>(__VA_ARGS__);                                       \
    if (B->nc == 2 && B->store == MCG_STORE_F32) return fn<2, float>(__VA_ARGS__);           \
    if (B->nc == 2 && B->store == MCG_STORE_F16) return fn<2, __half>(__VA_ARGS__);          \
    if (B->nc == 3 && B->store == MCG_STORE_F32) return fn<3, float>(__VA_ARGS__);           \
    if (B->nc == 3 && B->store == MCG_STORE_F16) return fn<3, __half>(__VA_ARGS__);          \
    return fail("unsupported nc/store combination");                                         \
  } while (0)

extern "C" int mcg_init(const mcg_batch* B, void* stream) {
  if (check_batch(B)) return -1;
  hipStream_t s = (hipStream_t)stream;
  DISPATCH(init_typed, B, s);
}

extern "C" int mcg_run(const mcg_batch* B, const mcg_plan* P, void* stream) {
  if (check_batch(B)) return -1;
  if (!P) return fail("null plan");
  if (P->nthermal < 0 || P->nsweep < 0) return fail("negative sweep counts");
  if (P->algorithm != MCG_METROPOLIS && P->algorithm != MCG_WOLFF) return fail("unknown algorithm %d", P->algorithm);
  hipStream_t s = (hipStream_t)stream;
  DISPATCH(run_typed, B, P, s);
}

// A prepared run (mcg_runner_*): the RunCtx and the region it owns.
struct mcg_runner {
  RunCtx X;
};

namespace {
template <int NC, typename ST>
int runner_create_typed(const mcg_batch* B, const mcg_plan* P, hipStream_t s, mcg_runner* R) {
  return prepare_runner<NC, ST>(B, P, s, R->X);
}
template <int NC, typename ST>
int runner_run_typed(const mcg_batch* B, const mcg_plan* P, hipStream_t s, mcg_runner* R) {
  if (check_key(B, P, R->X)) return -1;
  return exec_typed<NC, ST>(B, P, s, R->X);
}
void runner_free(mcg_runner* R) {
  if (!R) return;
  if (R->X.dev) {
    int cur = 0;
    (void)hipGetDevice(&cur);
    (void)hipSetDevice(R->X.device);
    (void)hipDeviceSynchronize();  // no launch of this run may still read the region
    (void)hipFree(R->X.dev);
    (void)hipSetDevice(cur);
  }
  delete R;
}
}  // namespace

extern "C" int mcg_runner_create(const mcg_batch* B, const mcg_plan* P, void* stream, mcg_runner** out) {
  if (!out) return fail("null runner out-pointer");
  *out = nullptr;
  if (check_batch(B)) return -1;
  if (!P) return fail("null plan");
  if (P->algorithm != MCG_METROPOLIS && P->algorithm != MCG_WOLFF) return fail("unknown algorithm %d", P->algorithm);
  mcg_runner* R = new (std::nothrow) mcg_runner();
  if (!R) return fail("out of host memory");
  hipStream_t s = (hipStream_t)stream;
  const int rc = [&]() -> int { DISPATCH(runner_create_typed, B, P, s, R); }();
  if (rc) {
    runner_free(R);
    return -1;
  }
  *out = R;
  return 0;
}

extern "C" int mcg_runner_run(mcg_runner* R, const mcg_batch* B, const mcg_plan* P, void* stream) {
  if (!R) return fail("null runner");
  if (check_batch(B)) return -1;
  if (!P) return fail("null plan");
  if (P->nthermal < 0 || P->nsweep < 0) return fail("negative sweep counts");
  if (P->algorithm != MCG_METROPOLIS && P->algorithm != MCG_WOLFF) return fail("unknown algorithm %d", P->algorithm);
  hipStream_t s = (hipStream_t)stream;
  DISPATCH(runner_run_typed, B, P, s, R);
}

extern "C" int mcg_runner_destroy(mcg_runner* R) {
  runner_free(R);
  return 0;
}

extern "C" int mcg_run_noalloc(const mcg_batch* B, const mcg_plan* P, void* stream) {
  if (check_batch(B)) return -1;
  if (!P) return fail("null plan");
  if (P->nthermal < 0 || P->nsweep < 0) return fail("negative sweep counts");
  if (P->algorithm != MCG_METROPOLIS && P->algorithm != MCG_WOLFF) return fail("unknown algorithm %d", P->algorithm);
  hipStream_t s = (hipStream_t)stream;
  DISPATCH(run_noalloc_typed, B, P, s);
}

extern "C" int mcg_sweeps(const mcg_batch* B, const mcg_plan* P, int64_t sweep0, int32_t nsweeps, void* stream) {
  if (check_batch(B)) return -1;
  if (!P) return fail("null plan");
  mcg_plan q = *P;
  q.nthermal = nsweeps;  // all sweeps unmeasured
  q.nsweep = 0;
  q.sweep0 = sweep0;
  q.pt_every = 0;
  hipStream_t s = (hipStream_t)stream;
  DISPATCH(run_typed, B, &q, s);
}

extern "C" int mcg_measure(const mcg_batch* B, int64_t frame, void* stream) {
  if (check_batch(B)) return -1;
  hipStream_t s = (hipStream_t)stream;
  DISPATCH(measure_typed, B, frame, s);
}

// greedy colouring in site order: each site takes the smallest colour not
// used by an already-coloured neighbour (in- and out-links both count)
// DSatur (Brelaz 1979): colour next the uncoloured vertex with the most
// distinct colours among its neighbours (ties: most neighbours, then lowest
// index) with the lowest colour none of them has.  Returns the colour count.
static int dsatur_colour(int32_t n, const std::vector<std::vector<int32_t>>& adj, std::vector<int32_t>& col) {
  col.assign(n, -1);
  std::vector<std::vector<char>> seen(n);
  std::vector<int32_t> sat(n, 0);
  // max-heap on (saturation, degree, -index)
  typedef std::tuple<int32_t, int32_t, int32_t> Key;
  std::priority_queue<Key> q;
  for (int32_t i = 0; i < n; ++i) q.push(Key(0, (int32_t)adj[i].size(), -i));
  int ncol = 0;
  while (!q.empty()) {
    const Key k = q.top();
    q.pop();
    const int32_t i = -std::get<2>(k);
    if (col[i] >= 0 || std::get<0>(k) != sat[i]) continue;  // stale entry
    int c = 0;
    while (c < (int)seen[i].size() && seen[i][c]) ++c;
    col[i] = c;
    ncol = std::max(ncol, c + 1);
    for (int32_t j : adj[i]) {
      if (col[j] >= 0) continue;
      if ((int)seen[j].size() <= c) seen[j].resize(c + 1, 0);
      if (!seen[j][c]) {
        seen[j][c] = 1;
        ++sat[j];
        q.push(Key(sat[j], (int32_t)adj[j].size(), -j));
      }
    }
  }
  return ncol;
}

// Proper colouring of the site graph: greedy in site order (the checkerboard
// of square and cubic lattices), or DSatur where that needs fewer colours
// (the honeycomb with second neighbours: 4 colours of 2048 sites against
// greedy's 6 on 64x64 cells).  Fewer colours mean fewer synchronised rounds
// per sweep and, for the streaming pass, fewer launches and neighbour reads.
extern "C" int mcg_colour_graph(int32_t n, int32_t zmax, const int32_t* nbr, int32_t* colour) {
  if (n < 0 || zmax < 0 || (!nbr && n * zmax) || !colour) return fail("bad arguments to mcg_colour_graph");
  std::vector<std::vector<int32_t>> adj(n);
  for (int32_t i = 0; i < n; ++i)
    for (int32_t l = 0; l < zmax; ++l) {
      const int32_t j = nbr[(size_t)i * zmax + l];
      if (j < 0 || j == i) continue;
      if (j >= n) return fail("neighbour index %d out of range", j);
      adj[i].push_back(j);
      adj[j].push_back(i);
    }
  std::vector<int32_t> mark;
  int ncol = 0;
  for (int32_t i = 0; i < n; ++i) colour[i] = -1;
  for (int32_t i = 0; i < n; ++i) {
    mark.assign(ncol + 1, 0);
    for (int32_t j : adj[i])
      if (colour[j] >= 0 && colour[j] <= ncol) mark[colour[j]] = 1;
    int c = 0;
    while (c <= ncol && mark[c]) ++c;
    colour[i] = c;
    if (c + 1 > ncol) ncol = c + 1;
  }
  if (ncol > 2) {
    std::vector<int32_t> ds;
    const int nd = dsatur_colour(n, adj, ds);
    if (nd < ncol) {
      for (int32_t i = 0; i < n; ++i) colour[i] = ds[i];
      ncol = nd;
    }
  }
  return ncol;
}
