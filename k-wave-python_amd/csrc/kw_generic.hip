// Generic-length family of the time-loop launchers.
//
// The fused kernels of kw_kernels.hpp are compiled for a fixed set of axis
// lengths (register-resident transforms with compile-time radix plans) and,
// along the contiguous axis, for even row counts.  Every other grid runs here:
// the same launcher entry points with the same argument blocks and results, so
// the step sequence, graphs, batching, sources and sensors of kw_abi.hip are
// unchanged.
//
// Transforms are Stockham passes over lines held in LDS with a radix plan chosen at
// run time: every radix from 2 to 16 as a butterfly in registers (few stages: 90 =
// 9 10, 108 = 9 12, 240 = 15 16), any larger prime factor as a direct stage over the
// sums and differences of mirrored inputs.  A kernel transforms all its lines at once -
// the axes of a density update, the jobs of a spectral pass - so that a stage fills the
// workgroup, and the contiguous-axis updates run between their inverse and forward
// transforms without leaving LDS.  Inverse transforms are forward ones with the real and
// imaginary parts exchanged on the way in and out, so one set of butterflies serves both.
// Lines too long for that (more LDS than a compute unit has) go through real temporaries
// (Fields::tmp) and a stash spectrum (Fields::gstash) instead.
//
// What bounds these kernels is latency on small grids (a 291 x 242 step: 14 launches of
// 0.9 ms together before, six of 75 us now) and, on larger ones, the loads, address
// arithmetic and LDS traffic around the butterflies (a copy of the 108 x 90 x 75 passes
// without any butterfly takes three quarters of their time; the radix limit, 5 to 16,
// changes it by a tenth).  Measured against unfused kernels with radices up to 8, one work
// item per output of a prime stage, twiddles in global memory and jobs one after the
// other: 291 x 242 (2 11 11 and 3 97) 890 -> 75 us a step, 108 x 90 x 75 with velocity
// records 440 -> 195 us.
//
// Arithmetic follows the fused kernels operation for operation (same operator
// tables, same order of the update terms), so the two families agree to FP32
// rounding of the transforms.
#include <algorithm>

#include "kw_host.hpp"
#include "kw_kernels.hpp"

namespace kw {

constexpr int kGenMaxN = 4096;
constexpr int kGenThreads = 256;
constexpr int kGenMaxStages = 16;
constexpr size_t kGenLds = 163840;     // LDS of a compute unit
// A workgroup's LDS where it can choose.  us a step with 32 KB -> 64 KB: 330 x 333 x 310 4221 ->
// 3708, 291 x 300 x 322 power law 5615 -> 5394, 200 x 180 x 170 and 108 x 90 x 75 with velocities
// 1063 -> 964 and 190 -> 181; 400^3 6800 -> 6905, 150^3 power law 452 -> 471, 360 x 420 x 64
// 966 -> 996; 2-D grids of 242 x 291 to 2000 x 1900 alike.  80 KB loses twice as much and gains less.
constexpr size_t kGenLdsShare = 32768;

struct GPlan {
  int n;
  int ns;
  int r[kGenMaxStages];
};

// Split m (no prime factor above 13) into the fewest factors of at most 16.
static void gsplit(int m, int top, GPlan& cur, GPlan& best) {
  if (m == 1) {
    if (best.ns < 0 || cur.ns < best.ns) best = cur;
    return;
  }
  if (cur.ns >= kGenMaxStages || (best.ns >= 0 && cur.ns + 1 >= best.ns)) return;
  for (int f = std::min(top, 16); f >= 2; --f) {
    if (m % f) continue;
    cur.r[cur.ns++] = f;
    gsplit(m / f, f, cur, best);
    --cur.ns;
  }
}

// Radix plan of n: prime factors above 13 first (direct stages, on the untwiddled
// first stages), then the fewest butterflies of at most 16, odd ones first: the first
// stage writes with a stride of its radix, which an odd one spreads over the LDS banks.
static GPlan gplan(int n) {
  GPlan p{};
  p.n = n;
  int m = n, rest = n;
  for (int f : {2, 3, 5, 7, 11, 13})
    while (rest % f == 0) rest /= f;
  for (int f = 17; rest > 1; f += 2)
    while (rest % f == 0) {
      p.r[p.ns++] = f;
      m /= f;
      rest /= f;
    }
  GPlan cur{}, best{};
  best.ns = -1;
  gsplit(m, 16, cur, best);
  std::stable_sort(best.r, best.r + best.ns, [](int x, int y) { return (x & 1) > (y & 1); });
  for (int i = 0; i < best.ns; ++i) p.r[p.ns++] = best.r[i];
  return p;
}

bool compiled_size(int n) { return size_supported_impl(n); }

bool size_supported(int n) { return compiled_size(n) || (n >= 2 && n <= kGenMaxN); }

// The fused contiguous-axis kernels need a compiled length and an even row count
// (they clamp a row pair into the grid).
bool generic_z(const Geom& g) { return !compiled_size(g.nz) || (g.rows & 1); }

// ---------------------------------------------------------------------------
// butterflies of any radix from 2 to 16 (forward)
// ---------------------------------------------------------------------------
// cos and sin of 2 pi m / n at compile time (Taylor series in double precision)
constexpr double gsin_series(double x) {
  double t = x, s = x;
  for (int i = 1; i < 20; ++i) { t *= -x * x / ((2 * i) * (2 * i + 1)); s += t; }
  return s;
}
constexpr double gcos_series(double x) {
  double t = 1, s = 1;
  for (int i = 1; i < 20; ++i) { t *= -x * x / ((2 * i - 1) * (2 * i)); s += t; }
  return s;
}
template <int R>
struct GRoots {  // cos and sin of 2 pi m / R
  float c[R], s[R];
  constexpr GRoots() : c(), s() {
    for (int m = 0; m < R; ++m) {
      const double x = 2.0 * 3.14159265358979323846 * (2 * m > R ? m - R : m) / R;
      c[m] = (float)gcos_series(x);
      s[m] = (float)gsin_series(x);
    }
  }
};

template <int R>
__device__ __forceinline__ void gdft(float2* v);

// prime radix 11 or 13: as dft_odd
template <int R>
__device__ __forceinline__ void gdft_prime(float2* v) {
  constexpr int H = (R - 1) / 2;
  constexpr GRoots<R> w{};
  float2 p[H], d[H];
  const float2 x0 = v[0];
  float2 sum = x0;
#pragma unroll
  for (int j = 0; j < H; ++j) {
    p[j] = cadd(v[j + 1], v[R - 1 - j]);
    d[j] = csub(v[j + 1], v[R - 1 - j]);
    sum = cadd(sum, p[j]);
  }
  v[0] = sum;
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    float2 a = x0, b = make_float2(0.f, 0.f);
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const int m = (k * (j + 1)) % R;
      a = make_float2(fmaf(w.c[m], p[j].x, a.x), fmaf(w.c[m], p[j].y, a.y));
      b = make_float2(fmaf(w.s[m], d[j].x, b.x), fmaf(w.s[m], d[j].y, b.y));
    }
    v[k] = make_float2(a.x + b.y, a.y - b.x);
    v[R - k] = make_float2(a.x - b.y, a.y + b.x);
  }
}

// radix R1 R2 from R1 butterflies of radix R2 and R2 of radix R1
template <int R1, int R2>
__device__ __forceinline__ void gdft_pair(float2* v) {
  constexpr int R = R1 * R2;
  constexpr GRoots<R> w{};
  float2 y[R];
#pragma unroll
  for (int n1 = 0; n1 < R1; ++n1) {
    float2 t[R2];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) t[n2] = v[n1 + R1 * n2];
    gdft<R2>(t);
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2)
      y[n1 * R2 + k2] = n1 * k2 == 0 ? t[k2] : cmul(t[k2], make_float2(w.c[(n1 * k2) % R], -w.s[(n1 * k2) % R]));
  }
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2) {
    float2 t[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) t[n1] = y[n1 * R2 + k2];
    gdft<R1>(t);
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) v[k2 + R2 * k1] = t[k1];
  }
}

template <int R>
__device__ __forceinline__ void gdft(float2* v) {
  if constexpr (R == 2 || R == 3 || R == 4 || R == 5 || R == 7 || R == 8) dft<R, -1>(v);
  else if constexpr (R == 11 || R == 13) gdft_prime<R>(v);
  else if constexpr (R % 4 == 0) gdft_pair<4, R / 4>(v);  // 12, 16
  else if constexpr (R % 2 == 0) gdft_pair<2, R / 2>(v);  // 6, 10, 14
  else gdft_pair<3, R / 3>(v);                            // 9, 15
}

// ---------------------------------------------------------------------------
// LDS transform of nl lines of length pl.n; element (n, line c) at buf[n * sp + c]
// (odd pitch sp >= nl).  Ping-pongs between A and B and returns the buffer that holds
// the result.  Every thread of the workgroup must call it.
// ---------------------------------------------------------------------------
// a / d for 0 <= a < 2^16 and a divisor whose reciprocal is given: the quotient's distance
// from an integer, at least 1 / (2 d), is far above the rounding of the product
__device__ __forceinline__ int gdiv(int a, float inv) { return (int)(((float)a + 0.5f) * inv); }

// lanes of the workgroup over (line, item) pairs: line c, first item i0, item step
struct GLanes {
  int c, i0, step;
  __device__ __forceinline__ explicit GLanes(int nl) {
    const float inv = 1.0f / (float)nl;
    step = max(1, gdiv(blockDim.x, inv));
    i0 = gdiv(threadIdx.x, inv);
    c = threadIdx.x - i0 * nl;
    if (i0 >= step) i0 = 1 << 30;  // a lane left over by nl does nothing
  }
};

// One Stockham stage of radix R over every line: butterfly j of a line reads elements
// j + r N/R, twiddles them by tw[r k N/(NS R)] (k = j mod NS), and writes its R-point DFT
// to positions o + r NS, o = (j / NS) NS R + k -- the stage of the fused transforms
// (reg_stage).
template <int R>
__device__ __forceinline__ void gstage(const float2* src, float2* dst, const float2* tw, int N, int NS, int sp, const GLanes& ln) {
  const int nbf = N / R, TWS = nbf / NS;
  const float ins = 1.0f / (float)NS;
#pragma unroll 1
  for (int j = ln.i0; j < nbf; j += ln.step) {
    const int q = gdiv(j, ins), k = j - q * NS;
    // strides the compiler must not multiply out ahead of the loop: the multiples of every
    // radix's strides would take a hundred registers
    int sst = nbf * sp, dst_st = NS * sp;
    asm("" : "+v"(sst), "+v"(dst_st));
    float2 x[R];
    const float2* ps = src + j * sp + ln.c;
#pragma unroll
    for (int r = 0; r < R; ++r, ps += sst) x[r] = *ps;
    if (NS > 1) {
      const int kt = k * TWS;
#pragma unroll
      for (int r = 1; r < R; ++r) x[r] = cmul(x[r], tw[r * kt]);
    }
    gdft<R>(x);
    float2* pd = dst + (q * NS * R + k) * sp + ln.c;
#pragma unroll
    for (int r = 0; r < R; ++r, pd += dst_st) *pd = x[r];
  }
}

// A stage of a prime radix R above 13, direct: the twiddled inputs r and R - r are
// replaced by their sum and difference, and outputs q and R - q come from one cosine sum
// over the sums and one sine sum over the differences (a quarter of the multiplications
// of the plain sum), QT of them per work item so that each operand read serves QT terms.
template <int QT>
__device__ __forceinline__ void gprime_sums(const float2* src, float2* dst, const float2* tw, int R, int NS, int nbf, int sp, const GLanes& ln);

__device__ __forceinline__ void gstage_prime(float2* src, float2* dst, const float2* tw, int N, int R, int NS, int sp, const GLanes& ln) {
  const int nbf = N / R, TWS = nbf / NS, H = (R - 1) / 2;
  const float ins = 1.0f / (float)NS, ibf = 1.0f / (float)nbf;
  for (int e = ln.i0; e < nbf * H; e += ln.step) {
    const int r = 1 + gdiv(e, ibf), j = e - (r - 1) * nbf;
    float2* const pa = src + (j + r * nbf) * sp + ln.c;
    float2* const pb = src + (j + (R - r) * nbf) * sp + ln.c;
    float2 a = *pa, b = *pb;
    if (NS > 1) {
      const int kt = (j - gdiv(j, ins) * NS) * TWS;
      a = cmul(a, tw[r * kt]);
      b = cmul(b, tw[(R - r) * kt]);
    }
    *pa = cadd(a, b);
    *pb = csub(a, b);
  }
  __syncthreads();
  // a small workgroup's share is spread over all its lanes instead
  if (nbf * H <= 2 * ln.step) gprime_sums<1>(src, dst, tw, R, NS, nbf, sp, ln);
  else gprime_sums<4>(src, dst, tw, R, NS, nbf, sp, ln);
}

template <int QT>
__device__ __forceinline__ void gprime_sums(const float2* src, float2* dst, const float2* tw, int R, int NS, int nbf, int sp, const GLanes& ln) {
  const int H = (R - 1) / 2, nqt = (H + QT) / QT;  // outputs 0..H
  const float ins = 1.0f / (float)NS, ibf = 1.0f / (float)nbf;
  for (int e = ln.i0; e < nbf * nqt; e += ln.step) {
    const int t = gdiv(e, ibf), j = e - t * nbf, q0 = t * QT;
    const float2 x0 = src[j * sp + ln.c];
    float2 a[QT], b[QT];
    int m[QT];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      a[i] = x0;
      b[i] = make_float2(0.f, 0.f);
      m[i] = 0;
    }
    const float2* ps = src + (j + nbf) * sp + ln.c;
    const float2* pd = src + (j + (R - 1) * nbf) * sp + ln.c;
    const int st = nbf * sp;
#pragma unroll 4
    for (int r = 1; r <= H; ++r, ps += st, pd -= st) {
      const float2 s = *ps, d = *pd;
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        m[i] += q0 + i;  // r q mod R
        if (m[i] >= R) m[i] -= R;
        const float2 w = tw[m[i] * nbf];  // (cos, -sin) of 2 pi r q / R
        a[i] = make_float2(fmaf(w.x, s.x, a[i].x), fmaf(w.x, s.y, a[i].y));
        b[i] = make_float2(fmaf(-w.y, d.x, b[i].x), fmaf(-w.y, d.y, b[i].y));
      }
    }
    const int q = gdiv(j, ins), k = j - q * NS;
    float2* const o = dst + (q * NS * R + k) * sp + ln.c;
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      if (q0 + i > H) continue;
      o[(q0 + i) * NS * sp] = make_float2(a[i].x + b[i].y, a[i].y - b[i].x);
      if (q0 + i > 0) o[(R - q0 - i) * NS * sp] = make_float2(a[i].x - b[i].y, a[i].y + b[i].x);
    }
  }
}

__device__ __forceinline__ float2* gfft(float2* A, float2* B, const GPlan& pl, const float2* tw, int nl, int sp) {
  const int N = pl.n;
  const GLanes ln(nl);
  float2* src = A;
  float2* dst = B;
  int NS = 1;
  for (int s = 0; s < pl.ns; ++s) {
    const int R = pl.r[s];
    switch (R) {
#define KW_GST(r) case r: gstage<r>(src, dst, tw, N, NS, sp, ln); break;
      KW_GST(2) KW_GST(3) KW_GST(4) KW_GST(5) KW_GST(6) KW_GST(7) KW_GST(8) KW_GST(9)
      KW_GST(10) KW_GST(11) KW_GST(12) KW_GST(13) KW_GST(14) KW_GST(15) KW_GST(16)
#undef KW_GST
      default: gstage_prime(src, dst, tw, N, R, NS, sp, ln); break;
    }
    __syncthreads();
    float2* t = src;
    src = dst;
    dst = t;
    NS *= R;
  }
  return src;
}

static int gpitch(int nl) { return nl | 1; }
static size_t glds_bytes(int n, int nl) { return sizeof(float2) * ((size_t)2 * n * gpitch(nl) + n); }

// Loops that move elements between global memory and LDS take them GB at a time, all
// loads of a batch before its first write (index clamped, writes guarded): one at a time,
// every element would wait for its own load.
constexpr int GB = 4;
template <class Load, class Put>
__device__ __forceinline__ void gbatch(int total, Load load, Put put) {
  const int nt = blockDim.x;
  for (int e0 = threadIdx.x; e0 < total; e0 += GB * nt) {
    decltype(load(0)) v[GB];
#pragma unroll
    for (int i = 0; i < GB; ++i) v[i] = load(min(e0 + i * nt, total - 1));
#pragma unroll
    for (int i = 0; i < GB; ++i)
      if (e0 + i * nt < total) put(e0 + i * nt, v[i]);
  }
}
struct GTwo { float2 a, b; };

// LDS of a kernel: n twiddles, then two buffers of n * sp.  The first twiddles of a lane
// are loaded when the object is made and put into LDS by put(), after the kernel has
// loaded its lines, so that the two do not wait for each other.
struct GTw {
  static constexpr int K = 2;
  const float2* src;
  float2* lds;
  float2 r[K];
  int N;
  __device__ __forceinline__ GTw(float2* smem, const float2* twg, int n) : src(twg), lds(smem), N(n) {
#pragma unroll
    for (int i = 0; i < K; ++i) r[i] = ld2(gp(twg), min((int)(threadIdx.x + i * blockDim.x), N - 1));
  }
  __device__ __forceinline__ void put() const {
#pragma unroll
    for (int i = 0; i < K; ++i)
      if ((int)(threadIdx.x + i * blockDim.x) < N) lds[threadIdx.x + i * blockDim.x] = r[i];
    for (int i = threadIdx.x + K * blockDim.x; i < N; i += blockDim.x) lds[i] = ld2(gp(src), i);
  }
};

__device__ __forceinline__ float2 gswap(float2 a) { return make_float2(a.y, a.x); }

// ---------------------------------------------------------------------------
// contiguous axis: real rows <-> half spectra, two rows per complex line
// ---------------------------------------------------------------------------
// Instance filter of a transform launch: skip instances that have finished
// (tdev), and, for source spectra, instances whose source `which` (-1: p,
// 0..2: u_i) is not an active spectral (CHAIN) source at this step.
enum { GF_ALL = -3, GF_ACTIVE = -2 };
__device__ __forceinline__ bool gen_skip(const int* tdev, int toff, const Inst* inst, int b, int which) {
  if (which == GF_ALL || !tdev) return false;
  const int t = gp(tdev)[b] + toff;
  const Inst& I = inst[b];
  if (t >= I.nt) return true;
  if (which == GF_ACTIVE) return false;
  const Src& s = which < 0 ? I.srcp : I.srcu[which];
  return !(s.mode == SRC_CHAIN && t < s.len);
}

// The half spectra of P row pairs into lines c0 .. c0 + P - 1 as the (exchanged) spectra of
// a + i b, Hermitian extension of each; after the transform, row a is the imaginary and row
// b the real part.  A missing second row (odd row count) or pair reads as zero.
__device__ __forceinline__ void gpairs_in(float2* A, int sp, int c0, const float2* __restrict__ spec, const Geom& g, int N, int pair0, int P) {
  const auto s = gp(spec);
  const int nh = g.nh;
  const float inh = 1.0f / (float)nh;
  gbatch(P * nh,
         [&](int e) {
           const int lp = gdiv(e, inh), k = e - lp * nh;
           const int ra = 2 * (pair0 + lp), rb = ra + 1;
           GTwo v{ld2(s, (int64_t)min(ra, g.rows - 1) * g.nhp + k), ld2(s, (int64_t)min(rb, g.rows - 1) * g.nhp + k)};
           if (ra >= g.rows) v.a = make_float2(0.f, 0.f);
           if (rb >= g.rows) v.b = make_float2(0.f, 0.f);
           return v;
         },
         [&](int e, const GTwo& v) {
           const int lp = gdiv(e, inh), k = e - lp * nh;
           const float2 a = v.a, c = v.b;
           const bool self = k == 0 || 2 * k == N;
           const float2 lo = self ? make_float2(c.x, a.x) : make_float2(a.y + c.x, a.x - c.y);
           const float2 hi = self ? lo : make_float2(c.x - a.y, a.x + c.y);
           A[k * sp + c0 + lp] = lo;
           A[(k == 0 ? 0 : N - k) * sp + c0 + lp] = hi;
         });
}
// lines c0 .. of transformed row pairs -> their half spectra
__device__ __forceinline__ void gpairs_out(const float2* Z, int sp, int c0, float2* __restrict__ spec, const Geom& g, int N, int pair0, int P) {
  const auto s = gw(spec);
  const int nh = g.nh;
  const float inh = 1.0f / (float)nh;
  for (int e = threadIdx.x; e < P * nh; e += blockDim.x) {
    const int lp = gdiv(e, inh), k = e - lp * nh;
    const int ra = 2 * (pair0 + lp), rb = ra + 1;
    const float2 z = Z[k * sp + c0 + lp], zc = Z[(k == 0 ? 0 : N - k) * sp + c0 + lp];
    if (ra < g.rows) st2(s, (int64_t)ra * g.nhp + k, make_float2(0.5f * (z.x + zc.x), 0.5f * (z.y - zc.y)));
    if (rb < g.rows) st2(s, (int64_t)rb * g.nhp + k, make_float2(0.5f * (z.y + zc.y), -0.5f * (z.x - zc.x)));
  }
}
// Update loop over P row pairs, GU positions of a thread at a time: load(r, n) for both rows
// of each (rows clamped into the grid), then apply(lp, n, ra, two rows?, operands).
constexpr int GU = 2;
template <class Load, class Apply>
__device__ __forceinline__ void gupdate(const Geom& g, int N, int pair0, int P, Load load, Apply apply) {
  const float in = 1.0f / (float)N;
  const int total = P * N, nt = blockDim.x;
  for (int e0 = threadIdx.x; e0 < total; e0 += GU * nt) {
    decltype(load(0, 0)) va[GU], vb[GU];
#pragma unroll
    for (int i = 0; i < GU; ++i) {
      const int e = min(e0 + i * nt, total - 1);
      const int lp = gdiv(e, in), n = e - lp * N, ra = 2 * (pair0 + lp);
      va[i] = load(min(ra, g.rows - 1), n);
      vb[i] = load(min(ra + 1, g.rows - 1), n);
    }
#pragma unroll
    for (int i = 0; i < GU; ++i) {
      const int e = e0 + i * nt;
      const int lp = gdiv(e, in), n = e - lp * N, ra = 2 * (pair0 + lp);
      if (e < total && ra < g.rows) apply(lp, n, ra, ra + 1 < g.rows, va[i], vb[i]);
    }
  }
}
// element loop over P row pairs: pair lp, position n, rows ra and rb = ra + 1
#define KW_GEN_PAIR_LOOP(N)                                              \
  for (int e = threadIdx.x; e < P * (N); e += blockDim.x)                \
    if (const int lp = gdiv(e, 1.0f / (float)(N)), n = e - lp * (N), ra = 2 * (pair0 + lp); ra < g.rows)

__global__ __launch_bounds__(kGenThreads) void k_gzfwd(Geom g, const float* __restrict__ f, int64_t fs, float2* __restrict__ spec,
                                                       int64_t ss, const float2* __restrict__ twg, GPlan pl, int P, int sp,
                                                       const int* tdev, int toff, const Inst* __restrict__ inst, int which) {
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y;
  if (gen_skip(tdev, toff, inst, b, which)) return;
  const int N = pl.n;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  float2* A = gsm + N;
  float2* B = A + N * sp;
  const auto fb = gp(f + b * fs);
  const int pair0 = blockIdx.x * P;
  const float in = 1.0f / (float)N;
  gbatch(P * N,
         [&](int e) {
           const int lp = gdiv(e, in), n = e - lp * N;
           const int ra = 2 * (pair0 + lp), rb = ra + 1;
           const float x = fb[(int64_t)min(ra, g.rows - 1) * N + n], y = fb[(int64_t)min(rb, g.rows - 1) * N + n];
           return make_float2(ra < g.rows ? x : 0.f, rb < g.rows ? y : 0.f);
         },
         [&](int e, float2 v) {
           const int lp = gdiv(e, in), n = e - lp * N;
           A[n * sp + lp] = v;
         });
  gt.put();
  __syncthreads();
  const float2* Z = gfft(A, B, pl, tw, P, sp);
  gpairs_out(Z, sp, 0, spec + b * ss, g, N, pair0, P);
}

__global__ __launch_bounds__(kGenThreads) void k_gzinv(Geom g, const float2* __restrict__ spec, int64_t ss, float* __restrict__ f,
                                                       int64_t fs, const float2* __restrict__ twg, GPlan pl, int P, int sp,
                                                       float scale, const int* tdev, int toff, const Inst* __restrict__ inst, int which) {
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y;
  if (gen_skip(tdev, toff, inst, b, which)) return;
  const int N = pl.n;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  float2* A = gsm + N;
  float2* B = A + N * sp;
  const auto fb = gw(f + b * fs);
  const int pair0 = blockIdx.x * P;
  gpairs_in(A, sp, 0, spec + b * ss, g, N, pair0, P);
  gt.put();
  __syncthreads();
  const float2* Z = gfft(A, B, pl, tw, P, sp);
  KW_GEN_PAIR_LOOP(N) {
    const float2 z = Z[n * sp + lp];
    fb[(int64_t)ra * N + n] = scale * z.y;
    if (ra + 1 < g.rows) fb[(int64_t)(ra + 1) * N + n] = scale * z.x;
  }
}

// Items (row pairs, columns) per workgroup when each takes `lines` lines of length n: the
// most, up to 16, that leave two workgroups per compute unit and fit the LDS; 0 when not
// even one fits.
static int gen_items(int n, int lines, int64_t items) {
  int best = 0;
  for (int p = 1; p <= 16; p *= 2) {
    if (glds_bytes(n, p * lines) > (p == 1 ? kGenLds : kGenLdsShare)) break;
    if (p > 1 && items / p < 512) break;
    best = p;
  }
  return best;
}
// Threads of a workgroup that holds `elems` elements: a wavefront for every 768 (12 a
// lane, about a butterfly each), as long as the launch fills the chip with that; a
// launch of fewer workgroups takes all the lanes it can use.  At least a lane per line
// (GLanes; at most 16 columns of kMaxJobs jobs).
static_assert(16 * kMaxJobs <= kGenThreads, "a lane per line");
static int gen_threads(int lines, int n, int64_t groups) {
  int nt = 64;
  while (nt < kGenThreads && (nt < lines || (int64_t)lines * n > 12 * nt || groups * nt < 131072)) nt *= 2;
  return nt;
}
static hipError_t gzfwd(const Geom& g, int nb, const float* f, int64_t fs, float2* spec, int64_t ss, const float2* tw,
                        const int* tdev, int toff, const Inst* inst, int which, hipStream_t st) {
  const GPlan pl = gplan(g.nz);
  const int npairs = (g.rows + 1) / 2, P = gen_items(g.nz, 1, (int64_t)npairs * nb);
  if (!P) return hipErrorInvalidValue;
  const int blocks = (npairs + P - 1) / P;
  hipLaunchKernelGGL(k_gzfwd, dim3(blocks, nb), dim3(gen_threads(P, g.nz, (int64_t)blocks * nb)), glds_bytes(g.nz, P), st, g, f, fs, spec,
                     ss, tw, pl, P, gpitch(P), tdev, toff, inst, which);
  return hipGetLastError();
}

static hipError_t gzinv(const Geom& g, int nb, const float2* spec, int64_t ss, float* f, int64_t fs, const float2* tw, float scale,
                        const int* tdev, int toff, const Inst* inst, int which, hipStream_t st) {
  const GPlan pl = gplan(g.nz);
  const int npairs = (g.rows + 1) / 2, P = gen_items(g.nz, 1, (int64_t)npairs * nb);
  if (!P) return hipErrorInvalidValue;
  const int blocks = (npairs + P - 1) / P;
  hipLaunchKernelGGL(k_gzinv, dim3(blocks, nb), dim3(gen_threads(P, g.nz, (int64_t)blocks * nb)), glds_bytes(g.nz, P), st, g, spec, ss, f,
                     fs, tw, pl, P, gpitch(P), scale, tdev, toff, inst, which);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// strided axes: column passes (k_col semantics)
// ---------------------------------------------------------------------------
// an axis's entry of an argument block by selects: indexed by a run-time axis, the whole
// block would be copied to scratch memory first
template <class T>
__device__ __forceinline__ T gpick(T const (&t)[3], int ax) { return ax == 0 ? t[0] : ax == 1 ? t[1] : t[2]; }

// operator value of a job at (x index n, column col of outer index o), without 1/ntot
__device__ __forceinline__ float2 gjob_op(const XJob& jb, const Ops& ops, const Geom& g, float kap, int n, int o, int col) {
  const float kx = gp(ops.k[0])[n];
  const float ky = gp(ops.k[1])[g.nd == 2 ? col : o];
  float km2 = fmaf(kx, kx, ky * ky);
  if (g.nd == 3) {
    const float kz = gp(ops.k[2])[col];
    km2 = fmaf(kx, kx, fmaf(kz, kz, ky * ky));
  }
  float2 op = make_float2(1.f, 0.f);
  if (jb.kind == XK_GRAD || jb.kind == XK_DIV || jb.kind == XK_UNSTAGGER) {
    const float2* t = jb.kind == XK_GRAD ? gpick(ops.grad, jb.axis) : jb.kind == XK_DIV ? gpick(ops.div, jb.axis) : gpick(ops.unst, jb.axis);
    op = ld2(gp(t), jb.axis == 0 ? n : ((jb.axis == 1 && g.nd == 3) ? o : col));
  }
  switch (jb.kind) {
    case XK_GRAD:
    case XK_DIV: return cscale(op, kap > 0.f ? sinc_k2(kap * kap * km2) : 1.f);
    case XK_FRAC1: return make_float2(kpow2(km2, ops.frac1), 0.f);
    case XK_FRAC2: return make_float2(kpow2(km2, ops.frac2), 0.f);
    case XK_SRCKAPPA: return make_float2(kap > 0.f ? cos_k2(kap * kap * km2) : 1.f, 0.f);
    default: return op;
  }
}

// L columns per workgroup, every buffer (FFT-only: blockIdx.z) or every job at once: the
// distinct inputs are transformed together as nin L lines, multiplied out into njob L lines
// and transformed back together.  All of a workgroup's inputs are in LDS before its first
// store, so jobs may write each other's inputs.
__global__ __launch_bounds__(kGenThreads) void k_gcol(Geom g, Fields fl, Ops ops, const Inst* __restrict__ inst, ColArgs a,
                                                      const float2* __restrict__ twg, GPlan pl, int L, int sp) {
  if (a.gath && (int)blockIdx.x >= a.gx) return gather_blocks(g, fl, inst, a);
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y;
  const int N = pl.n;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  const int t = fl.tdev ? step_of(fl, b) : -1, nt = inst[b].nt;
  float2* A = gsm + N;
  float2* B = A + N * sp;
  const int ntile = (a.ncols + L - 1) / L;
  const int lid = xcd_remap(blockIdx.x, a.gx);
  const int o = lid / ntile, col0 = (lid - o * ntile) * L;
  const int64_t base0 = (int64_t)b * g.nspec + (int64_t)o * a.ostride;
  const int ls = 31 - __clz(L);  // L is a power of two
  // (a column beyond the last one is a copy of it and is not stored)
  auto load = [&](const float2* buf, int c0, bool inverse) {
    const auto p = gp(buf);
    gbatch(N * L, [&](int e) { return ld2(p, base0 + min(col0 + (e & (L - 1)), a.ncols - 1) + (int64_t)(e >> ls) * a.estride); },
           [&](int e, float2 v) { A[(e >> ls) * sp + c0 + (e & (L - 1))] = inverse ? gswap(v) : v; });
  };
  auto store = [&](const float2* Z, int c0, float2* buf, bool inverse) {
    const auto p = gw(buf);
    for (int e = threadIdx.x; e < N * L; e += blockDim.x) {
      const int c = e & (L - 1), n = e >> ls;
      const float2 v = Z[n * sp + c0 + c];
      if (col0 + c < a.ncols) st2(p, base0 + col0 + c + (int64_t)n * a.estride, inverse ? gswap(v) : v);
    }
  };
  if (a.mode != 2) {
    float2* buf = fl.spec[a.bufs[blockIdx.z]];
    load(buf, 0, a.mode == 1);
    gt.put();
    if (t >= nt) return;
    __syncthreads();
    store(gfft(A, B, pl, tw, L, sp), 0, buf, a.mode == 1);
    return;
  }
  const float kap = inst[b].kap;
  int nin = 0;
  for (int j = 0, last = -1; j < a.njob; ++j)
    if (a.job[j].in != last) { last = a.job[j].in; load(fl.spec[last], L * nin++, false); }
  gt.put();
  if (t >= nt) return;
  __syncthreads();
  float2* X = gfft(A, B, pl, tw, nin * L, sp);
  float2* Y = X == A ? B : A;
  // gradients and divergences at any stable time step: kappa by its polynomial, straight-line
  const float kn0 = gp(ops.k[0])[N / 2], kn1 = gp(ops.k[1])[g.n[1] / 2], kn2 = g.nd == 3 ? gp(ops.k[2])[g.nz / 2] : 0.f;
  const float kap2 = kap * kap;
  const bool poly = kap2 * (kn0 * kn0 + kn1 * kn1 + kn2 * kn2) <= 3.9f;
  for (int j = 0, last = -1, in = -1; j < a.njob; ++j) {
    const XJob jb = a.job[j];
    if (jb.in != last) { last = jb.in; ++in; }
    auto put = [&](int e, float2 op) {
      const int c = e & (L - 1), n = e >> ls;
      Y[n * sp + j * L + c] = gswap(cscale(cmul(X[n * sp + in * L + c], op), ops.inv_ntot));
    };
    if (poly && (jb.kind == XK_GRAD || jb.kind == XK_DIV)) {
      const auto t = gp(jb.kind == XK_GRAD ? gpick(ops.grad, jb.axis) : gpick(ops.div, jb.axis));
      const auto k0 = gp(ops.k[0]), k1 = gp(ops.k[1]), k2 = gp(g.nd == 3 ? ops.k[2] : ops.k[1]);
      const float w2 = g.nd == 3 ? 1.f : 0.f;
      gbatch(N * L,
             [&](int e) {
               const int n = e >> ls, col = min(col0 + (e & (L - 1)), a.ncols - 1);
               const float kx = k0[n], ky = k1[g.nd == 2 ? col : o], kz = w2 * k2[col];
               const float f = sinc_k2<false>(kap2 * fmaf(kx, kx, fmaf(kz, kz, ky * ky)));
               return cscale(ld2(t, jb.axis == 0 ? n : ((jb.axis == 1 && g.nd == 3) ? o : col)), f);
             },
             put);
    } else {
      for (int e = threadIdx.x; e < N * L; e += (int)blockDim.x) put(e, gjob_op(jb, ops, g, kap, e >> ls, o, min(col0 + (e & (L - 1)), a.ncols - 1)));
    }
  }
  __syncthreads();
  const float2* Z = gfft(Y, X, pl, tw, a.njob * L, sp);
  for (int j = 0; j < a.njob; ++j) store(Z, j * L, fl.spec[a.job[j].out], true);
}

// One column and job at a time, the forward transform of the current input waiting in the
// stash spectrum: lines too long for all jobs' buffers in LDS.
__global__ __launch_bounds__(kGenThreads) void k_gcol_long(Geom g, Fields fl, Ops ops, const Inst* __restrict__ inst, ColArgs a,
                                                           const float2* __restrict__ twg, GPlan pl) {
  if (a.gath && (int)blockIdx.x >= a.gx) return gather_blocks(g, fl, inst, a);
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y;
  if (fl.tdev && step_of(fl, b) >= inst[b].nt) return;
  const int N = pl.n;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  float2* A = gsm + N;
  float2* B = A + N;
  gt.put();
  const int o = blockIdx.x / a.ncols, col = blockIdx.x % a.ncols;
  const int64_t base = (int64_t)b * g.nspec + (int64_t)o * a.ostride + col;
  const float kap = inst[b].kap;
  int cur_in = -1;
  for (int j = 0; j < a.njob; ++j) {
    const XJob jb = a.job[j];
    if (jb.in != cur_in) {
      cur_in = jb.in;
      for (int n = threadIdx.x; n < N; n += blockDim.x) A[n] = ld2(gp(fl.spec[jb.in]), base + (int64_t)n * a.estride);
      __syncthreads();
      const float2* R = gfft(A, B, pl, tw, 1, 1);
      for (int n = threadIdx.x; n < N; n += blockDim.x) st2(gw(fl.gstash), base + (int64_t)n * a.estride, R[n]);
      __syncthreads();
    }
    for (int n = threadIdx.x; n < N; n += blockDim.x)
      A[n] = gswap(cscale(cmul(ld2(gp(fl.gstash), base + (int64_t)n * a.estride), gjob_op(jb, ops, g, kap, n, o, col)), ops.inv_ntot));
    __syncthreads();
    const float2* R = gfft(A, B, pl, tw, 1, 1);
    for (int n = threadIdx.x; n < N; n += blockDim.x) st2(gw(fl.spec[jb.out]), base + (int64_t)n * a.estride, gswap(R[n]));
    __syncthreads();
  }
}

hipError_t launch_col_gen(const Geom& g, int nb, const Fields& fl, const Ops& ops, const Inst* inst, const ColArgs& a, int nline,
                          hipStream_t st) {
  if (a.mode == 2 && !fl.gstash) return hipErrorInvalidValue;
  const GPlan pl = gplan(nline);
  const int lines = a.mode == 2 ? a.njob : 1;  // never fewer than the distinct inputs
  const int L = gen_items(nline, lines, (int64_t)a.nouter * a.ncols * nb);
  if (!L) {
    if (a.mode != 2) return hipErrorInvalidValue;
    const ColArgs al = col_blocks(a, a.nouter * a.ncols);
    hipLaunchKernelGGL(k_gcol_long, dim3(col_gridx(al, kGenThreads), nb), dim3(kGenThreads), glds_bytes(nline, 1), st, g, fl, ops, inst, al,
                       ops.tw[a.axis], pl);
    return hipGetLastError();
  }
  const int ntile = (a.ncols + L - 1) / L, layers = a.mode == 2 ? 1 : a.nbuf;
  const int nt = gen_threads(lines * L, nline, (int64_t)a.nouter * ntile * nb * layers);
  const ColArgs al = col_blocks(a, a.nouter * ntile);
  hipLaunchKernelGGL(k_gcol, dim3(col_gridx(al, nt), nb, layers), dim3(nt), glds_bytes(nline, lines * L), st, g, fl, ops, inst, al,
                     ops.tw[a.axis], pl, L, gpitch(lines * L));
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// pointwise updates (the fused z-pass kernels' arithmetic, one element per thread)
// ---------------------------------------------------------------------------
// pml multiplier of axis ax at (row r, position n); 1 on the contiguous axis
// unless that is ax
__device__ __forceinline__ float gpml(const float* const* tab, const Geom& g, int ax, int r, int n) { return pml_at(tab, g, ax, r, n); }

#define KW_GEN_ELEMENT_LOOP                                                       \
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < g.ntot; \
       idx += (int64_t)gridDim.x * blockDim.x)

// Each update is split into the loads of its operands at an element and the update itself,
// so that a kernel can issue the loads of several elements together.
// pml multiplier of axis ax at (row r, position n), by selected indexes: a branch per axis
// would separate the loads around it
__device__ __forceinline__ float gpml_at(const float* const* tab, const Geom& g, int ax, int r, int n) {
  const int q = r / g.n[1];
  const int row = g.nd == 2 ? r : ax == 0 ? q : r - q * g.n[1];
  return gp(tab[ax])[ax == g.nd - 1 ? n : row];
}

struct GMomOps { float u, dr, s; };
__device__ __forceinline__ GMomOps gmomentum_load(const Geom& g, const Fields& fl, const Inst& I, int ax, int64_t off, int r, int n) {
  const int64_t idx = (int64_t)r * g.nz + n;
  return {gp(fl.u[ax] + off)[idx], ld(I.dtr0[ax], idx, I.dtr0_s), gpml_at(I.pmlsg, g, ax, r, n)};
}
// u_ax at (row r, position n) from the gradient value gv and the filtered source value chv
// (spectral sources); stores and returns it
__device__ __forceinline__ float gmomentum_elem(const Geom& g, const Fields& fl, const Inst& I, int ax, int64_t off, int t, int smode,
                                                float sig_t, int r, int n, const GMomOps& o, float gv, float chv) {
  const Src& src = I.srcu[ax];
  const int64_t idx = (int64_t)r * g.nz + n;
  float uv = pml_update(o.s, o.u, o.dr, gv);
  uv = src_inline(src, smode, uv, idx, src.fac[ax], sig_t, chv);
  if (src_is_point(smode)) {
    float v;
    if (csr_lookup(src, r, n, t, v)) uv = src_point(smode, uv, src.fac[ax], v);
  }
  gw(fl.u[ax] + off)[idx] = uv;
  return uv;
}

struct GMassOps { float r0, rs, c2, ba, rho[3], s[3]; };
__device__ __forceinline__ GMassOps gmass_load(const Geom& g, const Fields& fl, const Inst& I, int flags, int64_t off, int r, int n) {
  const int64_t idx = (int64_t)r * g.nz + n;
  GMassOps o;
  o.r0 = ld(I.rho0, idx, I.rho0_s);
  o.c2 = ld(I.c0sq, idx, I.c0sq_s);
  // (linear plans have neither array: the loads go to one that exists and are not used)
  const bool nl = flags & FLAG_NONLINEAR;
  o.rs = gp(nl ? fl.rhoi : fl.rho[0])[off + idx];
  o.ba = ld(nl ? I.bona : I.rho0, idx, nl ? I.bona_s : I.rho0_s);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int ax = i < g.nd ? i : 0;
    o.rho[i] = gp(fl.rho[ax] + off)[idx];
    o.s[i] = gpml_at(I.pml, g, ax, r, n);
  }
  return o;
}
// Density update at one element from its divergence terms dv; the split densities, their
// sum and, without power law, p are stored.  Returns what is transformed next: rho0 div u
// (power law) or p; rt: the density sum.
__device__ __forceinline__ float gmass_elem(const Geom& g, const Fields& fl, const Inst& I, int flags, int64_t nf, int64_t off, int t,
                                            int smode, float sig_t, int r, int n, const GMassOps& o, const float (&dv)[3], float chv,
                                            float& rt) {
  const int ND = g.nd;
  const Src& src = I.srcp;
  const int64_t idx = (int64_t)r * g.nz + n;
  float qa = o.r0;
  if (flags & FLAG_NONLINEAR) qa = fmaf(2.f, o.rs, qa);
  const float q = I.dt * qa;
  const bool filtered = smode == SRC_CHAIN || smode == SRC_PATTERN;
  const float ch = smode == SRC_PATTERN ? sig_t * gp(src.pattern)[idx] : chv;
  float rv[3], du = 0.f;
  rt = 0.f;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i >= ND) continue;
    if (fl.adjD) gw(fl.adjD)[(int64_t)i * nf + off + idx] = dv[i];  // adjoint replay: Dop_i u_i
    rv[i] = pml_update(o.s[i], o.rho[i], q, dv[i]);
    if (filtered) rv[i] = fmaf(src.fac[i], ch, rv[i]);
    rounded(rv[i]);
  }
  if (src_is_point(smode)) {
    float v;
    if (csr_lookup(src, r, n, t, v)) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (i < ND) rv[i] = src_point(smode, rv[i], src.fac[i], v);
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i >= ND) continue;
    gw(fl.rho[i] + off)[idx] = rv[i];
    du += dv[i];
    rt += rv[i];
  }
  if (fl.rhot) gw(fl.rhot)[off + idx] = rt;
  if (flags & (FLAG_POWERLAW_ABS | FLAG_POWERLAW_DISP)) return o.r0 * du;
  float qq = rt;
  if (flags & FLAG_STOKES) {
    qq = fmaf(tau_at(I, idx, o.c2) * o.r0, du, qq);
    if (fl.adjA) gw(fl.adjA)[off + idx] = o.r0 * du;  // adjoint replay: the Stokes operand
  }
  if (flags & FLAG_NONLINEAR) qq += o.ba * rt * rt / (2.f * o.r0);
  const float pv = o.c2 * qq;
  gw(fl.p)[off + idx] = pv;
  return pv;
}

struct GEosOps { float rt, c2, r0, ba; };
__device__ __forceinline__ GEosOps geos_load(const Fields& fl, const Inst& I, int flags, int64_t off, int64_t idx) {
  const bool nl = flags & FLAG_NONLINEAR;
  return {gp(fl.rhot)[off + idx], ld(I.c0sq, idx, I.c0sq_s), ld(I.rho0, idx, I.rho0_s),
          ld(nl ? I.bona : I.rho0, idx, nl ? I.bona_s : I.rho0_s)};
}
// equation of state at one element from the power-law operands av, bv; stores and returns p
__device__ __forceinline__ float geos_elem(const Fields& fl, const Inst& I, int flags, int64_t off, int64_t idx, const GEosOps& o, float av,
                                           float bv) {
  float q = o.rt;
  if (flags & FLAG_POWERLAW_ABS) q = fmaf(tau_at(I, idx, o.c2), av, q);
  if (flags & FLAG_POWERLAW_DISP) q = fmaf(-eta_at(I, idx, o.c2), bv, q);
  // adjoint replay: keep the absorption and dispersion operands
  if (fl.adjA && (flags & FLAG_POWERLAW_ABS)) gw(fl.adjA)[off + idx] = av;
  if (fl.adjB && (flags & FLAG_POWERLAW_DISP)) gw(fl.adjB)[off + idx] = bv;
  if (flags & FLAG_NONLINEAR) q += o.ba * o.rt * o.rt / (2.f * o.r0);
  const float pv = o.c2 * q;
  gw(fl.p)[off + idx] = pv;
  return pv;
}

// ---------------------------------------------------------------------------
// fused updates: inverse transforms, update, forward transforms on P row pairs in LDS
// ---------------------------------------------------------------------------
// momentum of axis blockIdx.z; the inverse transform of an active spectral source of that
// axis rides along as further lines
__global__ __launch_bounds__(kGenThreads) void k_gzmom(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ twg,
                                                       GPlan pl, int P, int sp) {
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y, ax = blockIdx.z;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  const int N = pl.n;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  float2* A = gsm + N;
  float2* B = A + N * sp;
  const int pair0 = blockIdx.x * P;
  const Src& src = I.srcu[ax];
  const int64_t off = (int64_t)b * g.ntot;
  float2* const spec = fl.spec[ax] + b * g.nspec;
  gpairs_in(A, sp, 0, spec, g, N, pair0, P);
  const int smode = src_mode_at(src, t);
  const bool chain = smode == SRC_CHAIN;
  const float sig_t = smode == SRC_PATTERN ? gp(src.sig)[t] : 0.f;
  if (chain) gpairs_in(A, sp, P, fl.spec[src.chain_buf] + b * g.nspec, g, N, pair0, P);
  gt.put();
  if (t >= I.nt) return;
  __syncthreads();
  float2* Z = gfft(A, B, pl, tw, chain ? 2 * P : P, sp);
  gupdate(g, N, pair0, P, [&](int r, int n) { return gmomentum_load(g, fl, I, ax, off, r, n); },
          [&](int lp, int n, int ra, bool two, const GMomOps& oa, const GMomOps& ob) {
            const float2 z = Z[n * sp + lp], ch = chain ? Z[n * sp + P + lp] : make_float2(0.f, 0.f);
            const float ua = gmomentum_elem(g, fl, I, ax, off, t, smode, sig_t, ra, n, oa, z.y, ch.y);
            const float ub = two ? gmomentum_elem(g, fl, I, ax, off, t, smode, sig_t, ra + 1, n, ob, z.x, ch.x) : 0.f;
            Z[n * sp + lp] = make_float2(ua, ub);
          });
  __syncthreads();
  const float2* F = gfft(Z, Z == A ? B : A, pl, tw, P, sp);
  gpairs_out(F, sp, 0, spec, g, N, pair0, P);
}

// mass conservation: the axes' divergence terms (and an active spectral source) are
// transformed together, axis i as lines i P ..
__global__ __launch_bounds__(kGenThreads) void k_gzmass(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ twg,
                                                        int flags, GPlan pl, int P, int sp) {
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  const int N = pl.n, ND = g.nd;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  float2* A = gsm + N;
  float2* B = A + N * sp;
  const int pair0 = blockIdx.x * P;
  const Src& src = I.srcp;
  const int64_t off = (int64_t)b * g.ntot, nf = (int64_t)gridDim.y * g.ntot;
  for (int i = 0; i < ND; ++i) gpairs_in(A, sp, i * P, fl.spec[i] + b * g.nspec, g, N, pair0, P);
  const int smode = src_mode_at(src, t);
  const bool chain = smode == SRC_CHAIN;
  const float sig_t = smode == SRC_PATTERN ? gp(src.sig)[t] : 0.f;
  if (chain) gpairs_in(A, sp, ND * P, fl.spec[src.chain_buf] + b * g.nspec, g, N, pair0, P);
  gt.put();
  if (t >= I.nt) return;
  __syncthreads();
  float2* Z = gfft(A, B, pl, tw, (chain ? ND + 1 : ND) * P, sp);
  const bool powerlaw = flags & (FLAG_POWERLAW_ABS | FLAG_POWERLAW_DISP);
  const bool f0 = !powerlaw || (flags & FLAG_POWERLAW_ABS), f1 = flags & FLAG_POWERLAW_DISP;
  gupdate(g, N, pair0, P, [&](int r, int n) { return gmass_load(g, fl, I, flags, off, r, n); },
          [&](int lp, int n, int ra, bool two, const GMassOps& oa, const GMassOps& ob) {
            float da[3], db[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const float2 z = i < ND ? Z[n * sp + i * P + lp] : make_float2(0.f, 0.f);
              da[i] = z.y;
              db[i] = z.x;
            }
            const float2 ch = chain ? Z[n * sp + ND * P + lp] : make_float2(0.f, 0.f);
            float2 out = make_float2(0.f, 0.f), rt = out;
            out.x = gmass_elem(g, fl, I, flags, nf, off, t, smode, sig_t, ra, n, oa, da, ch.y, rt.x);
            if (two) out.y = gmass_elem(g, fl, I, flags, nf, off, t, smode, sig_t, ra + 1, n, ob, db, ch.x, rt.y);
            if (f0) Z[n * sp + lp] = out;  // this element's own slots: axis 0's line, and axis 1's
            if (f1) Z[n * sp + (f0 ? P : 0) + lp] = rt;
          });
  __syncthreads();
  const float2* F = gfft(Z, Z == A ? B : A, pl, tw, f0 && f1 ? 2 * P : P, sp);
  if (f0) gpairs_out(F, sp, 0, fl.spec[0] + b * g.nspec, g, N, pair0, P);
  if (f1) gpairs_out(F, sp, f0 ? P : 0, fl.spec[1] + b * g.nspec, g, N, pair0, P);
}

// equation of state with power-law terms
__global__ __launch_bounds__(kGenThreads) void k_gzeos(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ twg,
                                                       int flags, GPlan pl, int P, int sp) {
  extern __shared__ float2 gsm[];
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  const int N = pl.n;
  const GTw gt(gsm, twg, N);
  const float2* const tw = gsm;
  float2* A = gsm + N;
  float2* B = A + N * sp;
  const int pair0 = blockIdx.x * P;
  const int64_t off = (int64_t)b * g.ntot;
  const bool fa = flags & FLAG_POWERLAW_ABS, fd = flags & FLAG_POWERLAW_DISP;
  const int cd = fa ? P : 0;  // first line of the dispersion operand
  if (fa) gpairs_in(A, sp, 0, fl.spec[0] + b * g.nspec, g, N, pair0, P);
  if (fd) gpairs_in(A, sp, cd, fl.spec[1] + b * g.nspec, g, N, pair0, P);
  gt.put();
  if (t >= I.nt) return;
  __syncthreads();
  float2* Z = gfft(A, B, pl, tw, fa && fd ? 2 * P : P, sp);
  gupdate(g, N, pair0, P, [&](int r, int n) { return geos_load(fl, I, flags, off, (int64_t)r * N + n); },
          [&](int lp, int n, int ra, bool two, const GEosOps& oa, const GEosOps& ob) {
            const float2 av = fa ? Z[n * sp + lp] : make_float2(0.f, 0.f), bv = fd ? Z[n * sp + cd + lp] : make_float2(0.f, 0.f);
            float2 out = make_float2(0.f, 0.f);
            out.x = geos_elem(fl, I, flags, off, (int64_t)ra * N + n, oa, av.y, bv.y);
            if (two) out.y = geos_elem(fl, I, flags, off, (int64_t)(ra + 1) * N + n, ob, av.x, bv.x);
            Z[n * sp + lp] = out;
          });
  __syncthreads();
  const float2* F = gfft(Z, Z == A ? B : A, pl, tw, P, sp);
  gpairs_out(F, sp, 0, fl.spec[0] + b * g.nspec, g, N, pair0, P);
}

// ---------------------------------------------------------------------------
// unfused updates (lines too long for the fused ones)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kGenThreads) void k_gmomentum(Geom g, Fields fl, const Inst* __restrict__ inst, int ax,
                                                           const float* __restrict__ gtmp, const float* __restrict__ ctmp) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  if (t >= I.nt) return;
  const Src& src = I.srcu[ax];
  const int smode = src_mode_at(src, t);
  const float sig_t = smode == SRC_PATTERN ? gp(src.sig)[t] : 0.f;
  const int64_t off = (int64_t)b * g.ntot;
  KW_GEN_ELEMENT_LOOP {
    const int r = (int)(idx / g.nz), n = (int)(idx % g.nz);
    gmomentum_elem(g, fl, I, ax, off, t, smode, sig_t, r, n, gmomentum_load(g, fl, I, ax, off, r, n), gp(gtmp)[off + idx], smode == SRC_CHAIN ? gp(ctmp)[off + idx] : 0.f);
  }
}

// mass conservation; with power law the outputs for the fractional Laplacians
// are rho0 div u (into aout) and the density sum (rhot), otherwise p.
__global__ __launch_bounds__(kGenThreads) void k_gmass(Geom g, Fields fl, const Inst* __restrict__ inst, int flags,
                                                       const float* d0, const float* d1, const float* d2,
                                                       const float* __restrict__ ctmp, float* aout) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  if (t >= I.nt) return;
  const Src& src = I.srcp;
  const int smode = src_mode_at(src, t);
  const float sig_t = smode == SRC_PATTERN ? gp(src.sig)[t] : 0.f;
  const int64_t off = (int64_t)b * g.ntot;
  KW_GEN_ELEMENT_LOOP {
    const int r = (int)(idx / g.nz), n = (int)(idx % g.nz);
    const float dv[3] = {gp(d0)[off + idx], gp(d1)[off + idx], g.nd > 2 ? gp(d2)[off + idx] : 0.f};
    float rt;
    const float a = gmass_elem(g, fl, I, flags, (int64_t)gridDim.y * g.ntot, off, t, smode, sig_t, r, n,
                               gmass_load(g, fl, I, flags, off, r, n), dv,
                               smode == SRC_CHAIN ? gp(ctmp)[off + idx] : 0.f, rt);
    if (flags & (FLAG_POWERLAW_ABS | FLAG_POWERLAW_DISP)) gw(aout)[off + idx] = a;
  }
}

__global__ __launch_bounds__(kGenThreads) void k_geos(Geom g, Fields fl, const Inst* __restrict__ inst, int flags,
                                                      const float* __restrict__ av, const float* __restrict__ bv) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  if (t >= I.nt) return;
  const int64_t off = (int64_t)b * g.ntot;
  KW_GEN_ELEMENT_LOOP {
    geos_elem(fl, I, flags, off, idx, geos_load(fl, I, flags, off, idx), (flags & FLAG_POWERLAW_ABS) ? gp(av)[off + idx] : 0.f,
              (flags & FLAG_POWERLAW_DISP) ? gp(bv)[off + idx] : 0.f);
  }
}

// t = 0 initial-value override: u_i = dt/(2 rho0_sg_i) grad_i p0, rho_j = p0 / (c0^2 D)
__global__ __launch_bounds__(kGenThreads) void k_ginit_u(Geom g, Fields fl, const Inst* __restrict__ inst, const float* __restrict__ g0,
                                                         const float* __restrict__ g1, const float* __restrict__ g2) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int64_t off = (int64_t)b * g.ntot;
  const float* gg[3] = {g0, g1, g2};
  KW_GEN_ELEMENT_LOOP {
    for (int ax = 0; ax < g.nd; ++ax) gw(fl.u[ax])[off + idx] = 0.5f * ld(I.dtr0[ax], idx, I.dtr0_s) * gp(gg[ax])[off + idx];
    const float pv = gw(fl.p)[off + idx], c2 = ld(I.c0sq, idx, I.c0sq_s);
    float rs = 0.f;
    for (int j = 0; j < g.nd; ++j) {
      const float rv = pv / (c2 * I.p0div[j]);
      gw(fl.rho[j])[off + idx] = rv;
      rs += rv;
    }
    if (fl.rhot) gw(fl.rhot)[off + idx] = rs;
  }
}

// dense field of a spectral (CHAIN) source at step t: scale * sig at the source
// points, 0 elsewhere (instances without an active CHAIN source are skipped)
__global__ __launch_bounds__(kGenThreads) void k_gsrc_scatter(Geom g, Fields fl, const Inst* __restrict__ inst, int which,
                                                              float* __restrict__ out) {
  const int b = blockIdx.y;
  if (gen_skip(fl.tdev, fl.toff, inst, b, which)) return;
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  const Src& s = which < 0 ? I.srcp : I.srcu[which];
  const int64_t off = (int64_t)b * g.ntot;
  KW_GEN_ELEMENT_LOOP {
    const int r = (int)(idx / g.nz), n = (int)(idx % g.nz);
    float v = 0.f;
    if (gp(s.row_ptr)[r] != gp(s.row_ptr)[r + 1]) {
      float x;
      if (csr_lookup(s, r, n, t, x)) v = x;
    }
    gw(out)[off + idx] = v;
  }
}

// ---------------------------------------------------------------------------
// reverse sweep: the arithmetic of kw_adjoint.hpp's kernels, one element per
// thread; their transforms run as the launchers below (every instance, no step
// filter: the reverse sweep runs all of them)
// ---------------------------------------------------------------------------
// power law: cbar += 2 p pbar / c + w ((y-1) tau A - y eta B) / c; tau w, eta w out
__global__ __launch_bounds__(kGenThreads) void k_gadj_abs1(Geom g, AdjFields af, const Inst* __restrict__ inst,
                                                           float* __restrict__ tout, float* __restrict__ eout) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int64_t off = (int64_t)b * g.ntot;
  KW_GEN_ELEMENT_LOOP {
    const float c2 = ld(I.c0sq, idx, I.c0sq_s), c = sqrtf(c2);
    const float pbar = gp(af.pb)[off + idx];
    const float w = c2 * pbar;
    const float tau = tau_at(I, idx, c2);
    const float eta = af.disp ? eta_at(I, idx, c2) : 0.f;
    float gc = 2.f * gp(af.pt)[off + idx] * pbar / c + w * af.ym1 * tau / c * gp(af.At)[off + idx];
    if (af.disp) gc -= w * af.y * eta / c * gp(af.Bt)[off + idx];
    gw(af.cb)[off + idx] += gc;
    gw(tout)[off + idx] = tau * w;
    if (af.disp) gw(eout)[off + idx] = eta * w;
  }
}

// equation of state, sources and mass update (k_adj_eos); l1, l2: L1[tau w], L2[eta w]
// on the grid (power law), w_i out for the gradient jobs
__global__ __launch_bounds__(kGenThreads) void k_gadj_eos(Geom g, AdjFields af, const Inst* __restrict__ inst, int t,
                                                          const float* __restrict__ l1, const float* __restrict__ l2, float* w0,
                                                          float* w1, float* w2) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int ND = g.nd;
  const int64_t off = (int64_t)b * g.ntot;
  const int64_t nf = (int64_t)gridDim.y * g.ntot;
  const Src& src = I.srcp;
  const bool srcon = src.mode != SRC_NONE && t < src.len;
  const bool dir = srcon && src.mode == SRC_DIRICHLET;
  float* const wo[3] = {w0, w1, w2};
  KW_GEN_ELEMENT_LOOP {
    const int r = (int)(idx / g.nz), n = (int)(idx % g.nz);
    const float c2 = ld(I.c0sq, idx, I.c0sq_s);
    const float pbar = gp(af.pb)[off + idx];
    const float wc = c2 * pbar;
    const float r0 = ld(I.rho0, idx, I.rho0_s);
    float gc = 0.f;
    if (af.absorb != 2) {  // the power law's speed terms are k_gadj_abs1's
      gc = 2.f * gp(af.pt)[off + idx] * pbar / sqrtf(c2);
      if (af.absorb == 1) gc += wc * tau_at(I, idx, c2) / sqrtf(c2) * gp(af.At)[off + idx];
    }
    float rs = 0.f, sb = 0.f, rn[3] = {0.f, 0.f, 0.f};
    for (int i = 0; i < ND; ++i) {
      const float s = gpml(I.pml, g, i, r, n);
      float rbt = gp(af.rb[i])[off + idx] + wc;
      float nl = 1.f;
      if (af.nonlin) {
        rbt += wc * ld(I.bona, idx, I.bona_s) * gp(af.St)[off + idx] / r0;
        nl = 1.f + 2.f * gp(af.Sp)[off + idx] / r0;
      }
      float dbar = 0.f;
      if (af.absorb == 1) dbar = tau_at(I, idx, c2) * wc;
      if (af.absorb == 2) {
        if (af.disp) rbt -= gp(l2)[off + idx];
        dbar = gp(l1)[off + idx];
      }
      if (dir) {
        float v;
        if (csr_lookup(src, r, n, t, v)) {
          gc += -2.f * src.fac[i] * v * rbt / sqrtf(c2);
          rbt = 0.f;
        }
      }
      rs += src.fac[i] * rbt;
      if (af.nonlin) sb += -2.f * I.dt * s * gp(af.Dt)[(int64_t)i * nf + off + idx] * rbt;
      gw(wo[i])[off + idx] = s * I.dt * r0 * nl * rbt - r0 * dbar;
      rn[i] = s * s * rbt;
    }
    for (int i = 0; i < ND; ++i) gw(af.rb[i])[off + idx] = rn[i] + sb;
    gw(af.cb)[off + idx] += gc;
    if (srcon) gw(af.R)[off + idx] = rs;
  }
}

// momentum (k_adj_mom) of axis ax: gin = Gop_ax w_ax on the grid, v out
__global__ __launch_bounds__(kGenThreads) void k_gadj_mom(Geom g, AdjFields af, const Inst* __restrict__ inst, int t, int ax,
                                                          const float* __restrict__ gin, float* __restrict__ vout) {
  const int b = blockIdx.y;
  const Inst& I = inst[b];
  const int64_t off = (int64_t)b * g.ntot;
  const Src& us = I.srcu[ax];
  const bool uon = us.mode != SRC_NONE && t < us.len;
  const bool udir = uon && us.mode == SRC_DIRICHLET;
  float* const Ub = uon && !udir && af.U[ax] ? af.U[ax] + off : nullptr;
  KW_GEN_ELEMENT_LOOP {
    const int r = (int)(idx / g.nz), n = (int)(idx % g.nz);
    const float s = gpml(I.pmlsg, g, ax, r, n);
    float u = gp(af.ub[ax])[off + idx] + gp(gin)[off + idx];
    if (udir) {
      float v;
      if (csr_lookup(us, r, n, t, v)) u = 0.f;
    }
    if (Ub) gw(Ub)[idx] = u;
    gw(vout)[off + idx] = s * ld(I.dtr0[ax], idx, I.dtr0_s) * u;
    gw(af.ub[ax])[off + idx] = s * s * u;
  }
}

// pbar = sum_i Dop_i v_i (k_adj_sum), the terms on the grid
__global__ __launch_bounds__(kGenThreads) void k_gadj_sum(Geom g, AdjFields af, const float* __restrict__ d0,
                                                          const float* __restrict__ d1, const float* __restrict__ d2) {
  const int b = blockIdx.y;
  const int64_t off = (int64_t)b * g.ntot;
  KW_GEN_ELEMENT_LOOP {
    float a = gp(d0)[off + idx];
    if (g.nd > 1) a += gp(d1)[off + idx];
    if (g.nd > 2) a += gp(d2)[off + idx];
    gw(af.pb)[off + idx] = a;
  }
}

static dim3 gen_elem_grid(const Geom& g, int nb) {
  const int64_t blocks = std::min<int64_t>((g.ntot + kGenThreads - 1) / kGenThreads, 4096);
  return dim3((unsigned)blocks, nb);
}

#define KW_GEN_CHECK(x)                    \
  do {                                     \
    const hipError_t e_ = (x);             \
    if (e_ != hipSuccess) return e_;       \
  } while (0)

// ---------------------------------------------------------------------------
// launchers (same contracts as the fused family in kw_launch.hpp)
// ---------------------------------------------------------------------------
hipError_t launch_zfwd_gen(const Geom& g, int nb, const float* f, int64_t fs, float2* spec, int64_t ss, const float2* tw, hipStream_t st) {
  return gzfwd(g, nb, f, fs, spec, ss, tw, nullptr, 0, nullptr, GF_ALL, st);
}

hipError_t launch_zinv_gen(const Geom& g, int nb, const float2* spec, int64_t ss, float* f, int64_t fs, const float2* tw, float scale,
                           hipStream_t st) {
  return gzinv(g, nb, spec, ss, f, fs, tw, scale, nullptr, 0, nullptr, GF_ALL, st);
}

// Launch shape of a fused update with `lines` lines per row pair; P = 0: does not fit.
struct GFused {
  GPlan pl;
  int P, sp, nt;
  unsigned blocks;
  size_t lds;
};
static GFused gfused(const Geom& g, int layers, int lines) {
  GFused f{};
  const int npairs = (g.rows + 1) / 2;
  f.P = gen_items(g.nz, lines, (int64_t)npairs * layers);
  if (!f.P) return f;
  f.pl = gplan(g.nz);
  f.sp = gpitch(lines * f.P);
  f.blocks = (unsigned)((npairs + f.P - 1) / f.P);
  f.nt = gen_threads(lines * f.P, g.nz, (int64_t)f.blocks * layers);
  f.lds = glds_bytes(g.nz, lines * f.P);
  return f;
}

hipError_t launch_momentum_gen(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[3]) return hipErrorInvalidValue;
  bool chain = false;  // some axis may have a spectral source
  for (int ax = 0; ax < g.nd; ++ax) chain = chain || fl.spec[g.nd + 1 + ax];
  if (const GFused f = gfused(g, nb * g.nd, chain ? 2 : 1); f.P) {
    hipLaunchKernelGGL(k_gzmom, dim3(f.blocks, nb, g.nd), dim3(f.nt), f.lds, st, g, fl, inst, tw, f.pl, f.P, f.sp);
    return hipGetLastError();
  }
  for (int ax = 0; ax < g.nd; ++ax) {
    KW_GEN_CHECK(gzinv(g, nb, fl.spec[ax], g.nspec, fl.tmp[0], g.ntot, tw, 1.f, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
    if (fl.spec[g.nd + 1 + ax])
      KW_GEN_CHECK(gzinv(g, nb, fl.spec[g.nd + 1 + ax], g.nspec, fl.tmp[3], g.ntot, tw, 1.f, fl.tdev, fl.toff, inst, ax, st));
    hipLaunchKernelGGL(k_gmomentum, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, fl, inst, ax, fl.tmp[0], fl.tmp[3]);
    KW_GEN_CHECK(hipGetLastError());
    KW_GEN_CHECK(gzfwd(g, nb, fl.u[ax], g.ntot, fl.spec[ax], g.nspec, tw, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
  }
  return hipSuccess;
}

hipError_t launch_mass_gen(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, int flags, hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[3]) return hipErrorInvalidValue;
  if (const GFused f = gfused(g, nb, fl.spec[g.nd] ? g.nd + 1 : g.nd); f.P) {
    hipLaunchKernelGGL(k_gzmass, dim3(f.blocks, nb), dim3(f.nt), f.lds, st, g, fl, inst, tw, flags, f.pl, f.P, f.sp);
    return hipGetLastError();
  }
  for (int i = 0; i < g.nd; ++i) KW_GEN_CHECK(gzinv(g, nb, fl.spec[i], g.nspec, fl.tmp[i], g.ntot, tw, 1.f, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
  if (fl.spec[g.nd]) KW_GEN_CHECK(gzinv(g, nb, fl.spec[g.nd], g.nspec, fl.tmp[3], g.ntot, tw, 1.f, fl.tdev, fl.toff, inst, -1, st));
  hipLaunchKernelGGL(k_gmass, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, fl, inst, flags, fl.tmp[0], fl.tmp[1], fl.tmp[2],
                     fl.tmp[3], fl.tmp[0]);
  KW_GEN_CHECK(hipGetLastError());
  if (flags & (FLAG_POWERLAW_ABS | FLAG_POWERLAW_DISP)) {
    if (flags & FLAG_POWERLAW_ABS) KW_GEN_CHECK(gzfwd(g, nb, fl.tmp[0], g.ntot, fl.spec[0], g.nspec, tw, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
    if (flags & FLAG_POWERLAW_DISP) KW_GEN_CHECK(gzfwd(g, nb, fl.rhot, g.ntot, fl.spec[1], g.nspec, tw, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
    return hipSuccess;
  }
  return gzfwd(g, nb, fl.p, g.ntot, fl.spec[0], g.nspec, tw, fl.tdev, fl.toff, inst, GF_ACTIVE, st);
}

hipError_t launch_eos_gen(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, int flags, hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[1]) return hipErrorInvalidValue;
  if (const GFused f = gfused(g, nb, 2); f.P) {
    hipLaunchKernelGGL(k_gzeos, dim3(f.blocks, nb), dim3(f.nt), f.lds, st, g, fl, inst, tw, flags, f.pl, f.P, f.sp);
    return hipGetLastError();
  }
  if (flags & FLAG_POWERLAW_ABS) KW_GEN_CHECK(gzinv(g, nb, fl.spec[0], g.nspec, fl.tmp[0], g.ntot, tw, 1.f, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
  if (flags & FLAG_POWERLAW_DISP) KW_GEN_CHECK(gzinv(g, nb, fl.spec[1], g.nspec, fl.tmp[1], g.ntot, tw, 1.f, fl.tdev, fl.toff, inst, GF_ACTIVE, st));
  hipLaunchKernelGGL(k_geos, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, fl, inst, flags, fl.tmp[0], fl.tmp[1]);
  KW_GEN_CHECK(hipGetLastError());
  return gzfwd(g, nb, fl.p, g.ntot, fl.spec[0], g.nspec, tw, fl.tdev, fl.toff, inst, GF_ACTIVE, st);
}

hipError_t launch_init_u_gen(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[2]) return hipErrorInvalidValue;
  for (int ax = 0; ax < g.nd; ++ax) KW_GEN_CHECK(gzinv(g, nb, fl.spec[ax], g.nspec, fl.tmp[ax], g.ntot, tw, 1.f, nullptr, 0, inst, GF_ALL, st));
  hipLaunchKernelGGL(k_ginit_u, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, fl, inst, fl.tmp[0], fl.tmp[1], fl.tmp[2]);
  return hipGetLastError();
}

hipError_t launch_src_build_gen(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, int which, hipStream_t st) {
  if (!fl.tmp[3]) return hipErrorInvalidValue;
  const int buf = which < 0 ? g.nd : g.nd + 1 + which;
  hipLaunchKernelGGL(k_gsrc_scatter, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, fl, inst, which, fl.tmp[3]);
  KW_GEN_CHECK(hipGetLastError());
  return gzfwd(g, nb, fl.tmp[3], g.ntot, fl.spec[buf], g.nspec, tw, fl.tdev, fl.toff, inst, which, st);
}

hipError_t launch_adj_abs1_gen(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw,
                               hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[1]) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gadj_abs1, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, af, inst, fl.tmp[0], fl.tmp[1]);
  KW_GEN_CHECK(hipGetLastError());
  KW_GEN_CHECK(gzfwd(g, nb, fl.tmp[0], g.ntot, fl.spec[0], g.nspec, tw, nullptr, 0, nullptr, GF_ALL, st));
  if (af.disp) KW_GEN_CHECK(gzfwd(g, nb, fl.tmp[1], g.ntot, fl.spec[1], g.nspec, tw, nullptr, 0, nullptr, GF_ALL, st));
  return hipSuccess;
}

hipError_t launch_adj_eos_gen(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw, int t,
                              hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[2]) return hipErrorInvalidValue;
  if (af.absorb == 2) {  // L1[tau w], L2[eta w] from spectra 0 and 1 (the fractional column passes' outputs)
    if (!af.gl[0] || !af.gl[1]) return hipErrorInvalidValue;
    KW_GEN_CHECK(gzinv(g, nb, fl.spec[0], g.nspec, af.gl[0], g.ntot, tw, 1.f, nullptr, 0, inst, GF_ALL, st));
    if (af.disp) KW_GEN_CHECK(gzinv(g, nb, fl.spec[1], g.nspec, af.gl[1], g.ntot, tw, 1.f, nullptr, 0, inst, GF_ALL, st));
  }
  hipLaunchKernelGGL(k_gadj_eos, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, af, inst, t, af.gl[0], af.gl[1], fl.tmp[0],
                     fl.tmp[1], fl.tmp[2]);
  KW_GEN_CHECK(hipGetLastError());
  for (int i = 0; i < g.nd; ++i)
    KW_GEN_CHECK(gzfwd(g, nb, fl.tmp[i], g.ntot, fl.spec[i], g.nspec, tw, nullptr, 0, nullptr, GF_ALL, st));
  return hipSuccess;
}

hipError_t launch_adj_mom_gen(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw, int t,
                              hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[1]) return hipErrorInvalidValue;
  for (int ax = 0; ax < g.nd; ++ax) {
    KW_GEN_CHECK(gzinv(g, nb, fl.spec[ax], g.nspec, fl.tmp[0], g.ntot, tw, 1.f, nullptr, 0, inst, GF_ALL, st));
    hipLaunchKernelGGL(k_gadj_mom, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, af, inst, t, ax, fl.tmp[0], fl.tmp[1]);
    KW_GEN_CHECK(hipGetLastError());
    KW_GEN_CHECK(gzfwd(g, nb, fl.tmp[1], g.ntot, fl.spec[ax], g.nspec, tw, nullptr, 0, nullptr, GF_ALL, st));
  }
  return hipSuccess;
}

hipError_t launch_adj_sum_gen(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw,
                              hipStream_t st) {
  if (!fl.tmp[0] || !fl.tmp[2]) return hipErrorInvalidValue;
  for (int i = 0; i < g.nd; ++i)
    KW_GEN_CHECK(gzinv(g, nb, fl.spec[i], g.nspec, fl.tmp[i], g.ntot, tw, 1.f, nullptr, 0, inst, GF_ALL, st));
  hipLaunchKernelGGL(k_gadj_sum, gen_elem_grid(g, nb), dim3(kGenThreads), 0, st, g, af, fl.tmp[0], fl.tmp[1], fl.tmp[2]);
  return hipGetLastError();
}

}  // namespace kw
