// The step before the solve: cell classification and level-set redistancing
// on the device, canonical C-order layout.
//
//   apply_markers   FluidSimulator.apply_markers (fluid_simulator.py:151-159)
//   init_boundary   FluidSimulator.init_boundary (fluid_simulator.py:337-341)
//   redistance      FastSweepingLevelSet.redistance (level_set.py:260-333):
//                   target_surface (level_set.py:66-86), then repeat_times x
//                   six directional sweeps of the Eikonal update
//                   update_from_neighbor (level_set.py:88-112).
//
// Sweeps: a grid line along the sweep axis is walked in the sweep direction,
// so the cells behind it on the line are already updated and the ones ahead
// are not, as in the reference's serial inner loop.  The reference runs the
// lines in parallel and reads the neighbouring lines while they change (the
// result depends on thread timing); here the neighbouring lines are read as
// they were before the sweep (a sweep reads one array and writes another),
// which makes the result deterministic.  Each axis is swept over its own
// extent (the reference bounds the axis-0 sweeps by res[1],
// level_set.py:297-303/323-327, which only differs on non-square grids).
#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>
#include <utility>

#include "../../include/mgpcg.h"
#include "mgpcg_common.h"

namespace {

constexpr int LB = 256;

struct Grid {
  int dim;
  int n[3];
  long st[3];          // C-order strides
  mg::FastDiv dn[3];   // division by n[a] (coords below 2^31)
  __host__ __device__ long cells() const { return (long)n[0] * n[1] * n[2]; }
};

Grid make_grid(int dim, const int32_t* res) {
  Grid g;
  g.dim = dim;
  for (int a = 0; a < 3; ++a) g.n[a] = a < dim ? res[a] : 1;
  g.st[dim - 1] = 1;
  for (int a = dim - 2; a >= 0; --a) g.st[a] = g.st[a + 1] * g.n[a + 1];
  for (int a = dim; a < 3; ++a) g.st[a] = 0;
  for (int a = 0; a < 3; ++a) g.dn[a] = mg::FastDiv((uint32_t)g.n[a]);
  return g;
}

__device__ __forceinline__ void coords(const Grid& g, long t, int* I) {
  if (t < 0x80000000L) {  // multiply-high division, no 64-bit divide
    uint32_t u = (uint32_t)t;
    for (int a = g.dim - 1; a >= 0; --a) {
      const uint32_t q = g.dn[a].div(u);
      I[a] = (int)(u - q * (uint32_t)g.n[a]);
      u = q;
    }
    for (int a = g.dim; a < 3; ++a) I[a] = 0;
    return;
  }
  for (int a = g.dim - 1; a >= 0; --a) {
    I[a] = (int)(t % g.n[a]);
    t /= g.n[a];
  }
  for (int a = g.dim; a < 3; ++a) I[a] = 0;
}

// taichi_glsl's sign: -1, 0 or 1
__device__ __forceinline__ float sgnf(float x) { return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f); }

__global__ void k_apply_markers(Grid g, const float* __restrict__ phi, int8_t* __restrict__ ct) {
  const long t = (long)blockIdx.x * LB + threadIdx.x;
  if (t >= g.cells()) return;
  if (ct[t] != MG_SOLID) ct[t] = phi[t] <= 0.0f ? (int8_t)MG_FLUID : (int8_t)MG_AIR;
}

__global__ void k_init_boundary(Grid g, int8_t* __restrict__ ct) {
  const long t = (long)blockIdx.x * LB + threadIdx.x;
  if (t >= g.cells()) return;
  int I[3];
  coords(g, t, I);
  for (int a = 0; a < g.dim; ++a)
    if (I[a] == 0 || I[a] + 1 == g.n[a]) ct[t] = MG_SOLID;
}

// What a sweep needs of a cell besides its distance, in one byte (the
// caller's `fixed` work array): bit 0 = fixed by target_surface, bits 1-2 =
// sign(phi) + 1.
__device__ __forceinline__ float code_sign(int code) { return (float)((code >> 1) - 1); }

// target_surface (level_set.py:66-86): cells with a sign change to a face
// neighbour take the signed distance estimate sign(phi) * theta * dx of the
// closest crossing and are fixed; the others start at 1e20.  Every neighbour
// is loaded before any is used (a missing one reads the cell itself, which
// has no sign change to it).  256^3: 141 us with a wait per neighbour -> 73 us,
// where the 9 B a cell reads and writes would take 32.
template <int DIM>
__global__ void __launch_bounds__(LB) k_target_surface(Grid g, const float* __restrict__ phi,
                                                       float dx, float* __restrict__ tmp,
                                                       int8_t* __restrict__ code) {
  const long t = (long)blockIdx.x * LB + threadIdx.x;
  if (t >= g.cells()) return;
  int I[3];
  coords(g, t, I);
  const float pi = phi[t];
  float pj[DIM][2];
#pragma unroll
  for (int k = 0; k < DIM; ++k) {
    pj[k][0] = phi[I[k] > 0 ? t - g.st[k] : t];
    pj[k][1] = phi[I[k] + 1 < g.n[k] ? t + g.st[k] : t];
  }
  const float si = sgnf(pi);
  bool change = false;
  float est = 1e20f;
#pragma unroll
  for (int k = 0; k < DIM; ++k)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (si != sgnf(pj[k][h])) {
        const float th = pi / (pi - pj[k][h]);
        const float est0 = si * th * dx;
        est = fabsf(est0) < fabsf(est) ? est0 : est;
        change = true;
      }
  tmp[t] = est;
  code[t] = (int8_t)((change ? 1 : 0) | (((int)si + 1) << 1));
}

struct EikonalConsts {
  float dx, two_dx2, dx2, half, third;
};

// The smaller and the larger of two magnitudes: their bit patterns order as
// they do, and an integer compare needs no quieting of NaNs first.
__device__ __forceinline__ float nearer(float a, float b) {
  const uint32_t x = __float_as_uint(a) & 0x7fffffffu, y = __float_as_uint(b) & 0x7fffffffu;
  return __uint_as_float(x < y ? x : y);
}
__device__ __forceinline__ float lesser(float a, float b) {
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  return __uint_as_float(x < y ? x : y);
}
__device__ __forceinline__ float larger(float a, float b) {
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  return __uint_as_float(x < y ? y : x);
}

// sqrtf, correctly rounded, for an argument that is 0, +inf or at least
// 2^-96: the hardware's root (within 1 ulp) and Tuckerman's test of its two
// neighbours (s is the rounded root of x when s (s - ulp) < x <= s (s + ulp)).
// The compiler's sqrtf spends six more instructions on scaling smaller
// arguments; the sweeps below are bound by the instructions of their chains.
__device__ __forceinline__ float root(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  const float s = __builtin_amdgcn_sqrtf(x);
  const float below = __uint_as_float(__float_as_uint(s) - 1u);
  const float above = __uint_as_float(__float_as_uint(s) + 1u);
  const float r = __builtin_fmaf(-below, s, x) <= 0.0f ? below : s;
  return __builtin_fmaf(-above, s, x) > 0.0f ? above : r;
#else
  return sqrtf(x);
#endif
}

// update_from_neighbor (level_set.py:88-112) from the nearer neighbour `a`
// along the line and the nearer ones across it, m1 <= m2 (2D: m1 alone).
// The three are merged in order (no distance is ever NaN: target_surface and
// the sweeps store a value only where it compares less than another one), and
// every candidate is formed, so nothing but the choice waits for a compare.
// ROOT: both roots' arguments are in root's range where their result counts.
template <int DIM, bool ROOT>
__device__ __forceinline__ float eikonal(float a, float m1, float m2, const EikonalConsts& c) {
  auto rt = [](float x) { return ROOT ? root(x) : sqrtf(x); };
  const float n0 = lesser(a, m1);
  const float n1 = DIM == 3 ? lesser(larger(a, m1), m2) : larger(a, m1);
  const float d1 = n0 + c.dx;
  const float df = n1 - n0;
  float d2 = c.half * (n0 + n1 + rt(c.two_dx2 - df * df));
  if (DIM == 3) {
    const float n2 = larger(a, m2);
    const float s = n0 + n1 + n2;
    const float q = n0 * n0 + n1 * n1 + n2 * n2 - c.dx2;
    const float d3 = c.third * (s + rt(fmaxf(0.0f, s * s - 3.0f * q)));
    d2 = d2 > n2 ? d3 : d2;
  }
  return d1 > n1 ? d2 : d1;
}

// Workgroup w of n works on part xcd_part(w, n): workgroups go to the 8 XCDs
// in turn, so this gives each XCD a contiguous range of parts, whose shared
// neighbour lines then meet in its L2.
__device__ __forceinline__ int xcd_part(int w, int n) {
  const int q = n / 8, r = n % 8, x = w % 8;
  return x * q + min(x, r) + w / 8;
}

// One directional sweep along axis AX.  A line is a serial chain, each cell
// waiting for the one before it, and a wave's chain is bound by the
// instructions it issues (4 cycles each, one wave per SIMD), so everything
// that does not wait is taken off it: a workgroup has SW_LINES lines in
// chunks of SW_STEPS steps; its last four waves read a chunk's cells and the
// lines across, coalesced, and leave in one of two LDS buffers each cell's
// distance and its two sorted cross neighbours, while the first wave walks
// the other buffer, a lane per line, on magnitudes alone.  The walked
// magnitudes replace the cross neighbours, and the filling waves sign and
// store them, coalesced, before that buffer is filled again (each thread the
// places it fills).  On the contiguous axis a line's steps are consecutive in
// LDS (17 words a line: no bank conflicts for the walk), on the others the
// lines of a step.  37 KB of LDS: four workgroups per CU.
// A sweep at 256^3: 77 us on the contiguous axis, 75 us on the others, bound
// by issue (one walking and four filling waves per SIMD); a thread per line
// on global memory, with a copy of the array before it, took 1390 and 600 us.
// At 131 x 97 x 150, 20-27 us, bound by the chain (about 150 ns a step in 3D,
// 70 ns in 2D).
constexpr int SW_LINES = 64;
constexpr int SW_STEPS = 16;
constexpr int SW_FILL = 256;
constexpr int SW_THREADS = 64 + SW_FILL;
constexpr int SW_MINE = SW_LINES * SW_STEPS / SW_FILL;  // places per filling thread
constexpr int SW_WORDS = SW_LINES * (SW_STEPS + 1);     // one step more: the chunk's next cell
// also: NULL, or (on axis 0, in the last sweep) a second array for the
// distances, which a copy after it would read again.
template <int DIM, int AX, bool ROOT, typename IX>
__global__ void __launch_bounds__(SW_THREADS, 5) k_sweep(Grid g, int dir,
                                                      const float* __restrict__ src,
                                                      float* __restrict__ dst,
                                                      float* __restrict__ also,
                                                      const int8_t* __restrict__ code,
                                                      EikonalConsts c) {
  constexpr bool CONTIG = AX == DIM - 1;
  // the axes across: B, and in 3D A
  constexpr int B = CONTIG ? DIM - 2 : DIM - 1, A = DIM == 2 ? B : (AX == 0 ? 1 : 0);
  __shared__ float own[2][SW_WORDS];   // the cells' distances, signed
  __shared__ float thr[2][SW_WORDS];   // |distance| to undercut: 0 where fixed
  __shared__ float m1[2][SW_WORDS];    // nearer neighbours across; the walked magnitudes
  __shared__ float m2[2][SW_WORDS];
  __shared__ int8_t cd[2][SW_WORDS];   // cell codes
  // chunk ch has an unfixed cell of sign 0 (its distance becomes 0): slot
  // ch & 3, cleared two chunks before it is filled
  __shared__ int flat[4];
  auto place = [](int line, int step) {
    return CONTIG ? line * (SW_STEPS + 1) + step : step * SW_LINES + line;
  };
  const int n = g.n[AX];
  const long nlines = g.cells() / n;
  const long line0 = (long)xcd_part((int)blockIdx.x, (int)gridDim.x) * SW_LINES;
  const int nchunks = (n + SW_STEPS - 1) / SW_STEPS;
  const int tid = (int)threadIdx.x;
  // filling thread f's places i: line fl + i * FL, step fs + i * FS of a chunk
  // (the walking wave computes them too and does not use them)
  constexpr int FL = CONTIG ? SW_FILL / SW_STEPS : 0, FS = CONTIG ? 0 : SW_FILL / SW_LINES;
  const int f = tid - 64;
  const int fl = CONTIG ? max(f, 0) / SW_STEPS : max(f, 0) & (SW_LINES - 1);
  const int fs = CONTIG ? f & (SW_STEPS - 1) : max(f, 0) / SW_LINES;
  // its lines' first cells in sweep order (a line past the last one reads the
  // last one and is not stored) and the offsets to the lines across; on a side
  // without one the other side's line is read twice (every axis has at least
  // two cells), which leaves the nearer of the two the same
  constexpr int NL = CONTIG ? SW_MINE : 1;
  const IX st = (IX)(dir > 0 ? g.st[AX] : -g.st[AX]), stb = (IX)g.st[B], sta = (IX)g.st[A];
  IX first[NL], obl[NL], obh[NL], oal[NL], oah[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const long line = min(line0 + fl + i * FL, nlines - 1);
    // the line's coordinates on B and A: C order over those axes
    constexpr int SLOW = DIM == 2 ? B : (A < B ? A : B), FAST = DIM == 2 ? B : (A < B ? B : A);
    const int is = DIM == 3 ? (int)(line / g.n[FAST]) : 0;
    const int ifa = (int)(line - (long)is * g.n[FAST]);
    first[i] = (IX)((DIM == 3 ? is * g.st[SLOW] : 0) + ifa * g.st[FAST] +
                    (dir > 0 ? 0 : (n - 1) * g.st[AX]));
    const int ib = FAST == B ? ifa : is, ia = FAST == B ? is : ifa;
    obl[i] = ib > 0 ? -stb : stb;
    obh[i] = ib + 1 < g.n[B] ? stb : -stb;
    oal[i] = ia > 0 ? -sta : sta;
    oah[i] = ia + 1 < g.n[A] ? sta : -sta;
  }
  auto at = [](auto* base, IX i) {
    if constexpr (sizeof(IX) == 4) return ldgi(base, i);
    else return ldg(base + i);
  };
  // A chunk that reaches the line's end (`tail`) clamps its steps there; the
  // others, and workgroups with all their lines, do without any test.
  const bool lines = line0 + SW_LINES <= nlines;
  auto tail = [&](int chunk) { return (chunk + 1) * SW_STEPS >= n; };
  auto store_t = [&](int chunk, auto test) {
    const int b = chunk & 1, s0 = chunk * SW_STEPS + fs;
#pragma unroll
    for (int i = 0; i < SW_MINE; ++i) {
      const int s = s0 + i * FS, w = place(fl + i * FL, fs + i * FS);
      if (decltype(test)::value && (line0 + fl + i * FL >= nlines || s >= n)) continue;
      const float mag = m1[b][w], was = own[b][w];
      const float v = mag < fabsf(was) ? mag * code_sign(cd[b][w]) : was;
      const IX t = first[CONTIG ? i : 0] + s * st;
      if constexpr (sizeof(IX) == 4) stgi(dst, t, v);
      else stg(dst + t, v);
      if (AX == 0 && also != nullptr) {
        if constexpr (sizeof(IX) == 4) stgi(also, t, v);
        else stg(also + t, v);
      }
    }
  };
  auto store = [&](int chunk) {
    if (lines && !tail(chunk)) store_t(chunk, std::false_type());
    else store_t(chunk, std::true_type());
  };
  // a chunk's values on their way to LDS: loaded a chunk ahead, so that their
  // latency passes behind the walk of the chunk between
  float v[SW_MINE], nx[SW_MINE], bl[SW_MINE], bh[SW_MINE], al[SW_MINE], ah[SW_MINE];
  int cv[SW_MINE];
  auto fetch_t = [&](int chunk, auto clamp) {
    const int s0 = chunk * SW_STEPS + fs;
#pragma unroll
    for (int i = 0; i < SW_MINE; ++i) {
      const int l = CONTIG ? i : 0;
      const int s = decltype(clamp)::value ? min(s0 + i * FS, n - 1) : s0 + i * FS;
      const IX t = first[l] + s * st;
      v[i] = at(src, t);
      bl[i] = at(src, t + obl[l]);
      bh[i] = at(src, t + obh[l]);
      if (DIM == 3) {
        al[i] = at(src, t + oal[l]);
        ah[i] = at(src, t + oah[l]);
      }
      cv[i] = at(code, t);
      // the chunk's last step carries the next cell of the line too
      if (CONTIG || i == SW_MINE - 1)
        nx[i] = at(src, !decltype(clamp)::value || s + 1 < n ? t + st : t);
    }
  };
  auto fetch = [&](int chunk) {
    if (tail(chunk)) fetch_t(chunk, std::true_type());
    else fetch_t(chunk, std::false_type());
  };
  auto put = [&](int chunk) {
    const int b = chunk & 1, s0 = chunk * SW_STEPS + fs;
    bool zero = false;
#pragma unroll
    for (int i = 0; i < SW_MINE; ++i) {
      const int step = fs + i * FS, w = place(fl + i * FL, step);
      const float mb = nearer(bl[i], bh[i]);
      const float ma = DIM == 3 ? nearer(al[i], ah[i]) : INFINITY;
      const bool fixed = (cv[i] & 1) != 0;
      // past the line's end: no neighbour ahead
      own[b][w] = s0 + i * FS < n ? v[i] : INFINITY;
      if ((CONTIG || i == SW_MINE - 1) && step == SW_STEPS - 1)
        own[b][place(fl + i * FL, SW_STEPS)] = s0 + i * FS + 1 < n ? nx[i] : INFINITY;
      thr[b][w] = fixed ? 0.0f : fabsf(v[i]);
      m1[b][w] = DIM == 3 ? lesser(mb, ma) : mb;
      if (DIM == 3) m2[b][w] = larger(mb, ma);
      cd[b][w] = (int8_t)cv[i];
      zero = zero || cv[i] == 2;  // not fixed, sign 0
    }
    if (zero) flat[chunk & 3] = 1;
  };
  // the walked magnitudes of chunk buffer b (steps past the line's end walk
  // over what the buffer holds, and are not stored)
  float prev = INFINITY;
  auto walk = [&](int b, auto zeros) {
    float nx[SW_STEPS], lim[SW_STEPS], a1[SW_STEPS], a2[SW_STEPS];
    const float here = own[b][place(tid, 0)];
#pragma unroll
    for (int u = 0; u < SW_STEPS; ++u) {
      nx[u] = own[b][place(tid, u + 1)];
      lim[u] = thr[b][place(tid, u)];
      a1[u] = m1[b][place(tid, u)];
      a2[u] = DIM == 3 ? m2[b][place(tid, u)] : INFINITY;
    }
#pragma unroll
    for (int u = 0; u < SW_STEPS; ++u) {
      const float was = fabsf(u == 0 ? here : nx[u - 1]);
      float d = eikonal<DIM, ROOT>(nearer(prev, nx[u]), a1[u], a2[u], c);
      const bool less = d < lim[u];
      if (decltype(zeros)::value) d = d * fabsf(code_sign(cd[b][place(tid, u)]));
      prev = less ? d : was;
      m1[b][place(tid, u)] = prev;
    }
  };
  if (tid < 4) flat[tid] = 0;
  // Both sides of the branch, each taken by whole waves, pass the same
  // barriers: one here, one before every chunk, one after the last.  (Two
  // loops rather than one keep the filling waves' values out of the walking
  // wave's registers.)
  __syncthreads();
  if (f >= 0) {
    fetch(0);
    put(0);
    fetch(1);
    for (int ch = 0; ch < nchunks; ++ch) {
      __syncthreads();  // buffer ch & 1 is filled, the other one walked
      if (ch > 0) store(ch - 1);
      if (ch + 1 < nchunks) {
        put(ch + 1);
        fetch(ch + 2);
      }
    }
    __syncthreads();
    store(nchunks - 1);
  } else {
    for (int ch = 0; ch < nchunks; ++ch) {
      __syncthreads();
      if (tid == 0) flat[(ch + 2) & 3] = 0;
      if (flat[ch & 3]) walk(ch & 1, std::true_type());
      else walk(ch & 1, std::false_type());
    }
    __syncthreads();
  }
}

__global__ void k_copy(long n, const float* __restrict__ src, float* __restrict__ dst) {
  const long t = (long)blockIdx.x * LB + threadIdx.x;
  if (t < n) dst[t] = src[t];
}

// ---------------------------------------------------------------------------
// FluidSimulator.extrap_velocity (fluid_simulator.py:240-270) for one MAC
// component k (shape res + e_k): mark_valid -- a face is valid when a cell on
// either side is FLUID (out of range is not) -- then `iterations` passes of
// diffuse_quantity, each averaging the valid faces of the 3^dim block around
// every invalid face (offsets in C order, FP32 sum then one division) into it
// and marking it valid; each pass reads the velocities and flags as they were
// before the pass.  Faces outside the component's own shape count as invalid
// (the reference's shared `valid` field is res + 1 in every axis and keeps
// other components' flags there, and it is read out of range at index -1).
// ---------------------------------------------------------------------------
// The flags of a component are a bit per face in C order, 32 to a word; a
// pass reads one copy and writes the other (every word of it).  Velocities
// are updated in place: a pass writes invalid faces only and reads valid ones
// only, and no face becomes both during a pass.  Each launch serves every
// component, a wave EX_GROUPS groups of 64 faces.  A pass changes few faces (the
// layer around the valid ones), and most rows that cross a body have one or
// two, so a workgroup first finds its candidates -- invalid, with a valid bit
// in the 3^dim block -- on whole words, 32 faces a lane, lists them, and then
// gives each lane one of the list: its 27 bits from the same words, and the
// velocities behind them, those without a bit as 0 (a sum that starts at +0
// is never -0, so adding +0 leaves it), all in flight together.  Bound by the
// latency of those few rounds of loads.  128^3, ten passes of three
// components: 5.3 ms with copies of the velocity and of byte flags and 27
// byte loads per invalid face, 0.45 ms on the flag bits with a lane per face
// -> 0.24 ms.
struct Faces3 {
  Grid f[3];           // each component's faces
  float* u[3];
  uint32_t* valid[2];  // flag words, every component's after the one before
  int word0[4];        // first word of each component
  int block0[4];       // first workgroup of each component (EX_FACES faces each)
  int dim;
};
// (4 groups a wave: 0.28 ms; eight waves per SIMD, which spills: 0.26 ms)
constexpr int EX_GROUPS = 8;
constexpr int EX_FACES = LB * EX_GROUPS;
__device__ __forceinline__ int component(const Faces3& F, int b) {
  return b < F.block0[1] ? 0 : (b < F.block0[2] ? 1 : 2);
}
// the first face of this wave's groups, of component k
__device__ __forceinline__ long wave_faces(const Faces3& F, int k) {
  return (long)((int)blockIdx.x - F.block0[k]) * EX_FACES +
         (long)(threadIdx.x / 64) * (64 * EX_GROUPS);
}

__global__ void __launch_bounds__(LB) k_mark_valid(Faces3 F, Grid c,
                                                   const int8_t* __restrict__ ct) {
  const int k = component(F, (int)blockIdx.x);
  const Grid& f = F.f[k];
  const long n = f.cells(), t0 = wave_faces(F, k);
  const int lane = threadIdx.x & 63;
  int above[EX_GROUPS], below[EX_GROUPS];
#pragma unroll
  for (int g = 0; g < EX_GROUPS; ++g) {  // every cell type before the first ballot
    const long t = t0 + 64 * g + lane;
    int I[3];
    coords(f, t < n ? t : 0, I);
    long u = 0;  // the cell above the face
    for (int a = 0; a < c.dim; ++a) u += I[a] * c.st[a];
    const bool up = t < n && I[k] < c.n[k], down = t < n && I[k] > 0;
    const int a = ct[up ? u : 0], b = ct[down ? u - c.st[k] : 0];
    above[g] = up ? a : MG_SOLID;
    below[g] = down ? b : MG_SOLID;
  }
#pragma unroll
  for (int g = 0; g < EX_GROUPS; ++g) {
    MG_KEEP(above[g]);
    MG_KEEP(below[g]);
  }
  uint32_t out = 0u;  // lanes 0 .. 2 EX_GROUPS - 1: the wave's words
#pragma unroll
  for (int g = 0; g < EX_GROUPS; ++g) {
    const unsigned long long m = __ballot(above[g] == MG_FLUID || below[g] == MG_FLUID);
    if ((lane >> 1) == g) out = (uint32_t)(m >> (32 * (lane & 1)));
  }
  const long w = (t0 >> 5) + lane;
  if (lane < 2 * EX_GROUPS && w < (n + 31) / 32) F.valid[0][F.word0[k] + w] = out;
}

template <int DIM>
__global__ void __launch_bounds__(LB, 6) k_diffuse(Faces3 F, int from) {
  constexpr int ROWS = DIM == 3 ? 9 : 3;   // rows around a face, in C order of the offsets
  constexpr int WORDS = 2 * EX_GROUPS;     // the wave's words
  constexpr int PARTS = 64 / WORDS;        // lanes that share the rows around a word
  __shared__ int count[LB / 64];      // candidates of each wave
  __shared__ uint16_t list[EX_FACES];  // the workgroup's candidates, from its first face
  __shared__ uint8_t made[EX_FACES];   // whether a candidate became valid
  const int k = component(F, (int)blockIdx.x);
  const Grid& f = F.f[k];
  const long n = f.cells(), t0 = wave_faces(F, k);
  const uint32_t* valid = F.valid[from] + F.word0[k];
  const int nwords = F.word0[k + 1] - F.word0[k];
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  // the offset of row r from the face's own
  auto row_of = [&](int r) -> long {
    return DIM == 3 ? (r / 3 - 1) * f.st[0] + (r % 3 - 1) * f.st[1] : (r - 1) * f.st[0];
  };
  // word w of the flags: 0 outside them, where a word inside is read instead
  // (no branch, so every load of a round is in flight before the first wait)
  auto word = [&](long w) -> uint32_t {
    const int wi = (int)w, in = min(max(wi, 0), nwords - 1);
    const uint32_t v = ldgi(valid, in);
    return wi == in ? v : 0u;
  };
  // candidates of word `lane % WORDS`: the rows' bits just below to just above
  // each face (34 from three words), a row for each of the PARTS in turn
  const long w0 = t0 >> 5, wl = w0 + (lane & (WORDS - 1));
  constexpr int MINE = (ROWS + PARTS - 1) / PARTS;
  const uint32_t own = word(wl);
  uint32_t a[MINE], b[MINE], c[MINE];
  long first[MINE];
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    const int r = lane / WORDS + i * PARTS;
    first[i] = 32 * wl + row_of(r < ROWS ? r : 0) - 1;  // row 0 once more changes nothing
    a[i] = word(first[i] >> 5);
    b[i] = word((first[i] >> 5) + 1);
    c[i] = word((first[i] >> 5) + 2);
  }
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    MG_KEEP(a[i]);
    MG_KEEP(b[i]);
    MG_KEEP(c[i]);
  }
  uint32_t cand = 0u;
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    const int sh = (int)(first[i] & 31);
    const unsigned long long v = (((unsigned long long)b[i] << 32 | a[i]) >> sh) |
                                 (sh ? (unsigned long long)c[i] << (64 - sh) : 0ull);
    cand |= (uint32_t)(v | v >> 1 | v >> 2);
  }
#pragma unroll
  for (int d = WORDS; d < 64; d <<= 1) cand |= (uint32_t)__shfl_xor((int)cand, d);
  cand &= ~own;
  if (32 * wl + 31 >= n) cand &= 32 * wl < n ? (1u << (n - 32 * wl)) - 1u : 0u;
  unsigned long long m[EX_GROUPS];  // candidates of each group
  int mine = 0;
#pragma unroll
  for (int g = 0; g < EX_GROUPS; ++g) {
    m[g] = (unsigned long long)(uint32_t)MG_READLANE((int)cand, 2 * g) |
           ((unsigned long long)(uint32_t)MG_READLANE((int)cand, 2 * g + 1) << 32);
    mine += __builtin_popcountll(m[g]);
  }
  if (lane == 0) count[wave] = mine;
  __syncthreads();
  int at0 = 0, total = 0;
#pragma unroll
  for (int w = 0; w < LB / 64; ++w) {
    if (w < wave) at0 += count[w];
    total += count[w];
  }
  const int here = wave * 64 * EX_GROUPS;  // the wave's first face, from the workgroup's
#pragma unroll
  for (int g = 0; g < EX_GROUPS; ++g) {
    if ((m[g] >> lane) & 1ull)
      list[at0 + __builtin_popcountll(m[g] & ((1ull << lane) - 1ull))] =
          (uint16_t)(here + 64 * g + lane);
    at0 += __builtin_popcountll(m[g]);
  }
  __syncthreads();
  for (int i = (int)threadIdx.x; i < total; i += LB) {
    const int at = list[i];
    const long t = t0 - here + at;
    int I[3];
    coords(f, t, I);
    unsigned long long two[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const long w = (t + row_of(r) - 1) >> 5;  // the row's first bit is in word w
      two[r] = (unsigned long long)word(w) | ((unsigned long long)word(w + 1) << 32);
    }
    uint32_t bits = 0u;  // the block's valid faces, in C order of the offsets
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int o0 = DIM == 3 ? r / 3 - 1 : r - 1, o1 = DIM == 3 ? r % 3 - 1 : 0;
      const bool in = I[0] + o0 >= 0 && I[0] + o0 < f.n[0] &&
                      (DIM == 2 || (I[1] + o1 >= 0 && I[1] + o1 < f.n[1]));
      uint32_t three = (uint32_t)(two[r] >> ((t + row_of(r) - 1) & 31)) & 7u;
      if (I[DIM - 1] == 0) three &= 6u;
      if (I[DIM - 1] + 1 == f.n[DIM - 1]) three &= 3u;
      if (in) bits |= three << (3 * r);
    }
    made[at] = bits != 0u;
    if (bits == 0u) continue;  // a row's end is next to another row's start
    float* u = F.u[k];
    float v[3 * ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int o = 0; o < 3; ++o)
        v[3 * r + o] = ldg(u + (((bits >> (3 * r + o)) & 1u) ? t + row_of(r) + (o - 1) : t));
#pragma unroll
    for (int j = 0; j < 3 * ROWS; ++j) MG_KEEP(v[j]);
    float tot = 0.0f;
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < 3 * ROWS; ++j) {
      const bool is = (bits >> j) & 1u;
      tot = tot + (is ? v[j] : 0.0f);
      cnt += is ? 1 : 0;
    }
    u[t] = tot / (float)cnt;
  }
  __syncthreads();
  uint32_t out = own;
#pragma unroll
  for (int g = 0; g < EX_GROUPS; ++g) {
    const bool on = ((m[g] >> lane) & 1ull) && made[here + 64 * g + lane];
    const unsigned long long v = __ballot(on);
    if ((lane >> 1) == g) out |= (uint32_t)(v >> (32 * (lane & 1)));
  }
  if (lane < WORDS && wl < nwords) F.valid[from ^ 1][F.word0[k] + wl] = out;
}

inline unsigned nblk(long n) { return (unsigned)((n + LB - 1) / LB); }

template <int DIM, int AX>
void sweep_t(hipStream_t s, const Grid& g, int dir, const float* src, float* dst, float* also,
             const int8_t* code, const EikonalConsts& c) {
  const long nlines = g.cells() / g.n[AX];
  const dim3 grid((unsigned)((nlines + SW_LINES - 1) / SW_LINES));
  // The roots' arguments are sums and products of distances rounded to 24
  // bits: 0 or at least dx^2 2^-24 where their result counts, so above root's
  // 2^-96 for every dx but the smallest.  32-bit offsets reach 2^30 cells.
  if (c.dx < 0x1p-32f)
    hipLaunchKernelGGL((k_sweep<DIM, AX, false, long>), grid, dim3(SW_THREADS), 0, s, g, dir, src,
                       dst, also, code, c);
  else if (g.cells() > (1l << 30))
    hipLaunchKernelGGL((k_sweep<DIM, AX, true, long>), grid, dim3(SW_THREADS), 0, s, g, dir, src,
                       dst, also, code, c);
  else
    hipLaunchKernelGGL((k_sweep<DIM, AX, true, int>), grid, dim3(SW_THREADS), 0, s, g, dir, src,
                       dst, also, code, c);
}

void sweep(hipStream_t s, const Grid& g, int ax, int dir, const float* src, float* dst,
           float* also, const int8_t* code, const EikonalConsts& c) {
  if (g.dim == 2) {
    if (ax == 0) sweep_t<2, 0>(s, g, dir, src, dst, also, code, c);
    else sweep_t<2, 1>(s, g, dir, src, dst, also, code, c);
  } else if (ax == 0) {
    sweep_t<3, 0>(s, g, dir, src, dst, also, code, c);
  } else if (ax == 1) {
    sweep_t<3, 1>(s, g, dir, src, dst, also, code, c);
  } else {
    sweep_t<3, 2>(s, g, dir, src, dst, also, code, c);
  }
}

int check_grid(int dim, const int32_t* res) {
  MG_REQUIRE(dim == 2 || dim == 3, "dim must be 2 or 3");
  MG_REQUIRE(res != nullptr, "res is NULL");
  for (int a = 0; a < dim; ++a) MG_REQUIRE(res[a] >= 2, "res[%d] = %d must be >= 2", a, res[a]);
  return 0;
}

}  // namespace

extern "C" int mgpcg_apply_markers(void* stream, int dim, const int32_t* res, const float* phi,
                                   int8_t* cell_type) {
  if (check_grid(dim, res)) return -1;
  MG_REQUIRE(phi && cell_type, "NULL argument");
  Grid g = make_grid(dim, res);
  hipLaunchKernelGGL(k_apply_markers, dim3(nblk(g.cells())), dim3(LB), 0, (hipStream_t)stream, g,
                     phi, cell_type);
  MG_HIP(hipGetLastError());
  return 0;
}

extern "C" int mgpcg_init_boundary(void* stream, int dim, const int32_t* res, int8_t* cell_type) {
  if (check_grid(dim, res)) return -1;
  MG_REQUIRE(cell_type, "NULL argument");
  Grid g = make_grid(dim, res);
  hipLaunchKernelGGL(k_init_boundary, dim3(nblk(g.cells())), dim3(LB), 0, (hipStream_t)stream,
                     g, cell_type);
  MG_HIP(hipGetLastError());
  return 0;
}

extern "C" int mgpcg_redistance(void* stream, int dim, const int32_t* res, double dx,
                                int repeat_times, float* phi, float* phi_temp, float* snap,
                                int8_t* fixed) {
  if (check_grid(dim, res)) return -1;
  MG_REQUIRE(phi && phi_temp && snap && fixed, "NULL argument");
  MG_REQUIRE(dx > 0.0, "dx must be positive");
  MG_REQUIRE(repeat_times >= 0, "repeat_times must be >= 0");
  hipStream_t s = (hipStream_t)stream;
  Grid g = make_grid(dim, res);
  const long n = g.cells();
  // Python-scope constants of update_from_neighbor, baked as FP32
  EikonalConsts c;
  c.dx = (float)dx;
  c.two_dx2 = (float)(2.0 * (dx * dx));
  c.dx2 = (float)(dx * dx);
  c.half = (float)(1.0 / 2.0);
  c.third = (float)(1.0 / 3.0);
  if (dim == 3)
    hipLaunchKernelGGL((k_target_surface<3>), dim3(nblk(n)), dim3(LB), 0, s, g,
                       (const float*)phi, (float)dx, phi_temp, fixed);
  else
    hipLaunchKernelGGL((k_target_surface<2>), dim3(nblk(n)), dim3(LB), 0, s, g,
                       (const float*)phi, (float)dx, phi_temp, fixed);
  // each sweep reads one work array and writes the other; the last one writes
  // phi, which nothing reads after target_surface, and phi_temp, which it does
  // not read (an even number of sweeps: the one before it wrote snap)
  float *src = phi_temp, *dst = snap;
  for (int rep = 0; rep < repeat_times; ++rep) {
    for (int ax = dim - 1; ax >= 0; --ax) {
      for (int dir = 1; dir >= -1; dir -= 2) {
        const bool last = rep == repeat_times - 1 && ax == 0 && dir == -1;
        sweep(s, g, ax, dir, src, last ? phi : dst, last ? dst : nullptr, (const int8_t*)fixed,
              c);
        std::swap(src, dst);
      }
    }
  }
  if (repeat_times == 0)
    hipLaunchKernelGGL(k_copy, dim3(nblk(n)), dim3(LB), 0, s, n, (const float*)phi_temp, phi);
  MG_HIP(hipGetLastError());
  return 0;
}

extern "C" int mgpcg_extrap_velocity(void* stream, int dim, const int32_t* res,
                                     const int8_t* cell_type, float* const* velocity,
                                     int iterations, float* backup, int8_t* valid,
                                     int8_t* valid_temp) {
  if (check_grid(dim, res)) return -1;
  MG_REQUIRE(cell_type && velocity && backup && valid && valid_temp, "NULL argument");
  for (int k = 0; k < dim; ++k) MG_REQUIRE(velocity[k], "velocity[%d] is NULL", k);
  MG_REQUIRE(iterations >= 0, "iterations must be >= 0");
  hipStream_t s = (hipStream_t)stream;
  const Grid c = make_grid(dim, res);
  // Both copies of the flag bits lie in `backup`: of the floats of the largest
  // component, n faces or more, they take 2 dim (n / 32 + 1) words, which is
  // less for every shape (n >= 6 in 2D, 12 in 3D).
  Faces3 F;
  F.dim = dim;
  long words = 0, blocks = 0;
  for (int k = 0; k < 3; ++k) {
    F.word0[k] = (int)words;
    F.block0[k] = (int)blocks;
    F.u[k] = k < dim ? velocity[k] : nullptr;
    if (k >= dim) {
      F.f[k] = c;
      continue;
    }
    int32_t fr[3] = {0, 0, 0};
    for (int a = 0; a < dim; ++a) fr[a] = res[a] + (a == k ? 1 : 0);
    F.f[k] = make_grid(dim, fr);
    words += (F.f[k].cells() + 31) / 32;
    blocks += (F.f[k].cells() + EX_FACES - 1) / EX_FACES;
  }
  MG_REQUIRE(blocks <= 0x7fffffffL && words <= 0x7fffffffL, "grid too large");
  F.word0[3] = (int)words;
  F.block0[3] = (int)blocks;
  F.valid[0] = (uint32_t*)backup;
  F.valid[1] = F.valid[0] + words;
  const dim3 grid((unsigned)blocks), block(LB);
  hipLaunchKernelGGL(k_mark_valid, grid, block, 0, s, F, c, cell_type);
  for (int it = 0; it < iterations; ++it) {
    if (dim == 3) hipLaunchKernelGGL((k_diffuse<3>), grid, block, 0, s, F, it & 1);
    else hipLaunchKernelGGL((k_diffuse<2>), grid, block, 0, s, F, it & 1);
  }
  MG_HIP(hipGetLastError());
  return 0;
}
