// Inverse 3D transform of a block of template-search products over the valid
// area only, with its neighbours in the pipeline joined to it: the template's
// forward z transform and the product by the tomogram spectrum come before the
// inverse z transform in one kernel, and the valid area's sums follow the x
// transform in another. (reference: alignment/BH_templateSearch3d_2.m:756-764)
//
// Each pass holds a tile of whole columns in LDS and runs a Stockham transform
// in place: a lane loads the butterflies it owns (at most 20 complex values)
// into registers, the workgroup meets, and they are stored at their sorted
// places. Per orientation and chunk the passes read and write
//   z: the template's partial DFT and the tomogram spectrum -> valid z
//   y: valid z -> valid (y, z)
//   x: valid (y, z) -> the valid map
// and nothing else. A general 3D inverse transform of the whole chunk moves the
// product, three transposes, three transforms and the whole map besides.
//
// What bounds them, 12 orientations of a 48^3 template over 360 x 384 x 324 (valid
// 312 x 336 x 276): z 1.6 ms, 62 % VALU (two transforms a column) with 2.2 GB
// moved; y 0.98 ms, 3.7 TB/s; x 0.98 ms, 3.1 TB/s. The kernels they replace took
// 1.9 ms (z product on the matrix cores) and 6.4 ms (library inverse) and 0.4 ms
// (sums).
#include <algorithm>
#include <cmath>

#include "ops.hpp"

namespace emc {

constexpr int kColThreads = 512;
constexpr int kColValues = 16;      // values of one column a lane holds
constexpr size_t kColLds = 65024;   // LDS of a workgroup's table and tile (64 KB with its sums)

// One axis: n = product of radix[0 .. count), e^{2 pi i j / (scale n)} tabled.
struct ColPlan {
  int n, count, scale;
  int radix[8];
};

static __device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
static __device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
static __device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
static __device__ __forceinline__ float2 muli(float2 a) { return make_float2(-a.y, a.x); }

static __device__ __forceinline__ void dft3(float2& a, float2& b, float2& c) {
  constexpr float s = 0.86602540378443864676f;
  const float2 t = cadd(b, c), d = csub(b, c);
  const float2 u = make_float2(fmaf(-0.5f, t.x, a.x), fmaf(-0.5f, t.y, a.y));
  a = cadd(a, t);
  b = make_float2(fmaf(-s, d.y, u.x), fmaf(s, d.x, u.y));
  c = make_float2(fmaf(s, d.y, u.x), fmaf(-s, d.x, u.y));
}

static __device__ __forceinline__ void dft4(float2& a, float2& b, float2& c, float2& d) {
  const float2 s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = muli(csub(b, d));
  a = cadd(s0, s2);
  b = cadd(s1, s3);
  c = csub(s0, s2);
  d = csub(s1, s3);
}

// v <- sum_j v[j] e^{2 pi i j k / R}
template <int R>
static __device__ __forceinline__ void dft(float2 (&v)[R]) {
  if constexpr (R == 2) {
    const float2 t = v[1];
    v[1] = csub(v[0], t);
    v[0] = cadd(v[0], t);
  } else if constexpr (R == 3) {
    dft3(v[0], v[1], v[2]);
  } else if constexpr (R == 4) {
    dft4(v[0], v[1], v[2], v[3]);
  } else if constexpr (R == 5) {
    constexpr float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
    constexpr float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
    const float2 t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]), t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
    const float2 m1 = make_float2(fmaf(c1, t1.x, fmaf(c2, t2.x, v[0].x)), fmaf(c1, t1.y, fmaf(c2, t2.y, v[0].y)));
    const float2 m2 = make_float2(fmaf(c2, t1.x, fmaf(c1, t2.x, v[0].x)), fmaf(c2, t1.y, fmaf(c1, t2.y, v[0].y)));
    const float2 u1 = make_float2(fmaf(s1, t3.x, s2 * t4.x), fmaf(s1, t3.y, s2 * t4.y));
    const float2 u2 = make_float2(fmaf(s2, t3.x, -(s1 * t4.x)), fmaf(s2, t3.y, -(s1 * t4.y)));
    v[0] = cadd(v[0], cadd(t1, t2));
    v[1] = cadd(m1, muli(u1));
    v[2] = cadd(m2, muli(u2));
    v[3] = csub(m2, muli(u2));
    v[4] = csub(m1, muli(u1));
  } else if constexpr (R == 6) {
    constexpr float s = 0.86602540378443864676f;
    dft3(v[0], v[2], v[4]);
    dft3(v[1], v[3], v[5]);
    const float2 o0 = v[1], o1 = cmul(v[3], make_float2(0.5f, s)), o2 = cmul(v[5], make_float2(-0.5f, s));
    const float2 e0 = v[0], e1 = v[2], e2 = v[4];
    v[0] = cadd(e0, o0);
    v[1] = cadd(e1, o1);
    v[2] = cadd(e2, o2);
    v[3] = csub(e0, o0);
    v[4] = csub(e1, o1);
    v[5] = csub(e2, o2);
  } else if constexpr (R == 8) {
    constexpr float h = 0.70710678118654752440f;
    dft4(v[0], v[2], v[4], v[6]);
    dft4(v[1], v[3], v[5], v[7]);
    const float2 o0 = v[1], o1 = make_float2(h * (v[3].x - v[3].y), h * (v[3].x + v[3].y)), o2 = muli(v[5]);
    const float2 o3 = make_float2(-h * (v[7].x + v[7].y), h * (v[7].x - v[7].y));
    const float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    v[0] = cadd(e0, o0);
    v[1] = cadd(e1, o1);
    v[2] = cadd(e2, o2);
    v[3] = cadd(e3, o3);
    v[4] = csub(e0, o0);
    v[5] = csub(e1, o1);
    v[6] = csub(e2, o2);
    v[7] = csub(e3, o3);
  } else {
    static_assert(R == 9, "radix");
    constexpr float c1 = 0.76604444311897803520f, s1 = 0.64278760968653932632f;  // 40 degrees
    constexpr float c2 = 0.17364817766693034885f, s2 = 0.98480775301220805937f;  // 80
    constexpr float c4 = -0.93969262078590838405f, s4 = 0.34202014332566873304f; // 160
    dft3(v[0], v[3], v[6]);
    dft3(v[1], v[4], v[7]);
    dft3(v[2], v[5], v[8]);
    v[4] = cmul(v[4], make_float2(c1, s1));
    v[7] = cmul(v[7], make_float2(c2, s2));
    v[5] = cmul(v[5], make_float2(c2, s2));
    v[8] = cmul(v[8], make_float2(c4, s4));
    dft3(v[0], v[1], v[2]);
    dft3(v[3], v[4], v[5]);
    dft3(v[6], v[7], v[8]);
    // v[3 k1 + k2] holds frequency k1 + 3 k2
    float2 t = v[1];
    v[1] = v[3];
    v[3] = t;
    t = v[2];
    v[2] = v[6];
    v[6] = t;
    t = v[5];
    v[5] = v[7];
    v[7] = t;
  }
}

// One Stockham pass over the tile's columns: loads by load(position), stores by
// store(position, value). L lanes share a column, lane j owning butterflies
// j, j + L, ... The barrier between lets the stores go to the loads' own tile.
template <int R, int L, class Load, class Store>
static __device__ __forceinline__ void col_pass(const ColPlan& p, int ns, int j, const float2* tw, Load load, Store store) {
  constexpr int NB = (kColValues + R - 1) / R;
  const int m = p.n / R, step = m / ns * p.scale;
  const unsigned inv = (1u << 20) / (unsigned)ns + 1;  // i / ns for i < n / R: i ns < 2^20
  // each pass's addresses are its own: hoisted out of the loop over the passes
  // those of every radix would be held at once
  asm volatile("" : "+v"(j));
  float2 v[NB][R];
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const int i = j + q * L;
    if (i >= m) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) v[q][r] = load(i + r * m);
  }
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const int i = j + q * L;
    if (i >= m) continue;
    const int k = i - ns * (int)(((unsigned)i * inv) >> 20);
    if (ns > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) v[q][r] = cmul(v[q][r], tw[r * k * step]);
    }
    dft<R>(v[q]);
    __builtin_amdgcn_sched_barrier(0);  // one butterfly's twiddles in registers at a time
  }
  __syncthreads();
  asm volatile("" : "+v"(j));
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const int i = j + q * L;
    if (i >= m) continue;
    const int k = i - ns * (int)(((unsigned)i * inv) >> 20);
    const int o = (i - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) store(o + r * ns, v[q][r]);
  }
  __syncthreads();
}

template <int L, class Load, class Store>
static __device__ __forceinline__ void col_pass_any(const ColPlan& p, int radix, int ns, int j, const float2* tw, Load load,
                                             Store store) {
  switch (radix) {  // uniform
    case 2: col_pass<2, L>(p, ns, j, tw, load, store); break;
    case 3: col_pass<3, L>(p, ns, j, tw, load, store); break;
    case 4: col_pass<4, L>(p, ns, j, tw, load, store); break;
    case 5: col_pass<5, L>(p, ns, j, tw, load, store); break;
    case 6: col_pass<6, L>(p, ns, j, tw, load, store); break;
    case 8: col_pass<8, L>(p, ns, j, tw, load, store); break;
    default: col_pass<9, L>(p, ns, j, tw, load, store); break;
  }
}

// consecutive tiles on one XCD (workgroups are dealt round-robin over the 8)
static __device__ __forceinline__ int64_t xcd_tile(int64_t per) { return (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8; }

__global__ void col_table_kernel(int n, float2* __restrict__ tw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s, c;
  sincospi(2.0 * (double)i / (double)n, &s, &c);
  tw[i] = make_float2((float)c, (float)s);
}

// z: out[b][z'][ky][kx] = sum_kz tomo conj(F) e^{2 pi i kz (z' + vz0) / nz}, with
// F(kz) = sum_z X2[b][z][ky][kx] e^{-2 pi i kz (p + z) / nz}, whose conjugate is
// the inverse transform of the conjugates. A tile is 16 (W) kx of one ky. The
// orientations of a tile are consecutive: its tomogram columns come from L2.
template <int L>
__global__ void __launch_bounds__(kColThreads, 4) ts_z_kernel(ColPlan p, const float2* __restrict__ twg,
                                                              const float2* __restrict__ X2, int zp, int tz, int pz,
                                                              const float2* __restrict__ tomo, int ny, int cx,
                                                              int pitch, int vz0, int vz, int nb, int64_t tiles,
                                                              int64_t per, float2* __restrict__ out) {
  constexpr int W = kColThreads / L;
  extern __shared__ float2 lds[];
  float2 *tw = lds, *tile = lds + p.n;
  const int64_t w = xcd_tile(per);
  if (w >= tiles * nb) return;
  const int b = (int)(w % nb);
  const int kt = (int)((w / nb) % (pitch / W)), ky = (int)((w / nb) / (pitch / W));
  const int t = threadIdx.x, c = t % W, j = t / W, kx = kt * W + c;
  const bool ok = kx < cx;
  for (int i = t; i < p.n; i += kColThreads) tw[i] = twg[i];
  const int64_t plane = (int64_t)ny * cx, col = (int64_t)ky * cx + (ok ? kx : cx - 1);
  const float2* xb = X2 + (int64_t)b * zp * plane + col;
  for (int z = j; z < p.n; z += L) {
    float2 v = make_float2(0.0f, 0.0f);
    if ((unsigned)(z - pz) < (unsigned)tz) {
      const float2 a = xb[(z - pz) * plane];
      v = make_float2(a.x, -a.y);
    }
    tile[z * W + c] = v;
  }
  __syncthreads();
  auto load = [&](int z) { return tile[z * W + c]; };
  auto store = [&](int z, float2 v) { tile[z * W + c] = v; };
  for (int half = 0; half < 2; ++half) {
    if (half == 1) {
      for (int z = j; z < p.n; z += L) tile[z * W + c] = cmul(tomo[z * plane + col], tile[z * W + c]);
      __syncthreads();
    }
    int ns = 1;
    for (int s = 0; s < p.count; ++s) {
      col_pass_any<L>(p, p.radix[s], ns, j, tw, load, store);
      ns *= p.radix[s];
    }
  }
  if (!ok) return;
  float2* ob = out + ((int64_t)b * vz * ny + ky) * pitch + kx;
  for (int z = j; z < vz; z += L) ob[(int64_t)z * ny * pitch] = tile[(z + vz0) * W + c];
}

// y, in place: T[b][z'][y][kx] for y in [vy0, vy0 + vy) from T[b][z'][ky][kx]
template <int L>
__global__ void __launch_bounds__(kColThreads, 4) ts_y_kernel(ColPlan p, const float2* __restrict__ twg, int pitch,
                                                              int vy0, int vy, int64_t tiles, int64_t per,
                                                              float2* __restrict__ T) {
  constexpr int W = kColThreads / L;
  extern __shared__ float2 lds[];
  float2 *tw = lds, *tile = lds + p.n;
  const int64_t w = xcd_tile(per);
  if (w >= tiles) return;
  const int kt = (int)(w % (pitch / W));
  const int64_t zb = w / (pitch / W);
  const int t = threadIdx.x, c = t % W, j = t / W;
  for (int i = t; i < p.n; i += kColThreads) tw[i] = twg[i];
  float2* tb = T + zb * p.n * pitch + kt * W + c;
  for (int y = j; y < p.n; y += L) tile[y * W + c] = tb[(int64_t)y * pitch];
  __syncthreads();
  auto load = [&](int y) { return tile[y * W + c]; };
  auto store = [&](int y, float2 v) { tile[y * W + c] = v; };
  int ns = 1;
  for (int s = 0; s < p.count; ++s) {
    col_pass_any<L>(p, p.radix[s], ns, j, tw, load, store);
    ns *= p.radix[s];
  }
  for (int y = vy0 + j; y < vy0 + vy; y += L) tb[(int64_t)y * pitch] = tile[y * W + c];
}

// x: cc[b][z'][y'][x'] of the valid area, from rows T[b][z'][y' + vy0][kx], and
// the sums of each tile's values and squares. With h = nx / 2 (p.n),
//   x[2 j] + i x[2 j + 1] = sum_{k < h} Z(k) e^{2 pi i j k / h},
//   Z(k) = X(k) + conj X(h - k) + i e^{2 pi i k / nx} (X(k) - conj X(h - k)).
// A tile is W rows (y', z'); its pitch in LDS is odd, as global memory is
// read and written along the row.
template <int L>
__global__ void __launch_bounds__(kColThreads, 4) ts_x_kernel(ColPlan p, const float2* __restrict__ twg,
                                                              const float2* __restrict__ T, int ny, int pitch,
                                                              int vx0, int vx, int vy0, int vy, int vz,
                                                              float* __restrict__ cc, double* __restrict__ part) {
  constexpr int W = kColThreads / L, P = W + 1;
  extern __shared__ float2 lds[];
  const int h = p.n;
  float2 *tw = lds, *tile = lds + 2 * h;
  const int b = blockIdx.y, t = threadIdx.x, wave = t / kWave, lane = t % kWave;
  const int rows = vy * vz, r0 = blockIdx.x * W;
  for (int i = t; i < 2 * h; i += kColThreads) tw[i] = twg[i];
  for (int q = wave; q < W; q += kColThreads / kWave) {
    const int r = r0 + q;
    if (r >= rows) break;  // uniform over the wave
    const float2* tb = T + (((int64_t)b * vz + r / vy) * ny + (r % vy + vy0)) * pitch;
    for (int k = lane; k <= h; k += kWave) {
      float2 v = tb[k];
      if (k == 0 || k == h) v.y = 0.0f;  // real for a real map
      tile[k * P + q] = v;
    }
  }
  __syncthreads();
  // columns of rows past the last hold what LDS held and are not written
  const int c = t % W, j = t / W;
  // X(k) and X(h - k) make Z(k) and Z(h - k) in place: one lane has the pair
  for (int k = j; 2 * k <= h; k += L) {
    const float2 a = tile[k * P + c], m = tile[(h - k) * P + c];
    const float2 s = make_float2(a.x + m.x, a.y - m.y), d = muli(cmul(make_float2(a.x - m.x, a.y + m.y), tw[k]));
    // Z(h - k) = conj(s) + i w(h - k) (m - conj a), w(h - k) = -conj w(k)
    tile[k * P + c] = cadd(s, d);
    if (k > 0) tile[(h - k) * P + c] = make_float2(s.x - d.x, d.y - s.y);
  }
  __syncthreads();
  auto load = [&](int k) { return tile[k * P + c]; };
  auto store = [&](int k, float2 v) { tile[k * P + c] = v; };
  int ns = 1;
  for (int s = 0; s < p.count; ++s) {
    col_pass_any<L>(p, p.radix[s], ns, j, tw, load, store);
    ns *= p.radix[s];
  }
  double v[2] = {0.0, 0.0};
  for (int q = wave; q < W; q += kColThreads / kWave) {
    const int r = r0 + q;
    if (r >= rows) break;
    float* ob = cc + ((int64_t)b * rows + r) * vx;
    for (int x = lane; x < vx; x += kWave) {
      const float2 z = tile[((x + vx0) / 2) * P + q];
      const float a = ((x + vx0) & 1) ? z.y : z.x;
      ob[x] = a;
      v[0] += (double)a;
      v[1] += (double)a * (double)a;
    }
  }
  block_sum<2>(v);
  if (t == 0) {
    double* o = part + 2 * ((int64_t)b * gridDim.x + blockIdx.x);
    o[0] = v[0];
    o[1] = v[1];
  }
}

// fewest passes over {9, 8, 6, 5, 4, 3, 2}, then the largest radices first;
// false if n has another factor
static bool col_radices(int n, ColPlan* p) {
  static const int kR[] = {9, 8, 6, 5, 4, 3, 2};
  p->n = n;
  p->scale = 1;
  for (int want = 1; want <= 8; ++want) {
    int at[8], d = 0, rest[9];
    rest[0] = n;
    at[0] = 0;
    // depth-first over non-increasing radices
    while (d >= 0) {
      if (d == want) {
        if (rest[d] == 1) {
          p->count = want;
          for (int k = 0; k < want; ++k) p->radix[k] = kR[at[k]];
          return true;
        }
        ++at[--d];
        continue;
      }
      while (at[d] < 7 && rest[d] % kR[at[d]] != 0) ++at[d];
      if (at[d] == 7) {
        if (--d >= 0) ++at[d];
        continue;
      }
      rest[d + 1] = rest[d] / kR[at[d]];
      if (d + 1 < want) at[d + 1] = at[d];
      ++d;
    }
  }
  return false;
}

// lanes a column: 32 (tiles of 16 columns, 128-byte segments) where the tile
// fits the LDS of a workgroup, else 64; 0 where neither does: along y and z up to
// 478 and 903 voxels, along x up to 852 and 1,476 (its columns are half as long)
static int col_lanes(int n, int table, bool padded) {
  for (int L : {32, 64}) {
    const int W = kColThreads / L;
    const size_t need = sizeof(float2) * ((size_t)table + (size_t)(padded ? (n + 1) * (W + 1) : n * W));
    if (need <= kColLds && n <= kColValues * L) return L;
  }
  return 0;
}

static const float2* col_table(emc_ctx* ctx, int n) {
  char key[32];
  snprintf(key, sizeof(key), "col_tw_%d", n);
  auto it = ctx->scratch.find(key);
  const bool fresh = it == ctx->scratch.end() || !it->second.ptr;
  float2* tw = (float2*)scratch(ctx, key, sizeof(float2) * n);
  if (fresh) {
    hipLaunchKernelGGL(col_table_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, ctx->stream, n, tw);
    EMC_HIP(hipGetLastError());
  }
  return tw;
}

constexpr int kPitch = 16;  // rows of the product are padded to whole tiles of either width

bool ts_inverse_supported(const int cd[3]) {
  ColPlan p;
  return cd[0] % 2 == 0 && col_radices(cd[0] / 2, &p) && col_radices(cd[1], &p) && col_radices(cd[2], &p) &&
         col_lanes(cd[0] / 2, cd[0], true) && col_lanes(cd[1], cd[1], false) && col_lanes(cd[2], cd[2], false);
}

int64_t ts_inverse_elems(const int cd[3], const int vd[3]) {
  return (int64_t)vd[2] * cd[1] * (ceil_div(cd[0] / 2 + 1, kPitch) * kPitch);
}

int ts_inverse_blocks(const int cd[3], const int vd[3]) {
  return ceil_div(vd[1] * vd[2], kColThreads / col_lanes(cd[0] / 2, cd[0], true));
}

void ts_inverse(emc_ctx* ctx, const float2* X2, int zp, int tz, int pz, const float2* tomo, const int cd[3],
                const int vlow[3], const int vd[3], int nb, float2* T, float* cc, double* part) {
  const int cx = cd[0] / 2 + 1, ny = cd[1], pitch = ceil_div(cx, kPitch) * kPitch;
  ColPlan px, py, pz_;
  EMC_REQUIRE(col_radices(cd[0] / 2, &px) && col_radices(ny, &py) && col_radices(cd[2], &pz_), "edge not supported");
  px.scale = 2;
  const float2 *wx = col_table(ctx, cd[0]), *wy = col_table(ctx, ny), *wz = col_table(ctx, cd[2]);
  {
    const int L = col_lanes(cd[2], cd[2], false), W = kColThreads / L;
    const int64_t tiles = (int64_t)ny * (pitch / W), per = ceil_div(tiles * nb, 8);
    const size_t lds = sizeof(float2) * (size_t)cd[2] * (W + 1);
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(8 * per), dim3(kColThreads), lds, ctx->stream, pz_, wz, X2, zp, tz, pz, tomo, ny,
                         cx, pitch, vlow[2], vd[2], nb, tiles, per, T);
    };
    L == 32 ? launch(ts_z_kernel<32>) : launch(ts_z_kernel<64>);
    EMC_HIP(hipGetLastError());
  }
  {
    const int L = col_lanes(ny, ny, false), W = kColThreads / L;
    const int64_t tiles = (int64_t)nb * vd[2] * (pitch / W), per = ceil_div(tiles, 8);
    const size_t lds = sizeof(float2) * (size_t)ny * (W + 1);
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(8 * per), dim3(kColThreads), lds, ctx->stream, py, wy, pitch, vlow[1], vd[1],
                         tiles, per, T);
    };
    L == 32 ? launch(ts_y_kernel<32>) : launch(ts_y_kernel<64>);
    EMC_HIP(hipGetLastError());
  }
  {
    const int h = cd[0] / 2, L = col_lanes(h, cd[0], true), W = kColThreads / L;
    const size_t lds = sizeof(float2) * ((size_t)cd[0] + (size_t)(h + 1) * (W + 1));
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(ts_inverse_blocks(cd, vd), nb), dim3(kColThreads), lds, ctx->stream, px, wx,
                         (const float2*)T, ny, pitch, vlow[0], vd[0], vlow[1], vd[1], vd[2], cc, part);
    };
    L == 32 ? launch(ts_x_kernel<32>) : launch(ts_x_kernel<64>);
    EMC_HIP(hipGetLastError());
  }
}

}  // namespace emc
