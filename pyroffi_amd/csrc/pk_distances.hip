// Output-shaped sphere distance kernels for gfx950: the reference FFI targets
// whose result is a full distance tensor ([B, K, M] per sphere, [B, N, M] per
// link over mixed obstacle kinds), and the JAX path's distance conventions.
//
// The flat kernels (per-sphere outputs, rows from placed spheres, and rows whose
// tables do not fit the LDS) are bound by the output write: a grid-stride loop gives
// consecutive lanes consecutive output elements (coalesced 256-byte rows per wave),
// and the inputs of an element (one robot sphere, one obstacle) come through the
// caches.  Rows from link poses (link_rows_kernel, self_rows_kernel) take a handful
// of sphere tests an element and are bound by those: they place a configuration's
// spheres into the LDS once.  The fused sweep in pk_collision.hip remains the fast
// path for sphere-only worlds and reduced outputs.
#include "pk_geom.h"
#include "pk_model.h"

#include <algorithm>

namespace pk {

constexpr float kNoSphere = 1e9f;  // the reference's "no sphere" value

// out[b, k, m] = distance of robot sphere k to obstacle m; padding (r < 0)
// writes 1e9 (_collision_cuda_kernel.cu:64-161).
__global__ __launch_bounds__(256) void world_sphere_full_kernel(const float* __restrict__ sc,
                                                                const float* __restrict__ sr,
                                                                long long BK, WorldPrims w,
                                                                float* __restrict__ out) {
  const long long M = w.total();
  const long long total = BK * M;
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long row = f / M;
    const int m = static_cast<int>(f - row * M);
    const float r = sr[row];
    float d = kNoSphere;
    if (r >= 0.f) d = dist_sphere_obstacle(sc[row], sc[BK + row], sc[2 * BK + row], r, w, m);
    __builtin_nontemporal_store(d, out + f);
  }
}

// out[b, n, m] = min over the link's sphere slots k = s * N + n (padding
// skipped, 1e9 when none is real) of the distance to obstacle m, for worlds
// with non-sphere obstacles (_collision_cuda_kernel.cu:169-407).
__global__ __launch_bounds__(256) void world_reduced_mixed_kernel(const float* __restrict__ sc,
                                                                  const float* __restrict__ sr,
                                                                  long long B, int K, int S, int N,
                                                                  WorldPrims w, float* __restrict__ out) {
  const long long M = w.total();
  const long long BK = B * K;
  const long long total = B * N * M;
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long bn = f / M;
    const int m = static_cast<int>(f - bn * M);
    const long long b = bn / N;
    const int n = static_cast<int>(bn - b * N);
    float best = kNoSphere;
    for (int s = 0; s < S; ++s) {
      const long long k = b * K + static_cast<long long>(s) * N + n;
      const float r = sr[k];
      if (r < 0.f) continue;
      best = fminf(best, dist_sphere_obstacle(sc[k], sc[BK + k], sc[2 * BK + k], r, w, m));
    }
    __builtin_nontemporal_store(best, out + f);
  }
}

// The JAX distance of two spheres (src/pyroffi/collision/_geometry_pairs.py:59-68
// with the 1e-6 added to each component inside the norm, _utils.py:45):
// |(p2 - p1) + 1e-6| - (r1 + r2).  Padding radii (-1e9) take part as they do
// in JAX and make the distance about +1e9.
__device__ __forceinline__ float jax_sphere_dist(float x1, float y1, float z1, float r1, float x2, float y2,
                                                 float z2, float r2) {
  const float dx = (x2 - x1) + 1e-6f, dy = (y2 - y1) + 1e-6f, dz = (z2 - z1) + 1e-6f;
  return sqrtf(dx * dx + dy * dy + dz * dz) - (r1 + r2);
}

// ---------------------------------------------------------------------------
// Per-link distances from link poses, out[b, l, m] = min over the link's
// spheres of the distance to obstacle m, in both conventions.
//
// An output element takes a handful of sphere tests and four bytes of write,
// so the work is the tests, not the write.  With one lane per element placing
// the link's spheres for itself (33 flop a sphere, padding slots included) the
// placement was most of the kernel: 403 us for 4099 Fetch configurations x 200
// obstacles (28 slots a link, 6.5 of them real), 410 us for 8191 UR5 ones x 195
// mixed obstacles.  Here a workgroup sorts the table once (by radius within a
// link, padding folded), places a configuration's spheres into LDS once, and
// its lanes run over (link, obstacle) with the spheres as near-broadcast LDS
// reads; spheres of one radius share a square root (sqrt and the subtraction
// are monotone, so the minimum is the same).  Obstacle kinds are taken one
// after the other, so the lanes of a wave test the same kind.  (The calls at
// those sizes: both collision residuals of Fetch 617 -> 163 us, the distances
// written as costs; the mixed world of UR5 491 -> 198 us.)
// ---------------------------------------------------------------------------

constexpr int kRowThreads = 256;
constexpr int kRowSlots = 2048;  // L * S slots the LDS tables hold (two float4 each)

// Activation of a distance into a collision cost: min(c(d), 0) * weight with
// c = d - half below zero, else quad (d - margin)^2, d capped at the margin
// (colldist_from_sdf).
struct RowCost {
  int on;
  float margin, half, quad, weight;
};

__device__ __forceinline__ float row_cost(const RowCost& c, float dist) {
  const float d = fminf(dist, c.margin);
  const float v = d < 0.f ? d - c.half : c.quad * ((d - c.margin) * (d - c.margin));
  return fminf(v, 0.f) * c.weight;
}

struct RowArgs {
  const float* poses;  // (B, L, 7)
  long long batch;
  int n_links, s_per_link;
  const float* table;  // (L, S, 4) link-frame spheres
  WorldPrims w;
  int parts;           // workgroups that share one configuration's rows
  RowCost cost;        // written instead of the distance when on
  float* out;
};

// Two floats' minimum that skips NaN, for values that are never negative: as
// unsigned integers, where every NaN is above +inf.
__device__ __forceinline__ unsigned min_bits(unsigned m, float v) { return min(m, __float_as_uint(v)); }

// Same-radius runs: the square root and the radius are applied when the radius
// changes.  `r` of the run that m2 belongs to.
template <bool JAX>
__device__ __forceinline__ float row_spheres(const float4* pos, int n, const float* o, float best) {
  const float ox = o[0], oy = o[1], oz = o[2], orad = o[3];
  if (n == 0) return best;
  unsigned m2 = 0x7f800000u;
  float r = pos[0].w;
  for (int i = 0; i < n; ++i) {
    const float4 c = pos[i];
    if (c.w != r) {
      best = fminf(best, sqrtf(__uint_as_float(m2)) - (r + orad));
      m2 = 0x7f800000u;
      r = c.w;
    }
    // The JAX path adds its bias to (obstacle - sphere).
    const float dx = JAX ? (ox - c.x) + 1e-6f : c.x - ox;
    const float dy = JAX ? (oy - c.y) + 1e-6f : c.y - oy;
    const float dz = JAX ? (oz - c.z) + 1e-6f : c.z - oz;
    m2 = min_bits(m2, dx * dx + dy * dy + dz * dz);
  }
  return fminf(best, sqrtf(__uint_as_float(m2)) - (r + orad));
}

__device__ __forceinline__ float row_capsule(const float4* pos, int n, const float* o, float best) {
  const float ax = o[0], ay = o[1], az = o[2];
  const float ux = o[3] - ax, uy = o[4] - ay, uz = o[5] - az, rad = o[6];
  const float uu = ux * ux + uy * uy + uz * uz;
  const float inv = uu > 1e-12f ? 1.f / uu : 0.f;  // a point: t = 0
  if (n == 0) return best;
  unsigned m2 = 0x7f800000u;
  float r = pos[0].w;
  for (int i = 0; i < n; ++i) {
    const float4 c = pos[i];
    if (c.w != r) {
      best = fminf(best, sqrtf(__uint_as_float(m2)) - (r + rad));
      m2 = 0x7f800000u;
      r = c.w;
    }
    const float wx = c.x - ax, wy = c.y - ay, wz = c.z - az;
    const float t = fminf(fmaxf((wx * ux + wy * uy + wz * uz) * inv, 0.f), 1.f);
    const float dx = wx - t * ux, dy = wy - t * uy, dz = wz - t * uz;
    m2 = min_bits(m2, dx * dx + dy * dy + dz * dz);
  }
  return fminf(best, sqrtf(__uint_as_float(m2)) - (r + rad));
}

// KIND of WorldPrims (0 spheres, 1 capsules, 2 boxes, 3 half-spaces): rows of
// obstacles [0, count) of that kind, written at column `col` of the M.
template <int KIND, bool JAX>
__device__ __forceinline__ void kind_rows(const RowArgs& a, const float4* pos, const int* cnt, int part,
                                          long long row0, int M, int col) {
  constexpr int width = KIND == 0 ? 4 : (KIND == 1 ? 7 : (KIND == 2 ? 15 : 6));
  const float* data = KIND == 0 ? a.w.data[0] : (KIND == 1 ? a.w.data[1] : (KIND == 2 ? a.w.data[2] : a.w.data[3]));
  const int n_obs = KIND == 0 ? a.w.count[0] : (KIND == 1 ? a.w.count[1] : (KIND == 2 ? a.w.count[2] : a.w.count[3]));
  if (n_obs == 0) return;
  const int S = a.s_per_link;
  // Lane strides of (link, obstacle), without a division in the loop.
  const int step = kRowThreads * a.parts;
  const int step_l = step / n_obs, step_m = step - step_l * n_obs;
  const int f0 = part * kRowThreads + static_cast<int>(threadIdx.x);
  int l = f0 / n_obs, m = f0 - l * n_obs;
  while (l < a.n_links) {
    const float* o = data + static_cast<long long>(width) * m;
    const float4* p = pos + l * S;
    const int n = cnt[l];
    float best = JAX ? INFINITY : kNoSphere;
    if (KIND == 0) {
      best = row_spheres<JAX>(p, n, o, best);
    } else if (KIND == 1) {
      best = row_capsule(p, n, o, best);
    } else {
      float obs[width];
#pragma unroll
      for (int i = 0; i < width; ++i) obs[i] = o[i];
      for (int i = 0; i < n; ++i) {
        const float4 c = p[i];
        best = fminf(best, KIND == 2 ? dist_sphere_box(c.x, c.y, c.z, c.w, obs)
                                     : dist_sphere_halfspace(c.x, c.y, c.z, c.w, obs));
      }
    }
    if (a.cost.on) best = row_cost(a.cost, best);
    __builtin_nontemporal_store(best, a.out + (row0 + l) * M + col + m);
    l += step_l;
    m += step_m;
    if (m >= n_obs) { m -= n_obs; ++l; }
  }
}

// The same rows with a wave per (link, 64 T obstacles): each lane keeps T
// obstacles in registers and every sphere is one broadcast LDS read for all of
// them, where kind_rows reads it per element and loads the obstacle per link.
// Links are taken by falling number of spheres, so the waves' shares are even.
template <int KIND, bool JAX, int T>
__device__ __forceinline__ void wave_rows(const RowArgs& a, const float4* pos, const int* cnt, const int* order,
                                          int part, long long row0, int M, int col) {
  constexpr int width = KIND == 0 ? 4 : (KIND == 1 ? 7 : 15);
  const float* data = KIND == 0 ? a.w.data[0] : (KIND == 1 ? a.w.data[1] : a.w.data[2]);
  const int n_obs = KIND == 0 ? a.w.count[0] : (KIND == 1 ? a.w.count[1] : a.w.count[2]);
  const int lane = threadIdx.x % kWave;
  const int worker = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) + part * (kRowThreads / kWave);
  const int n_workers = a.parts * (kRowThreads / kWave);
  const int S = a.s_per_link, L = a.n_links;
  const int n_chunks = (n_obs + kWave * T - 1) / (kWave * T);
  float o[T][width], inv[T];
  int held = -1;
  for (int task = worker; task < L * n_chunks; task += n_workers) {
    const int chunk = task / L;  // few chunks: the obstacles stay for most tasks
    const int l = __builtin_amdgcn_readfirstlane(order[task - chunk * L]);
    if (chunk != held) {
      held = chunk;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float* p = data + static_cast<long long>(width) * min((chunk * T + t) * kWave + lane, n_obs - 1);
#pragma unroll
        for (int c = 0; c < width; ++c) o[t][c] = p[c];
        if (KIND == 1) {  // segment end b -> direction, and 1 / |b - a|^2 (0 for a point)
#pragma unroll
          for (int c = 0; c < 3; ++c) o[t][3 + c] -= o[t][c];
          const float uu = o[t][3] * o[t][3] + o[t][4] * o[t][4] + o[t][5] * o[t][5];
          inv[t] = uu > 1e-12f ? 1.f / uu : 0.f;
        }
      }
    }
    const int n = __builtin_amdgcn_readfirstlane(cnt[l]);
    const float4* p = pos + l * S;
    float best[T];
    unsigned m2[T];
#pragma unroll
    for (int t = 0; t < T; ++t) { best[t] = JAX ? INFINITY : kNoSphere; m2[t] = 0x7f800000u; }
    float r = n > 0 ? p[0].w : 0.f;
    auto close_run = [&]() {  // a run of equal radii ends: its square roots
      if (KIND == 2) return;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        best[t] = fminf(best[t], sqrtf(__uint_as_float(m2[t])) - (r + o[t][KIND == 1 ? 6 : 3]));
        m2[t] = 0x7f800000u;
      }
    };
    for (int i = 0; i < n; ++i) {
      const float4 c = p[i];
      if (KIND != 2 && __builtin_amdgcn_readfirstlane(__float_as_int(c.w)) !=
                           __builtin_amdgcn_readfirstlane(__float_as_int(r))) {
        close_run();
        r = c.w;
      }
#pragma unroll
      for (int t = 0; t < T; ++t) {
        if (KIND == 0) {
          const float dx = JAX ? (o[t][0] - c.x) + 1e-6f : c.x - o[t][0];
          const float dy = JAX ? (o[t][1] - c.y) + 1e-6f : c.y - o[t][1];
          const float dz = JAX ? (o[t][2] - c.z) + 1e-6f : c.z - o[t][2];
          m2[t] = min_bits(m2[t], dx * dx + dy * dy + dz * dz);
        } else if (KIND == 1) {
          const float wx = c.x - o[t][0], wy = c.y - o[t][1], wz = c.z - o[t][2];
          const float s = fminf(fmaxf((wx * o[t][3] + wy * o[t][4] + wz * o[t][5]) * inv[t], 0.f), 1.f);
          const float dx = wx - s * o[t][3], dy = wy - s * o[t][4], dz = wz - s * o[t][5];
          m2[t] = min_bits(m2[t], dx * dx + dy * dy + dz * dz);
        } else {
          best[t] = fminf(best[t], dist_sphere_box(c.x, c.y, c.z, c.w, o[t]));
        }
      }
    }
    if (n > 0) close_run();
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int m = (chunk * T + t) * kWave + lane;
      if (a.cost.on) best[t] = row_cost(a.cost, best[t]);
      if (m < n_obs) __builtin_nontemporal_store(best[t], a.out + (row0 + l) * M + col + m);
    }
  }
}

// Rows of one obstacle kind.  A wave per link pays where it has two obstacles a lane:
// it takes whole passes of 128, so that its time steps where lane by lane it grows.
// 4096 configurations, lane by lane / a wave per link, us, 64, 65, 96, 128, 129, 256
// obstacles: spheres, Fetch 46 / 48, 59 / 49, 68 / 50, 72 / 49, 84 / 63, 122 / 63, UR5 26
// / 30, 30 / 31, 36 / 31, 42 / 31, 46 / 39, 69 / 39; capsules, Fetch 51 / 56, 66 / 58, 76
// / 58, 81 / 58, 96 / 90, 140 / 90, UR5 29 / 34, 34 / 35, 41 / 35, 47 / 35, 51 / 55, 79 /
// 56; boxes, which hold fifteen registers an obstacle and share no square root, Fetch 51
// / 78, 67 / 79, 76 / 80, 80 / 80, 95 / 136, 139 / 136, Baxter 43 / 57, 49 / 59, 60 / 59,
// 73 / 58, 81 / 103, 137 / 105 (112 obstacles 71 / 59): only passes at least seven eighths
// full pay.  Half-spaces, of which a scene has a handful, stay lane by lane.
constexpr int kWaveRowsMin = 65;

__device__ __forceinline__ bool box_waves_pay(int n) {
  const int places = (n + 2 * kWave - 1) / (2 * kWave) * (2 * kWave);
  return 8 * n >= 7 * places;
}

template <int KIND, bool JAX>
__device__ __forceinline__ void rows_of_kind(const RowArgs& a, const float4* pos, const int* cnt, const int* order,
                                             int part, long long row0, int M, int col) {
  const int n = KIND == 0 ? a.w.count[0] : (KIND == 1 ? a.w.count[1] : (KIND == 2 ? a.w.count[2] : a.w.count[3]));
  if constexpr (KIND < 3) {
    if (n >= kWaveRowsMin && (KIND != 2 || box_waves_pay(n))) {
      if (KIND != 0 || n <= 2 * kWave) wave_rows<KIND, JAX, 2>(a, pos, cnt, order, part, row0, M, col);
      else wave_rows<KIND, JAX, KIND == 0 ? 4 : 2>(a, pos, cnt, order, part, row0, M, col);
      return;
    }
  }
  kind_rows<KIND, JAX>(a, pos, cnt, part, row0, M, col);
}

template <bool JAX>
__global__ __launch_bounds__(kRowThreads) void link_rows_kernel(RowArgs a) {
  extern __shared__ float4 rsmem[];
  const int L = a.n_links, S = a.s_per_link, LS = L * S;
  float4* loc = rsmem;                             // sorted link-frame spheres, link l at l * S
  float4* pos = loc + LS;                          // the same in the world
  int* cnt = reinterpret_cast<int*>(pos + LS);     // spheres of each link
  int* order = cnt + L;                            // links by falling number of spheres
  const int tid = threadIdx.x;
  for (int t = tid; t < LS; t += kRowThreads) {
    const float* s = a.table + 4LL * t;
    pos[t] = make_float4(s[0], s[1], s[2], s[3]);  // staged here until sorted
  }
  for (int l = tid; l < L; l += kRowThreads) cnt[l] = 0;
  __syncthreads();
  // Which slots count.  CUDA conventions: those with r >= 0 (or NaN).  JAX:
  // padding takes part, but a slot equal to the one before it changes no
  // minimum, so of a run of padding one is kept.  A kept slot's place: larger
  // radii first, slot order within a radius (a NaN compares as smallest).
  for (int t = tid; t < LS; t += kRowThreads) {
    const int l = t / S, s = t - l * S;
    auto kept = [&](int i) {
      const float4 c = pos[l * S + i];
      if (!JAX) return !(c.w < 0.f);
      if (i == 0) return true;
      const float4 p = pos[l * S + i - 1];
      return !(c.x == p.x && c.y == p.y && c.z == p.z && c.w == p.w);
    };
    if (!kept(s)) continue;
    const float4 c = pos[t];
    auto above = [](float p, float q) { return p > q || (p == p && q != q); };
    int rank = 0;
    for (int i = 0; i < S; ++i) {
      const float r = pos[l * S + i].w;
      if ((above(r, c.w) || (!above(c.w, r) && i < s)) && kept(i)) ++rank;
    }
    loc[l * S + rank] = c;
    atomicAdd(&cnt[l], 1);
  }
  __syncthreads();
  for (int l = tid; l < L; l += kRowThreads) {
    int rank = 0;
    for (int i = 0; i < L; ++i) rank += cnt[i] > cnt[l] || (cnt[i] == cnt[l] && i < l);
    order[rank] = l;
  }
  __syncthreads();
  const int M = a.w.total();
  const long long n_items = a.batch * a.parts;
  for (long long item = blockIdx.x; item < n_items; item += gridDim.x) {
    const long long b = item / a.parts;
    const int part = static_cast<int>(item - b * a.parts);
    for (int t = tid; t < LS; t += kRowThreads) {
      const int l = t / S;
      if (t - l * S < cnt[l]) {
        const float* T = a.poses + (b * L + l) * 7;
        const float4 c = loc[t];
        float x, y, z;
        quat_rotate(T[0], T[1], T[2], T[3], c.x, c.y, c.z, x, y, z);
        pos[t] = make_float4(x + T[4], y + T[5], z + T[6], c.w);
      }
    }
    __syncthreads();
    int col = 0;
    rows_of_kind<0, JAX>(a, pos, cnt, order, part, b * L, M, col);
    if (!JAX) {
      col += a.w.count[0];
      rows_of_kind<1, false>(a, pos, cnt, order, part, b * L, M, col);
      col += a.w.count[1];
      rows_of_kind<2, false>(a, pos, cnt, order, part, b * L, M, col);
      col += a.w.count[2];
      rows_of_kind<3, false>(a, pos, cnt, order, part, b * L, M, col);
    }
    __syncthreads();
  }
}

// Same-slot self distances (jax_self_kernel's) with each configuration's
// spheres placed once into LDS: `tile` configurations at a time, lanes over
// (configuration, pair).  A link's slots past its last distinct one repeat it,
// so a pair stops at the longer of its two links.  (One lane per pair placing
// both links' 28 slots took 30 us for 4099 Fetch configurations.)
struct SelfRowArgs {
  const float* poses;
  long long batch;
  int n_links, s_per_link;
  const float* table;
  const int* pair_i;
  const int* pair_j;
  int n_pairs, tile;
  RowCost cost;
  float* out;
};

__global__ __launch_bounds__(kRowThreads) void self_rows_kernel(SelfRowArgs a) {
  extern __shared__ float4 rsmem[];
  const int L = a.n_links, S = a.s_per_link, LS = L * S, P = a.n_pairs;
  float4* loc = rsmem;                                    // link-frame slots
  float4* pos = loc + LS;                                 // tile x LS in the world
  int* cnt = reinterpret_cast<int*>(pos + a.tile * LS);   // slots of each link up to its last distinct one
  int* pairs = cnt + L;                                   // link i | link j << 16, -1 invalid
  const int tid = threadIdx.x;
  for (int t = tid; t < LS; t += kRowThreads) {
    const float* s = a.table + 4LL * t;
    loc[t] = make_float4(s[0], s[1], s[2], s[3]);
  }
  for (int l = tid; l < L; l += kRowThreads) cnt[l] = S > 0 ? 1 : 0;
  for (int p = tid; p < P; p += kRowThreads) {
    const int i = a.pair_i[p], j = a.pair_j[p];
    pairs[p] = (i >= 0 && i < L && j >= 0 && j < L) ? (i | (j << 16)) : -1;
  }
  __syncthreads();
  for (int t = tid; t < LS; t += kRowThreads) {
    const int l = t / S, s = t - l * S;
    if (s == 0) continue;
    const float4 c = loc[t], q = loc[t - 1];
    if (!(c.x == q.x && c.y == q.y && c.z == q.z && c.w == q.w)) atomicMax(&cnt[l], s + 1);
  }
  __syncthreads();
  const long long n_tiles = (a.batch + a.tile - 1) / a.tile;
  for (long long tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const long long b0 = tile * a.tile;
    const int nb = static_cast<int>(min(static_cast<long long>(a.tile), a.batch - b0));
    for (int t = tid; t < nb * LS; t += kRowThreads) {
      const int c = t / LS, k = t - c * LS, l = k / S;
      if (k - l * S >= cnt[l]) continue;
      const float* T = a.poses + ((b0 + c) * L + l) * 7;
      const float4 s = loc[k];
      float x, y, z;
      quat_rotate(T[0], T[1], T[2], T[3], s.x, s.y, s.z, x, y, z);
      pos[t] = make_float4(x + T[4], y + T[5], z + T[6], s.w);
    }
    __syncthreads();
    for (int t = tid; t < nb * P; t += kRowThreads) {
      const int c = t / P, en = pairs[t - c * P];
      float best = INFINITY;
      if (en >= 0) {
        const int li = en & 0xffff, lj = en >> 16;
        const int ni = cnt[li], nj = cnt[lj];
        const float4* pi = pos + c * LS + li * S;
        const float4* pj = pos + c * LS + lj * S;
        for (int s = 0; s < max(ni, nj); ++s) {
          const float4 u = pi[min(s, ni - 1)], v = pj[min(s, nj - 1)];
          best = fminf(best, jax_sphere_dist(u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w));
        }
      }
      if (a.cost.on) best = row_cost(a.cost, best);
      __builtin_nontemporal_store(best, a.out + b0 * P + t);
    }
    __syncthreads();
  }
}

// Where the kernels that place a configuration's spheres once pay against the flat
// ones, which place a link's slots for every element but have neither tables to sort
// nor barriers.  Flat / placed, us (JAX conventions; links x slots): 64 configurations
// among 128 obstacles Panda (13 x 18) 6 / 10, Fetch (17 x 28) 10 / 17; 1000 among 32, 64
// Panda 12 / 12, 19 / 14, UR5 (23 x 9) 11 / 10, 18 / 14, Fetch 20 / 21, 34 / 28, Baxter (44
// x 4) 10 / 13, 18 / 18; 16000 among 8, 16, 32 Panda 32 / 56, 60 / 60, 115 / 75, Fetch 60 /
// 82, 117 / 100, 224 / 120, Baxter 30 / 46, 57 / 64, 119 / 102.
inline bool placed_rows_pay(long long batch, int L, int S, int M) {
  const long long tests = static_cast<long long>(M) * S;  // of a link, padding included
  return M >= 24 && tests >= 192 && batch * L >= ((1LL << 23) + tests - 1) / tests;
}

// The same for the self pairs: 1000, 2000 and 4000 configurations Panda (66 pairs) 7 /
// 11, 9 / 11, 12 / 12, UR5 (231) 7 / 7, 10 / 9, 16 / 14, Fetch (120) 10 / 14, 15 / 14, 27 /
// 20, Baxter (903) 10 / 9, 18 / 14, 30 / 23.
inline bool placed_self_pays(long long batch, int S, int P) {
  const long long tests = static_cast<long long>(P) * S;
  return tests > 0 && batch >= ((1LL << 22) + tests - 1) / tests;
}

// False when that does not pay or the tables do not fit the LDS (jax_self_kernel then
// takes them).
static bool launch_self_rows(hipStream_t s, SelfRowArgs a) {
  const long long LS = static_cast<long long>(a.n_links) * a.s_per_link;
  if (LS > kRowSlots || a.n_links > kRowSlots || a.n_pairs > 8192) return false;
  if (!placed_self_pays(a.batch, a.s_per_link, a.n_pairs)) return false;
  // Enough configurations for two rounds of lanes, while their spheres take
  // at most 32 KiB.
  a.tile = std::max(1, std::min(2 * kRowThreads / a.n_pairs, LS > 0 ? static_cast<int>(2048 / LS) : 8));
  const size_t lds = sizeof(float4) * (1 + a.tile) * LS + sizeof(int) * (a.n_links + a.n_pairs);
  const unsigned grid = static_cast<unsigned>(std::min((a.batch + a.tile - 1) / a.tile, 256LL * 4));
  hipLaunchKernelGGL(self_rows_kernel, dim3(grid), dim3(kRowThreads), lds, s, a);
  return true;
}

// Launch of link_rows_kernel, or false when it does not pay or its tables do not fit
// the LDS.
// Four workgroups a CU loop over the configurations, which spreads the table's
// sorting; fewer configurations than that share each among workgroups.
template <bool JAX>
static bool launch_link_rows(hipStream_t s, RowArgs a) {
  const long long LS = static_cast<long long>(a.n_links) * a.s_per_link;
  const long long per = a.n_links * static_cast<long long>(a.w.total());
  // (Links without a slot have their two words each in the LDS all the same.)
  if (LS > kRowSlots || a.n_links > kRowSlots || per > 0x3fffffffLL) return false;
  if (!placed_rows_pay(a.batch, a.n_links, a.s_per_link, a.w.total())) return false;
  constexpr long long kGroups = 256LL * 4;
  long long parts = 1;
  if (a.batch < kGroups)
    parts = std::min((kGroups + a.batch - 1) / a.batch, (per + 4 * kRowThreads - 1) / (4 * kRowThreads));
  a.parts = static_cast<int>(parts);
  const size_t lds = sizeof(float4) * 2 * LS + sizeof(int) * 2 * a.n_links;
  const unsigned grid = static_cast<unsigned>(std::min(kGroups, a.batch * parts));
  hipLaunchKernelGGL((link_rows_kernel<JAX>), dim3(grid), dim3(kRowThreads), lds, s, a);
  return true;
}

// Centre of sphere slot s of link l for configuration b: T_l applied to the
// link-frame centre of the padded (L, S, 4) table.
__device__ __forceinline__ void placed(const float* __restrict__ poses, const float* __restrict__ table,
                                       long long b, int L, int S, int l, int s, float& x, float& y, float& z,
                                       float& r) {
  const float* T = poses + (b * L + l) * 7;
  const float* c = table + (static_cast<long long>(l) * S + s) * 4;
  quat_rotate(T[0], T[1], T[2], T[3], c[0], c[1], c[2], x, y, z);
  x += T[4];
  y += T[5];
  z += T[6];
  r = c[3];
}

// out[b, l, m] = min over slots s of jax_sphere_dist(sphere (l, s), world m)
// (RobotCollisionSpherized.compute_world_collision_distance,
// src/pyroffi/collision/_robot_collision.py:830-895).
__global__ __launch_bounds__(256) void jax_world_kernel(const float* __restrict__ poses, long long B, int L,
                                                        const float* __restrict__ table, int S,
                                                        const float* __restrict__ world, int M, RowCost cost,
                                                        float* __restrict__ out) {
  const long long total = B * L * static_cast<long long>(M);
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long bl = f / M;
    const int m = static_cast<int>(f - bl * M);
    const long long b = bl / L;
    const int l = static_cast<int>(bl - b * L);
    const float* o = world + 4 * m;
    float best = INFINITY;
    for (int s = 0; s < S; ++s) {
      float x, y, z, r;
      placed(poses, table, b, L, S, l, s, x, y, z, r);
      best = fminf(best, jax_sphere_dist(x, y, z, r, o[0], o[1], o[2], o[3]));
    }
    if (cost.on) best = row_cost(cost, best);
    __builtin_nontemporal_store(best, out + f);
  }
}

// out[b, p] = min over slots s of jax_sphere_dist(sphere (i_p, s), sphere (j_p, s)):
// the same-slot ("diagonal") pairs of
// RobotCollisionSpherized.compute_self_collision_distance
// (src/pyroffi/collision/_robot_collision.py:796-828).
__global__ __launch_bounds__(256) void jax_self_kernel(const float* __restrict__ poses, long long B, int L,
                                                       const float* __restrict__ table, int S,
                                                       const int* __restrict__ pair_i,
                                                       const int* __restrict__ pair_j, int P, RowCost cost,
                                                       float* __restrict__ out) {
  const long long total = B * static_cast<long long>(P);
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long b = f / P;
    const int p = static_cast<int>(f - b * P);
    const int li = pair_i[p], lj = pair_j[p];
    float best = INFINITY;
    if (li >= 0 && li < L && lj >= 0 && lj < L) {
      for (int s = 0; s < S; ++s) {
        float xi, yi, zi, ri, xj, yj, zj, rj;
        placed(poses, table, b, L, S, li, s, xi, yi, zi, ri);
        placed(poses, table, b, L, S, lj, s, xj, yj, zj, rj);
        best = fminf(best, jax_sphere_dist(xi, yi, zi, ri, xj, yj, zj, rj));
      }
    }
    if (cost.on) best = row_cost(cost, best);
    __builtin_nontemporal_store(best, out + f);
  }
}

// Capsule robot vs the world: out[b, n, m] for link capsule caps[:, b, n]
// (component-major [7, B, N]) (_collision_cuda_kernel.cu:203-407).
__global__ __launch_bounds__(256) void world_capsule_kernel(const float* __restrict__ caps, long long BN,
                                                            WorldPrims w, float* __restrict__ out) {
  const long long M = w.total();
  const long long total = BN * M;
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long bn = f / M;
    const int m = static_cast<int>(f - bn * M);
    float c[7];
#pragma unroll
    for (int i = 0; i < 7; ++i) c[i] = caps[i * BN + bn];
    __builtin_nontemporal_store(dist_capsule_obstacle(c, w, m), out + f);
  }
}

// Capsule robot self pairs: out[b, p] = capsule-capsule distance of links
// (pair_i[p], pair_j[p]) from AoS capsules [B, N, 7] (_collision_cuda_kernel.cu:474-495).
__global__ __launch_bounds__(256) void self_capsule_kernel(const float* __restrict__ caps, long long B, int N,
                                                           const int* __restrict__ pair_i,
                                                           const int* __restrict__ pair_j, int P,
                                                           float* __restrict__ out) {
  const long long total = B * static_cast<long long>(P);
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long b = f / P;
    const int p = static_cast<int>(f - b * P);
    const int li = pair_i[p], lj = pair_j[p];
    float d = kNoSphere;
    if (li >= 0 && li < N && lj >= 0 && lj < N) {
      float ci[7], cj[7];
#pragma unroll
      for (int i = 0; i < 7; ++i) {
        ci[i] = caps[(b * N + li) * 7 + i];
        cj[i] = caps[(b * N + lj) * 7 + i];
      }
      d = dist_capsule_capsule(ci, cj);
    }
    __builtin_nontemporal_store(d, out + f);
  }
}

// CUDA-semantics world distances from link poses over mixed obstacle kinds:
// out[b, l, m] = min over the link's real sphere slots (r >= 0) of the
// distance to obstacle m, 1e9 for a link without spheres; the spheres are
// placed from the padded (L, S, 4) link-frame table.
__global__ __launch_bounds__(256) void world_links_mixed_kernel(const float* __restrict__ poses, long long B,
                                                                int L, const float* __restrict__ table, int S,
                                                                WorldPrims w, float* __restrict__ out) {
  const long long M = w.total();
  const long long total = B * L * M;
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const long long bl = f / M;
    const int m = static_cast<int>(f - bl * M);
    const long long b = bl / L;
    const int l = static_cast<int>(bl - b * L);
    float best = kNoSphere;
    for (int s = 0; s < S; ++s) {
      float x, y, z, r;
      placed(poses, table, b, L, S, l, s, x, y, z, r);
      if (r < 0.f) continue;
      best = fminf(best, dist_sphere_obstacle(x, y, z, r, w, m));
    }
    __builtin_nontemporal_store(best, out + f);
  }
}

// Capsule robot at a configuration: each link-frame capsule [a, b, r] of the
// (N, 7) table moved by its link pose; written component-major [7, B, N]
// (the world kernel's layout) and/or AoS [B, N, 7] (the self kernel's).
__global__ __launch_bounds__(256) void capsule_place_kernel(const float* __restrict__ poses, long long B, int N,
                                                            const float* __restrict__ local,
                                                            float* __restrict__ out_soa,
                                                            float* __restrict__ out_aos) {
  const long long total = B * N;
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long f = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; f < total; f += stride) {
    const int n = static_cast<int>(f % N);
    const float* T = poses + f * 7;
    const float* c = local + static_cast<long long>(n) * 7;
    float v[7];
    quat_rotate(T[0], T[1], T[2], T[3], c[0], c[1], c[2], v[0], v[1], v[2]);
    quat_rotate(T[0], T[1], T[2], T[3], c[3], c[4], c[5], v[3], v[4], v[5]);
    v[0] += T[4];
    v[1] += T[5];
    v[2] += T[6];
    v[3] += T[4];
    v[4] += T[5];
    v[5] += T[6];
    v[6] = c[6];
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      if (out_soa) out_soa[k * total + f] = v[k];
      if (out_aos) out_aos[f * 7 + k] = v[k];
    }
  }
}

// Per-configuration minimum over the (L, M) block of world_links_mixed_kernel's
// output: one wave per configuration, a strided scan and a wave minimum.
__global__ __launch_bounds__(64) void row_min_kernel(const float* __restrict__ dist, long long B, long long LM,
                                                     float* __restrict__ out) {
  const long long b = blockIdx.x;
  if (b >= B) return;
  float v = kNoSphere;
  for (long long i = threadIdx.x; i < LM; i += kWave) v = fminf(v, dist[b * LM + i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, kWave));
  if (threadIdx.x == 0) out[b] = v;
}

// Grid for a flat grid-stride launch of `total` elements: enough 256-thread
// workgroups to fill the chip a few times over, never more than needed.
static unsigned flat_blocks(long long total) {
  const long long need = (total + 255) / 256;
  return static_cast<unsigned>(need < 256LL * 32 ? need : 256LL * 32);
}

static int world_prims(WorldPrims& w, const float* ws, int ms, const float* wc, int mc, const float* wb,
                       int mb, const float* wh, int mh) {
  PK_REQUIRE(ms >= 0 && mc >= 0 && mb >= 0 && mh >= 0, "negative obstacle count");
  PK_REQUIRE((ms == 0 || ws) && (mc == 0 || wc) && (mb == 0 || wb) && (mh == 0 || wh),
             "null world array");
  PK_REQUIRE(static_cast<long long>(ms) + mc + mb + mh <= 0x7fffffffLL, "too many obstacles");
  w.data[0] = ws; w.data[1] = wc; w.data[2] = wb; w.data[3] = wh;
  w.count[0] = ms; w.count[1] = mc; w.count[2] = mb; w.count[3] = mh;
  return PK_OK;
}

int launch_world_reduced_mixed(void* stream, const float* sc, const float* sr, long long batch, int k,
                               int n_links, const float* ws, int ms, const float* wc, int mc, const float* wb,
                               int mb, const float* wh, int mh, float* out) {
  WorldPrims w{};
  const int st = world_prims(w, ws, ms, wc, mc, wb, mb, wh, mh);
  if (st != PK_OK) return st;
  const long long total = batch * n_links * static_cast<long long>(w.total());
  if (total == 0) return PK_OK;
  hipLaunchKernelGGL(world_reduced_mixed_kernel, dim3(flat_blocks(total)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), sc, sr, batch, k, k / n_links, n_links, w, out);
  return check_launch("world_reduced_mixed_kernel");
}

}  // namespace pk

extern "C" int pk_collision_world_sphere_f32(void* stream, const float* sphere_centers,
                                             const float* sphere_radii, int64_t batch, int32_t k,
                                             const float* world_spheres, int32_t n_world_spheres,
                                             const float* world_capsules, int32_t n_world_capsules,
                                             const float* world_boxes, int32_t n_world_boxes,
                                             const float* world_halfspaces,
                                             int32_t n_world_halfspaces, float* out) {
  PK_REQUIRE(batch >= 0 && k >= 0 && n_world_spheres >= 0 && n_world_capsules >= 0 && n_world_boxes >= 0 &&
                 n_world_halfspaces >= 0,
             "negative size");
  const long long BK = batch * static_cast<long long>(k);
  if (BK == 0 || static_cast<long long>(n_world_spheres) + n_world_capsules + n_world_boxes +
                         n_world_halfspaces == 0)
    return PK_OK;
  pk::WorldPrims w{};
  const int st = pk::world_prims(w, world_spheres, n_world_spheres, world_capsules, n_world_capsules,
                                 world_boxes, n_world_boxes, world_halfspaces, n_world_halfspaces);
  if (st != PK_OK) return st;
  const long long total = BK * w.total();
  PK_REQUIRE(sphere_centers && sphere_radii && out, "null pointer");
  hipLaunchKernelGGL(pk::world_sphere_full_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), sphere_centers, sphere_radii, BK, w, out);
  return pk::check_launch("world_sphere_full_kernel");
}

namespace {

int distances_jax(void* stream, const float* link_poses, int64_t batch, int32_t n_links, const float* spheres_padded,
                  int32_t s_per_link, const float* world_spheres, int32_t n_world_spheres, const int32_t* pair_i,
                  const int32_t* pair_j, int32_t n_pairs, const pk::RowCost& cost, float* out_world,
                  float* out_self) {
  PK_REQUIRE(batch >= 0 && n_links >= 0 && s_per_link >= 0 && n_world_spheres >= 0 && n_pairs >= 0,
             "negative size");
  if (batch == 0 || n_links == 0) return PK_OK;
  PK_REQUIRE(link_poses && (s_per_link == 0 || spheres_padded), "null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (out_world && n_world_spheres > 0) {
    PK_REQUIRE(world_spheres != nullptr, "null world");
    pk::RowArgs a{};
    a.poses = link_poses;
    a.batch = batch;
    a.n_links = n_links;
    a.s_per_link = s_per_link;
    a.table = spheres_padded;
    a.w.data[0] = world_spheres;
    a.w.count[0] = n_world_spheres;
    a.cost = cost;
    a.out = out_world;
    if (!pk::launch_link_rows<true>(s, a)) {
      const long long total = batch * n_links * static_cast<long long>(n_world_spheres);
      hipLaunchKernelGGL(pk::jax_world_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0, s, link_poses,
                         static_cast<long long>(batch), n_links, spheres_padded, s_per_link, world_spheres,
                         n_world_spheres, cost, out_world);
    }
    const int st = pk::check_launch("link_rows_kernel");
    if (st != PK_OK) return st;
  }
  if (out_self && n_pairs > 0) {
    PK_REQUIRE(pair_i && pair_j, "null pair list");
    pk::SelfRowArgs a{};
    a.poses = link_poses;
    a.batch = batch;
    a.n_links = n_links;
    a.s_per_link = s_per_link;
    a.table = spheres_padded;
    a.pair_i = pair_i;
    a.pair_j = pair_j;
    a.n_pairs = n_pairs;
    a.cost = cost;
    a.out = out_self;
    if (!pk::launch_self_rows(s, a)) {
      const long long total = batch * static_cast<long long>(n_pairs);
      hipLaunchKernelGGL(pk::jax_self_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0, s, link_poses,
                         static_cast<long long>(batch), n_links, spheres_padded, s_per_link, pair_i, pair_j,
                         n_pairs, cost, out_self);
    }
    return pk::check_launch("self_rows_kernel");
  }
  return PK_OK;
}

}  // namespace

extern "C" int pk_sphere_distances_jax_f32(void* stream, const float* link_poses, int64_t batch,
                                           int32_t n_links, const float* spheres_padded,
                                           int32_t s_per_link, const float* world_spheres,
                                           int32_t n_world_spheres, const int32_t* pair_i,
                                           const int32_t* pair_j, int32_t n_pairs, float* out_world,
                                           float* out_self) {
  return distances_jax(stream, link_poses, batch, n_links, spheres_padded, s_per_link, world_spheres,
                       n_world_spheres, pair_i, pair_j, n_pairs, pk::RowCost{}, out_world, out_self);
}

extern "C" int pk_sphere_costs_jax_f32(void* stream, const float* link_poses, int64_t batch, int32_t n_links,
                                       const float* spheres_padded, int32_t s_per_link,
                                       const float* world_spheres, int32_t n_world_spheres,
                                       const int32_t* pair_i, const int32_t* pair_j, int32_t n_pairs,
                                       float margin, float half, float quad, float weight, float* out_world,
                                       float* out_self) {
  return distances_jax(stream, link_poses, batch, n_links, spheres_padded, s_per_link, world_spheres,
                       n_world_spheres, pair_i, pair_j, n_pairs, pk::RowCost{1, margin, half, quad, weight},
                       out_world, out_self);
}

extern "C" int pk_collision_world_capsule_f32(void* stream, const float* caps, int64_t batch, int32_t n_links,
                                              const float* world_spheres, int32_t n_world_spheres,
                                              const float* world_capsules, int32_t n_world_capsules,
                                              const float* world_boxes, int32_t n_world_boxes,
                                              const float* world_halfspaces, int32_t n_world_halfspaces,
                                              float* out) {
  PK_REQUIRE(batch >= 0 && n_links >= 0 && n_world_spheres >= 0 && n_world_capsules >= 0 && n_world_boxes >= 0 &&
                 n_world_halfspaces >= 0,
             "negative size");
  const long long BN = batch * static_cast<long long>(n_links);
  if (BN == 0 || static_cast<long long>(n_world_spheres) + n_world_capsules + n_world_boxes +
                         n_world_halfspaces == 0)
    return PK_OK;
  pk::WorldPrims w{};
  const int st = pk::world_prims(w, world_spheres, n_world_spheres, world_capsules, n_world_capsules,
                                 world_boxes, n_world_boxes, world_halfspaces, n_world_halfspaces);
  if (st != PK_OK) return st;
  PK_REQUIRE(caps && out, "null pointer");
  const long long total = BN * w.total();
  hipLaunchKernelGGL(pk::world_capsule_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), caps, BN, w, out);
  return pk::check_launch("world_capsule_kernel");
}

extern "C" int pk_collision_self_capsule_f32(void* stream, const float* caps, int64_t batch, int32_t n_links,
                                             const int32_t* pair_i, const int32_t* pair_j, int32_t n_pairs,
                                             float* out) {
  PK_REQUIRE(batch >= 0 && n_links >= 0 && n_pairs >= 0, "negative size");
  if (batch == 0 || n_pairs == 0) return PK_OK;
  PK_REQUIRE(caps && pair_i && pair_j && out, "null pointer");
  const long long total = batch * static_cast<long long>(n_pairs);
  hipLaunchKernelGGL(pk::self_capsule_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), caps, static_cast<long long>(batch), n_links, pair_i,
                     pair_j, n_pairs, out);
  return pk::check_launch("self_capsule_kernel");
}

extern "C" int pk_sphere_world_links_f32(void* stream, const float* link_poses, int64_t batch, int32_t n_links,
                                         const float* spheres_padded, int32_t s_per_link,
                                         const float* world_spheres, int32_t n_world_spheres,
                                         const float* world_capsules, int32_t n_world_capsules,
                                         const float* world_boxes, int32_t n_world_boxes,
                                         const float* world_halfspaces, int32_t n_world_halfspaces,
                                         float* out_world, float* out_world_min) {
  PK_REQUIRE(batch >= 0 && n_links >= 0 && s_per_link >= 0 && n_world_spheres >= 0 && n_world_capsules >= 0 &&
                 n_world_boxes >= 0 && n_world_halfspaces >= 0,
             "negative size");
  const long long M = static_cast<long long>(n_world_spheres) + n_world_capsules + n_world_boxes +
                      n_world_halfspaces;
  if (batch == 0) return PK_OK;
  PK_REQUIRE(out_world != nullptr, "out_world is required (the minimum is reduced from it)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (n_links > 0 && M > 0) {
    PK_REQUIRE(link_poses && (s_per_link == 0 || spheres_padded), "null pointer");
    pk::WorldPrims w{};
    const int ws = pk::world_prims(w, world_spheres, n_world_spheres, world_capsules, n_world_capsules,
                                   world_boxes, n_world_boxes, world_halfspaces, n_world_halfspaces);
    if (ws != PK_OK) return ws;
    pk::RowArgs a{};
    a.poses = link_poses;
    a.batch = batch;
    a.n_links = n_links;
    a.s_per_link = s_per_link;
    a.table = spheres_padded;
    a.w = w;
    a.out = out_world;
    if (!pk::launch_link_rows<false>(st, a)) {
      const long long total = batch * n_links * M;
      hipLaunchKernelGGL(pk::world_links_mixed_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0, st, link_poses,
                         static_cast<long long>(batch), n_links, spheres_padded, s_per_link, w, out_world);
    }
    const int e = pk::check_launch("link_rows_kernel");
    if (e != PK_OK) return e;
  }
  if (out_world_min) {
    PK_REQUIRE(batch <= 0x7fffffffLL, "batch too large");
    hipLaunchKernelGGL(pk::row_min_kernel, dim3(static_cast<unsigned>(batch)), dim3(pk::kWave), 0, st, out_world,
                       static_cast<long long>(batch), static_cast<long long>(n_links) * M, out_world_min);
    return pk::check_launch("row_min_kernel");
  }
  return PK_OK;
}

extern "C" int pk_capsules_place_f32(void* stream, const float* link_poses, int64_t batch, int32_t n_links,
                                     const float* capsules_local, float* out_soa, float* out_aos) {
  PK_REQUIRE(batch >= 0 && n_links >= 0, "negative size");
  if (batch == 0 || n_links == 0) return PK_OK;
  PK_REQUIRE(link_poses && capsules_local, "null pointer");
  PK_REQUIRE(out_soa || out_aos, "no output requested");
  const long long total = batch * n_links;
  hipLaunchKernelGGL(pk::capsule_place_kernel, dim3(pk::flat_blocks(total)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), link_poses, static_cast<long long>(batch), n_links,
                     capsules_local, out_soa, out_aos);
  return pk::check_launch("capsule_place_kernel");
}

extern "C" int pk_row_min_f32(void* stream, const float* dist, int64_t batch, int64_t row_len, float* out) {
  PK_REQUIRE(batch >= 0 && row_len >= 0, "negative size");
  if (batch == 0) return PK_OK;
  PK_REQUIRE(out && (row_len == 0 || dist), "null pointer");
  PK_REQUIRE(batch <= 0x7fffffffLL, "batch too large");
  hipLaunchKernelGGL(pk::row_min_kernel, dim3(static_cast<unsigned>(batch)), dim3(pk::kWave), 0,
                     static_cast<hipStream_t>(stream), dist, static_cast<long long>(batch),
                     static_cast<long long>(row_len), out);
  return pk::check_launch("row_min_kernel");
}
