// Pose + hinge collision cost and its hand-written adjoint, for gfx950.
//
// cost(q) = sum_c (W_c r_c)^2 + sum_{k,m} max(0, margin - d_km)^2
//   r     = [p_ee - p_t; log(q_ee q_t^-1)]  (the LM residual, _ik_cuda_helpers.cuh:471-494)
//   d_km  = |c_k - o_m| - r_k - R_m         (robot sphere k, world sphere m)
// The collision term is the CHOMP hinge^2 (src/pyroffi/optimization_engines/
// _chomp_optimization.py:140-154); the reference differentiates it with JAX AD.
//
// Adjoint (reverse accumulation over the kinematic tree, no Jacobians):
//   dcost/dc_k   = f_k = sum_m -2 h_km u_km,   u = (c - o)/|c - o|
//   per link L   : F_L = sum_{k in L} f_k,     T_L = sum_k c_k x f_k  (about the origin)
//   EE           : F += 2 W_p^2 r_pos at p_ee, T += p_ee x F + 2 W_o^2 r_ori
//                  (d|log E|^2 under a left perturbation w is 2 r_ori . w because
//                   J_l(r)^-T r = r)
//   subtree sums : (F, T)_sub(j) over the links below joint j (reverse topo order)
//   dcost/dq_a   = sum_{j : src(j) = a} mul_j (w_j . (T_sub - p_j x F_sub) + v_j . F_sub)
//                  with w_j = R_j omega_j, v_j = R_j v_j from the joint's twist
//                  and world pose (= pose of its child link).
//
// Work decomposition: workgroups of four waves share the per-launch tables; a
// wave owns a contiguous block of configurations and handles one at a time.
// Testing all spheres against all obstacles was most of the time (Panda, 59 x
// 512 pairs: 0.231 ms for 16384 configurations) though about one pair in a
// thousand is within the margin.  So each link carries a bounding sphere:
// lanes over obstacles (T per lane, resident in registers) test it link by
// link, the obstacles in reach are compacted into a list, and groups of eight
// lanes take the link's spheres against one listed obstacle each, with the
// exact hinge.  A link's wrench is a wavefront sum, taken only where a hinge is
// active, and the tree's adjoint has one lane per joint.  (The call, forward
// and backward, at that size: 238 -> 131 us.)
#include "pk_model.h"

#include <math.h>

#include <algorithm>

namespace pk {

struct HingeArgs {
  const float* link_poses;      // (B, L, 7)
  long long batch;
  int n_links;
  const float* spheres_local;   // (K, 4), grouped by link
  const int* link_sphere_start; // (L + 1)
  int n_spheres;
  const float* world;           // (M, 4)
  int n_world;
  float margin;
  int ee_link;                  // -1: no pose term
  const float* targets;         // (B, 7)
  float pos_weight, ori_weight;
  // tables for the adjoint
  const float* twists;
  const int* parent_idx;
  const int* act_idx;
  const int* mimic_act_idx;
  const float* mimic_mul;
  const int* topo_inv;
  const int* link_parent_joint;
  int n_joints, n_act;
  float* out_cost;              // (B)
  float* out_grad;              // (B, n_act) or null
};

struct JointAdj {
  float ang[3], lin[3];
  float mul;
  int src, parent, child_link;
  unsigned long long subtree;  // joints below this one, itself included
};

__device__ __forceinline__ float wave_sum(float v) { return wave_sum_dpp(v); }

constexpr int kHingeWaves = 4;  // at most; one where four waves' buffers do not fit the LDS

// Words of LDS: shared tables, then each wave's buffers (float4 regions first).
struct HingeLds {
  int spheres, bounds, joints, lstart, slink, waves;  // byte offsets
  int per_wave, total;
};

// T: obstacles per lane of a pass (a list entry is one of 64 T).
__host__ __device__ inline HingeLds hinge_lds(int L, int K, int J, int T, int n_waves) {
  HingeLds o;
  o.spheres = 0;                                                        // K float4, link frame
  o.bounds = o.spheres + static_cast<int>(sizeof(float4)) * K;          // L float4, link frame
  o.joints = o.bounds + static_cast<int>(sizeof(float4)) * L;           // J JointAdj
  o.lstart = o.joints + static_cast<int>(sizeof(JointAdj)) * J;         // L + 1 int
  o.slink = o.lstart + 4 * (L + 1);                                     // K int
  o.waves = (o.slink + 4 * K + 15) / 16 * 16;
  // per wave: K placed spheres, L placed bounds (float4), L * 7 poses, L * 6
  // wrenches, J joint gradients, the obstacle list
  o.per_wave = (16 * K + 16 * L + 4 * (13 * L + J) + 2 * kWave * T + 15) / 16 * 16;
  o.total = o.waves + n_waves * o.per_wave;
  return o;
}

template <int T>
__global__ __launch_bounds__(kWave * kHingeWaves, 4) void pose_hinge_kernel(HingeArgs a) {
  extern __shared__ float4 smem4[];
  char* base = reinterpret_cast<char*>(smem4);
  const int tid = threadIdx.x;
  const int lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int L = a.n_links, K = a.n_spheres, M = a.n_world, J = a.n_joints;
  const int nt = blockDim.x, wg_waves = nt / kWave;
  const HingeLds lay = hinge_lds(L, K, J, T, wg_waves);
  float4* sl = reinterpret_cast<float4*>(base + lay.spheres);
  float4* lb = reinterpret_cast<float4*>(base + lay.bounds);
  JointAdj* jt = reinterpret_cast<JointAdj*>(base + lay.joints);
  int* lstart = reinterpret_cast<int*>(base + lay.lstart);
  int* slink = reinterpret_cast<int*>(base + lay.slink);
  float4* sc = reinterpret_cast<float4*>(base + lay.waves + wave * lay.per_wave);
  float4* bc = sc + K;
  float* ptile = reinterpret_cast<float*>(bc + L);
  float* wl = ptile + 7 * L;
  float* gj = wl + 6 * L;
  unsigned short* list = reinterpret_cast<unsigned short*>(gj + J);

  for (int k = tid; k < K; k += nt) {
    const float* s = a.spheres_local + 4 * k;
    sl[k] = make_float4(s[0], s[1], s[2], s[3]);
    slink[k] = 0;
  }
  for (int n = tid; n <= L; n += nt) lstart[n] = (n == L) ? K : a.link_sphere_start[n];
  for (int j = tid; j < J; j += nt) {
    JointAdj r;
    for (int c = 0; c < 3; ++c) { r.lin[c] = a.twists[6 * j + c]; r.ang[c] = a.twists[6 * j + 3 + c]; }
    r.mul = a.mimic_mul[j];
    const int m = a.mimic_act_idx[j];
    int src = (m != -1) ? m : a.act_idx[j];
    r.src = (src >= 0 && src < a.n_act) ? src : -1;
    const int p = a.parent_idx[j];
    r.parent = (p >= 0 && p < J) ? p : -1;
    r.child_link = -1;
    r.subtree = 0;
    jt[j] = r;
  }
  __syncthreads();
  if (tid == 0) {  // clamp the CSR offsets into a monotone [0, K] sequence
    int prev = 0;
    for (int n = 0; n <= L; ++n) {
      prev = max(prev, min(lstart[n], K));
      lstart[n] = (n == 0) ? 0 : prev;
    }
  }
  for (int l = tid; l < L; l += nt) {
    const int j = a.link_parent_joint != nullptr ? a.link_parent_joint[l] : -1;
    if (j >= 0 && j < J) atomicMax(&jt[j].child_link, l);
  }
  // Each joint enters the subtree of itself and its ancestors (at most J steps,
  // whatever the table holds).
  for (int j = tid; j < J; j += nt) {
    int p = j;
    for (int i = 0; i < J && p >= 0; ++i) {
      atomicOr(&jt[p].subtree, 1ull << j);
      p = jt[p].parent;
    }
  }
  __syncthreads();
  for (int n = tid; n < L; n += nt) {
    float lx = INFINITY, ly = INFINITY, lz = INFINITY, hx = -INFINITY, hy = -INFINITY, hz = -INFINITY;
    for (int k = lstart[n]; k < lstart[n + 1]; ++k) {
      slink[k] = n;
      const float4 q = sl[k];
      lx = fminf(lx, q.x); ly = fminf(ly, q.y); lz = fminf(lz, q.z);
      hx = fmaxf(hx, q.x); hy = fmaxf(hy, q.y); hz = fmaxf(hz, q.z);
    }
    float4 b = make_float4(0.5f * (lx + hx), 0.5f * (ly + hy), 0.5f * (lz + hz), -1e30f);
    for (int k = lstart[n]; k < lstart[n + 1]; ++k) {
      const float4 q = sl[k];
      const float dx = q.x - b.x, dy = q.y - b.y, dz = q.z - b.z;
      b.w = fminf(fmaxf(b.w, sqrtf(dx * dx + dy * dy + dz * dz) + fmaxf(q.w, 0.f)), 1e29f);
    }
    if (lstart[n] == lstart[n + 1]) b = make_float4(0.f, 0.f, 0.f, -1e30f);
    lb[n] = b;
  }

  const int chunk = kWave * T;
  const int n_chunks = (M + chunk - 1) / chunk;
  float ox[T], oy[T], oz[T], orm[T];  // obstacle centre, radius + margin
  auto load_obstacles = [&](int c) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int m = c * chunk + t * kWave + lane;
      if (m < M) {
        ox[t] = a.world[4 * m]; oy[t] = a.world[4 * m + 1]; oz[t] = a.world[4 * m + 2];
        orm[t] = a.world[4 * m + 3] + a.margin;
      } else {  // reached by nothing
        ox[t] = 0.f; oy[t] = 0.f; oz[t] = 0.f; orm[t] = -1e30f;
      }
    }
  };
  if (n_chunks > 0) load_obstacles(0);
  __syncthreads();

  const long long n_waves = static_cast<long long>(gridDim.x) * wg_waves;
  const long long per = (a.batch + n_waves - 1) / n_waves;
  const long long b_begin = (static_cast<long long>(blockIdx.x) * wg_waves + wave) * per;
  const long long b_end = min(a.batch, b_begin + per);
  const bool want_grad = a.out_grad != nullptr;
  for (long long b = b_begin; b < b_end; ++b) {
    const float* pb = a.link_poses + b * L * 7;
    for (int f = lane; f < L * 7; f += kWave) ptile[f] = pb[f];
    for (int f = lane; f < L * 6; f += kWave) wl[f] = 0.f;
    wave_sync();
    for (int k = lane; k < K + L; k += kWave) {
      const float* p = ptile + 7 * (k < K ? slink[k] : k - K);
      const float4 s = k < K ? sl[k] : lb[k - K];
      float wx, wy, wz;
      quat_rotate(p[0], p[1], p[2], p[3], s.x, s.y, s.z, wx, wy, wz);
      float r = s.w;
      if (k >= K) {
        // A quaternion that is not of unit length stretches the link's offsets by at
        // most 1 + 4 ||q|^2 - 1| (finite also for a NaN pose).
        const float qq = p[0] * p[0] + p[1] * p[1] + p[2] * p[2] + p[3] * p[3];
        r = fminf(fmaf(4.f * fabsf(qq - 1.f), fmaxf(r, 0.f), r), 1e29f);
      }
      sc[k] = make_float4(wx + p[4], wy + p[5], wz + p[6], r);  // bc follows sc
    }
    wave_sync();

    float cost = 0.f;
    for (int c = 0; c < n_chunks; ++c) {
      if (c > 0) load_obstacles(c);
      for (int n = 0; n < L; ++n) {
        const int k0 = lstart[n], k1 = lstart[n + 1];
        if (k0 == k1) continue;
        const float4 bn = bc[n];
        // Slack for the rounding of the centres, by the size of the coordinates
        // (finite also for a NaN pose: lanes without an obstacle never hit).
        const float slack = fminf(1e-5f + 4e-6f * (fabsf(bn.x) + fabsf(bn.y) + fabsf(bn.z)), 1e20f);
        int cnt = 0;
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const float dx = bn.x - ox[t], dy = bn.y - oy[t], dz = bn.z - oz[t];
          float reach = bn.w + orm[t];
          reach = fmaf(4e-6f, fabsf(reach), reach + slack);
          // A pair the test cannot decide (NaN) is kept for the exact one.
          const bool hit = !(reach < 0.f) && !(dx * dx + dy * dy + dz * dz > reach * reach);
          const unsigned long long mask = __ballot(hit);
          if (mask != 0) {
            if (hit)
              list[cnt + __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                                   __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u))] =
                  static_cast<unsigned short>(t * kWave + lane);
            cnt += __popcll(mask);
          }
        }
        if (cnt == 0) continue;
        wave_sync();
        float F0 = 0.f, F1 = 0.f, F2 = 0.f, T0 = 0.f, T1 = 0.f, T2 = 0.f;
        bool active = false;
        for (int e = lane / 8; e < cnt; e += kWave / 8) {
          const float* o = a.world + 4 * (static_cast<long long>(c) * chunk + list[e]);
          const float qx = o[0], qy = o[1], qz = o[2], qr = o[3] + a.margin;
          for (int k = k0 + lane % 8; k < k1; k += 8) {
            const float4 s = sc[k];
            const float dx = s.x - qx, dy = s.y - qy, dz = s.z - qz;
            const float d2 = fmaxf(dx * dx + dy * dy + dz * dz, 1e-20f);
            const float rs = __builtin_amdgcn_rsqf(d2);
            const float h = (s.w + qr) - d2 * rs;  // margin - d
            if (h > 0.f) {
              active = true;
              cost = fmaf(h, h, cost);
              const float g = -2.f * h * rs;
              const float fx = g * dx, fy = g * dy, fz = g * dz;
              F0 += fx; F1 += fy; F2 += fz;
              T0 += s.y * fz - s.z * fy;
              T1 += s.z * fx - s.x * fz;
              T2 += s.x * fy - s.y * fx;
            }
          }
        }
        if (want_grad && __any(active)) {
          const float w0 = wave_sum(F0), w1 = wave_sum(F1), w2 = wave_sum(F2);
          const float w3 = wave_sum(T0), w4 = wave_sum(T1), w5 = wave_sum(T2);
          if (lane == 0) {
            wl[6 * n] += w0; wl[6 * n + 1] += w1; wl[6 * n + 2] += w2;
            wl[6 * n + 3] += w3; wl[6 * n + 4] += w4; wl[6 * n + 5] += w5;
          }
        }
        wave_sync();
      }
    }
    if (n_chunks > 1) load_obstacles(0);
    cost = wave_sum(cost);

    if (lane == 0) {
      // Pose term at the end effector.
      if (a.ee_link >= 0 && a.ee_link < L) {
        const float* pe = ptile + 7 * a.ee_link;
        const float* tg = a.targets + b * 7;
        float r[6];
        r[0] = pe[4] - tg[4]; r[1] = pe[5] - tg[5]; r[2] = pe[6] - tg[6];
        float ew, ex, ey, ez;
        quat_mul(pe[0], pe[1], pe[2], pe[3], tg[0], -tg[1], -tg[2], -tg[3], ew, ex, ey, ez);
        if (ew < 0.f) { ew = -ew; ex = -ex; ey = -ey; ez = -ez; }
        const float shn = sqrtf(ex * ex + ey * ey + ez * ez);
        const float kk = (shn > 1e-6f) ? 2.f * atan2f(shn, ew) / shn : 2.f;
        r[3] = ex * kk; r[4] = ey * kk; r[5] = ez * kk;
        const float wp2 = a.pos_weight * a.pos_weight, wo2 = a.ori_weight * a.ori_weight;
        cost += wp2 * (r[0] * r[0] + r[1] * r[1] + r[2] * r[2]) + wo2 * (r[3] * r[3] + r[4] * r[4] + r[5] * r[5]);
        if (want_grad) {
          const float Fx = 2.f * wp2 * r[0], Fy = 2.f * wp2 * r[1], Fz = 2.f * wp2 * r[2];
          float* w = wl + 6 * a.ee_link;
          w[0] += Fx; w[1] += Fy; w[2] += Fz;
          w[3] += pe[5] * Fz - pe[6] * Fy + 2.f * wo2 * r[3];
          w[4] += pe[6] * Fx - pe[4] * Fz + 2.f * wo2 * r[4];
          w[5] += pe[4] * Fy - pe[5] * Fx + 2.f * wo2 * r[5];
        }
      }
      a.out_cost[b] = cost;
    }
    if (want_grad) {
      wave_sync();
      // One lane per joint: the wrench of its subtree's links, then dcost/dq_j.
      if (lane < J) {
        const JointAdj& r = jt[lane];
        float w[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float g = 0.f;
        if (r.src >= 0 && r.child_link >= 0) {
          for (unsigned long long m = r.subtree; m != 0; m &= m - 1) {
            const int l = jt[__builtin_ctzll(m)].child_link;
            if (l >= 0)
#pragma unroll
              for (int i = 0; i < 6; ++i) w[i] += wl[6 * l + i];
          }
          const float* pj = ptile + 7 * r.child_link;
          float wx, wy, wz, vx, vy, vz;
          quat_rotate(pj[0], pj[1], pj[2], pj[3], r.ang[0], r.ang[1], r.ang[2], wx, wy, wz);
          quat_rotate(pj[0], pj[1], pj[2], pj[3], r.lin[0], r.lin[1], r.lin[2], vx, vy, vz);
          const float tx = w[3] - (pj[5] * w[2] - pj[6] * w[1]);
          const float ty = w[4] - (pj[6] * w[0] - pj[4] * w[2]);
          const float tz = w[5] - (pj[4] * w[1] - pj[5] * w[0]);
          g = r.mul * (wx * tx + wy * ty + wz * tz + vx * w[0] + vy * w[1] + vz * w[2]);
        }
        gj[lane] = g;
      }
      wave_sync();
      if (lane < a.n_act) {
        float g = 0.f;
        for (int j = 0; j < J; ++j)
          if (jt[j].src == lane) g += gj[j];
        a.out_grad[b * a.n_act + lane] = g;
      }
    }
    wave_sync();
  }
}

static int pick_t(int M) {
  if (M <= 64) return 1;
  if (M <= 128) return 2;
  if (M <= 256) return 4;
  return 8;
}

}  // namespace pk

extern "C" int pk_pose_hinge_cost_f32(
    void* stream, const float* link_poses, int64_t batch, int32_t n_links,
    const float* spheres_local, const int32_t* link_sphere_start, int32_t n_spheres,
    const float* world_spheres, int32_t n_world_spheres, float margin, int32_t ee_link,
    const float* targets, float pos_weight, float ori_weight, const float* twists,
    const int32_t* parent_idx, const int32_t* act_idx, const int32_t* mimic_act_idx,
    const float* mimic_mul, const int32_t* topo_inv, const int32_t* link_parent_joint,
    int32_t n_joints, int32_t n_act, float* out_cost, float* out_grad) {
  PK_REQUIRE(batch >= 0 && n_links >= 0 && n_spheres >= 0 && n_world_spheres >= 0, "negative size");
  PK_REQUIRE(n_joints >= 0 && n_joints <= pk::kMaxJoints, "n_joints=%d outside [0, %d]", n_joints,
             pk::kMaxJoints);
  PK_REQUIRE(n_act >= 0 && n_act <= pk::kMaxAct, "n_act=%d outside [0, %d]", n_act, pk::kMaxAct);
  PK_REQUIRE(n_links <= pk::kMaxJoints + 1, "n_links=%d too large", n_links);
  PK_REQUIRE(ee_link < n_links, "ee_link=%d outside the %d links", ee_link, n_links);
  if (batch == 0) return PK_OK;
  PK_REQUIRE(link_poses && link_sphere_start && out_cost && (n_spheres == 0 || spheres_local) &&
                 (n_world_spheres == 0 || world_spheres) && (ee_link < 0 || targets),
             "null pointer");
  if (out_grad)
    PK_REQUIRE(twists && parent_idx && act_idx && mimic_act_idx && mimic_mul && topo_inv &&
                   link_parent_joint,
               "null adjoint table");
  pk::HingeArgs a{link_poses, batch, n_links, spheres_local, link_sphere_start, n_spheres,
                  world_spheres, n_world_spheres, margin, ee_link, targets, pos_weight,
                  ori_weight, twists, parent_idx, act_idx, mimic_act_idx, mimic_mul,
                  topo_inv, link_parent_joint, out_grad ? n_joints : 0, n_act, out_cost, out_grad};
  const int T = pk::pick_t(n_world_spheres);
  int waves = pk::kHingeWaves;
  if (n_spheres > 0x10000 || pk::hinge_lds(n_links, n_spheres, a.n_joints, T, waves).total > 64 * 1024) waves = 1;
  const size_t need = 48 * static_cast<size_t>(n_spheres);
  const size_t lds = need > 150 * 1024 ? need
                                       : static_cast<size_t>(pk::hinge_lds(n_links, n_spheres, a.n_joints, T, waves).total);
  PK_REQUIRE(lds <= 150 * 1024, "tables need %zu bytes of LDS", lds);
  // Up to four workgroups a CU (16 waves), each wave looping over its block of
  // configurations.
  const long long want = (batch + waves - 1) / waves;
  const unsigned grid = static_cast<unsigned>(std::max(1LL, std::min(want, 256LL * 4)));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 block(pk::kWave * waves);
  switch (T) {
    case 1: hipLaunchKernelGGL(pk::pose_hinge_kernel<1>, dim3(grid), block, lds, s, a); break;
    case 2: hipLaunchKernelGGL(pk::pose_hinge_kernel<2>, dim3(grid), block, lds, s, a); break;
    case 4: hipLaunchKernelGGL(pk::pose_hinge_kernel<4>, dim3(grid), block, lds, s, a); break;
    default: hipLaunchKernelGGL(pk::pose_hinge_kernel<8>, dim3(grid), block, lds, s, a); break;
  }
  return pk::check_launch("pose_hinge_kernel");
}
