// d2_learned.hpp -- device code of the learned pair gate (included by
// d2_kernels.hip inside namespace d2).
//
// A 24 -> 64 -> 64 -> 2 MLP (ReLU, bf16 weights, FP32 accumulation) reads a
// pair's relative pose and motion and proposes
//   y0: the pair's conservative-advancement step scale (the TOI -> step rule's
//       scale; 1 = the pair does not limit the step),
//   y1: a lower bound on the pair's time of impact as a fraction of the CCD
//       interval (labels are 1.25 for pairs with no CCD contact at all).
// A pair proposed as contact-free (y1 and y0 above their gates) is checked by
// a sound certificate instead of being traversed: its bodies' vertex sets are
// separated, along axes found by support-point refinement, by more than the
// search distance plus every rounding and float-barycentric margin, in every
// frame the reference's sub-tests measure in.  Certified pairs provably give
// the plain path's result (no contact, scale 1, min_time = max_time); every
// other pair runs the plain traversal.

constexpr int MLP_IN = 24, MLP_H = 64, MLP_OUT = 2;
constexpr int OFF_W1 = 0;                            // W1[24][64], row = input
constexpr int OFF_B1 = OFF_W1 + MLP_IN * MLP_H;      // b1[64]
constexpr int OFF_W2 = OFF_B1 + MLP_H;               // W2[64][64]
constexpr int OFF_B2 = OFF_W2 + MLP_H * MLP_H;       // b2[64]
constexpr int OFF_W3 = OFF_B2 + MLP_H;               // W3[64][2]
constexpr int OFF_B3 = OFF_W3 + MLP_H * MLP_OUT;     // b3[2]
constexpr int MLP_PARAMS = OFF_B3 + MLP_OUT;         // 5890

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// float -> bf16, round to nearest even (inputs are finite).
__device__ __forceinline__ short f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}
__device__ __forceinline__ float bf2f(short h) { return __uint_as_float(((unsigned)(unsigned short)h) << 16); }

// ------------------------------------------------------------------ features
// Per pair, in body a's frame at the start of the interval, lengths in units
// of Lc = r_a + r_b (bounding radii), times in units of the interval:
//   0-2 centre offset, 3-6 relative rotation (w >= 0), 7-9 relative velocity,
//   10-12 / 13-15 angular velocities of a / b, 16-17 radii, 18 search
//   distance, 19 centre distance, 20 gap between the bounding spheres,
//   21 closing speed, 22 rotational sweep (|w_a| r_a + |w_b| r_b), 23 |v_rel|.
__device__ __forceinline__ void pair_features(int p, const int32_t* pairs, const double* bodies,
                                              const int32_t* body_tree, const float* tree_radius,
                                              const double* max_time, float* x) {
  {
    const int a = pairs[2 * p], b = pairs[2 * p + 1];
    const double* ra = bodies + 40 * (size_t)a;
    const double* rb = bodies + 40 * (size_t)b;
    const body_state sa = load_state(ra), sb = load_state(rb);
    const double mt = max_time ? max_time[p] : ((rb[39] < ra[39]) ? rb[39] : ra[39]);
    const double rA = tree_radius[body_tree[a]], rB = tree_radius[body_tree[b]];
    const double Lc = rA + rB > 1e-12 ? rA + rB : 1e-12;
    double R[9], Iw[9];
    qrot(sa.q, R);
    auto to_a = [&](v3<double> v) {  // R^T v
      return v3<double>{(R[0] * v.x + R[3] * v.y) + R[6] * v.z, (R[1] * v.x + R[4] * v.y) + R[7] * v.z,
                        (R[2] * v.x + R[5] * v.y) + R[8] * v.z};
    };
    world_inv_inertia(sa.q, ra + 28, Iw);
    const v3<double> wa = mul33v(Iw, sa.L);
    world_inv_inertia(sb.q, rb + 28, Iw);
    const v3<double> wb = mul33v(Iw, sb.L);
    const v3<double> dw = sub(sb.t, sa.t);
    const v3<double> d = to_a(dw);
    quat qc{sa.q.w, -sa.q.x, -sa.q.y, -sa.q.z};
    quat qr = qmul(qc, sb.q);
    if (qr.w < 0.0) qr = quat{-qr.w, -qr.x, -qr.y, -qr.z};
    const v3<double> vr = to_a(sub(sb.v, sa.v));
    const v3<double> wa_a = to_a(wa), wb_a = to_a(wb);
    const double dist = vlen(d), vlenr = vlen(vr);
    const double closing = dist > 0.0 ? -dot(d, vr) / dist : 0.0;
    const double il = 1.0 / Lc, vt = mt / Lc;
    x[0] = (float)(d.x * il), x[1] = (float)(d.y * il), x[2] = (float)(d.z * il);
    x[3] = (float)qr.w, x[4] = (float)qr.x, x[5] = (float)qr.y, x[6] = (float)qr.z;
    x[7] = (float)(vr.x * vt), x[8] = (float)(vr.y * vt), x[9] = (float)(vr.z * vt);
    x[10] = (float)(wa_a.x * mt), x[11] = (float)(wa_a.y * mt), x[12] = (float)(wa_a.z * mt);
    x[13] = (float)(wb_a.x * mt), x[14] = (float)(wb_a.y * mt), x[15] = (float)(wb_a.z * mt);
    x[16] = (float)(rA * il), x[17] = (float)(rB * il);
    x[18] = (float)((double)(float)(ra[37] + rb[37]) * il);
    x[19] = (float)(dist * il);
    x[20] = (float)((dist - rA - rB) * il);
    x[21] = (float)(closing * vt);
    x[22] = (float)((vlen(wa) * rA + vlen(wb) * rB) * vt);
    x[23] = (float)(vlenr * vt);
  }
}
__global__ void k_pair_features(int n_pairs, const int32_t* pairs, const double* bodies, const int32_t* body_tree,
                                const float* tree_radius, const double* max_time, float* X) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n_pairs; p += gridDim.x * blockDim.x)
    pair_features(p, pairs, bodies, body_tree, tree_radius, max_time, X + (size_t)MLP_IN * p);
}

// --------------------------------------------------------- MFMA inference
// One wavefront per tile of 16 pairs, v_mfma_f32_16x16x16_bf16 (FP32
// accumulation).  Operand layout: lane l supplies A[l%16][4(l/16)+i] and
// B[4(l/16)+i][l%16], i = 0..3, and receives D[4(l/16)+i][l%16].
// Activations go through LDS (bf16) between layers.  wb: bf16 parameters.
// FEAT: the inputs are the pairs' features, computed here (lanes 0-15 of the
// wavefront, one pair each, into LDS) instead of read from X.
struct FeatIn {
  const int32_t* pairs;
  const double* bodies;
  const int32_t* body_tree;
  const float* tree_radius;
  const double* max_time;
};
template <bool FEAT>
__global__ void __launch_bounds__(256) k_mlp_infer(int n, const float* X, const short* wb, float* Y, FeatIn F) {
  __shared__ float s_x[FEAT ? 4 : 1][16 * MLP_IN];
  __shared__ short w1[32 * MLP_H];  // K padded to 32
  __shared__ short w2[MLP_H * MLP_H];
  __shared__ short w3[MLP_H * 16];  // N padded to 16
  __shared__ float bias[2 * MLP_H + MLP_OUT];
  __shared__ short act[4][16 * MLP_H];
  for (int i = threadIdx.x; i < 32 * MLP_H; i += blockDim.x) {
    const int k = i / MLP_H;
    w1[i] = k < MLP_IN ? wb[OFF_W1 + i] : (short)0;
  }
  for (int i = threadIdx.x; i < MLP_H * MLP_H; i += blockDim.x) w2[i] = wb[OFF_W2 + i];
  for (int i = threadIdx.x; i < MLP_H * 16; i += blockDim.x) {
    const int k = i / 16, c = i % 16;
    w3[i] = c < MLP_OUT ? wb[OFF_W3 + k * MLP_OUT + c] : (short)0;
  }
  for (int i = threadIdx.x; i < MLP_H; i += blockDim.x) bias[i] = bf2f(wb[OFF_B1 + i]), bias[MLP_H + i] = bf2f(wb[OFF_B2 + i]);
  if (threadIdx.x < MLP_OUT) bias[2 * MLP_H + threadIdx.x] = bf2f(wb[OFF_B3 + threadIdx.x]);
  __syncthreads();
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  const int r = lane & 15, kq = lane >> 4;
  short* A = act[wid];
  const int n_tiles = (n + 15) / 16;
  for (int base = blockIdx.x * 4; base < n_tiles; base += gridDim.x * 4) {  // same trip count in every wave
    const int tile = base + wid;
    const int row = tile * 16 + r;
    const bool valid_row = tile < n_tiles && row < n;
    floatx4 acc[4];
    if (FEAT) {
      if (kq == 0 && valid_row)
        pair_features(row, F.pairs, F.bodies, F.body_tree, F.tree_radius, F.max_time, s_x[wid] + MLP_IN * r);
      wave_sync_lds();
    }
    // layer 1
    for (int nt = 0; nt < 4; ++nt) acc[nt] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < 2; ++ks) {
      bf16x4 a;
      for (int i = 0; i < 4; ++i) {
        const int k = ks * 16 + 4 * kq + i;
        const float xv = !(valid_row && k < MLP_IN) ? 0.f : FEAT ? s_x[FEAT ? wid : 0][MLP_IN * r + k]
                                                                  : X[(size_t)row * MLP_IN + k];
        a[i] = (valid_row && k < MLP_IN) ? f2bf(xv) : (short)0;
      }
      for (int nt = 0; nt < 4; ++nt) {
        bf16x4 b;
        for (int i = 0; i < 4; ++i) b[i] = w1[(ks * 16 + 4 * kq + i) * MLP_H + nt * 16 + r];
        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[nt], 0, 0, 0);
      }
    }
    for (int nt = 0; nt < 4; ++nt)
      for (int i = 0; i < 4; ++i) {
        const int m = 4 * kq + i, c = nt * 16 + r;
        const float v = acc[nt][i] + bias[c];
        A[m * MLP_H + c] = f2bf(v > 0.f ? v : 0.f);
      }
    __syncthreads();
    // layer 2
    for (int nt = 0; nt < 4; ++nt) acc[nt] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < 4; ++ks) {
      bf16x4 a;
      for (int i = 0; i < 4; ++i) a[i] = A[r * MLP_H + ks * 16 + 4 * kq + i];
      for (int nt = 0; nt < 4; ++nt) {
        bf16x4 b;
        for (int i = 0; i < 4; ++i) b[i] = w2[(ks * 16 + 4 * kq + i) * MLP_H + nt * 16 + r];
        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[nt], 0, 0, 0);
      }
    }
    __syncthreads();
    for (int nt = 0; nt < 4; ++nt)
      for (int i = 0; i < 4; ++i) {
        const int m = 4 * kq + i, c = nt * 16 + r;
        const float v = acc[nt][i] + bias[MLP_H + c];
        A[m * MLP_H + c] = f2bf(v > 0.f ? v : 0.f);
      }
    __syncthreads();
    // layer 3
    floatx4 out{0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < 4; ++ks) {
      bf16x4 a, b;
      for (int i = 0; i < 4; ++i) {
        a[i] = A[r * MLP_H + ks * 16 + 4 * kq + i];
        b[i] = w3[(ks * 16 + 4 * kq + i) * 16 + r];
      }
      out = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, out, 0, 0, 0);
    }
    if (r < MLP_OUT && tile < n_tiles)
      for (int i = 0; i < 4; ++i) {
        const int orow = tile * 16 + 4 * kq + i;
        if (orow < n) Y[(size_t)orow * MLP_OUT + r] = out[i] + bias[2 * MLP_H + r];
      }
    __syncthreads();
  }
}

// --------------------------------------------------------------- training
// Forward, backward and parameter gradient of a minibatch in FP32 with the
// bf16-rounded weights wf (the network inference evaluates).  Loss per
// sample: sum_o lw_o * huber_delta(y_o - t_o); the batch loss is its mean.
//
// A block takes tiles of MLP_TILE samples: weights, activations and deltas
// stay in LDS, thread (tx, ty) owns columns tx + 16 c of its two samples in
// the layers and a 4 x 4 patch of W2's gradient (2 x 4 of W1's) that it keeps
// in registers over its tiles.  Each block writes one partial gradient, and
// k_mlp_grad_sum adds the partials in a fixed order (deterministic).  The
// products are 24 MFLOP per 1000 samples, so what bounds it is filling the
// chip: tiles of 32 give 129 blocks at 4099 samples.  Before, one thread per
// sample (17 blocks) and one thread per parameter summing over the whole
// batch (23 blocks) took 85.9 + 1126 us there; now 21.1 + 4.0 us, and the
// shorter sums are closer to the exact gradient (8e-8 against 6e-6
// relative).
constexpr int MLP_TILE = 32;
constexpr int MLP_MAX_PART = 256;  // partial gradients (blocks) at most
__global__ void __launch_bounds__(256) k_mlp_fwd_bwd(int nb, const int* idx, const float* X, const float* T,
                                                     const float* wf, float lw0, float lw1, float delta_h, float* part,
                                                     float* loss) {
  constexpr int TS = MLP_TILE, LD = MLP_H + 1;  // rows padded by one: columns of a row and of W2 fall in different banks
  __shared__ float w1[MLP_IN * MLP_H], w2[MLP_H * LD], w3[MLP_H * MLP_OUT], bias[2 * MLP_H + MLP_OUT];
  __shared__ float sx[TS][MLP_IN + 1], h1[TS][LD], h2[TS][LD], d1[TS][LD], d2[TS][LD], d3[TS][MLP_OUT];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  for (int i = tid; i < MLP_IN * MLP_H; i += 256) w1[i] = wf[OFF_W1 + i];
  for (int i = tid; i < MLP_H * MLP_H; i += 256) w2[(i / MLP_H) * LD + i % MLP_H] = wf[OFF_W2 + i];
  if (tid < MLP_H * MLP_OUT) w3[tid] = wf[OFF_W3 + tid];
  if (tid < MLP_H) bias[tid] = wf[OFF_B1 + tid], bias[MLP_H + tid] = wf[OFF_B2 + tid];
  if (tid < MLP_OUT) bias[2 * MLP_H + tid] = wf[OFF_B3 + tid];
  float g2[4][4] = {}, g1[2][4] = {}, g3 = 0.f, gb = 0.f, gb3 = 0.f;
  for (int t0 = blockIdx.x * TS; t0 < nb; t0 += gridDim.x * TS) {
    __syncthreads();
    for (int i = tid; i < TS * MLP_IN; i += 256) {
      const int s = t0 + i / MLP_IN, k = i % MLP_IN;
      sx[i / MLP_IN][k] = s < nb ? X[(size_t)(idx ? idx[s] : s) * MLP_IN + k] : 0.f;
    }
    __syncthreads();
    float z[2][4];
    for (int c = 0; c < 4; ++c) z[0][c] = z[1][c] = bias[tx + 16 * c];
#pragma unroll 4
    for (int k = 0; k < MLP_IN; ++k) {
      const float x0 = sx[2 * ty][k], x1 = sx[2 * ty + 1][k];
      for (int c = 0; c < 4; ++c) {
        const float w = w1[k * MLP_H + tx + 16 * c];
        z[0][c] = fmaf(x0, w, z[0][c]), z[1][c] = fmaf(x1, w, z[1][c]);
      }
    }
    for (int q = 0; q < 2; ++q)
      for (int c = 0; c < 4; ++c) h1[2 * ty + q][tx + 16 * c] = z[q][c] > 0.f ? z[q][c] : 0.f;
    __syncthreads();
    for (int c = 0; c < 4; ++c) z[0][c] = z[1][c] = bias[MLP_H + tx + 16 * c];
#pragma unroll 8
    for (int k = 0; k < MLP_H; ++k) {
      const float x0 = h1[2 * ty][k], x1 = h1[2 * ty + 1][k];
      for (int c = 0; c < 4; ++c) {
        const float w = w2[k * LD + tx + 16 * c];
        z[0][c] = fmaf(x0, w, z[0][c]), z[1][c] = fmaf(x1, w, z[1][c]);
      }
    }
    for (int q = 0; q < 2; ++q)
      for (int c = 0; c < 4; ++c) h2[2 * ty + q][tx + 16 * c] = z[q][c] > 0.f ? z[q][c] : 0.f;
    __syncthreads();
    {  // outputs: a quarter of the sum per lane, then the loss and its derivative
      const int q = tid & 3, o = (tid >> 2) & 1, s = tid >> 3;
      float y = q == 0 ? bias[2 * MLP_H + o] : 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) y = fmaf(h2[s][16 * q + k], w3[(16 * q + k) * MLP_OUT + o], y);
      y += __shfl_xor(y, 1);
      y += __shfl_xor(y, 2);
      const bool valid = t0 + s < nb;
      const int src = valid ? (idx ? idx[t0 + s] : t0 + s) : 0;
      const float r = y - T[(size_t)src * MLP_OUT + o], ar = fabsf(r), lw = o ? lw1 : lw0;
      const float l = lw * (ar <= delta_h ? 0.5f * r * r : delta_h * (ar - 0.5f * delta_h));
      const float g = ar <= delta_h ? r : (r > 0.f ? delta_h : -delta_h);
      const float lo = __shfl_xor(l, 4);
      if (q == 0) d3[s][o] = valid ? lw * g / (float)nb : 0.f;
      if (q == 0 && o == 0 && valid) loss[t0 + s] = l + lo;
    }
    __syncthreads();
    for (int q = 0; q < 2; ++q) {
      const float e0 = d3[2 * ty + q][0], e1 = d3[2 * ty + q][1];
      for (int c = 0; c < 4; ++c) {
        const int j = tx + 16 * c;
        d2[2 * ty + q][j] = h2[2 * ty + q][j] > 0.f ? fmaf(w3[j * MLP_OUT + 1], e1, w3[j * MLP_OUT] * e0) : 0.f;
      }
    }
    __syncthreads();
    for (int c = 0; c < 4; ++c) z[0][c] = z[1][c] = 0.f;
#pragma unroll 8
    for (int j = 0; j < MLP_H; ++j) {
      const float x0 = d2[2 * ty][j], x1 = d2[2 * ty + 1][j];
      for (int c = 0; c < 4; ++c) {
        const float w = w2[(tx + 16 * c) * LD + j];
        z[0][c] = fmaf(x0, w, z[0][c]), z[1][c] = fmaf(x1, w, z[1][c]);
      }
    }
    for (int q = 0; q < 2; ++q)
      for (int c = 0; c < 4; ++c) d1[2 * ty + q][tx + 16 * c] = h1[2 * ty + q][tx + 16 * c] > 0.f ? z[q][c] : 0.f;
    __syncthreads();
#pragma unroll 4
    for (int s = 0; s < TS; ++s) {
      float a[4], e[4], f[4];
      for (int c = 0; c < 4; ++c) a[c] = h1[s][ty + 16 * c], e[c] = d2[s][tx + 16 * c], f[c] = d1[s][tx + 16 * c];
      const float x0 = sx[s][ty], x1 = ty < MLP_IN - 16 ? sx[s][ty + 16] : 0.f;
      for (int i = 0; i < 4; ++i)
        for (int c = 0; c < 4; ++c) g2[i][c] = fmaf(a[i], e[c], g2[i][c]);
      for (int c = 0; c < 4; ++c) g1[0][c] = fmaf(x0, f[c], g1[0][c]), g1[1][c] = fmaf(x1, f[c], g1[1][c]);
    }
    if (tid < MLP_H * MLP_OUT) {
      for (int s = 0; s < TS; ++s) g3 = fmaf(h2[s][tid >> 1], d3[s][tid & 1], g3);
    } else {
      const int j = tid & (MLP_H - 1);
      for (int s = 0; s < TS; ++s) gb += (tid & MLP_H) ? d2[s][j] : d1[s][j];
    }
    if (tid < MLP_OUT)
      for (int s = 0; s < TS; ++s) gb3 += d3[s][tid];
  }
  float* o = part + (size_t)blockIdx.x * MLP_PARAMS;
  for (int i = 0; i < 4; ++i)
    for (int c = 0; c < 4; ++c) o[OFF_W2 + (ty + 16 * i) * MLP_H + tx + 16 * c] = g2[i][c];
  for (int c = 0; c < 4; ++c) {
    o[OFF_W1 + ty * MLP_H + tx + 16 * c] = g1[0][c];
    if (ty < MLP_IN - 16) o[OFF_W1 + (ty + 16) * MLP_H + tx + 16 * c] = g1[1][c];
  }
  if (tid < MLP_H * MLP_OUT) o[OFF_W3 + tid] = g3;
  else o[((tid & MLP_H) ? OFF_B2 : OFF_B1) + (tid & (MLP_H - 1))] = gb;
  if (tid < MLP_OUT) o[OFF_B3 + tid] = gb3;
}

// The partial gradients' sum: 64 parameters per block, its eight wavefronts
// take every eighth partial and their sums are added in order.
__global__ void __launch_bounds__(512) k_mlp_grad_sum(int n_part, const float* part, float* grad) {
  __shared__ float s[8][64];
  const int lane = lane_id(), w = threadIdx.x >> 6, q = blockIdx.x * 64 + lane;
  float g = 0.f;
  if (q < MLP_PARAMS) {
#pragma unroll 4
    for (int p = w; p < n_part; p += 8) g += part[(size_t)p * MLP_PARAMS + q];
  }
  s[w][lane] = g;
  __syncthreads();
  if (w == 0 && q < MLP_PARAMS) {
    for (int k = 1; k < 8; ++k) g += s[k][lane];
    grad[q] = g;
  }
}

// Adam on the FP32 master weights; refreshes the bf16 copy and its float view.
__global__ void k_mlp_adam(float* w, float* m, float* v, const float* g, float lr, float beta1, float beta2, float eps,
                           float c1, float c2, short* wb, float* wf) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= MLP_PARAMS) return;
  const float gq = g[q];
  const float mq = beta1 * m[q] + (1.f - beta1) * gq;
  const float vq = beta2 * v[q] + (1.f - beta2) * gq * gq;
  m[q] = mq, v[q] = vq;
  const float wq = w[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
  w[q] = wq;
  const short h = f2bf(wq);
  wb[q] = h;
  wf[q] = bf2f(h);
}
__global__ void k_mlp_round(const float* w, short* wb, float* wf) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= MLP_PARAMS) return;
  const short h = f2bf(w[q]);
  wb[q] = h;
  wf[q] = bf2f(h);
}

// ------------------------------------------------------------- certificate
// Lower bounds of the distances the reference's sub-tests can report, from
// separating axes.  Along a unit axis u, set P lies below set Q by
// min_Q u.q - max_P u.p, a lower bound of their distance.  Three bounds:
//   world, per time: the CCD's edge-edge sub-tests lerp world positions, so a
//     point pair's offset at time t is the lerp of its offsets at the ends and
//     min(gap at start, gap at end) along one axis bounds every t;
//   b's frame: a point of a lerps between its start and end positions in b's
//     frame (point-triangle sub-tests) while b is fixed: the gap between the
//     union of a's two poses and b;
//   a's frame: the same with the bodies swapped.
// The discrete phase needs one bound: the two bodies at the future poses.
// A set's vertices are transformed once; axes come from Gilbert's minimum-norm-point iteration on the difference set
// (every iterate's axis gives a sound bound, the best one is kept).
constexpr int CERT_MAXV = 1024;  // vertices per body held in LDS; larger bodies are not certified
__device__ __forceinline__ void cert_mat(const double* m, const double* origin, float* o) {
  for (int r = 0; r < 3; ++r) {
    o[4 * r] = (float)m[4 * r], o[4 * r + 1] = (float)m[4 * r + 1], o[4 * r + 2] = (float)m[4 * r + 2];
    o[4 * r + 3] = (float)(m[4 * r + 3] - (origin ? origin[r] : 0.0));
  }
}
// A vertex set under a pose.  CertBlock: a block's, in LDS; CertWave: a
// wavefront's, in registers (vertex lane + 64 k in slot k), up to CERT_WAVEV.
constexpr int CERT_SLOTS = 4, CERT_WAVEV = 64 * CERT_SLOTS;
struct CertBlock {
  float* v;
  int n;
};
struct CertWave {
  float v[CERT_SLOTS][3];
  int n;
};
__device__ __forceinline__ void cert_move(const float* v, const float* m, float* o, float& mag) {
  const float x = v[0], y = v[1], z = v[2];
  o[0] = x, o[1] = y, o[2] = z;
  if (m) {
    o[0] = (m[0] * x + m[1] * y) + (m[2] * z + m[3]);
    o[1] = (m[4] * x + m[5] * y) + (m[6] * z + m[7]);
    o[2] = (m[8] * x + m[9] * y) + (m[10] * z + m[11]);
  }
  mag = fmaxf(mag, fmaxf(fabsf(o[0]), fmaxf(fabsf(o[1]), fabsf(o[2]))));
}
// n body-frame vertices under the 3x4 matrix m (as they are when null).
__device__ __forceinline__ void cert_load(const float* v, int n, const float* m, CertBlock& S, float& mag) {
  S.n = n;
  for (int k = threadIdx.x; k < n; k += blockDim.x) cert_move(v + 3 * k, m, S.v + 3 * k, mag);
}
__device__ __forceinline__ void cert_load(const float* v, int n, const float* m, CertWave& S, float& mag) {
  S.n = n;
#pragma unroll
  for (int k = 0; k < CERT_SLOTS; ++k) {
    S.v[k][0] = S.v[k][1] = S.v[k][2] = 0.f;
    if (lane_id() + 64 * k < n) cert_move(v + 3 * (lane_id() + 64 * k), m, S.v[k], mag);
  }
}
// Largest magnitude of all lanes' (block: and the sets are complete).
__device__ __forceinline__ float cert_mag(const CertBlock&, float m, float* mag_red) {
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) mag_red[threadIdx.x >> 6] = m;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r = fmaxf(r, mag_red[i]);
  return r;
}
__device__ __forceinline__ float cert_mag(const CertWave&, float m, float*) {
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  return m;
}
__device__ __forceinline__ void cert_reuse(const CertBlock&) { __syncthreads(); }  // before a set is loaded anew
__device__ __forceinline__ void cert_reuse(const CertWave&) {}
// Extreme of u.x over A (and B: TWO) (sign +1: max, -1: min) and the point
// attaining it; of equal ones the first vertex's, A's before B's.
template <bool TWO>
__device__ float cert_extreme(const CertBlock& A, const CertBlock& B, const float* u, float sign, float* pt, float* red) {
  float best = -3.4e38f, bp[3] = {0.f, 0.f, 0.f};
  for (int s = 0; s < (TWO ? 2 : 1); ++s) {
    const CertBlock& S = s ? B : A;
    for (int k = threadIdx.x; k < S.n; k += blockDim.x) {
      const float* q = S.v + 3 * k;
      const float pr = sign * ((u[0] * q[0] + u[1] * q[1]) + u[2] * q[2]);
      if (pr > best) best = pr, bp[0] = q[0], bp[1] = q[1], bp[2] = q[2];
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    const float ob = __shfl_xor(best, off);
    const float o0 = __shfl_xor(bp[0], off), o1 = __shfl_xor(bp[1], off), o2 = __shfl_xor(bp[2], off);
    if (ob > best) best = ob, bp[0] = o0, bp[1] = o1, bp[2] = o2;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    float* r = red + 4 * (threadIdx.x >> 6);
    r[0] = best, r[1] = bp[0], r[2] = bp[1], r[3] = bp[2];
  }
  __syncthreads();
  int w = 0;
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i)
    if (red[4 * i] > red[4 * w]) w = i;
  pt[0] = red[4 * w + 1], pt[1] = red[4 * w + 2], pt[2] = red[4 * w + 3];
  return sign * red[4 * w];
}
template <bool TWO>
__device__ __forceinline__ float cert_extreme(const CertWave& A, const CertWave& B, const float* u, float sign, float* pt,
                                              float*) {
  float best = -3.4e38f, bp[3] = {0.f, 0.f, 0.f};
  int bv = 1 << 20;
#pragma unroll
  for (int k = 0; k < CERT_SLOTS; ++k) {
    const int v = lane_id() + 64 * k;
#pragma unroll
    for (int s = 0; s < (TWO ? 2 : 1); ++s) {
      const CertWave& S = s ? B : A;
      const float* q = S.v[k];
      const float pr = sign * ((u[0] * q[0] + u[1] * q[1]) + u[2] * q[2]);
      if (v < S.n && pr > best) best = pr, bp[0] = q[0], bp[1] = q[1], bp[2] = q[2], bv = v;
    }
  }
  float top = best;
  for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
  unsigned long long m = __ballot(best == top);
  int l = __ffsll((long long)m) - 1;
  for (m &= m - 1ull; m; m &= m - 1ull) {
    const int o = __ffsll((long long)m) - 1;
    if (rl(bv, o) < rl(bv, l)) l = o;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) pt[k] = __int_as_float(rl(__float_as_int(bp[k]), l));
  return sign * top;
}
// Separation bound of P (P0, P1: TWO) below Q along u: (min_Q u.q - max_P u.p)
// / |u|, and the support points.
template <bool TWO, class Set>
__device__ __forceinline__ float cert_axis(const Set& P0, const Set& P1, const Set& Q, const float* u, float* pp, float* qq,
                                           float* red) {
  const float nu = sqrtf((u[0] * u[0] + u[1] * u[1]) + u[2] * u[2]);
  const float hp = cert_extreme<TWO>(P0, P1, u, 1.f, pp, red);
  const float lq = cert_extreme<false>(Q, Q, u, -1.f, qq, red);
  return nu > 1e-30f ? (lq - hp) / nu : -3.4e38f;
}
// Gilbert's minimum-norm-point iteration on the difference set Q - P from the
// point x0 (a member of its hull): the support point s = argmin (x.d) over
// Q - P bounds the distance by x.s / |x| at every step (kept as the best
// bound), and x moves to the point of segment [x, s] closest to the origin.
// Returns the best bound; u_out = its axis.
// With stop >= 0 the iteration ends as soon as the answer to "best > stop"
// is known: a gap above stop, or an iterate x with |x| <= stop (x lies in the
// hull of the difference set, so no axis can separate it by more than |x|).
template <bool TWO, class Set>
__device__ __forceinline__ float cert_gilbert(const Set& P0, const Set& P1, const Set& Q, const float* x0, int iters,
                                              float* u_out, float* red, float stop = -1.f) {
  float x[3] = {x0[0], x0[1], x0[2]};
  float best = -3.4e38f;
  u_out[0] = x[0], u_out[1] = x[1], u_out[2] = x[2];
#pragma unroll 1
  for (int it = 0; it < iters; ++it) {
    const float xx = (x[0] * x[0] + x[1] * x[1]) + x[2] * x[2];
    if (!(xx > 1e-30f)) break;
    if (stop >= 0.f && it > 0 && xx <= stop * stop) break;
    float pp[3], qq[3];
    const float g = cert_axis<TWO>(P0, P1, Q, x, pp, qq, red);
    if (g > best) best = g, u_out[0] = x[0], u_out[1] = x[1], u_out[2] = x[2];
    if (stop >= 0.f && best > stop) break;
    const float sd[3] = {qq[0] - pp[0], qq[1] - pp[1], qq[2] - pp[2]};
    const float xs = (x[0] * sd[0] + x[1] * sd[1]) + x[2] * sd[2];
    if (xx - xs <= 1e-7f * xx) break;  // x is (nearly) the minimum-norm point
    const float e[3] = {x[0] - sd[0], x[1] - sd[1], x[2] - sd[2]};
    const float ee = (e[0] * e[0] + e[1] * e[1]) + e[2] * e[2];
    float lam = ee > 0.f ? (xx - xs) / ee : 0.f;  // x + lam (s - x) is closest to the origin
    lam = fminf(fmaxf(lam, 0.f), 1.f);
    x[0] += lam * (sd[0] - x[0]), x[1] += lam * (sd[1] - x[1]), x[2] += lam * (sd[2] - x[2]);
  }
  return best;
}
// Per-time world bound: min over the two instants of the separation along one
// axis, the axis taken from each instant's own Gilbert iteration.
template <class Set>
__device__ __forceinline__ float cert_gap_timed(const Set& P0, const Set& P1, const Set& Q0, const Set& Q1, const float* x0,
                                                const float* x1, int iters, float* red) {
  float ax[3][3];
  (void)cert_gilbert<false>(P0, P0, Q0, x0, iters, ax[0], red);
  (void)cert_gilbert<false>(P1, P1, Q1, x1, iters, ax[1], red);
  const float n0 = sqrtf((ax[0][0] * ax[0][0] + ax[0][1] * ax[0][1]) + ax[0][2] * ax[0][2]);
  const float n1 = sqrtf((ax[1][0] * ax[1][0] + ax[1][1] * ax[1][1]) + ax[1][2] * ax[1][2]);
#pragma unroll
  for (int r = 0; r < 3; ++r) ax[2][r] = (n0 > 0.f ? ax[0][r] / n0 : 0.f) + (n1 > 0.f ? ax[1][r] / n1 : 0.f);
  float best = -3.4e38f;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float pp[3], qq[3];
    const float g0 = cert_axis<false>(P0, P0, Q0, ax[c], pp, qq, red);
    const float g1 = cert_axis<false>(P1, P1, Q1, ax[c], pp, qq, red);
    best = fmaxf(best, fminf(g0, g1));
  }
  return best;
}
constexpr int CERT_ITERS = 16;
constexpr int CERT_LIST = 1024;  // pairs per block at most (the grids are sized for it)
// Whether a pair's bodies (hull vertices va, vb) are provably apart by more
// than thr: CCD (mode 0) or at the future poses (mode 1).  S: the sets' storage.
template <class Set>
__device__ __forceinline__ bool cert_pair(int mode, const double* pr, const float* va, int na, const float* vb, int nb,
                                          float thr, Set (&S)[4], float* red, float* mag_red) {
  const float EPSF = 5.9604645e-08f;
  float m0[12], m1[12], m2[12], m3[12], u[3], ax[3];
  float mag = 0.f;
  if (mode != 0) {
    const double o[3] = {pr[PR_TB1 + 3], pr[PR_TB1 + 7], pr[PR_TB1 + 11]};
    cert_mat(pr + PR_TA1, o, m0), cert_mat(pr + PR_TB1, o, m1);
    cert_load(va, na, m0, S[0], mag), cert_load(vb, nb, m1, S[1], mag);
    const float M = cert_mag(S[0], mag, mag_red);
    for (int k = 0; k < 3; ++k) u[k] = m1[4 * k + 3] - m0[4 * k + 3];
    const float margin = 1e-6f + 64.f * EPSF * M;
    return cert_gilbert<false>(S[0], S[0], S[1], u, CERT_ITERS, ax, red, thr + margin) - margin > thr;
  }
  const double o[3] = {pr[PR_TB0 + 3], pr[PR_TB0 + 7], pr[PR_TB0 + 11]};
  cert_mat(pr + PR_TA0, o, m0), cert_mat(pr + PR_TA1, o, m1), cert_mat(pr + PR_TB0, o, m2), cert_mat(pr + PR_TB1, o, m3);
  cert_load(va, na, m0, S[0], mag), cert_load(va, na, m1, S[1], mag);
  cert_load(vb, nb, m2, S[2], mag), cert_load(vb, nb, m3, S[3], mag);
  const float M = cert_mag(S[0], mag, mag_red);
  {  // world, per instant: (a at start, b at start), (a at end, b at end)
    float x0[3], x1[3];
    for (int k = 0; k < 3; ++k) x0[k] = m2[4 * k + 3] - m0[4 * k + 3], x1[k] = m3[4 * k + 3] - m1[4 * k + 3];
    if (!(cert_gap_timed(S[0], S[1], S[2], S[3], x0, x1, CERT_ITERS, red) - (1e-6f + 64.f * EPSF * M) > thr)) return false;
  }
#pragma unroll 1
  for (int f = 0; f < 2; ++f) {  // a's two poses in b's frame against b, then the other way round
    cert_reuse(S[0]);
    mag = 0.f;
    cert_mat(pr + (f ? PR_MBA0 : PR_MAB0), nullptr, m0), cert_mat(pr + (f ? PR_MBA1 : PR_MAB1), nullptr, m1);
    const float* v = f ? vb : va;
    const int n = f ? nb : na;
    cert_load(v, n, m0, S[0], mag), cert_load(v, n, m1, S[1], mag);
    cert_load(f ? va : vb, f ? na : nb, nullptr, S[2], mag);
    const float M2 = cert_mag(S[0], mag, mag_red);
    for (int k = 0; k < 3; ++k) u[k] = -0.5f * (m0[4 * k + 3] + m1[4 * k + 3]);
    if (!(cert_gilbert<true>(S[0], S[1], S[2], u, CERT_ITERS, ax, red) - (1e-6f + 64.f * EPSF * M2) > thr)) return false;
  }
  return true;
}
struct CertIn {
  int n_pairs;
  const int32_t *pair_info, *body_tree;
  const double* pair_rec;
  const float* Y;
  float t_gate, s_gate;
  const int32_t* hv_off;
  const float *hv, *tree_eps_out;
  int mode;
};
// A pair's part in the certificate: 0 not proposed, or proposed with hulls
// beyond CERT_MAXV (kept); 1 a wavefront's, 2 a block's.
__device__ __forceinline__ int cert_kind(const CertIn& C, int p, bool& gated, int& ta, int& tb, int& na, int& nb) {
  gated = !C.Y || (C.Y[2 * p] >= C.s_gate && C.Y[2 * p + 1] >= C.t_gate);
  ta = C.body_tree[C.pair_info[4 * p]], tb = C.body_tree[C.pair_info[4 * p + 1]];
  na = C.hv_off[ta + 1] - C.hv_off[ta], nb = C.hv_off[tb + 1] - C.hv_off[tb];
  const int m = na > nb ? na : nb;
  return !gated || m > CERT_MAXV ? 0 : m > CERT_WAVEV ? 2 : 1;
}

// gate: the MLP outputs (y0 >= s_gate and y1 >= t_gate), or every pair when
// null.  keep[p] = 0 for a certified pair, 1 otherwise.  counters[0..1]:
// proposed / certified pairs.  The kept pairs are the phase's roots: each
// block appends its kept pairs to soup with one atomic on *n_soup (zeroed by
// the phase's set-up; the discrete and CCD lists need no order).
//
// A wavefront per pair while both hulls have at most 256 vertices: they sit in
// its registers, and a support point is a few products and one reduction.  A
// block per pair met two barriers for each of the ~100 support points of a CCD
// certificate (1,773 pairs, 548 of them proposed: 183 -> 78 us); k_certify_block still takes the larger hulls.
__global__ void __launch_bounds__(256) k_certify(CertIn C, int* keep, unsigned long long* counters, NP* soup,
                                                 unsigned long long* n_soup) {
  __shared__ int s_kept[CERT_LIST];
  __shared__ int s_nk, s_cnt[2];
  __shared__ unsigned long long s_base;
  if (threadIdx.x == 0) s_nk = 0, s_cnt[0] = 0, s_cnt[1] = 0;
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (int p = 4 * (int)blockIdx.x + wv; p < C.n_pairs; p += 4 * (int)gridDim.x) {
    bool gated;
    int ta, tb, na, nb;
    const int kind = cert_kind(C, p, gated, ta, tb, na, nb);
    if (kind == 2) continue;
    bool ok = false;
    if (kind == 1) {
      CertWave S[4];
      ok = cert_pair(C.mode, C.pair_rec + (size_t)PR_STRIDE * p, C.hv + 3 * (size_t)C.hv_off[ta], na,
                     C.hv + 3 * (size_t)C.hv_off[tb], nb,
                     (float)C.pair_rec[(size_t)PR_STRIDE * p + PR_SEARCH] + C.tree_eps_out[ta] + C.tree_eps_out[tb], S,
                     nullptr, nullptr);
    }
    if (lane_id() == 0) {
      keep[p] = ok ? 0 : 1;
      if (!ok) s_kept[atomicAdd(&s_nk, 1)] = p;
      if (gated) atomicAdd(&s_cnt[0], 1);
      if (ok) atomicAdd(&s_cnt[1], 1);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    s_base = s_nk ? atomicAdd(n_soup, (unsigned long long)s_nk) : 0ull;
    if (s_cnt[0]) atomicAdd(&counters[0], (unsigned long long)s_cnt[0]);
    if (s_cnt[1]) atomicAdd(&counters[1], (unsigned long long)s_cnt[1]);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < s_nk; i += blockDim.x)
    soup[s_base + i] = NP{(uint32_t)s_kept[i], 0u, 0u, 0u, 0ull};
}
// The pairs k_certify leaves: a hull of more than 256 vertices (a block each).
__global__ void __launch_bounds__(256) k_certify_block(CertIn C, int* keep, unsigned long long* counters, NP* soup,
                                                       unsigned long long* n_soup) {
  __shared__ float buf[4][3 * CERT_MAXV];
  __shared__ float red[4 * 16];
  __shared__ float mag_red[16];
  __shared__ int s_kept[CERT_LIST];
  __shared__ int s_nk;
  __shared__ unsigned long long s_base;
  if (threadIdx.x == 0) s_nk = 0;
  for (int p = blockIdx.x; p < C.n_pairs; p += gridDim.x) {
    bool gated;
    int ta, tb, na, nb;
    if (cert_kind(C, p, gated, ta, tb, na, nb) != 2) continue;
    CertBlock S[4] = {{buf[0], 0}, {buf[1], 0}, {buf[2], 0}, {buf[3], 0}};
    const bool ok = cert_pair(C.mode, C.pair_rec + (size_t)PR_STRIDE * p, C.hv + 3 * (size_t)C.hv_off[ta], na,
                              C.hv + 3 * (size_t)C.hv_off[tb], nb,
                              (float)C.pair_rec[(size_t)PR_STRIDE * p + PR_SEARCH] + C.tree_eps_out[ta] +
                                  C.tree_eps_out[tb],
                              S, red, mag_red);
    if (threadIdx.x == 0) {
      keep[p] = ok ? 0 : 1;
      if (!ok) s_kept[s_nk++] = p;
      atomicAdd(&counters[0], 1ull);
      if (ok) atomicAdd(&counters[1], 1ull);
    }
    __syncthreads();  // LDS reuse by the next pair
  }
  __syncthreads();
  if (threadIdx.x == 0) s_base = s_nk ? atomicAdd(n_soup, (unsigned long long)s_nk) : 0ull;
  __syncthreads();
  for (int i = threadIdx.x; i < s_nk; i += blockDim.x)
    soup[s_base + i] = NP{(uint32_t)s_kept[i], 0u, 0u, 0u, 0ull};
}

