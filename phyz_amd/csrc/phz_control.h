// phz_control.h — the device-resident control loop for gfx950 (CDNA4):
// FK readout, observation ops and the MLP policy pass.
//
// Behaviour follows crates/phyz-gpu/src/policy_pipeline.rs (ObsOp, PolicySpec,
// observe_reference, policy_reference, KernelRng) and the reference passes
// crates/phyz-gpu/cuda/phyz_kernels.cu:1423-1715 (fk_thread, obs_thread,
// policy_thread). The layout here is this library's own:
//
//   phz_obs     one lane per world, model and op table compiled in (the host
//               emits `struct Model` and `struct Obs` of constexpr tables).
//               FK in registers; the FK readout rows and the observation row
//               are stored structure-of-arrays ([j][stride]) so a wave's
//               stores coalesce.
//   phz_policy  one wave per 16*CB worlds. The three MLP layers run on MFMA
//               with the weights as the A operand and the activations as the
//               B operand, so a layer's 16x16 output tiles are already laid
//               out as the next layer's B fragments: hidden activations never
//               leave registers. The first layer is f32 (16x16x4f32); the
//               second and third take both operands as three bf16 pieces
//               (tanh_layer_split). Only the per-world prologue (input noise)
//               and epilogue (Gaussian sample, log-prob, PD targets) go
//               through LDS, because each world's random stream is sequential
//               and lives in one lane. Small launches give a tile of 16 or 32
//               worlds to a workgroup of 4 or 8 waves instead (policy_team).
#pragma once

namespace phz {

// ── FK readout and observations ──────────────────────────────────────────────

// Observation op kinds: the packed table row [kind, a, b, c] of ObsOp::pack
// (crates/phyz-gpu/src/policy_pipeline.rs:115-137).
enum {
  OBS_CONST = 0,    // c
  OBS_QMINUS = 1,   // q[a] - c
  OBS_V = 2,        // v[a]
  OBS_PITCH = 3,    // atan2(-r02, r22), r = world->body rotation of body a
  OBS_ROLL = 4,     // atan2(r12, r22)
  OBS_YAWERR = 5,   // wrap(c - atan2(r01, r00))
  OBS_POSZ = 6,     // body a origin z, world
  OBS_POS = 7,      // body a origin, world axis b
  OBS_COM_SUPPORT = 8  // centre of mass minus mean support point, axis c; aux window (a, b)
};

constexpr int XF_STRIDE = 18;  // rotation world->body (9, row-major), origin (3), omega (3), v (3), body frame

struct ObsArgs {
  const void* q;  // [nq][stride] T
  const void* v;  // [nv][stride] T
  void* kin;      // [nb * XF_STRIDE][stride] T, written when write_kin
  float* obs;     // [n_in][stride] f32, the history row of this control step, written when write_obs
  void* hq;       // state-history rows ([nq][stride], [nv][stride] T) of the control step before,
  void* hv;       // whose final state is the one read here; null to record nothing
  int nworld;
  int stride;
  int write_kin;
  int write_obs;
};

template <class M, class T> struct FKState {
  R3<T> Rw[M::NB];  // body -> world rotation
  V3<T> Pw[M::NB];  // body origin in world
  SV<T> vel[M::NB]; // body-frame spatial velocity
};

// Forward kinematics of every body (crates/phyz-rigid/src/kinematics.rs:10-50,
// the same chain as the reference's fk_world).
template <class M, class T> __device__ __forceinline__ void fk_all(const T* q, const T* v, FKState<M, T>& f) {
  sfor<0, M::NB>([&](auto I) {
    constexpr int i = decltype(I)::value;
    constexpr int p = M::parent[i];
    Xf<T> X;
    SV<T> vj;
    joint_xf<M, T, i>(q, v, X, vj);
    if constexpr (p < 0) {
      f.vel[i] = vj;
      f.Rw[i] = transpose(X.E);
      f.Pw[i] = X.r;
    } else {
      f.vel[i] = apply_motion(X, f.vel[p]) + vj;
      f.Rw[i] = mul_bt(f.Rw[p], X.E);
      f.Pw[i] = f.Pw[p] + mul(f.Rw[p], X.r);
    }
  });
}

template <class T> __device__ __forceinline__ T wrap_pi(T a) {
  const T pi = T(3.14159265358979323846);
  while (a > pi) a -= T(2) * pi;
  while (a < -pi) a += T(2) * pi;
  return a;
}

template <class T> __device__ __forceinline__ T axis_of(V3<T> p, int axis) {
  return axis == 0 ? p.x : (axis == 1 ? p.y : p.z);
}

// One feature (ObsOp::eval, policy_pipeline.rs:189-249). The world->body
// rotation r is Rw^T, so r[i][j] = Rw.m[3 j + i].
template <class M, class O, class T, int k>
__device__ __forceinline__ T obs_feature(const T* q, const T* v, const FKState<M, T>& f) {
  constexpr int kind = O::kind[k], a = O::a[k], b = O::b[k];
  if constexpr (kind == OBS_CONST) {
    return T(O::c[k]);
  } else if constexpr (kind == OBS_QMINUS) {
    return q[a] - T(O::c[k]);
  } else if constexpr (kind == OBS_V) {
    return v[a];
  } else if constexpr (kind == OBS_PITCH) {
    return datan2(-f.Rw[a].m[6], f.Rw[a].m[8]);
  } else if constexpr (kind == OBS_ROLL) {
    return datan2(f.Rw[a].m[7], f.Rw[a].m[8]);
  } else if constexpr (kind == OBS_YAWERR) {
    return wrap_pi(T(O::c[k]) - datan2(f.Rw[a].m[3], f.Rw[a].m[0]));
  } else if constexpr (kind == OBS_POSZ) {
    return f.Pw[a].z;
  } else if constexpr (kind == OBS_POS) {
    return axis_of(f.Pw[a], b > 2 ? 2 : b);
  } else {
    // ComOverSupport: aux window [heading_flag, heading_body, (body, ox, oy, oz) x b] at a.
    if constexpr (b == 0) {
      return T(0);
    } else {
      V3<T> com = v3(T(0), T(0), T(0));
      T mt = T(0);
      sfor<0, M::NB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if constexpr (M::mass[i] > 0.0) {
          const V3<T> c = v3(T(M::com[i][0]), T(M::com[i][1]), T(M::com[i][2]));
          com = com + (f.Pw[i] + mul(f.Rw[i], c)) * T(M::mass[i]);
          mt = mt + T(M::mass[i]);
        }
      });
      if (mt > T(0)) com = com * (T(1) / dmax(mt, T(1e-30)));
      V3<T> tgt = v3(T(0), T(0), T(0));
      sfor<0, b>([&](auto J) {
        constexpr int base = a + 2 + 4 * decltype(J)::value;
        constexpr int body = (int)O::aux[base];
        const V3<T> o = v3(T(O::aux[base + 1]), T(O::aux[base + 2]), T(O::aux[base + 3]));
        tgt = tgt + f.Pw[body] + mul(f.Rw[body], o);
      });
      const V3<T> e = com - tgt * (T(1) / T(b));
      constexpr int axis = (int)O::c[k];
      if constexpr (O::aux[a] != 0.0) {
        constexpr int h = (int)O::aux[a + 1];
        const T yaw = datan2(f.Rw[h].m[3], f.Rw[h].m[0]);
        T sy, cy;
        dsincos(yaw, &sy, &cy);
        if constexpr (axis == 0) return cy * e.x + sy * e.y;
        else if constexpr (axis == 1) return -sy * e.x + cy * e.y;
        else return e.z;
      } else {
        return axis_of(e, axis);
      }
    }
  }
}

template <class M, class O, class T> __device__ __forceinline__ void obs_world(const ObsArgs& a, int w) {
  const T* gq = (const T*)a.q;
  const T* gv = (const T*)a.v;
  const int S = a.stride;
  T q[M::NQ], v[M::NV];
#pragma unroll
  for (int j = 0; j < M::NQ; j++) q[j] = gq[j * S + w];
#pragma unroll
  for (int j = 0; j < M::NV; j++) v[j] = gv[j * S + w];
  if (a.hq != nullptr) {
#pragma unroll
    for (int j = 0; j < M::NQ; j++) ((T*)a.hq)[j * S + w] = q[j];
#pragma unroll
    for (int j = 0; j < M::NV; j++) ((T*)a.hv)[j * S + w] = v[j];
  }
  FKState<M, T> f;
  fk_all<M, T>(q, v, f);
  if (a.write_kin) {
    T* kin = (T*)a.kin;
    sfor<0, M::NB>([&](auto I) {
      constexpr int i = decltype(I)::value;
      T* r = kin + (size_t)(i * XF_STRIDE) * S + w;
      const R3<T> wb = transpose(f.Rw[i]);
#pragma unroll
      for (int k = 0; k < 9; k++) r[k * S] = wb.m[k];
      r[9 * S] = f.Pw[i].x;
      r[10 * S] = f.Pw[i].y;
      r[11 * S] = f.Pw[i].z;
      r[12 * S] = f.vel[i].a.x;
      r[13 * S] = f.vel[i].a.y;
      r[14 * S] = f.vel[i].a.z;
      r[15 * S] = f.vel[i].l.x;
      r[16 * S] = f.vel[i].l.y;
      r[17 * S] = f.vel[i].l.z;
    });
  }
  if constexpr (O::N > 0) {
    if (a.write_obs) {
      sfor<0, O::N>([&](auto K) {
        constexpr int k = decltype(K)::value;
        a.obs[(size_t)k * S + w] = (float)obs_feature<M, O, T, k>(q, v, f);
      });
    }
  }
}

// ── policy: two-hidden-layer tanh MLP, diagonal Gaussian, PD targets ─────────

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct PolicyArgs {
  const f32x4* w1;     // [KU][NHB][64] x 4 fragments of W1 (host re-layout, zero padded)
  const f32x4* w2;     // W2, input block major: [KB2][NHB][3][64] x 8 bf16 pieces (P::SPLIT), or
                       // [NHB][NHB][64] x 4 floats
  const f32x4* w3;     // W3 likewise, NOB output blocks
  const float* bias;   // b1[NHB*16] b2[NHB*16] b3[NOB*16], zero padded
  const float* stdv;   // [NO]
  float* obs;          // [NI][stride], this control step's history row (noised in place)
  float* out;          // [NO + 1][stride], actions then log-prob
  u64* rng;            // [stride] policy streams
  float* z;            // [NO][stride] AR(1) noise state
  const void* base;    // [NPD][stride] T, base PD targets
  void* targets;       // [NPD][stride] T, PD targets the step kernel reads
  int nworld;
  int stride;
};

// KernelRng::uniform / normal (policy_pipeline.rs:441-456): 53-bit uniform,
// Box-Muller on two uniforms, cosine branch, in double: sqrt(-2 ln u1) cos(2 pi
// u2) with u1 >= 1e-300. The uniforms come from the draws' 32-bit words in one
// exact fma each; ln is tab_log and the root nr_sqrt (the step kernels' f64
// Box-Muller, within 1 ulp each); the cosine is taken in turns, where the
// reduction is exact (t = 64 u2, k = rint(t), r = (t - k) 2 pi / 64) and the
// LDS table gives cos(2 pi k / 64), within 2 ulp of the cosine of the exact
// angle. These 37 normals per world and control step are the part of the
// policy kernel that does not overlap its MFMAs; the kernel fills the tables
// at its start.
__device__ __forceinline__ double uniform_of(u64 x) {
  return fma((double)(unsigned)(x >> 32), 0x1p-32, (double)((unsigned)x >> 11) * 0x1p-53);
}
__device__ __forceinline__ double turns_of(u64 x) {
  return fma((double)(unsigned)(x >> 32), 0x1p-26, (double)((unsigned)x >> 11) * 0x1p-47);
}
__device__ __forceinline__ void policy_uniforms(u64& s, double& u1, double& t) {
  u1 = uniform_of(xorshift64(s));
  t = turns_of(xorshift64(s));
}
__device__ __forceinline__ double policy_transform(double u1, double t) {
  const double k = rint(t);
  double sn, cs;
  tab_sincos_at((t - k) * 0x1.921fb54442d18p-4, cvt_sat_i32(k) & 63, &sn, &cs);
  return nr_sqrt(-2.0 * tab_log(fmax(u1, 1e-300))) * cs;
}
__device__ __forceinline__ double policy_normal(u64& s) {
  double u1, t;
  policy_uniforms(s, u1, t);
  return policy_transform(u1, t);
}

// A double from lane `lane ^ 32`, the other half of the wave (ds_bpermute,
// which every lane of the wave executes).
__device__ __forceinline__ double from_other_half(double v, int lane) {
  const u64 b = __builtin_bit_cast(u64, v);
  const int addr = (lane ^ 32) << 2;
  const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)b);
  const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((u64)hi << 32) | lo);
}

// The next N normals of the stream in lanes 0..31 (one world each; lanes
// 32..63 own none), the same values as N calls of policy_normal there. The
// world's lane draws every pair of uniforms in order; the transforms, the
// costly part, run two at a time: normal 2j in the world's lane and normal
// 2j + 1 in lane + 32, whose uniforms and result cross the wave's halves.
// Lanes 32..63 advance a stream of their own that nothing reads. Every lane
// of the wave calls it, outside any branch.
template <int N> __device__ __forceinline__ void policy_normals_paired(u64& s, int lane, double (&n)[N]) {
#pragma unroll
  for (int j = 0; j < N; j += 2) {
    double u1a, ta, u1b = 0.5, tb = 0.0;
    policy_uniforms(s, u1a, ta);
    if (j + 1 < N) policy_uniforms(s, u1b, tb);
    const double pu = from_other_half(u1b, lane), pt = from_other_half(tb, lane);
    const bool upper = lane >= 32;
    const double r = policy_transform(upper ? pu : u1a, upper ? pt : ta);
    n[j] = r;
    if (j + 1 < N) n[j + 1] = from_other_half(r, lane);
  }
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// tanh without branches, from tanh|x| = (1 - t) / (1 + t), t = e^(-2|x|) = 2^(-2|x| log2 e)
// (hardware exp2 and reciprocal, about 1 ulp each), and the odd series
// x - x^3/3 + 2x^5/15 - 17x^7/315 below |x| = 1/16, where 1 - t cancels; the
// series' first omitted term is under 1e-12 relative there. Absolute error
// stays near 2e-7 over the whole range; NaN propagates.
__device__ __forceinline__ float tanh_mlp(float x) {
  const float ax = fabsf(x);
  const float t = __builtin_amdgcn_exp2f(-2.88539008177792681f * ax);
  const float big = (1.0f - t) * __builtin_amdgcn_rcpf(1.0f + t);
  const float x2 = x * x;
  const float small = ax * (1.0f + x2 * (-0.333333333333f + x2 * (0.133333333333f + x2 * -0.0539682539683f)));
  return copysignf(ax < 0.0625f ? small : big, x);
}

template <int NB_, int CB> __device__ __forceinline__ void bias_tiles(const float* bias, int g, f32x4 (&acc)[NB_][CB]) {
#pragma unroll
  for (int ob = 0; ob < NB_; ob++) {
    f32x4 b0;
#pragma unroll
    for (int j = 0; j < 4; j++) b0[j] = bias[ob * 16 + 4 * g + j];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) acc[ob][cb] = b0;
  }
}

template <int NB_, int CB> __device__ __forceinline__ void tanh_tiles(f32x4 (&h)[NB_][CB]) {
#pragma unroll
  for (int ob = 0; ob < NB_; ob++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int j = 0; j < 4; j++) h[ob][cb][j] = tanh_mlp(h[ob][cb][j]);
}

// acc[ob][cb] += sum over k of W[ob block][k] B[k][cb block]. The weights are
// fragments [kb][ob][lane] x 4 (component s = k-step s of input block kb), read
// in that order as one contiguous stream with PF fragments in flight; the
// sched_barrier keeps the compiler from sinking the prefetches to their use,
// which would expose a full L2 round trip per fragment. bfrag(kb, s, cb) is
// the B operand (this lane's input value) of k-step s of block kb for world
// block cb.
template <int NKB, int NOB_, int CB, class BF>
__device__ __forceinline__ void mfma_layer(const f32x4* __restrict__ w, int lane, f32x4 (&acc)[NOB_][CB], BF bfrag) {
  constexpr int NT = NKB * NOB_;
  constexpr int PF = NT < 6 ? NT : 6;
  f32x4 ring[PF];
#pragma unroll
  for (int t = 0; t < PF; t++) ring[t] = w[t * 64 + lane];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int kb = t / NOB_, ob = t % NOB_;
    const f32x4 wa = ring[t % PF];
    if (t + PF < NT) ring[t % PF] = w[(t + PF) * 64 + lane];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int cb = 0; cb < CB; cb++) acc[ob][cb] = mfma4(wa[s], bfrag(kb, s, cb), acc[ob][cb]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ── layers 2 and 3 in three bf16 pieces ──
// An f32 is the exact sum of three bf16 values, each the rounding of what the
// ones before it left (8 significant bits each, signed remainders):
// x = h + m + l with |m| <= 2^-8 |x|, |l| <= 2^-17 |x|. A product takes the
// six partial products hh, hm, mh, hl, lh, mm; the dropped ml and lm are up to
// 2^-25 of it each (ll 2^-34), half a unit in the last place of an f32 product
// together where both operands' pieces are at their largest with one sign. In
// return bf16 products are exact in f32 and the MFMA sums 32 of them with one
// rounding where the f32 MFMA rounds per 4: six roundings per 32 inputs
// against eight. That the layer's error against 64 bits is no larger is
// measured (tests/test_gpu_policy_split.py): 0.69-0.99 of the f32 MFMA's over
// random weights, 0.75-0.93 with every weight at 2^-8 and 2^-17 pieces of one
// sign, 0.05-1.01 with equal activations of that kind too. Six 16x16x32 bf16
// MFMAs (16 cycles each) replace eight 16x16x4 f32 ones (32 cycles each) per
// 32 inputs: 96 against 256 cycles of matrix core, for 5.5 more VALU
// instructions per activation. 29-256-256-8 in one wave per tile, us per
// launch at steady clocks (f32, split): 56, 38 at 4096 worlds, 112, 71 at
// 65536, 215, 139 at 131072, the large two in the build for two waves per SIMD
// (154 at 131072 without its parked tiles). What bounds the large launch now
// is VALU issue and MFMA together: 8300 VALU instructions (the normals' f64,
// tanh, the split) and 34000 cycles of MFMA per wave, which keep the matrix
// cores busy 49% of the launch; the two waves of a SIMD overlap by little.
// Taken where every weight of the two layers is zero or of magnitude in
// [2^-100, 2^100] (the host checks on upload), so that none of its pieces
// overflows or is subnormal. Their inputs are tanh values, at most 1; of one
// below 2^-103 the bits under 2^-126 may be lost. The first layer stays f32: its
// inputs are the caller's observations, of any range.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

struct Split3 { bf16x8 h, m, l; };
__device__ __forceinline__ Split3 split3(f32x4 a, f32x4 b) {
  const f32x8 x = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  Split3 s;
  s.h = __builtin_convertvector(x, bf16x8);
  const f32x8 r = x - __builtin_convertvector(s.h, f32x8);
  s.m = __builtin_convertvector(r, bf16x8);
  s.l = __builtin_convertvector(r - __builtin_convertvector(s.m, f32x8), bf16x8);
  return s;
}
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// acc[cb] += W B over one block of 32 inputs, the small partial products
// first; the columns alternate, so consecutive MFMAs do not depend.
template <int CB>
__device__ __forceinline__ void mfma_split(const Split3& w, const Split3 (&b)[CB], f32x4 (&acc)[CB]) {
#pragma unroll
  for (int cb = 0; cb < CB; cb++) acc[cb] = mfma32(w.l, b[cb].h, acc[cb]);
#pragma unroll
  for (int cb = 0; cb < CB; cb++) acc[cb] = mfma32(w.h, b[cb].l, acc[cb]);
#pragma unroll
  for (int cb = 0; cb < CB; cb++) acc[cb] = mfma32(w.m, b[cb].m, acc[cb]);
#pragma unroll
  for (int cb = 0; cb < CB; cb++) acc[cb] = mfma32(w.m, b[cb].h, acc[cb]);
#pragma unroll
  for (int cb = 0; cb < CB; cb++) acc[cb] = mfma32(w.h, b[cb].m, acc[cb]);
#pragma unroll
  for (int cb = 0; cb < CB; cb++) acc[cb] = mfma32(w.h, b[cb].h, acc[cb]);
}
__device__ __forceinline__ Split3 weight_pieces(const f32x4* w, int t, int lane) {
  const bf16x8* p = (const bf16x8*)w + (size_t)t * 192 + lane;
  return Split3{p[0], p[64], p[128]};
}

// As mfma_layer, on tanh of the input tiles h, taken two at a time (32 inputs;
// an odd last tile is paired with zeros). The weights are [kb2][ob] triples of
// pieces, streamed in that order with PF triples in flight (4 to 6 measured
// the same). PARK = 0: the tanh of the next pair of tiles is spread over this
// pair's output blocks, where it issues while the MFMAs run. PARK > 0: every
// tanh first, and the last PARK tiles wait for their turn in LDS (`park`), for
// a wave that would have to spill them.
template <int PARK, int NHB_, int NOB_, int CB>
__device__ __forceinline__ void tanh_layer_split(const f32x4* __restrict__ w, int lane, f32x4 (&acc)[NOB_][CB],
                                                 f32x4 (&h)[NHB_][CB], f32x4* park) {
  constexpr int KB2 = (NHB_ + 1) / 2, NT = KB2 * NOB_;
  constexpr int PF = NT < 3 ? NT : 3;
  constexpr int KEEP = NHB_ - PARK;  // tiles that stay in registers
  Split3 ring[PF];
#pragma unroll
  for (int t = 0; t < PF; t++) ring[t] = weight_pieces(w, t, lane);
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  // Value e of a pair of tiles: tile, column, register.
  auto squash = [&](auto K, auto E) {
    constexpr int e = decltype(E)::value, tile = 2 * decltype(K)::value + e / (4 * CB);
    if constexpr (tile < NHB_) {
      float& x = *((float*)&h[tile][(e / 4) % CB] + e % 4);
      x = tanh_mlp(x);
    }
  };
  sfor<0, (PARK > 0 ? KB2 : 1)>([&](auto K) { sfor<0, 8 * CB>([&](auto E) { squash(K, E); }); });
  sfor<KEEP, NHB_>([&](auto I) {
    constexpr int i = decltype(I)::value;
#pragma unroll
    for (int cb = 0; cb < CB; cb++) park[((i - KEEP) * CB + cb) * 64 + lane] = h[i][cb];
  });
  auto tile = [&](auto I, int cb) {
    constexpr int i = decltype(I)::value;
    if constexpr (i >= NHB_) return zero;
    else if constexpr (i < KEEP) return h[i][cb];
    else return park[((i - KEEP) * CB + cb) * 64 + lane];
  };
  sfor<0, KB2>([&](auto K) {
    constexpr int kb = decltype(K)::value;
    Split3 b[CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) b[cb] = split3(tile(ic<2 * kb>{}, cb), tile(ic<2 * kb + 1>{}, cb));
    sfor<0, NOB_>([&](auto O) {
      constexpr int o = decltype(O)::value, t = kb * NOB_ + o;
      const Split3 wa = ring[t % PF];
      if constexpr (t + PF < NT) ring[t % PF] = weight_pieces(w, t + PF, lane);
      mfma_split<CB>(wa, b, acc[o]);
      if constexpr (PARK == 0 && kb + 1 < KB2)
        sfor<8 * CB * o / NOB_, 8 * CB * (o + 1) / NOB_>([&](auto E) { squash(ic<kb + 1>{}, E); });
      __builtin_amdgcn_sched_barrier(0);
    });
  });
}

// v_mfma_f32_16x16x4f32 lane layout: A[i][k] in lane i + 16 k, B[k][j] in
// lane j + 16 k, D[i][j] in lane j + 16 (i / 4), register i % 4.
// Layer l computes H_l^T = tanh(W_l H_{l-1}^T + b_l): rows are neurons, columns
// worlds. For the next layer, k-step s of input block kb uses register s of
// the previous output tile, i.e. lane j + 16 g supplies neuron 16 kb + 4 g + s
// of world j; the host lays W out to match (phz_host.cpp, policy_fragments).
// The bf16 16x16x32 takes 8 values per lane, k = 8 g + s in lane group g, of
// both operands: components 0..3 are neurons 32 kb + 4 g + s, components 4..7
// neurons 32 kb + 16 + 4 g + (s - 4), the two tiles of the pair.
// Inputs with observation noise, the prologue's normals per world.
template <class P> constexpr int noised_inputs() {
  int c = 0;
  for (int i = 0; i < P::NI; i++) c += P::noise[i] != 0.0 ? 1 : 0;
  return c;
}

// One world's sample (policy_reference, policy_pipeline.rs:488-520): every
// servo gets its base target, then each action k: AR(1) noise, sample,
// log-prob, the clamped action onto its slot's base. normal(k) is action k's
// normal; the calls come in order (products and sums are fused as written, so
// that every form of the kernel rounds alike). base[j] is servo j's base target and z[k]
// the AR(1) state before the step.
template <class P, class T, class NF>
__device__ __forceinline__ void policy_sample(const PolicyArgs& a, int my, const float* mean, const T (&base)[P::NPD],
                                              const float (&z)[P::NO], NF normal) {
  constexpr int NO = P::NO, NPD = P::NPD;
  const int S = a.stride;
  T* tgt = (T*)a.targets;
#pragma unroll
  for (int j = 0; j < NPD; j++) tgt[(size_t)j * S + my] = base[j];
  const float rho = float(P::rho);
  const float keep = sqrtf(fmaxf(0.0f, 1.0f - rho * rho));
  const float half_ln_2pi = 0.91893853320467274178f;
  float logp = 0.0f;
#pragma unroll
  for (int k = 0; k < NO; k++) {
    const float mk = mean[k];
    const float zk = fmaf(rho, z[k], keep * normal(k));
    a.z[(size_t)k * S + my] = zk;
    const float sd = a.stdv[k];
    const float act = fmaf(sd, zk, mk);
    const float zi = (act - mk) / sd;
    logp += fmaf(-0.5f * zi, zi, -logf(sd)) - half_ln_2pi;
    a.out[(size_t)k * S + my] = act;
    const float lim = float(P::clamp[k]);
    // clamp(-lim, lim) that passes NaN through, as f64::clamp does.
    const float applied = act < -lim ? -lim : (act > lim ? lim : act);
    const int slot = P::slot[k];
    tgt[(size_t)slot * S + my] = base[slot] + T(applied);
  }
  a.out[(size_t)NO * S + my] = logp;
}

template <class P, class T>
__device__ __forceinline__ void sample_state(const PolicyArgs& a, int my, T (&base)[P::NPD], float (&z)[P::NO]) {
#pragma unroll
  for (int j = 0; j < P::NPD; j++) base[j] = ((const T*)a.base)[(size_t)j * a.stride + my];
#pragma unroll
  for (int k = 0; k < P::NO; k++) z[k] = a.z[(size_t)k * a.stride + my];
}

template <class P, class T> __device__ __forceinline__ void policy_wave(const PolicyArgs& a, float* lds) {
  constexpr int NI = P::NI, NO = P::NO, CB = P::CB, NHB = P::NHB, NOB = P::NOB, KU = P::KU;
  constexpr int WPW = 16 * CB;     // worlds per wave
  constexpr int XS = 16 * KU + 1;  // LDS row stride of the input tile (floats)
  constexpr int MS = 16 * NOB + 1; // LDS row stride of the output tile
  const int lane = threadIdx.x & 63;
  const int w0 = blockIdx.x * WPW;
  const int S = a.stride;
  const int my = w0 + lane;
  const bool own = lane < WPW && my < a.nworld;
  u64 rs = 0;
  // Two-wave builds: the second wave of a SIMD issues first where both can, so
  // that the two leave lockstep and one's VALU phases fall into the other's
  // MFMAs (workgroups fill a SIMD's first wave, then its second; the order is
  // no more than a hint): 71.9 -> 71.2 us at 65536 worlds, 138-142 either way
  // at 131072, and 100 -> 52 B of spills per lane.
  if constexpr (P::PARK > 0) {
    if ((blockIdx.x >> 10) & 1) __builtin_amdgcn_s_setprio(3);
  }

  // Prologue: world w0 + lane reads its observation row, adds input noise in
  // index order (the noised value is what the history keeps), stages x in LDS.
  if constexpr (WPW == 32) {
    // Half the lanes own a world: the normals' transforms are paired across
    // the wave's halves (policy_normals_paired).
    constexpr int NN = noised_inputs<P>();
    if (own) rs = a.rng[my];
    float x[16 * KU];
#pragma unroll
    for (int i = 0; i < 16 * KU; i++) x[i] = (i < NI && own) ? a.obs[(size_t)i * S + my] : 0.0f;
    if constexpr (NN > 0) {
      double nz[NN];
      policy_normals_paired<NN>(rs, lane, nz);
      int c = 0;
#pragma unroll
      for (int i = 0; i < NI; i++)
        if (P::noise[i] != 0.0) {
          x[i] = fmaf(float(P::noise[i]), (float)nz[c++], x[i]);
          if (own) a.obs[(size_t)i * S + my] = x[i];
        }
    }
    if (lane < WPW) {
#pragma unroll
      for (int i = 0; i < 16 * KU; i++) lds[lane * XS + i] = x[i];
    }
  } else if (lane < WPW) {
    if (own) rs = a.rng[my];
#pragma unroll
    for (int i = 0; i < 16 * KU; i++) {
      float x = 0.0f;
      if (i < NI && own) {
        x = a.obs[(size_t)i * S + my];
        if (P::noise[i] != 0.0) {
          x = fmaf(float(P::noise[i]), (float)policy_normal(rs), x);
          a.obs[(size_t)i * S + my] = x;
        }
      }
      lds[lane * XS + i] = x;
    }
  }
  __syncthreads();

  const int r = lane & 15, g = lane >> 4;
  // Layer 1: B = the input tile in LDS; k-step s of input group u is inputs
  // 16 u + 4 s + g in lane group g.
  f32x4 h[NHB][CB];
  bias_tiles<NHB, CB>(a.bias, g, h);
  mfma_layer<KU, NHB, CB>(a.w1, lane, h, [&](int kb, int s, int cb) { return lds[(cb * 16 + r) * XS + 16 * kb + 4 * s + g]; });
  // Layer 2: B = layer 1's output tiles, straight from registers.
  f32x4 h2[NHB][CB];
  bias_tiles<NHB, CB>(a.bias + 16 * NHB, g, h2);
  if constexpr (P::SPLIT) {
    __syncthreads();  // the input tile's LDS is the parked tiles' now
    tanh_layer_split<P::PARK, NHB, NHB, CB>(a.w2, lane, h2, h, (f32x4*)lds);
  } else {
    tanh_tiles<NHB, CB>(h);
    mfma_layer<NHB, NHB, CB>(a.w2, lane, h2, [&](int kb, int s, int cb) { return h[kb][cb][s]; });
  }
  // Layer 3: the action means.
  f32x4 m[NOB][CB];
  bias_tiles<NOB, CB>(a.bias + 32 * NHB, g, m);
  if constexpr (P::SPLIT) {
    tanh_layer_split<0, NHB, NOB, CB>(a.w3, lane, m, h2, nullptr);
  } else {
    tanh_tiles<NHB, CB>(h2);
    mfma_layer<NHB, NOB, CB>(a.w3, lane, m, [&](int kb, int s, int cb) { return h2[kb][cb][s]; });
  }
  // Means to LDS, world-major, for the per-world epilogue.
  __syncthreads();
#pragma unroll
  for (int ob = 0; ob < NOB; ob++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int j = 0; j < 4; j++) lds[(cb * 16 + r) * MS + ob * 16 + 4 * g + j] = m[ob][cb][j];
  __syncthreads();

  // With half the lanes owning a world the actions' normals are drawn first,
  // paired across the halves.
  double na[NO];
  if constexpr (WPW == 32) policy_normals_paired<NO>(rs, lane, na);
  if (own) {
    T base[P::NPD];
    float z[NO];
    sample_state<P, T>(a, my, base, z);
    policy_sample<P, T>(a, my, lds + lane * MS, base, z, [&](int k) { return (float)(WPW == 32 ? na[k] : policy_normal(rs)); });
    a.rng[my] = rs;
  }
}

// ── small launches: a tile of 16 CB worlds to a workgroup of TW waves ──
// One wave per tile leaves most SIMDs idle when a launch has few tiles, and
// the launch then lasts as long as one wave's stream (29-256-256-8: 38 us at
// 64 worlds, 42 at 16384; here 16 and 29). Here wave k computes the hidden neurons of blocks
// k * BPW .. of both hidden layers for the whole tile, and passes them to the
// others through LDS, already split into bf16 pieces and laid out as B
// fragments. The streams' raw draws are one lane's work per world, the
// Box-Muller transforms are spread over every lane. Every sum runs in
// policy_wave's order: the two give the same bits.
//
// LDS: the draws (8 bytes each, kTeamDraws normals at a time, later the hidden pieces: KB2 x 3 x CB x 1 KB),
// the input tile [world][XS], the means [world][MS] and the actions' normals.
constexpr int kTeamDraws = 40;  // normals drawn at a time
template <class P> constexpr int team_draws() {
  const int n = noised_inputs<P>() + P::NO;
  return 2 * (n < kTeamDraws ? n : kTeamDraws) * 16 * P::CB * 8;
}
template <class P> constexpr int team_pieces() { return ((P::NHB + 1) / 2) * 3 * P::CB * 1024; }
template <class P> constexpr int team_front() {
  return team_draws<P>() > team_pieces<P>() ? team_draws<P>() : team_pieces<P>();
}
template <class P> constexpr int team_lds_bytes() {
  return team_front<P>() + 16 * P::CB * (16 * P::KU + 1 + 16 * P::NOB + 1 + P::NO) * 4;
}

// h[j] is tile blk0 + j: its pieces into the halves of fragment (blk / 2).
template <int CB, int BPW>
__device__ __forceinline__ void put_pieces(bf16x8* pieces, const f32x4 (&h)[BPW][CB], int blk0, int nhb, int lane) {
#pragma unroll
  for (int j = 0; j < BPW; j += 2) {
    const int blk = blk0 + j;
    if (blk >= nhb) continue;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
      const Split3 s = split3(h[j][cb], blk + 1 < nhb ? h[j + 1][cb] : zero);
      bf16x8* p = pieces + ((size_t)(blk / 2) * 3 * CB + cb) * 64 + lane;
      p[0] = s.h;
      p[CB * 64] = s.m;
      p[2 * CB * 64] = s.l;
    }
  }
}
template <int CB> __device__ __forceinline__ void get_pieces(const bf16x8* pieces, int kb, int lane, Split3 (&b)[CB]) {
#pragma unroll
  for (int cb = 0; cb < CB; cb++) {
    const bf16x8* p = pieces + ((size_t)kb * 3 * CB + cb) * 64 + lane;
    b[cb] = Split3{p[0], p[CB * 64], p[2 * CB * 64]};
  }
}

template <class P, class T> __device__ __forceinline__ void policy_team(const PolicyArgs& a, char* lds) {
  constexpr int NI = P::NI, NO = P::NO, CB = P::CB, NHB = P::NHB, NOB = P::NOB, KU = P::KU, TW = P::TW;
  constexpr int W = 16 * CB, XS = 16 * KU + 1, MS = 16 * NOB + 1, KB2 = (NHB + 1) / 2;
  constexpr int BPW = 2 * ((KB2 + TW - 1) / TW);  // hidden blocks per wave, whole pairs
  constexpr int NN = noised_inputs<P>(), ND = NN + NO;
  u64* draws = (u64*)lds;                          // [ND][2][W]
  bf16x8* pieces = (bf16x8*)lds;                   // [KB2][3][CB][64]
  float* x = (float*)(lds + team_front<P>());      // [W][XS]
  float* mean = x + W * XS;                        // [W][MS]
  float* nact = mean + W * MS;                     // [NO][W]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w0 = blockIdx.x * W, S = a.stride;

  // What later phases read from memory is loaded ahead of the barriers before
  // them: layer 1's weights (of a narrow input) and the sample's state here,
  // layer 2's first weights before layer 1, layer 3's before its inputs are
  // exchanged.
  constexpr bool PRE = KU <= 2;
  f32x4 w1f[BPW][PRE ? KU : 1];
  const int blk0 = wave * BPW;
  auto block = [&](int j) { return blk0 + j < NHB ? blk0 + j : NHB - 1; };
  if constexpr (PRE) {
#pragma unroll
    for (int j = 0; j < BPW; j++)
#pragma unroll
      for (int kb = 0; kb < KU; kb++) w1f[j][kb] = a.w1[(kb * NHB + block(j)) * 64 + lane];
  }
  const bool sampler = tid < W && w0 + tid < a.nworld;
  T base[P::NPD];
  float z[NO];
  if (sampler) sample_state<P, T>(a, w0 + tid, base, z);

  for (int e = tid; e < 16 * KU * W; e += 64 * TW) {
    const int i = e / W, w = e % W;
    x[w * XS + i] = i < NI && w0 + w < a.nworld ? a.obs[(size_t)i * S + w0 + w] : 0.0f;
  }
  // Raw draws in stream order (inputs, then actions) by one lane per world of
  // the first wave, then their transforms on every lane.
  u64 rs = 1;
  if (sampler) rs = a.rng[w0 + tid];
  for (int d0 = 0; d0 < ND; d0 += kTeamDraws) {
    const int nd = ND - d0 < kTeamDraws ? ND - d0 : kTeamDraws;
    if (d0 > 0) __syncthreads();  // the transforms of the draws before are done
    if (tid < W) {
#pragma unroll 4
      for (int d = 0; d < 2 * nd; d++) draws[d * W + tid] = xorshift64(rs);
    }
    __syncthreads();
    for (int e = tid; e < nd * W; e += 64 * TW) {
      const int d = e / W, w = e % W, k = d0 + d;
      const u64 x1 = draws[(2 * d) * W + w], x2 = draws[(2 * d + 1) * W + w];
      const float n = (float)policy_transform(uniform_of(x1), turns_of(x2));
      if (k < NN) {
        const int i = P::noised[k];
        const float xi = fmaf(P::scale[k], n, x[w * XS + i]);
        x[w * XS + i] = xi;
        if (w0 + w < a.nworld) a.obs[(size_t)i * S + w0 + w] = xi;
      } else {
        nact[(k - NN) * W + w] = n;
      }
    }
  }
  if (sampler) a.rng[w0 + tid] = rs;
  __syncthreads();

  const int r = lane & 15, g = lane >> 4;
  auto w2_at = [&](int kb, int j) { return weight_pieces(a.w2, kb * NHB + block(j), lane); };
  Split3 wn[BPW];
#pragma unroll
  for (int j = 0; j < BPW; j++) wn[j] = w2_at(0, j);
  // Layer 1, this wave's blocks (one past the last block repeats it and is
  // not stored).
  f32x4 h[BPW][CB];
#pragma unroll
  for (int j = 0; j < BPW; j++) {
    f32x4 acc[1][CB];
    bias_tiles<1, CB>(a.bias + 16 * block(j), g, acc);
#pragma unroll
    for (int kb = 0; kb < KU; kb++) {
      f32x4 wa;
      if constexpr (PRE) wa = w1f[j][kb];
      else wa = a.w1[(kb * NHB + block(j)) * 64 + lane];
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) acc[0][cb] = mfma4(wa[s], x[(cb * 16 + r) * XS + 16 * kb + 4 * s + g], acc[0][cb]);
    }
#pragma unroll
    for (int cb = 0; cb < CB; cb++) h[j][cb] = acc[0][cb];
  }
  tanh_tiles<BPW, CB>(h);
  put_pieces<CB, BPW>(pieces, h, blk0, NHB, lane);
  __syncthreads();
  // Layer 2: every input pair, this wave's output blocks; the next pair's
  // weights load while this one multiplies.
  f32x4 h2[BPW][CB];
#pragma unroll
  for (int j = 0; j < BPW; j++) {
    f32x4 acc[1][CB];
    bias_tiles<1, CB>(a.bias + 16 * NHB + 16 * block(j), g, acc);
#pragma unroll
    for (int cb = 0; cb < CB; cb++) h2[j][cb] = acc[0][cb];
  }
#pragma unroll
  for (int kb = 0; kb < KB2; kb++) {
    Split3 b[CB];
    get_pieces<CB>(pieces, kb, lane, b);
#pragma unroll
    for (int j = 0; j < BPW; j++) {
      const Split3 wa = wn[j];
      if (kb + 1 < KB2) wn[j] = w2_at(kb + 1, j);
      mfma_split<CB>(wa, b, h2[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  constexpr int P3 = KB2 < 3 ? KB2 : 3;  // layer 3's weights in flight
  Split3 w3[P3];
  if (wave < NOB) {
#pragma unroll
    for (int kb = 0; kb < P3; kb++) w3[kb] = weight_pieces(a.w3, kb * NOB + wave, lane);
  }
  tanh_tiles<BPW, CB>(h2);
  __syncthreads();  // every wave is past its reads of layer 1's pieces
  put_pieces<CB, BPW>(pieces, h2, blk0, NHB, lane);
  __syncthreads();
  // Layer 3: output block k on wave k.
  if (wave < NOB) {
    f32x4 acc[1][CB];
    bias_tiles<1, CB>(a.bias + 32 * NHB + 16 * wave, g, acc);
#pragma unroll
    for (int kb = 0; kb < KB2; kb++) {
      const Split3 wa = w3[kb % P3];
      if (kb + P3 < KB2) w3[kb % P3] = weight_pieces(a.w3, (kb + P3) * NOB + wave, lane);
      Split3 b[CB];
      get_pieces<CB>(pieces, kb, lane, b);
      mfma_split<CB>(wa, b, acc[0]);
    }
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int j = 0; j < 4; j++) mean[(cb * 16 + r) * MS + wave * 16 + 4 * g + j] = acc[0][cb][j];
  }
  __syncthreads();
  if (sampler)
    policy_sample<P, T>(a, w0 + tid, mean + tid * MS, base, z, [&](int k) { return nact[k * W + tid]; });
}

}  // namespace phz
