// Gated DeltaNet (GDN) recurrent step for gfx950: gate, q/k L2 norm and the delta-rule state update.
//
// Per (sequence b, value head h), token by token (T >= 1; T = 1 is decode):
//   q, k  <- L2-normalised key-head vectors (x / sqrt(sum x^2 + 1e-6)), q *= DK^-0.5
//            (l2norm_lastdim, sgl_kernel_axera/attention/gdn.py:919-931; models/.../q35_step.py:164-169)
//   g      = -exp(A_log[h]) * softplus(a + dt_bias[h]);  beta = sigmoid(b)          (gdn_gate, gdn.py:934-949)
//   S     <- exp(g) S;  pred = k^T S;  err = beta (v - pred);  S <- S + k err^T;  o = q^T S
//            (gdn_recurrent_step, gdn.py:952-989)
// Value head h reads key head (h / kdiv) % NK: kdiv = NV / NK in the grouped order (h / (NV / NK), the operators'
// order, test_gdn_attn.py:268-277), kdiv = 1 in the tiled order (h % NK, the layer kernels' default order,
// models/qwen35_35b_a3b/src/70b0fbc/q35_step.py:82-85, 171).
// The state S [DK, DV] fp32 is the kernels' whole HBM traffic: a workgroup holds its 128 x 128 tile in
// registers (64 floats per thread, float4 loads along DV) from one read to one write, across all T tokens.
// Arithmetic is fp32 throughout (the reference rounds the state to bf16 for its two products; the
// difference is well inside the bf16 output tolerance and is checked against both formulations).
// With GATE (the decode layer), the output row of each head goes through the GDN output norm before it is
// stored: out = bf16(bf16(rmsnorm(bf16 o) * norm_w) * silu(z)) (q35_step.py:179-180), the same rounding points
// as the separate gated-norm kernel.
#include "axk_common.h"
#include "axk_host.h"

namespace {

constexpr int kDK = 128, kDV = 128;
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kWaveCols = kDV / kWaves;  // 32 state columns a wave: 8 lanes of 4 columns
constexpr int kRowGroups = 8;            // the other 3 lane bits: row group rg holds rows rg, rg + 8, ..
constexpr int kRows = kDK / kRowGroups;  // 16 state rows per thread
constexpr int kLdRow = kRows + 4;        // floats between row groups of k / q in LDS (16-byte reads, no conflicts)

constexpr int kStepCols = kDV / 4;                  // gdn_recurrent_kernel: 32 threads across DV, 4 columns each
constexpr int kStepRowGroups = kThreads / kStepCols;  // 8 row groups of kRows rows
constexpr int kColsMaxWgs = 512, kEarlyMaxWgs = 256, kStepFullWgs = 2560;  // see axk_gdn_recurrent_strided
constexpr int kStepPadLds = 54 * 1024;  // dynamic LDS that leaves room for two workgroups a CU

struct GdnArgs {
  const uint16_t* q;   // [B, T, NK, DK] bf16
  const uint16_t* k;   // [B, T, NK, DK] bf16
  const uint16_t* v;   // [B, T, NV, DV] bf16
  const uint16_t* a;   // [B, T, NV] bf16
  const uint16_t* b;   // [B, T, NV] bf16
  const float* a_log;  // [NV]
  const float* dt_bias;  // [NV]
  const float* state_in;  // [B, NV, DK, DV]
  float* state_out;       // [B, NV, DK, DV] (may alias state_in)
  uint16_t* out;          // [B, T, NV, DV] bf16
  int B, T, NK, NV;
  int64_t ldq, ldk, ldv, ldab;  // elements between consecutive (sequence, token) rows of q, k, v, a / b
  const float* norm_w;          // GATE: the output norm's weight [DV] and gate z [B, T, NV, DV]
  const uint16_t* z;
  float eps;
  float* snap;                  // optional: the state after token t at snap + t * snap_ld, [B, NV, DK, DV] each
  int64_t snap_ld;
  int kdiv;                     // value head h reads key head (h / kdiv) % NK
  int out_over_qk;              // out overlaps q or k
};

// One token's inputs as a wave loads them: two rows of k and q a lane, v of the lane's columns, the gate inputs.
struct GdnTok {
  uint32_t k0, k1, q0, q1, v[4], a, b;  // a register each: packed halves would wait for the load before
};

AXK_DEV GdnTok gdn_load_tok(const GdnArgs& p, int64_t tok, int kh, int h, uint32_t lane, uint32_t c0) {
  GdnTok x;
  // opaque, so that no lane pointer is kept across the token loop: the state leaves no registers for ten of them
  asm volatile("" : "+v"(lane), "+v"(c0));
  const uint16_t* kr = p.k + tok * p.ldk + kh * kDK;
  const uint16_t* qr = p.q + tok * p.ldq + kh * kDK;
  const uint16_t* vr = p.v + tok * p.ldv + h * kDV;
  x.k0 = kr[lane];
  x.k1 = kr[lane + 64];
  x.q0 = qr[lane];
  x.q1 = qr[lane + 64];
#pragma unroll
  for (int j = 0; j < 4; ++j) x.v[j] = vr[c0 + j];
  x.a = p.a[tok * p.ldab + h];
  x.b = p.b[tok * p.ldab + h];
  return x;
}

// The column sum over the 8 row groups (lane bits 3 .. 5), the same value in each of them.
AXK_DEV float row_group_sum(float v) {
  v += dpp_move<0x128>(v, v);  // row_ror:8, the lane 8 away in its row of 16
  return xor32_sum(xor16_sum(v));
}

// Few sequences, or several tokens: bound by one token's chain as much as by the state's read and write. A state column
// evolves by itself, so a wave carries 32 columns of all 128 rows and its sums stay inside the wave: no barrier (one a
// token with GATE, whose norm spans the head). EARLY: the first token's inputs are loaded ahead of the state, and the
// norms and gates are done while it arrives. A call of one token (!MULTI) keeps no addresses for a next one (97
// registers against 117). 1 sequence x 32 heads: 4.65 us (5.27 with the sums through LDS and the inputs behind the
// state), 4 tokens 9.7 us (10.5).
template <bool GATE, bool MULTI, bool EARLY>
__global__ __launch_bounds__(kThreads, GATE && MULTI ? 3 : 4) void gdn_columns_kernel(GdnArgs p) {
  __shared__ __align__(16) float s_kq[kWaves][2][kRowGroups * kLdRow];  // each wave's own normalised k and q
  __shared__ float s_gn[2][kWaves];                                     // by token parity

  const int bh = blockIdx.x;
  const int b = bh / p.NV, h = bh - (bh / p.NV) * p.NV;
  const int kh = (h / p.kdiv) % p.NK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cg = lane & 7, rg = lane >> 3;
  const int c0 = kWaveCols * wave + 4 * cg;
  const int64_t tok0 = (int64_t)b * p.T;
  float* sk = s_kq[wave][0];
  float* sq = s_kq[wave][1];

  GdnTok in;
  if (EARLY) in = gdn_load_tok(p, tok0, kh, h, lane, c0);
  const float a_log = p.a_log[h], dt_bias = p.dt_bias[h];
  const int col = c0 + (rg & 3);
  uint32_t z = 0;
  float nw = 0.f;
  if (GATE) {
    nw = p.norm_w[col];
    if (!MULTI) z = (p.z + (tok0 * p.NV + h) * kDV)[col];
  }
  __builtin_amdgcn_sched_barrier(0);

  // state tile in registers: rows rg + 8 r, columns c0 .. c0 + 3 (a load instruction covers 8 rows of 128 bytes)
  const int64_t tile = ((int64_t)b * p.NV + h) * kDK * kDV;
  const float* sin = p.state_in + tile + rg * kDV + c0;
  float4 S[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {  // the tile is read once and written once: non-temporal
    const axk_u32x4 u = load_nt(sin + r * kRowGroups * kDV);
    S[r] = make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
  }
  __builtin_amdgcn_sched_barrier(0);
  if (!EARLY) in = gdn_load_tok(p, tok0, kh, h, lane, c0);

  const float gscale = -__expf(a_log);
  const float qscale = rsqrtf((float)kDK);
  const int pos = (lane & 7) * kLdRow + (lane >> 3);  // row `lane` in k / q's LDS order; row lane + 64 is 8 further

  const int T = MULTI ? p.T : 1;
  for (int t = 0; t < T; ++t) {
    if (MULTI && t > 0) in = gdn_load_tok(p, tok0 + t, kh, h, lane, c0);
    // ---- q / k L2 norm, gate ----
    const float k0 = bf16_bits_to_f32(in.k0), k1 = bf16_bits_to_f32(in.k1);
    const float q0 = bf16_bits_to_f32(in.q0), q1 = bf16_bits_to_f32(in.q1);
    const float kn = sqrtf(wave_sum(k0 * k0) + wave_sum(k1 * k1) + 1e-6f);
    const float qn = sqrtf(wave_sum(q0 * q0) + wave_sum(q1 * q1) + 1e-6f);
    sk[pos] = k0 / kn;
    sk[pos + 8] = k1 / kn;
    sq[pos] = q0 / qn * qscale;
    sq[pos + 8] = q1 / qn * qscale;
    const float decay = __expf(gscale * softplus_f32(bf16_bits_to_f32(in.a) + dt_bias));
    const float beta = sigmoid_f32(bf16_bits_to_f32(in.b));
    const float4 vv = make_float4(bf16_bits_to_f32(in.v[0]), bf16_bits_to_f32(in.v[1]), bf16_bits_to_f32(in.v[2]),
                                  bf16_bits_to_f32(in.v[3]));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own LDS writes above, reads below
    __builtin_amdgcn_wave_barrier();

    // ---- S <- decay S; pred = k^T S (column sums over this thread's rows, then over row groups) ----
    float4 pr = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int r4 = 0; r4 < kRows; r4 += 4) {
      const float4 k4 = *reinterpret_cast<const float4*>(sk + rg * kLdRow + r4);
      const float kr[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float4& s = S[r4 + i];
        s.x *= decay; s.y *= decay; s.z *= decay; s.w *= decay;
        pr.x += kr[i] * s.x; pr.y += kr[i] * s.y; pr.z += kr[i] * s.z; pr.w += kr[i] * s.w;
      }
    }
    pr.x = row_group_sum(pr.x); pr.y = row_group_sum(pr.y);
    pr.z = row_group_sum(pr.z); pr.w = row_group_sum(pr.w);
    // ---- err = beta (v - pred); S += k err^T; o = q^T S ----
    const float4 er = make_float4(beta * (vv.x - pr.x), beta * (vv.y - pr.y), beta * (vv.z - pr.z), beta * (vv.w - pr.w));
    float4 ov = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int r4 = 0; r4 < kRows; r4 += 4) {
      const float4 k4 = *reinterpret_cast<const float4*>(sk + rg * kLdRow + r4);
      const float4 q4 = *reinterpret_cast<const float4*>(sq + rg * kLdRow + r4);
      const float kr[4] = {k4.x, k4.y, k4.z, k4.w}, qr[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float4& s = S[r4 + i];
        s.x += kr[i] * er.x; s.y += kr[i] * er.y; s.z += kr[i] * er.z; s.w += kr[i] * er.w;
        ov.x += qr[i] * s.x; ov.y += qr[i] * s.y; ov.z += qr[i] * s.z; ov.w += qr[i] * s.w;
      }
      if (r4 & 4) __builtin_amdgcn_sched_barrier(0);  // half of k and q in registers at a time
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the reads above precede the next token's writes
    __builtin_amdgcn_wave_barrier();
    const int64_t vh = ((tok0 + t) * p.NV + h) * kDV;  // output row; lane (rg < 4, cg) stores column c0 + rg
    if (GATE && MULTI) z = (p.z + vh)[col];
    ov.x = row_group_sum(ov.x); ov.y = row_group_sum(ov.y);
    ov.z = row_group_sum(ov.z); ov.w = row_group_sum(ov.w);
    const float o = rg == 0 ? ov.x : rg == 1 ? ov.y : rg == 2 ? ov.z : ov.w;
    if (!GATE) {
      if (p.out_over_qk) __syncthreads();  // every wave has this token's q and k before they are written over
      if (rg < 4) (p.out + vh)[col] = (uint16_t)f32_to_bf16_bits(o);
    } else {
      const float core = round_bf16(o);  // the head's bf16 output
      const float ss = wave_sum(rg < 4 ? core * core : 0.f);
      if (lane == 0) s_gn[t & 1][wave] = ss;
      __syncthreads();  // a wave writes this half again only after the next token's barrier
      if (rg < 4) {
        const float* gn = s_gn[t & 1];
        const float inv = rsqrtf((gn[0] + gn[1] + gn[2] + gn[3]) / (float)kDV + p.eps);
        (p.out + vh)[col] = (uint16_t)f32_to_bf16_bits(round_bf16(core * inv * nw) * silu_f32(bf16_bits_to_f32(z)));
      }
    }
    if (MULTI && p.snap) {  // the state after this token (speculative verification's per-row snapshots)
      uint32_t lo = rg * kDV + c0;
      asm volatile("" : "+v"(lo));
      float* sn = p.snap + t * p.snap_ld + tile + lo;
#pragma unroll
      for (int r = 0; r < kRows; ++r)
        store_nt(sn + r * kRowGroups * kDV, axk_u32x4{__float_as_uint(S[r].x), __float_as_uint(S[r].y),
                                                      __float_as_uint(S[r].z), __float_as_uint(S[r].w)});
    }
  }

  uint32_t lo = rg * kDV + c0;
  asm volatile("" : "+v"(lo));
  float* sout = p.state_out + tile + lo;
#pragma unroll
  for (int r = 0; r < kRows; ++r)
    store_nt(sout + r * kRowGroups * kDV, axk_u32x4{__float_as_uint(S[r].x), __float_as_uint(S[r].y),
                                                    __float_as_uint(S[r].z), __float_as_uint(S[r].w)});
}

// One token for many sequences: the state's read and write fill the chip, and what counts is the order in which HBM
// sees them. A wave reads and writes whole rows (two of 512 bytes an instruction), a workgroup's stores follow all of
// its loads and start together. Thread = 16 rows x 4 columns; the column sums meet in LDS. (32 / 64 / 256 sequences of 32
// heads: 24.1 / 47.2 / 190.7 us; without the barrier before the stores 24.2 / 48.4 / 195.9, with the compiler aiming at four
// workgroups a CU 23.9 / 47.8 / 192.2.)
template <bool GATE>
__global__ __launch_bounds__(kThreads, 3) void gdn_recurrent_kernel(GdnArgs p) {
  __shared__ float s_k[kDK], s_q[kDK];
  __shared__ float s_gn[2];
  __shared__ __align__(16) float s_red[kStepRowGroups / 2][kDV];  // per-wave partial column sums
  __shared__ __align__(16) float s_vec[kDV];
  __shared__ float s_norm[4];

  const int bh = blockIdx.x;
  const int b = bh / p.NV, h = bh - (bh / p.NV) * p.NV;
  const int kh = (h / p.kdiv) % p.NK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cg = tid % kStepCols, rg = tid / kStepCols;
  const int c0 = 4 * cg, r0 = kRows * rg;

  // state tile in registers: rows r0 .. r0 + 15, columns c0 .. c0 + 3
  const float* sin = p.state_in + ((int64_t)b * p.NV + h) * kDK * kDV;
  float4 S[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {  // the tile is read once and written once: non-temporal
    const axk_u32x4 u = load_nt(sin + (r0 + r) * kDV + c0);
    S[r] = make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
  }

  const float a_log = p.a_log[h], dt_bias = p.dt_bias[h];
  const float qscale = rsqrtf((float)kDK);

  const int64_t tok = b;  // one token a sequence
  // ---- q / k L2 norm (threads 0..127 own one element of each) ----
  float kx = 0.f, qx = 0.f;
  if (tid < kDK) {
    kx = bf16_bits_to_f32(p.k[tok * p.ldk + kh * kDK + tid]);
    qx = bf16_bits_to_f32(p.q[tok * p.ldq + kh * kDK + tid]);
  }
  float ks = wave_sum(kx * kx), qs = wave_sum(qx * qx);
  if (lane == 0 && wave < 2) {
    s_norm[wave] = ks;
    s_norm[2 + wave] = qs;
  }
  const int64_t vh = tok * p.NV + h;  // output row
  const float a = bf16_bits_to_f32(p.a[tok * p.ldab + h]), bb = bf16_bits_to_f32(p.b[tok * p.ldab + h]);
  const uint16_t* vr = p.v + tok * p.ldv + h * kDV + c0;
  const float4 vv = make_float4(bf16_bits_to_f32(vr[0]), bf16_bits_to_f32(vr[1]), bf16_bits_to_f32(vr[2]),
                                bf16_bits_to_f32(vr[3]));
  __syncthreads();
  if (tid < kDK) {
    const float kn = sqrtf(s_norm[0] + s_norm[1] + 1e-6f), qn = sqrtf(s_norm[2] + s_norm[3] + 1e-6f);
    s_k[tid] = kx / kn;
    s_q[tid] = qx / qn * qscale;
  }
  // ---- gate ----
  const float g = -__expf(a_log) * softplus_f32(a + dt_bias);
  const float decay = __expf(g);
  const float beta = sigmoid_f32(bb);
  __syncthreads();

  // ---- S <- decay S; pred = k^T S (column sums over this thread's rows, then over row groups) ----
  float4 pr = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const float kr = s_k[r0 + r];
    S[r].x *= decay; S[r].y *= decay; S[r].z *= decay; S[r].w *= decay;
    pr.x += kr * S[r].x; pr.y += kr * S[r].y; pr.z += kr * S[r].z; pr.w += kr * S[r].w;
  }
  // the two row groups of a wave: lanes l and l ^ 32
  pr.x = xor32_sum(pr.x); pr.y = xor32_sum(pr.y);
  pr.z = xor32_sum(pr.z); pr.w = xor32_sum(pr.w);
  if (lane < 32) *reinterpret_cast<float4*>(&s_red[wave][c0]) = pr;
  __syncthreads();
  if (tid < kDV) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kStepRowGroups / 2; ++w) sum += s_red[w][tid];
    s_vec[tid] = sum;
  }
  __syncthreads();
  // ---- err = beta (v - pred); S += k err^T; o = q^T S ----
  const float4 pd = *reinterpret_cast<const float4*>(&s_vec[c0]);
  const float4 er = make_float4(beta * (vv.x - pd.x), beta * (vv.y - pd.y), beta * (vv.z - pd.z), beta * (vv.w - pd.w));
  float4 ov = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const float kr = s_k[r0 + r], qr = s_q[r0 + r];
    S[r].x += kr * er.x; S[r].y += kr * er.y; S[r].z += kr * er.z; S[r].w += kr * er.w;
    ov.x += qr * S[r].x; ov.y += qr * S[r].y; ov.z += qr * S[r].z; ov.w += qr * S[r].w;
  }
  ov.x = xor32_sum(ov.x); ov.y = xor32_sum(ov.y);
  ov.z = xor32_sum(ov.z); ov.w = xor32_sum(ov.w);
  __syncthreads();  // s_red / s_vec reuse
  if (lane < 32) *reinterpret_cast<float4*>(&s_red[wave][c0]) = ov;
  __syncthreads();
  if (!GATE) {
    if (tid < kDV) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kStepRowGroups / 2; ++w) sum += s_red[w][tid];
      p.out[vh * kDV + tid] = (uint16_t)f32_to_bf16_bits(sum);
    }
  } else {
    float core = 0.f;  // the head's bf16 output, element tid (threads 0 .. 127: waves 0 and 1)
    if (tid < kDV) {
#pragma unroll
      for (int w = 0; w < kStepRowGroups / 2; ++w) core += s_red[w][tid];
      core = round_bf16(core);
    }
    const float ss = wave_sum(core * core);
    if (lane == 0 && wave < 2) s_gn[wave] = ss;
    __syncthreads();
    if (tid < kDV) {
      const float inv = rsqrtf((s_gn[0] + s_gn[1]) / (float)kDV + p.eps);
      const float zz = bf16_bits_to_f32(p.z[vh * kDV + tid]);
      p.out[vh * kDV + tid] = (uint16_t)f32_to_bf16_bits(round_bf16(core * inv * p.norm_w[tid]) * silu_f32(zz));
    }
  }

  __syncthreads();  // the workgroup's stores start together
  float* sout = p.state_out + ((int64_t)b * p.NV + h) * kDK * kDV;
#pragma unroll
  for (int r = 0; r < kRows; ++r)
    store_nt(sout + (r0 + r) * kDV + c0, axk_u32x4{__float_as_uint(S[r].x), __float_as_uint(S[r].y), __float_as_uint(S[r].z), __float_as_uint(S[r].w)});
}

}  // namespace

int axk_gdn_recurrent_strided(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint16_t* a,
                              const uint16_t* b, const float* a_log, const float* dt_bias, const float* state_in,
                              float* state_out, uint16_t* out, int64_t batch, int64_t tokens, int64_t num_k_heads,
                              int64_t num_v_heads, const AxkGdnStrides& ld, const AxkGdnGate* gate, int v_order,
                              hipStream_t stream, float* state_snap, int64_t snap_ld) {
  AXK_REQUIRE(q && k && v && a && b && a_log && dt_bias && state_in && state_out && out, AXK_E_NULL);
  AXK_REQUIRE(v_order == AXK_VORDER_GROUPED || v_order == AXK_VORDER_TILED, AXK_E_SHAPE);
  AXK_REQUIRE(!gate || (gate->norm_w && gate->z), AXK_E_NULL);
  AXK_REQUIRE(batch > 0 && tokens > 0 && num_k_heads > 0 && num_v_heads > 0, AXK_E_SHAPE);
  AXK_REQUIRE(num_v_heads % num_k_heads == 0, AXK_E_SHAPE);
  AXK_REQUIRE(batch * num_v_heads <= INT32_MAX && tokens <= INT32_MAX, AXK_E_SHAPE);
  AXK_REQUIRE(ld.q >= num_k_heads * kDK && ld.k >= num_k_heads * kDK && ld.v >= num_v_heads * kDV &&
                  ld.ab >= num_v_heads,
              AXK_E_SHAPE);
  AXK_REQUIRE(axk_aligned(state_in, 16) && axk_aligned(state_out, 16), AXK_E_ALIGN);
  const size_t sbytes = (size_t)batch * num_v_heads * kDK * kDV * 4;
  // in place is allowed (each thread writes what it alone read, after all of its reads); partial overlap is not
  AXK_REQUIRE(state_in == state_out || !axk_overlap(state_in, sbytes, state_out, sbytes), AXK_E_ALIAS);
  const size_t obytes = (size_t)batch * tokens * num_v_heads * kDV * 2;
  AXK_REQUIRE(!axk_overlap(out, obytes, state_out, sbytes), AXK_E_ALIAS);
  if (state_snap) {  // snapshot t: [B, NV, DK, DV] at state_snap + t * snap_ld, none overlapping the states
    const int64_t per = batch * num_v_heads * kDK * kDV;
    AXK_REQUIRE(snap_ld >= per && axk_aligned(state_snap, 16) && snap_ld % 4 == 0, AXK_E_SHAPE);
    const size_t nbytes = (size_t)((tokens - 1) * snap_ld + per) * 4;
    AXK_REQUIRE(!axk_overlap(state_snap, nbytes, state_in, sbytes) && !axk_overlap(state_snap, nbytes, state_out, sbytes) &&
                    !axk_overlap(state_snap, nbytes, out, obytes),
                AXK_E_ALIAS);
  }
  GdnArgs p{q, k, v, a, b, a_log, dt_bias, state_in, state_out, out, (int)batch, (int)tokens, (int)num_k_heads,
            (int)num_v_heads, ld.q, ld.k, ld.v, ld.ab, gate ? gate->norm_w : nullptr, gate ? gate->z : nullptr,
            gate ? gate->eps : 0.f, state_snap, snap_ld,
            v_order == AXK_VORDER_TILED ? 1 : (int)(num_v_heads / num_k_heads)};
  // out may take the place of q, k or v (with as many key heads as value heads): a head's workgroup reads its token's
  // rows before it writes them
  auto over = [&](const uint16_t* x, int64_t row) {
    return axk_overlap(out, obytes, x, (size_t)((batch * tokens - 1) * row + num_k_heads * kDK) * 2);
  };
  p.out_over_qk = over(q, ld.q) || over(k, ld.k);
  AXK_LAUNCH_GATE();
  // Which kernel, measured (32 value heads; us, rows in a loop over the tokens -> gdn_columns_kernel):
  //   1 token:  1 sequence 5.27 -> 4.65, 4 6.24 -> 5.37, 8 8.4 -> 7.5, 16 12.9 -> 11.8
  //   4 tokens: 1 sequence 10.5 -> 9.7, 8 14.3 -> 13.4, 32 34.4 -> 32;  64 x 2 tokens of 16 heads 28.3 -> 27.8
  // From 257 workgroups, more than one a CU, the state is loaded first (16 sequences: 11.8 us, inputs first 13.8); up to
  // 256 the inputs, whose chain is then the longer one. Above 512 workgroups of one token the state's traffic is all there
  // is, and whole rows are the better order for it (32 sequences: 24.1 us, 24.8 by columns; 64: 47.2, 49.1; rows in a loop
  // over the tokens took 25.3 and 47.8, and 35.9 at 48 sequences, where this takes 36.4). Above 2560, where every CU has
  // several rounds of them, two at a time are better than three: fewer reads and writes mix in HBM (96 sequences 70.0 ->
  // 69.2 us, 128 92.9 -> 90.9, 256 190.7 -> 180.8; 80 58.7 -> 58.8, 64 47.2 -> 48.1).
  const dim3 grid((unsigned)(batch * num_v_heads));
  auto launch = [&](auto kernel, int lds = 0) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, stream, p); };
  const int pad = grid.x > kStepFullWgs ? kStepPadLds : 0;
  if (tokens > 1 || state_snap)
    gate ? launch(gdn_columns_kernel<true, true, true>) : launch(gdn_columns_kernel<false, true, true>);
  else if (grid.x <= kEarlyMaxWgs)
    gate ? launch(gdn_columns_kernel<true, false, true>) : launch(gdn_columns_kernel<false, false, true>);
  else if (grid.x <= kColsMaxWgs)
    gate ? launch(gdn_columns_kernel<true, false, false>) : launch(gdn_columns_kernel<false, false, false>);
  else
    gate ? launch(gdn_recurrent_kernel<true>, pad) : launch(gdn_recurrent_kernel<false>, pad);
  return axk_launch_status();
}

extern "C" int axk_gdn_recurrent(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint16_t* a,
                                 const uint16_t* b, const float* a_log, const float* dt_bias, const float* state_in,
                                 float* state_out, uint16_t* out, int64_t batch, int64_t tokens, int64_t num_k_heads,
                                 int64_t num_v_heads, int64_t head_k_dim, int64_t head_v_dim, axk_stream_t stream) {
  AXK_REQUIRE(head_k_dim == kDK && head_v_dim == kDV, AXK_E_SHAPE);
  const AxkGdnStrides ld{num_k_heads * kDK, num_k_heads * kDK, num_v_heads * kDV, num_v_heads};
  return axk_gdn_recurrent_strided(q, k, v, a, b, a_log, dt_bias, state_in, state_out, out, batch, tokens,
                                   num_k_heads, num_v_heads, ld, nullptr, AXK_VORDER_GROUPED, axk_stream(stream));
}
