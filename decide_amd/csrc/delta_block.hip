// The gated delta recurrence 16 tokens at a time, in one kernel (decide:
// kernels/delta_fast.metal; cpu_ref.rs:101-129). Per value head, with
// γ_i = g_0 … g_i inside a block of 16 tokens and S the state before it:
//   A_ij = β_i (γ_i/γ_j) k_i·k_j (i > j),  T = (I + A)⁻¹,
//   D = T · β(v − γ S k),                  the block's 16 state updates,
//   O_i = γ_i S q_i + Σ_{j<=i} (γ_i/γ_j)(q_i·k_j) D_j,
//   S ← γ_15 S + Σ_i (γ_15/γ_i) D_i k_iᵀ,
// every product an fp32 matrix product on v_mfma_f32_16x16x4_f32. The token
// by token form of the same recurrence waits about 160 ns per token for its
// chain of two dot products and two cross-lane sums; here the chain (products,
// one LDS exchange and a barrier, all in sequence) is paid once per 16 tokens.
// Measured: 169 tokens 31.4 → 22.0 µs, 319 tokens 55.5 → 35.3, 41 tokens
// 10.9 → 10.2; 1.5 µs per block.
//
// Accuracy is no less than token by token: no sum runs longer than it must in
// one accumulator (T·x in four, the update and M·D in two, K Kᵀ and Q Kᵀ in
// 16), and log g, β and the γ ratios come from fp64. Against 64 bits, over 17
// to 319 tokens of inputs as the conv forms them: output 0.99e-7 and state
// 0.73e-7 (token by token 1.05e-7 and 0.84e-7); with one accumulator each, two
// for K Kᵀ and Q Kᵀ, and fp32 gates 1.60e-7 and 0.93e-7, at 20.7 µs for 169.
//
//   * A workgroup is one value head × 16 value rows: 256 workgroups, one per
//     CU, the 8 of a head (and of the two value heads that share a key head)
//     on one XCD, whose L2 serves their common q and k rows.
//   * Waves 0-3 carry the recurrence, wave w the keys [32w, 32w + 32). They
//     hold Sᵀ as MFMA accumulators and the products are arranged so that no
//     operand ever changes lanes: an accumulator's lane (r, g) has rows
//     4g .. 4g + 3 of column r, which is the B operand of four 4-deep steps
//     when step e takes rows {4g + e}; so S feeds S·kᵀ and S·qᵀ, x feeds T·x,
//     and D feeds M·D and the state update, all from the registers they were
//     formed in. Only S·kᵀ and S·qᵀ, summed over the waves' key ranges, go
//     through LDS: one barrier per block.
//   * Waves 4-7 prepare the next two blocks meanwhile, two waves each: one
//     K Kᵀ, the gates, and T by forward substitution (T's columns in lanes,
//     A's rows broadcast from LDS; powers of A would need fewer steps but
//     cancel badly when keys repeat), the other Q Kᵀ and its weights. Sums of log g run in fp64: the γ ratios are exponentials of their
//     differences.
//   * Waves 8-11 form and store the output, a block behind the recurrence,
//     every fourth block each.
//   * The recurrence's own q, k and v come a ring of six blocks ahead by DMA
//     into LDS, 16 KB of q and k in 16 instructions per block: loaded into
//     registers by every wave that uses them they took 64, and the CU passes
//     a vector-memory instruction in about 30 clocks, so they set the pace.
//     The 16-byte chunk c of row t sits at chunk c ^ t (values: at c ^ t / 4),
//     which keeps both the row and the column reads free of bank conflicts.
//   * Rows past T load row T - 1 and take β = 0, g = 1: they change nothing.
//   * A non-finite x (x = β(v − γ S k)) or D (finite inputs whose products
//     overflow) may reach only its own token and later ones, as token by
//     token; the zeros above T's and M's diagonals would spread it to earlier
//     tokens of the block, so such a block takes its products from cleaned
//     operands and marks the later tokens afterwards.
#include "tile_common.h"

namespace dh {

namespace {
constexpr int NK = 16, DK = 128, NV = 32, DV = 128;
constexpr int kTok = 16;   // tokens per block
constexpr int kAhead = 2;  // blocks prepared together, two prep waves each
constexpr int kLD = 20;    // row stride of a 16 x 16 LDS matrix: conflict-free 4-byte writes and 16-byte reads
constexpr double kMinLogG = -1e4;  // exp of it is 0 in fp32; keeps differences of -inf out of the ratios

struct Prepared {  // what the recurrence and the output need of one block besides q, k, v
  float t[kTok * kLD];
  float m[kTok * kLD];
  float beta[kTok], gam[kTok], rest[kTok];  // β_i, γ_i, γ_15/γ_i
  double sum[kTok];                         // Σ log g over tokens 0 .. i
};

// x of the lane o places below in its row of 16 lanes (0 past the row's start).
template <int O>
__device__ __forceinline__ double row_shr(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x110 + O, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x110 + O, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Lane M of this lane's row of 16.
template <int M>
__device__ __forceinline__ float row_lane(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + M, 0xF, 0xF, true));
}

__device__ __forceinline__ f4 mfma4(float a, float b, const f4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// exp of an fp64 argument to fp32 accuracy: that of its fp32 part, corrected for what the rounding left off.
__device__ __forceinline__ float exp_of(double x) {
  const float hi = (float)x, e = expf(hi);
  return fmaf(e, (float)(x - hi), e);
}
__device__ __forceinline__ bool finite(float x) { return __builtin_fabsf(x) < __builtin_inff(); }

constexpr int kRing = 6;             // blocks of q, k and v in LDS
struct Rows {                        // one of them
  float k[kTok * DK], q[kTok * DK];  // [token][128 keys], 16-byte chunk c of token t at chunk c ^ t
  float v[kTok * 16];                // [token][16 value rows], chunk c of token t at c ^ t / 4
};

// What becomes of one block's keys (Q false: T) and of its queries and gates (Q true: M, β, γ), a wave each. start()
// runs during one block of the recurrence, finish() during the next; the gates come before either.
template <bool Q>
struct PrepWave {
  uint32_t T;
  int r, g;
  f4 gram;  // K Kᵀ or Q Kᵀ: rows 4g .., column r

  // The 128 terms in kChains sums of their own, added in pairs: in two they were most of the output's error.
  __device__ __forceinline__ void start(const Rows& R) {
    constexpr int kChains = 16;
    f4 c[kChains];
#pragma unroll
    for (int i = 0; i < kChains; ++i) c[i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int x = r * DK + 4 * ((4 * i + g) ^ r);
      const f4 kf = *(const f4*)(R.k + x);
      const f4 lf = Q ? *(const f4*)(R.q + x) : kf;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f4& to = c[(4 * i + e) % kChains];
        to = mfma4(lf[e], kf[e], to);
      }
    }
#pragma unroll
    for (int n = kChains / 2; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; ++i) c[i] += c[i + n];
    gram = c[0];
  }
  // av, bv: the gate inputs of token t0 + r (of the last token past T).
  // log g and β in fp64: their fp32 roundings reach every ratio and product of the block.
  __device__ __forceinline__ void gates(float av, float bv, double negA, double bias, uint32_t t0, Prepared& p) {
    const bool valid = t0 + r < T;
    const double z = (double)av + bias;
    double lg = negA * (z > 20.0 ? z : log(1.0 + exp(z)));
    lg = lg < kMinLogG ? kMinLogG : lg;
    double sum = valid ? lg : 0.0;
    sum += row_shr<1>(sum);
    sum += row_shr<2>(sum);
    sum += row_shr<4>(sum);
    sum += row_shr<8>(sum);
    if (g == 0) {
      p.sum[r] = sum;
      p.beta[r] = valid ? (float)(1.0 / (1.0 + exp(-(double)bv))) : 0.0f;
      p.gam[r] = exp_of(sum);
    }
    __builtin_amdgcn_wave_barrier();
    if (g == 0) p.rest[r] = exp_of(p.sum[kTok - 1] - sum);
  }
  __device__ __forceinline__ void finish(Prepared& p) {
    const double mine = p.sum[r];
    f4 beta;
    if constexpr (!Q) beta = *(const f4*)(p.beta + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * g + e;  // row; column r
      const float ratio = exp_of(p.sum[i] - mine);
      if constexpr (Q)
        p.m[i * kLD + r] = i >= r ? ratio * gram[e] : 0.0f;
      else
        p.t[i * kLD + r] = i > r ? -(beta[e] * ratio * gram[e]) : 0.0f;
    }
    if constexpr (!Q) {
      __builtin_amdgcn_wave_barrier();
      invert(p);
    }
  }
  // T = (I + A)⁻¹ in place of -A: lane r has column r of T, and of -A, whose row i it takes from its row of lanes.
  __device__ __forceinline__ void invert(Prepared& p) {
    float n[kTok], t[kTok];
#pragma unroll
    for (int i = 1; i < kTok; ++i) n[i] = p.t[i * kLD + r];
    static_for<0, kTok>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      float s0 = i == r ? 1.0f : 0.0f, s1 = 0.0f;
      static_for<0, i>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        if constexpr (m & 1)
          s1 = fmaf(row_lane<m>(n[i]), t[m], s1);
        else
          s0 = fmaf(row_lane<m>(n[i]), t[m], s0);
      });
      t[i] = s0 + s1;
    });
#pragma unroll
    for (int i = 0; i < kTok; ++i)
      if (g == i / 4) p.t[i * kLD + r] = t[i];
  }
};

// One block's q, k and v in a recurrence wave.
struct BlockRows {
  f4 ka[2], qa[2];  // token r, keys 32w + 16t + 4g ..
  f4 kt[2];         // tokens 4g .., key 32w + 16t + r
  f4 v;             // tokens 4g .., value row dv0 + r
};

constexpr int kRowDmas = 5;  // DMAs per recurrence wave and block: two of k, two of q, one of v

// 4-byte-per-lane DMA global → LDS (dma16's counterpart for v, which need only be 4-byte aligned).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma4(uint32_t m0, uint32_t voff, const void* sbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2 offset:0" ::"s"(m0), "v"(voff), "s"(sbase)
               : "memory", "m0");
}
#pragma clang diagnostic pop
}  // namespace

__global__ __launch_bounds__(768) void delta_block_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, const float* __restrict__ a,
                                                          const float* __restrict__ b, const float* __restrict__ a_log,
                                                          const float* __restrict__ dt_bias, const float* state_in,
                                                          float* state_out, float* __restrict__ o, uint32_t T,
                                                          uint32_t ldab, uint32_t write_state) {
  __shared__ __attribute__((aligned(1024))) Rows rows[kRing];
  __shared__ __attribute__((aligned(16))) Prepared prep[4][kAhead];  // by pair of blocks, mod 4
  __shared__ f4 sk[2][4][64], sq[2][4][64];  // the waves' parts of S·kᵀ and S·qᵀ, by the block's parity
  __shared__ f4 upd[2][64];                  // D, zero from a value row's first non-finite token on
  __shared__ uint32_t first_bad[2][64];      // that token (kTok: none)
  const uint32_t h = 4 * (blockIdx.x & 7) + (blockIdx.x >> 6), hk = h >> 1;
  const uint32_t dv0 = 16 * ((blockIdx.x >> 3) & 7);
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t nblk = (T + kTok - 1) / kTok;
  const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
  // Barriers, the same number in every wave: three until the first blocks have landed and are prepared, one per
  // block c (after which every wave's part of S·kᵀ(c) and all of S·qᵀ(c - 1) and D(c - 1) can be read), one after
  // the last. What is prepared for a pair of blocks is written from three blocks before the pair on (its gates)
  // and read until one block after it (by the output): four buffers.

  if (wave >= 8) {
    const uint32_t i = wave - 8;
    for (int n = 0; n < 4; ++n) __syncthreads();
    for (uint32_t c = 0; c < nblk; ++c) {
      __syncthreads();
      if ((c & 3) != i) continue;
      const int par = c & 1;
      const Prepared& p = prep[c / kAhead % 4][c % kAhead];
      const f4 mm = *(const f4*)(p.m + r * kLD + 4 * g), gam = *(const f4*)(p.gam + 4 * g);
      const f4 d = upd[par][lane];
      const uint32_t bad = first_bad[par][lane];
      f4 o1 = zero, ov = gam * ((sq[par][0][lane] + sq[par][1][lane]) + (sq[par][2][lane] + sq[par][3][lane]));
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        ov = mfma4(mm[e], d[e], ov);
        o1 = mfma4(mm[e + 1], d[e + 1], o1);
      }
      ov += o1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t tok = c * kTok + 4 * g + e;
        if (tok < T)
          o[((size_t)tok * NV + h) * DV + dv0 + r] = (uint32_t)(4 * g + e) >= bad ? __builtin_nanf("") : ov[e];
      }
    }
    return;
  }

  if (wave >= 4) {
    const uint32_t j = (wave >> 1) & 1;
    if (wave & 1) {
      const double negA = -exp((double)a_log[h]), bias = dt_bias[h];
      PrepWave<true> w{T, r, g, zero};
      float av, bv;
      auto gates_in = [&](uint32_t t0) {
        const size_t row = min(t0 + r, T - 1);
        av = a[row * ldab + h];
        bv = b[row * ldab + h];
      };
      gates_in(j * kTok);
      w.gates(av, bv, negA, bias, j * kTok, prep[0][j]);
      gates_in((kAhead + j) * kTok);
      __syncthreads();
      w.start(rows[j]);
      __syncthreads();
      w.finish(prep[0][j]);
      w.gates(av, bv, negA, bias, (kAhead + j) * kTok, prep[1][j]);
      gates_in((2 * kAhead + j) * kTok);
      __syncthreads();
      for (uint32_t c = 0; c < nblk; ++c) {
        // during blocks 2s and 2s + 1: block 2s + 2 + j, and the gates of block 2s + 4 + j (past the last block
        // there is nothing to be used of them)
        const uint32_t s = c / kAhead;
        if (c % kAhead == 0) {
          w.start(rows[(c + kAhead + j) % kRing]);
        } else {
          w.finish(prep[(s + 1) % 4][j]);
          w.gates(av, bv, negA, bias, ((s + 2) * kAhead + j) * kTok, prep[(s + 2) % 4][j]);
          gates_in(((s + 3) * kAhead + j) * kTok);
        }
        __syncthreads();
      }
    } else {
      PrepWave<false> w{T, r, g, zero};
      __syncthreads();
      w.start(rows[j]);
      __syncthreads();
      w.finish(prep[0][j]);
      __syncthreads();
      for (uint32_t c = 0; c < nblk; ++c) {
        if (c % kAhead == 0)
          w.start(rows[(c + kAhead + j) % kRing]);
        else
          w.finish(prep[(c / kAhead + 1) % 4][j]);
        __syncthreads();
      }
    }
    __syncthreads();
    return;
  }

  __builtin_amdgcn_s_setprio(3);
  const uint32_t d0 = 32 * wave;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)rows;
  // Issues this wave's DMAs of block blk (rows past T: row T - 1, so any blk is in range).
  auto dma = [&](uint32_t blk) {
    const uint32_t tb = min(blk * kTok, T - 1), most = T - 1 - tb;
    const float* kb = k + ((size_t)tb * NK + hk) * DK;
    const float* qb = q + ((size_t)tb * NK + hk) * DK;
    const float* vb = v + ((size_t)tb * NV + h) * DV + dv0;
    const uint32_t slot = lds0 + (blk % kRing) * (uint32_t)sizeof(Rows);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const uint32_t t = 4 * wave + 2 * n + (lane >> 5);  // two rows per DMA
      const uint32_t off = min(t, most) * (NK * DK * 4) + ((lane & 31) ^ t) * 16;
      const uint32_t to = slot + (4 * wave + 2 * n) * (DK * 4);
      dma16(to, off, kb);
      dma16(to + (uint32_t)sizeof(Rows::k), off, qb);
    }
    const uint32_t t = 4 * wave + g;
    dma4(slot + 2 * (uint32_t)sizeof(Rows::k) + wave * 256, min(t, most) * (NV * DV * 4) + (r ^ (4 * wave)) * 4, vb);
  };
  auto load = [&](BlockRows& x, uint32_t blk) {
    const Rows& R = rows[blk % kRing];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int c = (8 * wave + 4 * t + g) ^ r;
      x.ka[t] = *(const f4*)(R.k + r * DK + 4 * c);
      x.qa[t] = *(const f4*)(R.q + r * DK + 4 * c);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 4 * g + e;
      x.kt[0][e] = R.k[t * DK + 4 * ((8 * wave + (r >> 2)) ^ t) + (r & 3)];
      x.kt[1][e] = R.k[t * DK + 4 * ((8 * wave + 4 + (r >> 2)) ^ t) + (r & 3)];
      x.v[e] = R.v[t * 16 + (r ^ (4 * g))];
    }
  };
  f4 s[2];  // Sᵀ: keys d0 + 16t + 4g .., value row dv0 + r
  const size_t srow = ((size_t)h * DV + dv0 + r) * DK + d0 + 4 * g;
#pragma unroll
  for (int t = 0; t < 2; ++t) s[t] = *(const f4*)(state_in + srow + 16 * t);

  auto block = [&](uint32_t c, BlockRows& x, BlockRows& next) {
    const int par = c & 1;
    f4 p0 = zero, p1 = zero, q0 = zero, q1 = zero;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p0 = mfma4(x.ka[0][e], s[0][e], p0);
      p1 = mfma4(x.ka[1][e], s[1][e], p1);
    }
    const Prepared& p = prep[c / kAhead % 4][c % kAhead];
    const f4 tt = *(const f4*)(p.t + r * kLD + 4 * g);
    const f4 beta = *(const f4*)(p.beta + 4 * g), gam = *(const f4*)(p.gam + 4 * g);
    const f4 rest = *(const f4*)(p.rest + 4 * g);
    const float gend = p.gam[kTok - 1];
    sk[par][wave][lane] = p0 + p1;
    wait_vm<kRowDmas>();  // blocks up to c + 4 have landed (the next pair's preparation reads them); c + 5 may not
    __syncthreads();
    const f4 k0 = sk[par][0][lane], k1 = sk[par][1][lane], k2 = sk[par][2][lane], k3 = sk[par][3][lane];
    load(next, c + 1);
    dma(c + kRing);  // into this block's slot: every wave has its rows in registers
    // S·qᵀ while the parts of S·kᵀ come back from LDS
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      q0 = mfma4(x.qa[0][e], s[0][e], q0);
      q1 = mfma4(x.qa[1][e], s[1][e], q1);
    }
    f4 xv = beta * (x.v - gam * ((k0 + k1) + (k2 + k3)));
    // T · x, a sum per step of four tokens
    auto update = [&] {
      return (mfma4(tt[0], xv[0], zero) + mfma4(tt[1], xv[1], zero)) +
             (mfma4(tt[2], xv[2], zero) + mfma4(tt[3], xv[3], zero));
    };
    f4 d = update();
    uint32_t bad = kTok;  // this value row's first token whose x or D is not finite
    if (__any(!finite((d[0] + d[1]) + (d[2] + d[3])))) {
      auto first_not_finite = [&](const f4& y) {
        uint32_t n = kTok;
#pragma unroll
        for (int e = 3; e >= 0; --e)
          if (!finite(y[e])) n = 4 * g + e;
        n = min(n, (uint32_t)__shfl_xor((int)n, 16, 64));
        return min(n, (uint32_t)__shfl_xor((int)n, 32, 64));
      };
      bad = first_not_finite(xv);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!finite(xv[e])) xv[e] = 0.0f;
      d = update();
      bad = min(bad, first_not_finite(d));
    }
    sq[par][wave][lane] = q0 + q1;
#pragma unroll
    for (int t = 0; t < 2; ++t) s[t] *= gend;
    f4 dd = d * rest;
    if (bad < (uint32_t)kTok) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * g + e >= bad) {
          d[e] = 0.0f;
          dd[e] = __builtin_nanf("");
        }
    }
    f4 u[2] = {zero, zero};
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      s[0] = mfma4(x.kt[0][e], dd[e], s[0]);
      s[1] = mfma4(x.kt[1][e], dd[e], s[1]);
      u[0] = mfma4(x.kt[0][e + 1], dd[e + 1], u[0]);
      u[1] = mfma4(x.kt[1][e + 1], dd[e + 1], u[1]);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) s[t] += u[t];
    if (wave == 0) {
      upd[par][lane] = d;
      first_bad[par][lane] = bad;
    }
  };
  BlockRows x0, x1;
  for (uint32_t c = 0; c < (uint32_t)kRing; ++c) dma(c);
  wait_vm<(kRing - kAhead) * kRowDmas>();
  __syncthreads();
  load(x0, 0);
  wait_vm<(kRing - 2 * kAhead) * kRowDmas>();
  __syncthreads();
  __syncthreads();
  for (uint32_t c = 0; c < nblk; c += 2) {
    block(c, x0, x1);
    if (c + 1 >= nblk) break;
    block(c + 1, x1, x0);
  }
  wait_vm<0>();  // no DMA may land after this workgroup's LDS is given away
  __syncthreads();
  if (write_state) {
#pragma unroll
    for (int t = 0; t < 2; ++t) *(f4*)(state_out + srow + 16 * t) = s[t];
  }
}

hipError_t launch_gated_delta_block(const float* q, const float* k, const float* v, const float* a, const float* b,
                                    const float* a_log, const float* dt_bias, const float* state_in,
                                    float* state_out, float* o, uint32_t t, uint32_t ldab, bool write_state,
                                    hipStream_t s) {
  hipLaunchKernelGGL(delta_block_kernel, dim3(NV * DV / 16), dim3(768), 0, s, q, k, v, a, b, a_log, dt_bias, state_in,
                     state_out, o, t, ldab, write_state ? 1u : 0u);
  return hipGetLastError();
}

}  // namespace dh
