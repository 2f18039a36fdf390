// Causal GQA attention with the sigmoid output gate, for gfx950 MFMA
// (decide: kernels/attn_fast.metal; cpu_ref.rs:167-188):
//   y[r, h·256 + d] = (softmax_j(q_r,h · k_j,h/4 / 16) · v_·,h/4)[d] · σ(gate[r, h·256 + d]),
// over cache rows j = 0 ..= qpos[r]; q, K, V fp16, scores and softmax fp32,
// the softmax weights rounded to fp16 once as the P·V operand, y fp16.
//
// Design (MI355X's own):
//   * A workgroup is one kv head × 32 query rows; its 8 waves are the 4 query
//     heads sharing that kv head × 2 halves of a staged tile of 64 keys, each
//     wave taking all 32 rows on v_mfma_f32_32x32x16_f16. A wave reads every K
//     and Vᵀ fragment it multiplies from LDS, 32 KB per 32 keys, so a fragment
//     serves 32 rows. With 16 rows per wave and the waves split over rows
//     instead of keys, 2,307 causal rows took 99 µs against 73, 16 rows at
//     position 2,000 92 against 53, 169 rows behind 107 keys 24.0 against 20.0
//     (and 8 rows at the start of a prompt 8.6 against 9.7). 64 keys are 64
//     products of 32 clocks per SIMD, and as long in LDS reads at 128 bytes a
//     clock; over 2,307 rows a tile takes 5,100 CU clocks, starts and ends
//     included: the matrix cores are busy for 40 % of them, without a bank
//     conflict. The two key halves of a head meet once, at the end, through
//     LDS: each wave takes half of the dims.
//   * Everything is computed transposed: Sᵀ = K·Qᵀ (A = K rows from LDS,
//     B = the wave's Q rows held in registers for the whole kernel) and
//     Oᵀ += Vᵀ·Pᵀ. In the MFMA output layout lane (r, f), r = lane % 32,
//     f = lane / 32, then holds 16 scores of ONE query row, for keys
//     {8b + 4f .. + 3}, which are the B operands Pᵀ needs if the 32 keys are
//     taken in that order — so P goes from scores to MFMA operand without
//     leaving registers, and each Vᵀ fragment is two transposing LDS reads
//     (ds_read_b64_tr_b16) of 4 consecutive keys each.
//   * K and V go straight into LDS by DMA as they lie in the cache, two tiles of
//     each, one barrier per 64 keys. 16-byte chunk c of key t sits at chunk
//     c ^ t % 16 (K: 16 rows' reads hit all banks) or c ^ 4 (t % 4) (V: so do a
//     transposing read's 4 keys). Nothing of them is held in registers, which Q
//     (64) and O (128) nearly fill.
//   * Online softmax in the exp2 domain; a row's max is reduced across the
//     two lanes that hold it; the running sum stays per lane and is reduced
//     once at the end. The reference point moves (and O is rescaled) only when
//     a score passes it by more than 2^8, which after the first blocks almost
//     never happens. Tiles wholly before every row skip the causal mask.
//   * One workgroup per CU (two waves per SIMD), so a causal prompt's longest
//     query block (all of its keys) would set the kernel's time while most
//     CUs sit idle. A query block's keys are therefore cut into pieces of L
//     key blocks at fixed offsets (piece p covers blocks [pL, pL + L), the
//     last piece the rest), one workgroup each, dispatched longest-first;
//     a query block with more than one piece writes each piece's (max,
//     sum, unnormalised O) per row and head, and attention_combine_kernel
//     merges them. The cut points depend only on L (chosen on the host from
//     the row count and the key bound), never on the neighbouring rows, so a
//     row whose keys end before a cut gets bit for bit the one-piece result.
//   * Rows past `rows` are clamped for loads and skipped for stores; keys past
//     the block's last position are masked (their staged rows are clamped
//     reads of valid cache rows).
#include <algorithm>

#include "tile_common.h"

namespace dh {

namespace {
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr int kHD = 256, kNQ = 16, kQDim = kNQ * kHD;
constexpr int kBQ = 32;     // query rows per workgroup
constexpr int kBKey = 32;   // keys per block: the unit of the key pieces, and a wave's share of a tile
constexpr int kTile = 64;   // keys staged together
constexpr int kTileBytes = kTile * kHD * 2;
constexpr float kScaleLog2 = 0.0625f * 1.4426950408889634f;  // 1/16 · log2(e)
constexpr float kNeg = -1e30f;
constexpr float kLazy = 8.0f;  // log2 headroom of the softmax reference point (weights up to 256)

typedef float f16v __attribute__((ext_vector_type(16)));

// The two lanes (r, 0) and (r, 1) that hold one query row, combined with gfx950's half-wave swap (no LDS round
// trip): called with the same value twice, the two results are x and its partner.
__device__ __forceinline__ float max_halves(float x) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Transposing LDS read: the 16 lanes of a row group read a 4 x 16 block of halves, 8 bytes each (lane s: row s / 4,
// columns 4 (s % 4) ..), and lane s gets column s.
typedef short s4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ s4 read_tr(const char* at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(at));
}

// The gate's σ: the hardware exp, and 1 / d from the hardware reciprocal (one ulp off at worst) and a Newton step, which
// makes it the full division's value. For the 64 outputs of a lane the step takes 0.3 µs at 16 rows and none that shows
// from 32 on; the division took 1.7 at 16 and 1.6 at 2,307 rows. Past 2^100 d is held there (at
// infinity the step is inf · 0; σ is 0 in fp16 by far).
__device__ __forceinline__ float sigmoid(float x) {
  const float d = __builtin_elementwise_minimum(1.0f + __expf(-x), 0x1p100f);  // NaN stays NaN
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.0f), r, r);
}

__device__ __forceinline__ f16v mfma32(const h8& a, const h8& b, const f16v& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
}  // namespace

// The largest position over query block qb's 32 rows (rows past `rows` clamped
// to the last one): its last key, the same in both kernels.
__device__ __forceinline__ uint32_t block_kmax(const uint32_t* __restrict__ qpos, uint32_t qb, uint32_t rows,
                                               uint32_t lane) {
  uint32_t v = qpos[min(qb * kBQ + (lane & 31), rows - 1)];
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, 64));
  return v;
}

// Pieces query block qb really has: ceil(nblk / L), at most np (the last one
// takes the remainder).
__device__ __forceinline__ uint32_t block_pieces(uint32_t nblk, uint32_t L, uint32_t np) {
  return min(np, (nblk + L - 1) / L);
}

__global__ __launch_bounds__(512) void attention_kernel(const _Float16* __restrict__ q, const _Float16* __restrict__ kc,
                                                        const _Float16* __restrict__ vc, const float* __restrict__ pq,
                                                        const uint32_t* __restrict__ qpos, _Float16* __restrict__ y,
                                                        float* __restrict__ part, uint32_t ldq, uint32_t rows,
                                                        uint32_t L, uint32_t np) {
  // two tiles of K, two of V; at the end the halves' states
  __shared__ __attribute__((aligned(1024))) char lds[4 * kTileBytes + 8 * 64 * 8];
  static_assert(8 * 16 * 64 * 16 + 8 * 64 * 8 <= sizeof(lds), "the halves' exchange fits the tiles");
  // Work item: kv head fastest, then query blocks longest (last) first, then pieces. The hardware deals
  // workgroups round-robin over the 8 XCDs, so each XCD gets every 8th item: with pieces outermost, any 8
  // consecutive items are two query blocks' worth of the same piece, of about the same length.
  const uint32_t nqb = (rows + kBQ - 1) / kBQ;
  const uint32_t kvh = blockIdx.x & 3;
  const uint32_t qb = nqb - 1 - (blockIdx.x >> 2) % nqb;
  const uint32_t piece = (blockIdx.x >> 2) / nqb;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2;
  const uint32_t h = kvh * 4 + (wave & 3);
  const int r = lane & 31, f = lane >> 5;
  const uint32_t row = min(qb * kBQ + r, rows - 1);
  const uint32_t mypos = qpos[row];
  // Q by DMA into the second tiles (free until the loop), half a head per wave, chunk c of row t at c ^ t % 16: a
  // fragment loaded straight into registers would touch 32 rows per instruction
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const uint32_t qlds = (wave & 2 ? 3 : 1) * kTileBytes + (wave & 1) * (kBQ * kHD * 2);  // this head's 32 rows
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const uint32_t t = 16 * half + 2 * n + f;
    dma16(lds0 + qlds + (16 * half + 2 * n) * (kHD * 2),
          min(t, rows - 1 - qb * kBQ) * (kQDim * 2) + (r ^ (t & 15)) * 16, q + ((size_t)qb * kBQ * kNQ + h) * kHD);
  }
  // the workgroup's last key: the largest position over its 32 rows (loads past it are clamped to it)
  uint32_t kmax = mypos, minpos = mypos;
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) {
    kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o, 64));
    minpos = min(minpos, (uint32_t)__shfl_xor((int)minpos, o, 64));
  }
  kmax = __builtin_amdgcn_readfirstlane(kmax);
  minpos = __builtin_amdgcn_readfirstlane(minpos);
  const uint32_t nblk = kmax / kBKey + 1;
  const uint32_t npieces = block_pieces(nblk, L, np);
  if (piece >= npieces) {  // uniform over the workgroup: every wave read the same rows
    wait_vm<0>();          // no DMA may land after this workgroup's LDS is given away
    return;
  }
  // this piece's key blocks: L of them (L even, so whole tiles), the last piece the rest (its last tile may hold one
  // block past nblk, which is wholly masked)
  const uint32_t b0 = piece * L;
  const uint32_t b1 = piece + 1 == npieces ? nblk : b0 + L;

  // K and V of the block pair at blk into buffer buf: two keys per DMA, four of each per wave
  auto stage = [&](uint32_t blk, uint32_t buf) {
    const uint32_t kb0 = blk * kBKey, most = kmax - kb0;
    const _Float16* kb = kc + ((size_t)kb0 * 4 + kvh) * kHD;
    const _Float16* vb = vc + ((size_t)kb0 * 4 + kvh) * kHD;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const uint32_t t = 8 * wave + 2 * n + f, off = min(t, most) * (4 * kHD * 2);
      const uint32_t to = lds0 + buf * kTileBytes + (8 * wave + 2 * n) * (kHD * 2);
      dma16(to, off + (r ^ (t & 15)) * 16, kb);
      dma16(to + 2 * kTileBytes, off + (r ^ (t & 3) * 4) * 16, vb);
    }
  };
  // this lane's 8 bytes of a transposing read: key 4f + s / 4 of 8, dims 16 (lane / 16 % 2) + 4 (s % 4) of 32, for
  // s = lane % 16; the lane gets dim r of the 32 for keys 4f .. 4f + 3
  const int trk = 4 * f + (lane >> 2 & 3), trc = 2 * (lane >> 4 & 1) + (lane >> 1 & 1);
  const int tr0 = trk * (kHD * 2) + (lane & 1) * 8, trx = (lane >> 2 & 3) * 64 ^ half * 256;

  f16v oacc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[i][e] = 0.f;
  float m = kNeg, lsum = 0.f;

  stage(b0, 0);
  wait_vm<0>();
  __syncthreads();
  h8 qf[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) qf[c] = *(const h8*)(lds + qlds + r * (kHD * 2) + (((2 * c + f) ^ (r & 15)) * 16));
#pragma unroll
  for (int c = 0; c < 16; ++c) tie(qf[c]);
  __syncthreads();
  for (uint32_t blk = b0, buf = 0; blk < b1; blk += 2, buf ^= 1) {
    if (blk + 2 < b1) stage(blk + 2, buf ^ 1);  // into the buffer every wave left before the last barrier
    const char* ks = lds + buf * kTileBytes + (32 * half + r) * (kHD * 2);
    int sw = (f ^ (r & 15)) * 16;  // chunk 2c + f of the row sits at byte 32c ^ sw
    asm volatile("" : "+v"(sw));   // formed in the loop: 16 hoisted addresses would spill
    f16v st;
#pragma unroll
    for (int e = 0; e < 16; ++e) st[e] = 0.f;
    // fragments are read three products ahead; the barriers keep the compiler from moving the reads to their use
    h8 kf[4];
#pragma unroll
    for (int c = 0; c < 3; ++c) kf[c] = *(const h8*)(ks + ((32 * c) ^ sw));
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      if (c + 3 < 16) kf[(c + 3) % 4] = *(const h8*)(ks + ((32 * (c + 3)) ^ sw));
      __builtin_amdgcn_sched_barrier(0);
      st = mfma32(kf[c % 4], qf[c], st);
    }
    const uint32_t kb0 = blk * kBKey + 32 * half;  // this wave's first key
    float sv[16];
    if (kb0 + kBKey - 1 <= minpos) {  // every key is visible to every row
#pragma unroll
      for (int i = 0; i < 16; ++i) sv[i] = st[i] * kScaleLog2;
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t key = kb0 + 8 * (i / 4) + 4 * f + i % 4;
        sv[i] = key <= mypos ? st[i] * kScaleLog2 : kNeg;
      }
    }
    float bm = sv[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) bm = fmaxf(bm, sv[i]);
    bm = max_halves(bm);
    // Lazy rescale: the reference point m moves only when a score exceeds it by more than 2^kLazy, so
    // the weights stay <= 2^kLazy (well inside fp16) and O and the sum are rescaled only on the rare
    // tile that moves it (the normalisation uses the same m, so the result does not depend on when).
    if (__any(bm > m + kLazy)) {
      const float mnew = bm > m + kLazy ? bm : m;
      const float alpha = exp2f(m - mnew);
      lsum *= alpha;
      m = mnew;
#pragma unroll
      for (int i = 0; i < 8; ++i) oacc[i] *= alpha;
    }
    h8 pb[2];
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float pv = __builtin_amdgcn_exp2f(sv[i] - m);  // below 2^-126: 0, as in its fp16 operand
      ps += pv;
      pb[i / 8][i % 8] = (_Float16)pv;
    }
    lsum += ps;
    // Vᵀ fragment i = 8a + dt: keys 16a + 4f .. and 16a + 8 + 4f .. of dims 32 (dt ^ 4 half) ..
    const char* vs = lds + (2 + buf) * kTileBytes + 32 * half * (kHD * 2) + tr0;
    s4 vf[4][2];
    auto read_v = [&](int i) {
      const char* at = vs + ((64 * (i % 8) + 16 * trc) ^ trx) + 16 * (i / 8) * (kHD * 2);
      vf[i % 4][0] = read_tr(at);
      vf[i % 4][1] = read_tr(at + 8 * kHD * 2);
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) read_v(i);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i + 3 < 16) read_v(i + 3);
      __builtin_amdgcn_sched_barrier(0);
      const h8 va = __builtin_bit_cast(h8, __builtin_shufflevector(vf[i % 4][0], vf[i % 4][1], 0, 1, 2, 3, 4, 5, 6, 7));
      oacc[i % 8] = mfma32(va, pb[i / 8], oacc[i % 8]);
    }
    wait_vm<0>();
    __syncthreads();
  }

  // The halves' states meet: each wave keeps its oacc[0..3] (dims 128 half ..) and gives its partner the rest. A half
  // whose first key lies past a row's position has nothing for that row (its weights are exp2(0) on masked scores):
  // l = 0 and m = kNeg give it no weight. (Its O is finite: cache rows are.)
  float l = sum_halves(lsum);
  if ((uint64_t)mypos < (uint64_t)b0 * kBKey + 32 * half) {
    l = 0.f;
    m = kNeg;
  }
  const bool whole = npieces == 1;
  const float* gp = pq + (size_t)row * ldq + kQDim + h * kHD + 128 * half + 4 * f;
  f4 gate[16];
  if (whole) {  // in flight through the exchange; two float2s: 8-byte alignment suffices (decide's contract)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f2 g01 = *(const f2*)(gp + 8 * i), g23 = *(const f2*)(gp + 8 * i + 2);
      gate[i] = f4{g01[0], g01[1], g23[0], g23[1]};
    }
  }
  f4* xo = (f4*)lds;                        // [wave][16 pieces of 4 dims][64 lanes]
  f2* xml = (f2*)(lds + 8 * 16 * 64 * 16);  // [wave][64 lanes]
  const int partner = wave ^ 4;
  xml[wave * 64 + lane] = f2{m, l};
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const f16v& o = oacc[4 + i / 4];
    const int e = 4 * (i % 4);
    xo[(wave * 16 + i) * 64 + lane] = f4{o[e], o[e + 1], o[e + 2], o[e + 3]};
  }
  // For up to four rows σ is formed here, where the wave would wait for its partner, for more it overlaps the exchange's
  // reads below. Here and below: 1 row 9.4 and 13.0 µs, 3 rows at position 600 22.6 and 26.3, 6 and 8 rows alike, 32 rows
  // 13.0 and 11.8.
  const bool few = rows - qb * kBQ <= 4;
  if (whole && few) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) gate[i][e] = sigmoid(gate[i][e]);
  }
  __syncthreads();
  if (qb * kBQ + r >= rows) return;
  const f2 pml = xml[partner * 64 + lane];
  const float mx = fmaxf(m, pml[0]);
  const float wme = exp2f(m - mx), wpa = exp2f(pml[0] - mx);
  const float lt = l * wme + pml[1] * wpa;
  // dims 128 half + 8i + 4f .. + 3; which product is fused is written out: left to the compiler it differed between the
  // two uses below, and with it a row's bits by how many rows it is called with
  auto merged = [&](int i) {
    const f4 po = xo[(partner * 16 + i) * 64 + lane];
    f4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(po[e], wpa, oacc[i / 4][4 * (i % 4) + e] * wme);
    return o;
  };
  if (!whole) {
    // This piece's state for the combine: O unnormalised (relative to mx), and (mx, lt), where a row with no key in
    // the piece (position before its first key) has l = 0: the combine skips the piece for that row by the same
    // position test.
    const uint32_t prow = nqb * kBQ;
    const size_t slot = ((size_t)piece * prow + qb * kBQ + r) * kNQ + h;
    float* op = part + slot * kHD + 128 * half + 4 * f;
#pragma unroll
    for (int i = 0; i < 16; ++i) *(f4*)(op + 8 * i) = merged(i);
    if (half == 0 && f == 0) {
      float* ml = part + (size_t)np * prow * kNQ * kHD + 2 * slot;
      *(f2*)ml = f2{mx, lt};
    }
    return;
  }
  const float inv = 1.0f / lt;
  _Float16* yp = y + (size_t)row * kQDim + h * kHD + 128 * half + 4 * f;
  auto store = [&](auto sigma) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f4 o = merged(i);
      _Float16 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (_Float16)(o[e] * inv * sigma(gate[i][e]));
      *(h2*)(yp + 8 * i) = h2{v[0], v[1]};  // 4-byte alignment suffices (decide's contract)
      *(h2*)(yp + 8 * i + 2) = h2{v[2], v[3]};
    }
  };
  if (few)
    store([](float x) { return x; });
  else
    store([](float x) { return sigmoid(x); });
}

// Merges the pieces of every query block that has more than one: a workgroup
// per row, a lane per (query head, 16 dims). Only the pieces whose first key
// the row can see take part (the attention kernel's position test); with one
// such piece the arithmetic is the one-piece path's own (weight exp2(0) = 1),
// so the result is identical.
__global__ __launch_bounds__(256) void attention_combine_kernel(const float* __restrict__ part,
                                                                const float* __restrict__ pq,
                                                                const uint32_t* __restrict__ qpos,
                                                                _Float16* __restrict__ y, uint32_t ldq, uint32_t rows,
                                                                uint32_t L, uint32_t np) {
  const uint32_t r = blockIdx.x, qb = r / kBQ;
  const int tid = threadIdx.x;
  const uint32_t kmax = block_kmax(qpos, qb, rows, tid & 63);
  const uint32_t npieces = block_pieces(kmax / kBKey + 1, L, np);
  if (npieces <= 1) return;  // written by the attention kernel itself
  const uint32_t mypos = qpos[r];
  const uint32_t nv = (uint32_t)min((uint64_t)npieces, (uint64_t)mypos / ((uint64_t)L * kBKey) + 1);
  const uint32_t h = tid >> 4, d0 = 16 * (tid & 15);
  const uint32_t prow = (rows + kBQ - 1) / kBQ * kBQ;
  const size_t pstride = (size_t)prow * kNQ;  // (row, head) slots per piece
  const size_t slot0 = (size_t)r * kNQ + h;
  const float* ml = part + (size_t)np * pstride * kHD;
  float mv[kAttnMaxPieces], lv[kAttnMaxPieces];
#pragma unroll
  for (uint32_t p = 0; p < kAttnMaxPieces; ++p)
    if (p < nv) {
      const f2 st = *(const f2*)(ml + 2 * (p * pstride + slot0));
      mv[p] = st[0];
      lv[p] = st[1];
    }
  float mx = mv[0];
#pragma unroll
  for (uint32_t p = 1; p < kAttnMaxPieces; ++p)
    if (p < nv) mx = fmaxf(mx, mv[p]);
  f4 o[4];
  float l;
  {  // piece 0 holds every row's first key
    const float w = exp2f(mv[0] - mx);
    const f4* op = (const f4*)(part + slot0 * kHD + d0);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = op[j] * w;
    l = lv[0] * w;
  }
#pragma unroll
  for (uint32_t p = 1; p < kAttnMaxPieces; ++p)
    if (p < nv) {
      const float w = exp2f(mv[p] - mx);
      const f4* op = (const f4*)(part + (p * pstride + slot0) * kHD + d0);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += op[j] * w;
      l += lv[p] * w;
    }
  const float inv = 1.0f / l;
  const float* gp = pq + (size_t)r * ldq + kQDim + h * kHD + d0;
  _Float16* yp = y + (size_t)r * kQDim + h * kHD + d0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const f2 gt = *(const f2*)(gp + 2 * j);
    const float o0 = o[j / 2][2 * (j % 2)], o1 = o[j / 2][2 * (j % 2) + 1];
    *(h2*)(yp + 2 * j) = h2{(_Float16)(o0 * inv * sigmoid(gt[0])),
                            (_Float16)(o1 * inv * sigmoid(gt[1]))};
  }
}

AttnSplit attention_split(uint32_t rows, uint32_t npos, uint32_t cus) {
  AttnSplit sp;
  if (rows == 0) return sp;
  npos = std::max(npos, rows);
  const uint32_t nqb = (rows + kBQ - 1) / kBQ;
  const uint32_t nbm = (npos + kBKey - 1) / kBKey;  // key blocks of the furthest row
  // key blocks over every query block if the rows sit at positions npos - rows .. npos - 1 (a prompt chunk)
  uint64_t est = 0;
  for (uint32_t qb = 0; qb < nqb; ++qb) {
    const uint64_t last = std::min<uint64_t>(npos - 1, (uint64_t)(npos - rows) + (uint64_t)qb * kBQ + kBQ - 1);
    est += last / kBKey + 1;
  }
  // Pieces of 1.5x one CU's even share of the work (4 kv heads), even length, at most kAttnMaxPieceRows / 32
  // query-block pieces in all (the workspace bound). Measured, with the combine: 850 causal rows 1.0x 40.7 us, 1.3x
  // 35.2, 1.6x 30.9; 1,200 rows 48.7, 38.3, 36.9; 2,307 rows 84, 72, 72; 603 rows 26.8 at any. Fewer, longer pieces
  // write fewer partial states for the combine; shorter ones balance the CUs better.
  auto even_up = [](uint64_t v) { return (uint32_t)std::max<uint64_t>(2, (v + 1) & ~1ull); };
  const uint32_t cap = std::min<uint32_t>(kAttnMaxPieces, std::max<uint32_t>(1, kAttnMaxPieceRows / kBQ / nqb));
  uint32_t L = even_up((est * 4 * 15 / 10 + cus - 1) / std::max(1u, cus));
  uint32_t np = (nbm + L - 1) / L;
  if (np > cap) {
    L = even_up((nbm + cap - 1) / cap);
    np = (nbm + L - 1) / L;
  }
  if (np <= 1) return sp;
  sp.L = L;
  sp.np = np;
  return sp;
}

uint64_t attention_ws_bytes(uint32_t rows, const AttnSplit& sp) {
  if (sp.np <= 1) return 0;
  const uint64_t prow = (uint64_t)(rows + kBQ - 1) / kBQ * kBQ;
  return (uint64_t)sp.np * prow * kNQ * (kHD + 2) * sizeof(float);
}

uint64_t attention_ws_max(uint32_t max_rows) {
  uint64_t most = 0;
  for (uint32_t nqb = 1; nqb <= (std::max(1u, max_rows) + kBQ - 1) / kBQ; ++nqb) {
    AttnSplit sp;
    sp.np = std::min<uint32_t>(kAttnMaxPieces, std::max<uint32_t>(1, kAttnMaxPieceRows / kBQ / nqb));
    most = std::max(most, attention_ws_bytes(nqb * kBQ, sp));
  }
  return most;
}

hipError_t launch_attention(const _Float16* q, const _Float16* kc, const _Float16* vc, const float* pq,
                            const uint32_t* qpos, _Float16* y, float* part, uint32_t rows, uint32_t ldq,
                            const AttnSplit& sp, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  if (sp.np == 0 || sp.L == 0 || sp.L % 2 != 0 || (sp.np > 1 && !part)) return hipErrorInvalidValue;
  const uint32_t nqb = (rows + kBQ - 1) / kBQ;
  hipLaunchKernelGGL(attention_kernel, dim3(nqb * sp.np * 4), dim3(512), 0, s, q, kc, vc, pq, qpos, y, part, ldq,
                     rows, sp.L, sp.np);
  if (sp.np > 1) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(attention_combine_kernel, dim3(rows), dim3(256), 0, s, part, pq, qpos, y, ldq, rows, sp.L,
                       sp.np);
  }
  return hipGetLastError();
}

}  // namespace dh
