// The flat search's candidate pass on the f16 matrix cores (split.hpp): rows
// and queries go in as two f16 parts each, three products per f32 one.
// Included by flat.hip only (it uses that file's tile helpers).
//
// Scales: one for the rows from the largest norm in the index (every |x_i| is
// below it), one per query from its own. What the parts of smaller rows lose
// is far inside the certificate's bound, which is relative to the largest
// norm.
#pragma once

#include "split.hpp"

// flat_prep_search_queries for the split pass: also each query's parts, as
// records of 32 hi then 32 lo halves per 32 dimensions (nK records per query,
// zeros past dim), and the factor cq that takes an accumulated product back
// to scale * (q . x), scale / sq / sx (down to 2^-148: a power of two, so
// exact as a subnormal float too). qn becomes the norm that the certificate
// counts with; where the squares overflow it is infinite, and the query is
// scanned exactly.
static __global__ __launch_bounds__(64) void flat_prep_split_queries(
    const float* __restrict__ raw, int dim, int ld, int metric, int do_prepare, float* __restrict__ Qp,
    float* __restrict__ qb, float* __restrict__ qn, unsigned long long* __restrict__ bad,
    unsigned long long* __restrict__ gthr, int* __restrict__ flag_count, _Float16* __restrict__ Qs, int nK,
    float scale, float sx,
    float* __restrict__ cq) {
  const int q = blockIdx.x, lane = threadIdx.x;
  __shared__ float s_sq;
  const bool alone = gridDim.x == 1;
  if (lane == 0) {
    gthr[q] = ~0ull;
    if (alone) *flag_count = 0;
  }
  prep_query_row(raw, dim, ld, metric, do_prepare, Qp, qb, qn, bad, alone);
  if (lane == 0) {  // the lane that wrote qn[q]
    // A norm below the scales' range stands as its lower end: f32 squares may
    // have underflowed (up to sqrt(dim) 2^-75 is missing, 0.1% of 2^-60 at
    // 2^20 dimensions, inside merge_certified's 1%), also in a norm of zero,
    // so neither the scale nor the certificate may rest on it.
    const float nv = qn[q] < 0x1p-60f ? 0x1p-60f : qn[q];
    // above it the scale and the factor stay normal floats up to the largest
    // norm there is, 2^64
    const bool ok = nv <= 0x1p+64f;
    const float sq = ok ? split_scale(nv) : 0.0f;
    s_sq = sq;
    cq[q] = ok ? scale / sq / sx : 0.0f;  // sq * sx may exceed f32
    qn[q] = ok ? nv : INFINITY;
  }
  __syncthreads();
  const float sq = s_sq;
  const float* row = Qp + (size_t)q * ld;
  _Float16* out = Qs + (size_t)q * nK * 64;
  for (int i = lane; i < nK * 32; i += 64) {
    _Float16 hi = (_Float16)0.0f, lo = (_Float16)0.0f;
    if (i < dim && sq != 0.0f) split_f16(row[i], sq, hi, lo);
    out[(i >> 5) * 64 + (i & 31)] = hi;
    out[(i >> 5) * 64 + 32 + (i & 31)] = lo;
  }
}

// Row biases of a filtered search: those of the accepted slots, +inf for the
// others (and past N, to the end of the last tile).
static __global__ __launch_bounds__(256) void flat_mask_bias(const float* __restrict__ xb,
                                                             const uint8_t* __restrict__ accept, int N, int n_pad,
                                                             float* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n_pad) out[i] = i < N && accept[i] != 0 ? xb[i] : INFINITY;
}

// The stored first tile (see flat_stored_tile): words of usable slots only
// are below 0xFFFFFFFF here, so no liveness is read.
template <int CAP, int R>
__device__ __attribute__((noinline)) void split_stored_tile(uint64_t* __restrict__ cand, int S, int split, int q0,
                                                            int nq, int n0, const uint64_t* thr, int* cnt, int tid) {
  constexpr int U = R / 8;
  const int c = tid & 31;
  uint4 w[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int qr = min(q0 + (tid >> 5) + 8 * u, nq - 1);  // unconditional loads
    w[u] = reinterpret_cast<const uint4*>(cand + ((size_t)qr * S + split) * CAP + (CAP - FB_N / 2))[c];
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int row = (tid >> 5) + 8 * u;
    if (q0 + row >= nq) continue;
    const uint64_t t = thr[row];
    const uint32_t th = (uint32_t)(t >> 32);
    const uint32_t kk[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (kk[e] <= th && kk[e] != 0xFFFFFFFFu) {
        const uint64_t key = ((uint64_t)kk[e] << 32) | (uint32_t)(n0 + 4 * c + e);
        if (key < t) {
          const int pos = atomicAdd(&cnt[row], 1);
          cand[((size_t)(q0 + row) * S + split) * CAP + 1 + pos] = key;
        }
      }
    }
  }
}

// The float a lane compares scores with for a threshold key: the key's
// distance part, or the largest finite float where that part is no number
// (no threshold yet), so that a usable slot passes and +inf never does.
__device__ __forceinline__ float split_thr_float(uint64_t thr) {
  const float f = key_float((uint32_t)(thr >> 32));
  return f < 3.4028235e38f ? f : 3.4028235e38f;
}

// Candidate pass over one (split, block of 32 QT queries): the same tiling
// along the store, buffers, thresholds, seeding and compaction as
// flat_mfma_candidates; what differs is the product and who holds what.
//
// What bounds it: with three f16 products per f32 one the matrix pipe needs
// 768 cycles per 128 x 128 x 32 slice of a workgroup (against 4096 for f32),
// so everything else has to stay below that. Rows are the MFMA's A operand
// and each of the four waves owns 32 of a tile's 128 rows for all the block's
// queries: a row's parts are then made once per workgroup, in registers, from
// the f32 slice that the copies put in LDS (two fused instructions per
// element, beside the other wave's MFMAs), and the store keeps its one f32
// copy. Queries are the B operand, split once per search. A lane ends up with
// one query's scores of 16 rows per 32 x 32 block, so the query's factor and
// threshold sit in two registers, and the filter is an fma and half a min3
// per score with one compare per 16 (an fma, a compare, a select and an or
// per score with the threshold per row, 5 instructions, in the f32 pass).
//
// Against the f32 pass on one card (whole searches, k = 10): 100k x 128 with
// 1000 queries 310 -> 167 us, with 48 queries (64-query blocks) 111 -> 75 us,
// cosine 1M x 768 with 1024 queries 11.50 -> 5.29 ms (893 TFLOP/s of f16
// products; the card's large f16 matrix product reaches 1140).
//
// A score is xb - scale q.x: the query's own term, the same for every row, is
// left to the merge. Unusable slots (removed, filtered out, past the end)
// have xb = +inf.
template <int CAP, int QT, bool SEED>
__global__ __launch_bounds__(256, 2) void flat_split_candidates(
    const _Float16* __restrict__ Qs, int nq, int nK, const float* __restrict__ X, int N, int ld,
    const float* __restrict__ cq, const float* __restrict__ xb, float sx, int S, int QB, int per_split, int Kp,
    uint64_t* __restrict__ cand, unsigned long long* __restrict__ gthr, int seeded) {
  constexpr int R = 32 * QT;              // queries per workgroup
  constexpr int XW = FB_N * FB_K;         // words of a row slice
  constexpr int QW = R * FB_K;            // words of a query slice
  __shared__ __align__(16) float smem[2 * XW + 2 * QW];
  __shared__ uint64_t thr[R];
  __shared__ int cnt[R];
  __shared__ float thr_f[R];

  // XCD-aware mapping, as flat_mfma_candidates
  const int total = QB * S;
  const int per_xcd = (total + 7) / 8;
  const int g = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (g >= total) return;
  const int qblk = g % QB, split = g / QB;
  const int q0 = qblk * R;
  const int s_begin = split * per_split;
  const int s_end = min(N, s_begin + (SEED ? FB_N : per_split));

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int h = lane >> 5, r = lane & 31, r7 = r & 7;

  for (int i = tid; i < R; i += 256) {
    thr[i] = KEY_MAX;
    thr_f[i] = split_thr_float(KEY_MAX);
    cnt[i] = 0;
  }
  float cqv[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) cqv[t] = cq[min(q0 + 32 * t + r, nq - 1)];
  __syncthreads();

  float* const sX = smem;
  float* const sQ = smem + 2 * XW;
  [[maybe_unused]] const int wid_s = __builtin_amdgcn_readfirstlane(wid);
  int gs = 0;

  for (int n0 = s_begin; n0 < s_end; n0 += FB_N) {
    // published thresholds and this lane's 16 row biases (rows 8 vb + 4 h + e
    // of the wave's 32), read before the k loop
    const uint64_t g_thr = tid < R && q0 + tid < nq
                               ? __hip_atomic_load(gthr + q0 + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                               : KEY_MAX;
    float4 xbv[4];
#pragma unroll
    for (int vb = 0; vb < 4; ++vb)
      xbv[vb] = *reinterpret_cast<const float4*>(xb + n0 + 32 * wid + 8 * vb + 4 * h);
    const bool stored = !SEED && seeded != 0 && n0 == s_begin;
    f16v acc[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;

    // slice kt of the tile starting at slot t0, into buffer buf: rows of 128
    // bytes, eight per copy instruction, 16-byte chunk c at c ^ (row & 7)
    auto gload = [&](int t0, int kt, int buf) {
#if defined(__HIP_DEVICE_COMPILE__)
      const float* x_rows = X + (size_t)t0 * ld;
      const int x_bytes = max(min(s_end - t0, FB_N), 0) * ld * 4;
      const _Float16* q_rows = Qs + (size_t)q0 * nK * 64;
      const int q_bytes = max(min(nq - q0, R), 0) * nK * 128;
      const __amdgpu_buffer_rsrc_t rs_q = uniform_rsrc(q_rows, q_bytes);
      const __amdgpu_buffer_rsrc_t rs_x = uniform_rsrc(x_rows, x_bytes);
      const int r8 = lane >> 3, ch = (lane & 7) ^ r8;
      const int kc = kt * FB_K + ch * 4;
      // a chunk past the row's end, and a row past the valid ones, is given an
      // offset outside the resource and lands as zeros
      const uint32_t xoff = kc < ld ? (uint32_t)((r8 * ld + kc) * 4) : 0x7FFFFFF0u;
      const uint32_t qoff = (uint32_t)(r8 * nK * 128 + kt * 128 + ch * 16);
      const uint32_t x_lds = lds_u32(sX + buf * XW), q_lds = lds_u32(sQ + buf * QW);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int gr = 4 * wid_s + u;
        lds_dma16(rs_x, xoff, (uint32_t)(8 * gr * ld * 4), x_lds + (uint32_t)(gr * 8 * FB_K * 4));
      }
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        const int gr = QT * wid_s + u;
        lds_dma16(rs_q, qoff, (uint32_t)(8 * gr * nK * 128), q_lds + (uint32_t)(gr * 8 * FB_K * 4));
      }
#endif
    };

    if (stored) {
      if (n0 + FB_N < s_end) gload(n0 + FB_N, 0, gs & 1);
    } else {
      if (n0 == s_begin) {
        gload(n0, 0, gs & 1);
        vm_wait0();
        __syncthreads();
      }
      for (int kt = 0; kt < nK; ++kt) {
        const int cur = (gs + kt) & 1;
        if (kt + 1 < nK) gload(n0, kt + 1, cur ^ 1);
        else if (n0 + FB_N < s_end) gload(n0 + FB_N, 0, cur ^ 1);
        const float* xp = sX + cur * XW + (32 * wid + r) * FB_K;
        const float* qp = sQ + cur * QW + r * FB_K;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          // lane half h takes dimensions 16 t + 8 h .. + 7 of both operands
          const float4 x0 = *reinterpret_cast<const float4*>(xp + (((4 * t + 2 * h) ^ r7) << 2));
          const float4 x1 = *reinterpret_cast<const float4*>(xp + (((4 * t + 2 * h + 1) ^ r7) << 2));
          h8v bh[QT], bl[QT];
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            const float* row = qp + qt * 32 * FB_K;
            bh[qt] = *reinterpret_cast<const h8v*>(row + (((2 * t + h) ^ r7) << 2));
            bl[qt] = *reinterpret_cast<const h8v*>(row + (((4 + 2 * t + h) ^ r7) << 2));
          }
          const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
          h8v ah, al;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            _Float16 hi, lo;
            split_f16(xs[j], sx, hi, lo);
            ah[j] = hi;
            al[j] = lo;
          }
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) acc[qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[qt], acc[qt], 0, 0, 0);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) acc[qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[qt], acc[qt], 0, 0, 0);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) acc[qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[qt], acc[qt], 0, 0, 0);
        }
        vm_wait0();  // this wave's copies of the next slice have landed
        __syncthreads();
      }
      gs += nK;
    }
    if (tid < R && g_thr < thr[tid]) {
      thr[tid] = g_thr;
      thr_f[tid] = split_thr_float(g_thr);
    }
    __syncthreads();

    const float xbf[16] = {xbv[0].x, xbv[0].y, xbv[0].z, xbv[0].w, xbv[1].x, xbv[1].y, xbv[1].z, xbv[1].w,
                           xbv[2].x, xbv[2].y, xbv[2].z, xbv[2].w, xbv[3].x, xbv[3].y, xbv[3].z, xbv[3].w};
    if constexpr (SEED) {
      // The tile's scores as ordered words (unusable: 0xFFFFFFFF), through
      // LDS (all of smem is free after a one-tile k loop): query row of 128
      // words, 16-byte chunk c at c ^ (query & 31), so that the lanes of a
      // store (different queries, the same chunk) use different banks.
      uint32_t* words = reinterpret_cast<uint32_t*>(smem);
#pragma unroll
      for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int vb = 0; vb < 4; ++vb) {
          uint32_t w[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = __builtin_fmaf(-cqv[qt], acc[qt][vb * 4 + e], xbf[vb * 4 + e]);
            w[e] = p <= 3.4028235e38f ? ord_key(p) : 0xFFFFFFFFu;
          }
          const int chunk = 8 * wid + 2 * vb + h;
          *reinterpret_cast<uint4*>(words + (32 * qt + r) * FB_N + ((chunk ^ r) << 2)) =
              make_uint4(w[0], w[1], w[2], w[3]);
        }
      __syncthreads();
#pragma unroll 4
      for (int u = 0; u < R / 8; ++u) {
        const int row = (tid >> 5) + 8 * u, c = tid & 31;
        if (q0 + row < nq) {
          const uint4 w4 = *reinterpret_cast<const uint4*>(words + row * FB_N + ((c ^ (row & 31)) << 2));
          reinterpret_cast<uint4*>(cand + ((size_t)(q0 + row) * S + split) * CAP + (CAP - FB_N / 2))[c] = w4;
        }
      }
      // each row's two smallest words in the entry below (two threads per
      // row, starting at different chunks so that reads spread over banks)
      if (tid < 2 * R) {
        const int row = tid >> 1, half = tid & 1;
        const uint32_t* rw = words + row * FB_N;
        uint32_t m1 = 0xFFFFFFFFu, m2 = 0xFFFFFFFFu;
#pragma unroll
        for (int u = 0; u < FB_N / 8; ++u) {
          const int c = half * (FB_N / 8) + ((u + row) & (FB_N / 8 - 1));
          const uint4 w = *reinterpret_cast<const uint4*>(rw + (c << 2));
          const uint32_t x4[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            m2 = min(m2, max(m1, x4[e]));
            m1 = min(m1, x4[e]);
          }
        }
        const uint32_t p1 = __shfl_xor(m1, 1), p2 = __shfl_xor(m2, 1);
        const uint32_t a1 = min(m1, p1), a2 = min(max(m1, p1), min(m2, p2));
        if (half == 0 && q0 + row < nq)
          cand[((size_t)(q0 + row) * S + split) * CAP + (CAP - FB_N / 2 - 1)] = ((uint64_t)a2 << 32) | a1;
      }
    } else if (stored) {
      split_stored_tile<CAP, R>(cand, S, split, q0, nq, n0, thr, cnt, tid);
      vm_wait0();  // the prefetched slice
    } else {
      // Filter: the least of a lane's 16 scores of a query tile against the
      // query's threshold; where some lane of the wave passes, the scores go
      // through the wave's 4 KB of the finished row slice and each lane takes
      // its own marked ones, lowest row first.
      float* slab = sX + ((gs - 1) & 1) * XW + wid * (WAVE * 16);
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const int row = 32 * qt + r;
        const float tf = q0 + row < nq ? thr_f[row] : -INFINITY;
        float p[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) p[v] = __builtin_fmaf(-cqv[qt], acc[qt][v], xbf[v]);
        float m = p[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) m = fminf(m, p[v]);
        if (__ballot(m <= tf)) {
          uint32_t pass = 0u;
#pragma unroll
          for (int v = 0; v < 16; ++v) pass |= p[v] <= tf ? 1u << v : 0u;
#pragma unroll
          for (int vb = 0; vb < 4; ++vb)
            *reinterpret_cast<float4*>(&slab[(vb * WAVE + lane) * 4]) =
                make_float4(p[vb * 4], p[vb * 4 + 1], p[vb * 4 + 2], p[vb * 4 + 3]);
          while (__ballot(pass != 0u)) {
            if (pass != 0u) {
              const int v = __builtin_ctz(pass);
              pass &= pass - 1u;
              const float a = slab[((v >> 2) * WAVE + lane) * 4 + (v & 3)];
              const int slot = n0 + 32 * wid + 8 * (v >> 2) + 4 * h + (v & 3);
              const uint64_t key = ((uint64_t)ord_key(a) << 32) | (uint32_t)slot;
              if (key < thr[row]) {
                const int pos = atomicAdd(&cnt[row], 1);
                cand[((size_t)(q0 + row) * S + split) * CAP + 1 + pos] = key;
              }
            }
          }
        }
      }
    }
    __syncthreads();
    if constexpr (!SEED) {
      // this wave's rows wid, wid + 4, ...: a compaction for each row that
      // might not take another tile's appends
      const int c_l = lane < R / 4 ? cnt[wid + 4 * lane] : 0;
      uint64_t full = __ballot(c_l > CAP - 1 - FB_N);
      while (full) {
        const int l = __builtin_ctzll(full);
        full &= full - 1;
        const int row = wid + 4 * l;
        compact_row<CAP>(cand + ((size_t)(q0 + row) * S + split) * CAP + 1, __builtin_amdgcn_readlane(c_l, l), Kp, lane,
                         &thr[row], &thr_f[row], &cnt[row], gthr + q0 + row);
      }
      __syncthreads();
    }
  }
  if constexpr (SEED) return;
  if (tid < R && q0 + tid < nq) cand[((size_t)(q0 + tid) * S + split) * CAP] = (uint64_t)cnt[tid];
}
