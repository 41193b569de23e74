// Attention of a long chunk of queries over laid-out keys: a first launch
// lays every page's keys and values out once, dequantised, in the order the
// matrix cores read them, and the second multiplies every query block
// against them. (reference: attention.cu:449-746 and kv_pages.h:86-93, the
// same semantics as prefill.hip, whose kernel stages and dequantises the
// pages once a query block.)
//
// Why: at 2,048 queries a page is read by 32 to 114 query blocks, and
// dequantising, transposing and staging it in each was a third of the
// kernel's instructions, between barriers. Laid out once (a 16K-position
// Llama layer: 38 MB written), a block's staging is 16-byte copies straight
// into LDS with no registers and no arithmetic, and its LDS reads are linear.
//
// The laid-out page of a KV head (page_block halves), as 1 KiB fragments of
// 16 bytes a lane:
//   K    HD/16 fragments, one a 16-channel slice: lane l holds key l % 32,
//        channels 16 c + 8 (l / 32) .. +7 (the A operand of 32x32x16); with
//        a key bias the high parts' fragments, then the low parts'.
//   V^T  fragment 2 dt + ks: lane l holds channel 32 dt + l % 32 of keys
//        16 ks + 4 h + {0..3, 8..11}, h = l / 32: the keys whose scores the
//        lane's half holds, so that P needs no movement.
//
// The main kernel. A workgroup of four waves takes one KV head and `qb`
// consecutive queries; its rows are the (query, head) pairs of those queries
// and the KV head's `group` heads, 32 rows a wave. A step is NP pages, double
// buffered in LDS behind one barrier:
//   S^T (32 keys x 32 rows) = K . Q^T     lane l holds row l % 32 and half
//                                         of the keys: the softmax is in the
//                                         lane but for one exchange
//   O^T (32 ch x 32 rows)  += V^T . P^T   P from the lane's own scores
// Two such workgroups a CU drift apart, so that one's softmax runs while the
// other's products do: at head_dim 64 a wave issues 192 MFMA cycles and
// about 300 VALU cycles for 512 scores.
//
// Precision as in prefill.hip: Q and the dequantised K and V exact in fp16,
// k + bias as fp16 high and low parts of the fp32 sum, the probabilities as
// high and low parts of p * 2^14 (kProbScale2), sums in fp32.
//
// Causality: rows read each page before their own sealed and their own at
// FP16 (both versions of the chunk's own pages are laid out). A step no row
// of the workgroup masks runs without a branch; any other goes page by page,
// and a wave skips a page none of its rows reads.

#include "chunk_pages.hpp"
#include "lane_ops.hpp"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>

namespace mi
{
  namespace
  {
    typedef float f32x16 __attribute__((ext_vector_type(16)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef _Float16 half2v __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) void *lds_void;
    typedef const __attribute__((address_space(1))) void *global_void;

    constexpr int kChunkWaves = 4;
    constexpr int kChunkThreads = 64 * kChunkWaves;
    constexpr int kTileRows = 32; // rows a product takes
    // A row's probabilities are held x 2^14 against its reference, which is
    // never above the row's maximum so far: the low part's last bit is then at
    // most 2^-38 of the largest probability's weight, as where the reference
    // is the maximum itself (prefill.hip). A step whose probabilities stay
    // within fp16 (a part of their sum, no less than any in it, shows it)
    // leaves the reference, so that the maximum of most steps is never formed
    // and a row's maximum may rise by two powers of two before it moves: a
    // wave's rows then move it in a sixth of its steps. (A 2,048-query chunk
    // at 16K: 416 us; 420 with every step's maximum formed; 386 with the
    // probabilities held x 2^5, which leaves the maximum ten powers to rise
    // but the low part nine bits fewer.)
    constexpr float kProbScale2 = 14.0f;
    constexpr float kProbUnscale = 1.0f / 16384.0f;
    constexpr float kMostProb = 65504.0f; // fp16's largest value
    constexpr int kMaxSplits = 32;

    struct ChunkArgs
    {
      KVSource kv;
      PageLayout lay[kTierCount];
      const std::uint16_t *q;
      std::uint16_t *out;
      const std::uint16_t *k_bias;
      const float *rope;
      // The laid-out pages: [kv head][slot] of page_block halves. A sealing
      // cache's sealed pages 0 .. sealed-1 are slots 0 .. sealed-1; the FP16
      // pages first_own .. first_own + owned - 1 follow from own_slot.
      std::uint16_t *pages;
      std::uint8_t *live; // slot's page has keys to read
      int slots;
      int sealed;
      int own_slot;
      int first_own;
      int owned;
      // With splits > 1: [split][query][head] maxima and sums, and outputs.
      float *part_ml;
      float *part_o;
      int splits;
      int seq_q;
      int seq_k;
      int heads;
      int kv_heads;
      int group;
      int qb;       // queries a workgroup
      float scale2; // log2(e) / sqrt(head_dim)
    };

    // Halves of a laid-out page of a KV head.
    template <int HD, bool kBias>
    __host__ __device__ constexpr int page_block()
    {
      return (kBias ? 3 : 2) * kP * HD;
    }

    __device__ inline half8 as_half8(u32x4 v) { return __builtin_bit_cast(half8, v); }

    // ---- laying the pages out ------------------------------------------------

    // A workgroup lays out one slot of one KV head: a thread an (8-channel
    // chunk, key) item, K straight to its fragment, V through LDS.
    template <int HD, bool kBias>
    __global__ void __launch_bounds__(256) lay_out_kernel(ChunkArgs a)
    {
      constexpr int kItems = kP * HD / 8;
      constexpr int kPer = (kItems + 255) / 256;
      constexpr int kVRow = HD + 2; // halves: odd dwords, so that a column's reads spread
      __shared__ std::uint16_t v_lds[kP * kVRow];
      const int slot = blockIdx.x;
      const int kvh = blockIdx.y;
      const bool sealed = slot < a.sealed;
      const int p = sealed ? slot : a.first_own + slot - a.own_slot;
      const int version = sealed ? kSealed : kOwn;
      const bool gap = !sealed && slot < a.own_slot; // padding between the two
      if (gap)
      {
        return; // never read
      }
      Entry e = entry_of(a.kv, p, version, p + 1);
      const bool live = !(sealed && e.tier == kUnreadPage);
      if (kvh == 0 && threadIdx.x == 0)
      {
        a.live[slot] = live ? 1 : 0;
      }
      if (!live)
      {
        return;
      }
      e.tier = __builtin_amdgcn_readfirstlane(e.tier);
      std::uint16_t *block =
          a.pages + (static_cast<std::size_t>(kvh) * a.slots + slot) * page_block<HD, kBias>();
      Fetched f[kPer];
      f32x4 cs[kPer][4];
#pragma unroll
      for (int u = 0; u < kPer; ++u)
      {
        const int item = threadIdx.x + 256 * u;
        if (item < kItems)
        {
          const int t = item % kP, c = item / kP;
          fetch<HD>(a, p, version, e, kvh, t, c, f[u]);
          if constexpr (kBias)
          {
            fetch_rope<HD>(a.rope, min(p * kP + t, a.seq_k - 1), 8 * c, cs[u]);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u)
      {
        const int item = threadIdx.x + 256 * u;
        if (item < kItems)
        {
          const int t = item % kP, c = item / kP;
          u32x4 kw, vw;
          values_of(f[u], kw, vw);
          std::uint16_t *at = block + 512 * (c / 2) + 8 * (t + 32 * (c % 2));
          if constexpr (kBias)
          {
            const int d0 = 8 * c;
            const int j0 = d0 < HD / 2 ? d0 : d0 - HD / 2;
            const std::uint16_t *b = a.k_bias + static_cast<std::size_t>(kvh) * HD;
            u32x4 wh, wl;
            biased_keys(f[u].tier, kw, cs[u], load_global<u32x4>(b + j0),
                        load_global<u32x4>(b + j0 + HD / 2), d0 < HD / 2, wh, wl);
            *reinterpret_cast<u32x4 *>(at) = wh;
            *reinterpret_cast<u32x4 *>(at + kP * HD) = wl;
          }
          else
          {
            *reinterpret_cast<u32x4 *>(at) = kw;
          }
          unsigned *row = reinterpret_cast<unsigned *>(v_lds + t * kVRow + 8 * c);
          row[0] = vw.x;
          row[1] = vw.y;
          row[2] = vw.z;
          row[3] = vw.w;
        }
      }
      __syncthreads();
      std::uint16_t *vt = block + (kBias ? 2 : 1) * kP * HD;
#pragma unroll
      for (int u = 0; u < kPer; ++u)
      {
        const int item = threadIdx.x + 256 * u;
        if (item < kItems)
        {
          const int frag = item / 64, l = item % 64;
          const int ch = 32 * (frag / 2) + l % 32;
          const int key = 16 * (frag % 2) + 4 * (l / 32);
          u32x4 w;
#pragma unroll
          for (int i = 0; i < 4; ++i)
          {
            const int k = key + 2 * i + (i >= 2 ? 4 : 0);
            w[i] = v_lds[k * kVRow + ch] |
                   (static_cast<unsigned>(v_lds[(k + 1) * kVRow + ch]) << 16);
          }
          *reinterpret_cast<u32x4 *>(vt + 8 * item) = w;
        }
      }
    }

    // ---- the chunk -----------------------------------------------------------

    __device__ inline f32x16 mfma32(half8 a, half8 b, f32x16 c)
    {
      return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }

    // Two values as fp16 high and low parts, packed: split_half's bits. The
    // low parts are kept in fp32 until one packed conversion takes both:
    // v_fma_mix_f32 and half a v_cvt_pk are 6.9 cycles a value where
    // v_fma_mixlo_f16, which rounds by itself, is 8.8.
    __device__ inline void split_pair(float x, float y, unsigned &hi, unsigned &lo)
    {
      float neg_one = -1.0f;
      asm("" : "+s"(neg_one));
      const half2v h = __builtin_convertvector(f32x2{x, y}, half2v);
      f32x2 rest = {__builtin_fmaf(static_cast<float>(h[0]), neg_one, x),
                    __builtin_fmaf(static_cast<float>(h[1]), neg_one, y)};
      asm("" : "+v"(rest[0]), "+v"(rest[1]));
      hi = __builtin_bit_cast(unsigned, h);
      lo = __builtin_bit_cast(unsigned, __builtin_convertvector(rest, half2v));
    }

    // The running softmax and output of a wave's rows (lane l: row l % 32,
    // the keys and channels of its half).
    template <int HD>
    struct Rows
    {
      float m; // the reference: base 2, scaled
      float l; // x 2^kProbScale2
      f32x16 o[HD / 32];
    };

    // N pages' scores: S^T = K . Q^T from the stage, each operand read for
    // every row tile, the products in turn so that none waits on the one
    // before it.
    template <int HD, int RT, int N, bool kBias>
    __device__ inline void page_scores(f32x16 (&s)[RT][N], const std::uint16_t *page,
                                       const half8 (&qf)[RT][HD / 16], int lane)
    {
      constexpr int kBlock = page_block<HD, kBias>();
#pragma unroll
      for (int t = 0; t < RT; ++t)
      {
#pragma unroll
        for (int j = 0; j < N; ++j)
        {
#pragma unroll
          for (int i = 0; i < 16; ++i)
          {
            s[t][j][i] = 0.0f;
          }
        }
      }
#pragma unroll
      for (int c = 0; c < HD / 16; ++c)
      {
#pragma unroll
        for (int part = 0; part < (kBias ? 2 : 1); ++part)
        {
#pragma unroll
          for (int j = 0; j < N; ++j)
          {
            const std::uint16_t *at = page + j * kBlock + part * kP * HD + 512 * c + 8 * lane;
            const half8 k = as_half8(*reinterpret_cast<const u32x4 *>(at));
#pragma unroll
            for (int t = 0; t < RT; ++t)
            {
              s[t][j] = mfma32(k, qf[t][c], s[t][j]);
            }
          }
        }
      }
    }

    // The rows' reference moved up to the maximum of scores of N pages, the
    // sums and outputs rescaled.
    template <int HD, int N>
    __device__ inline void move_reference(const f32x16 (&s)[N], float scale2, Rows<HD> &run)
    {
      float top = s[0][0];
#pragma unroll
      for (int j = 0; j < N; ++j)
      {
#pragma unroll
        for (int i = j == 0 ? 1 : 0; i < 16; ++i)
        {
          top = fmaxf(top, s[j][i]);
        }
      }
      top = fmaxf(run.m, lane_max32(top) * scale2); // the scale is positive
      const float keep = run.m < top ? __builtin_amdgcn_exp2f(run.m - top) : 1.0f;
      run.m = top;
      run.l *= keep;
#pragma unroll
      for (int dt = 0; dt < HD / 32; ++dt)
      {
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
          run.o[dt][i] *= keep;
        }
      }
    }

    // What a score's exponent takes on: a row that has seen no key (its
    // scores all -inf) stays at zero.
    __device__ inline float shift_of(float m)
    {
      return kProbScale2 - (m == -INFINITY ? 0.0f : m);
    }

    // Scores of N pages to probabilities (x 2^kProbScale2) in place; returns
    // the lane's sum of them, and in `most` the largest of its four parts, no
    // less than any probability.
    template <int N>
    __device__ inline float exponentiate(f32x16 (&s)[N], float scale2, float shift2, float &most)
    {
      float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < N; ++j)
      {
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
          s[j][i] = __builtin_amdgcn_exp2f(fmaf(s[j][i], scale2, shift2));
          part[i % 4] += s[j][i];
        }
      }
      most = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
      return (part[0] + part[1]) + (part[2] + part[3]);
    }

    // Probabilities of N pages (finite) brought back within fp16, with their
    // sum and the row's sum and outputs, by the power of two that puts the
    // row's largest, where it is larger, in [2^14, 2^15): nothing is rounded.
    template <int HD, int N>
    __device__ inline void lower(f32x16 (&p)[N], float &sum, Rows<HD> &run)
    {
      float top = 0.0f;
#pragma unroll
      for (int j = 0; j < N; ++j)
      {
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
          top = fmaxf(top, p[j][i]);
        }
      }
      const int by = max(__builtin_amdgcn_frexp_expf(lane_max32(top)) - 15, 0);
      const float factor = __builtin_ldexpf(1.0f, -by);
      run.m += static_cast<float>(by);
      run.l *= factor;
      sum *= factor;
#pragma unroll
      for (int dt = 0; dt < HD / 32; ++dt)
      {
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
          run.o[dt][i] *= factor;
        }
      }
#pragma unroll
      for (int j = 0; j < N; ++j)
      {
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
          p[j][i] *= factor;
        }
      }
    }

    // P.V of a page added, each operand read for every row tile, the outputs'
    // products in turn so that none waits on the one before it.
    template <int HD, int RT, int N>
    __device__ inline void page_values(const std::uint16_t *vt, const f32x16 (&p)[RT][N], int j,
                                       Rows<HD> (&run)[RT], int lane)
    {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
      {
        u32x4 hi[RT], lo[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t)
        {
#pragma unroll
          for (int i = 0; i < 4; ++i)
          {
            unsigned h, l;
            split_pair(p[t][j][8 * ks + 2 * i], p[t][j][8 * ks + 2 * i + 1], h, l);
            hi[t][i] = h;
            lo[t][i] = l;
          }
        }
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
        {
          const half8 v = as_half8(*reinterpret_cast<const u32x4 *>(vt + 512 * (2 * dt + ks) +
                                                                    8 * lane));
#pragma unroll
          for (int t = 0; t < RT; ++t)
          {
            run[t].o[dt] = mfma32(v, as_half8(hi[t]), run[t].o[dt]);
          }
#pragma unroll
          for (int t = 0; t < RT; ++t)
          {
            run[t].o[dt] = mfma32(v, as_half8(lo[t]), run[t].o[dt]);
          }
        }
      }
    }

    template <int HD, int RT, int NP, bool kBias, int kWavesASimd>
    __global__ void __launch_bounds__(kChunkThreads, kWavesASimd) chunk_kernel(ChunkArgs a)
    {
      constexpr int kBlock = page_block<HD, kBias>();
      constexpr int kStage = NP * kBlock;
      constexpr int kV = (kBias ? 2 : 1) * kP * HD; // V^T's place in a block
      constexpr int kWaveRows = RT * kTileRows;
      extern __shared__ u32x4 stage_words[];
      auto *const stages = reinterpret_cast<std::uint16_t *>(stage_words);
      const int lane = threadIdx.x & 63;
      const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
      const int half = lane >> 5;
      // KV heads fastest: workgroups are handed to the XCDs in turn, so that
      // an XCD's L2 holds the pages of few KV heads.
      const int kvh = static_cast<int>(blockIdx.x) % a.kv_heads;
      const int rest = static_cast<int>(blockIdx.x) / a.kv_heads;
      const int split = rest % a.splits;
      const int q_first = rest / a.splits * a.qb;
      const int q_last = min(q_first + a.qb, a.seq_q) - 1;
      const int shift = a.seq_k - a.seq_q;
      const bool causal = a.kv.layout == Layout::kCausal;
      const int rows = (q_last - q_first + 1) * a.group;

      // The lane's rows: whether there is one, its position, its own page,
      // its place in q and the output.
      bool valid[RT];
      int pos[RT], own[RT], row_at[RT];
      half8 qf[RT][HD / 16];
      Rows<HD> run[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t)
      {
        const int r = wave * kWaveRows + t * kTileRows + lane % 32;
        valid[t] = r < rows;
        const int query = q_first + (valid[t] ? r / a.group : 0);
        row_at[t] = query * a.heads + kvh * a.group + (valid[t] ? r % a.group : 0);
        pos[t] = valid[t] ? shift + query : -1;
        own[t] = valid[t] ? pos[t] / kP : -1;
        const std::uint16_t *q = a.q + static_cast<std::size_t>(row_at[t]) * HD + 8 * half;
#pragma unroll
        for (int c = 0; c < HD / 16; ++c)
        {
          qf[t][c] = as_half8(valid[t] ? load_global<u32x4>(q + 16 * c) : u32x4{0u, 0u, 0u, 0u});
        }
        // (A lane with no row: every probability 0, so that it moves nothing.)
        run[t].m = valid[t] ? -INFINITY : 1e30f;
        run[t].l = 0.0f;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
        {
#pragma unroll
          for (int i = 0; i < 16; ++i)
          {
            run[t].o[dt][i] = 0.0f;
          }
        }
      }
      // The wave's rows' own pages (rows are in order of position).
      const int wave_rows = min(kWaveRows, rows - wave * kWaveRows);
      const bool computes = wave_rows > 0;
      const int wave_lo = (shift + q_first + wave * kWaveRows / a.group) / kP;
      const int wave_hi =
          computes ? (shift + q_first + (wave * kWaveRows + wave_rows - 1) / a.group) / kP : 0;
      const int first_pos = shift + q_first;
      const int o_lo = first_pos / kP;
      const int o_hi = (shift + q_last) / kP;

      // The workgroup's steps, NP slots each: first over the sealed pages
      // before its last row's own page, then over its rows' own pages
      // (without a cache that seals, over every page up to it); the split's
      // share of them.
      const int own_from = causal ? o_lo : 0;
      const int sealed_steps = causal ? (o_hi + NP - 1) / NP : 0;
      const int total = sealed_steps + (o_hi - own_from + NP) / NP;
      const int per = (total + a.splits - 1) / a.splits;
      const int begin = min(split * per, total);
      const int end = min(begin + per, total);

      const std::uint16_t *laid =
          a.pages + static_cast<std::size_t>(kvh) * a.slots * kBlock;
      // A step's copies into LDS: 1 KiB a wave at a time, lane l's 16 bytes
      // at 16 l. (Slots are padded so that every step's are there.)
      const auto copy = [&](int step, int buf) {
        const int slot = step < sealed_steps
                             ? NP * step
                             : a.own_slot + own_from - a.first_own + NP * (step - sealed_steps);
        const std::uint16_t *src =
            laid + static_cast<std::size_t>(slot) * kBlock + wave * 512 + 8 * lane;
        std::uint16_t *dst = stages + buf * kStage + wave * 512;
#pragma unroll
        for (int i = 0; i < kStage / 512 / kChunkWaves; ++i)
        {
          __builtin_amdgcn_global_load_lds((global_void)(src + i * 512 * kChunkWaves),
                                           (lds_void)(dst + i * 512 * kChunkWaves), 16, 0, 0);
        }
      };
      if (begin < end)
      {
        copy(begin, 0);
      }
      // Whether any sealed page has nothing to read, once (a page a cache
      // evicted or masked).
      bool dead = false;
      for (int p = threadIdx.x; causal && p < o_hi; p += kChunkThreads)
      {
        dead = dead || a.live[p] == 0;
      }
      dead = __syncthreads_or(dead) != 0;
      // The steps that no row masks come first: sealed pages before every
      // row's own, or without sealing pages wholly before the first query.
      const int whole_steps = dead ? 0 : (causal ? o_lo : (first_pos + 1) / kP) / NP;
      // Step `step` is in LDS and the next on its way: its own copies have
      // landed (each wave waits for its own before the barrier), and every
      // wave is done with the other buffer.
      const auto turn = [&](int step) -> const std::uint16_t * {
        const int buf = (step - begin) & 1;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        if (step + 1 < end)
        {
          copy(step + 1, buf ^ 1);
        }
        return stages + buf * kStage;
      };
      int step = begin;
      const std::uint16_t *stage = begin < end ? turn(begin) : stages;
      const int whole_end = min(end, whole_steps);
      // The rows' first reference: their maximum over the first page, which
      // every row reads.
      if (step < whole_end)
      {
        f32x16 s[RT][1];
        page_scores<HD, RT, 1, kBias>(s, stage, qf, lane);
#pragma unroll
        for (int t = 0; t < RT; ++t)
        {
          move_reference<HD, 1>(s[t], a.scale2, run[t]);
        }
      }
      while (step < whole_end)
      {
        f32x16 s[RT][NP];
        // A wave in its products goes before one in its softmax, so that the
        // two workgroups of a CU alternate (a 2,048-query chunk at 16K, the
        // probabilities x 2^5: 398 to 382 us).
        __builtin_amdgcn_s_setprio(1);
        page_scores<HD, RT, NP, kBias>(s, stage, qf, lane);
        __builtin_amdgcn_s_setprio(0);
        float sum[RT], most[RT];
        bool finite = true;
#pragma unroll
        for (int t = 0; t < RT; ++t)
        {
          sum[t] = exponentiate<NP>(s[t], a.scale2, kProbScale2 - run[t].m, most[t]);
          finite = finite && sum[t] < INFINITY;
        }
        // A rise past fp32's range, a row whose first page had no finite score,
        // or values that are not finite: the wave goes on below.
        if (!__all(finite))
        {
          break;
        }
#pragma unroll
        for (int t = 0; t < RT; ++t)
        {
          if (__any(most[t] > kMostProb))
          {
            lower<HD, NP>(s[t], sum[t], run[t]);
          }
        }
#pragma unroll
        for (int t = 0; t < RT; ++t)
        {
          run[t].l += sum[t];
        }
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < NP; ++j)
        {
          page_values<HD, RT, NP>(stage + j * kBlock + kV, s, j, run, lane);
        }
        __builtin_amdgcn_s_setprio(0);
        if (++step < end)
        {
          stage = turn(step);
        }
      }
      // The rest page by page, against the exact maximum: a page no row of
      // the wave reads is left out, whatever it holds; a masked key's score
      // is -inf.
      while (step < end)
      {
        const bool sealed = step < sealed_steps;
        const int p0 = sealed ? NP * step : own_from + NP * (step - sealed_steps);
        for (int j = 0; j < NP; ++j)
        {
          const int p = p0 + j;
          const bool read = sealed   ? p < wave_hi && (!dead || a.live[p] != 0)
                            : causal ? p >= wave_lo && p <= wave_hi
                                     : p <= wave_hi;
          if (!computes || !read)
          {
            continue;
          }
          f32x16 s[RT][1];
          page_scores<HD, RT, 1, kBias>(s, stage + j * kBlock, qf, lane);
#pragma unroll
          for (int t = 0; t < RT; ++t)
          {
            const int limit = sealed   ? (p < own[t] ? 0x7fffffff : -1)
                              : causal ? (p == own[t] ? pos[t] : -1)
                                       : pos[t];
#pragma unroll
            for (int i = 0; i < 16; ++i)
            {
              const int key = p * kP + 8 * (i / 4) + 4 * half + i % 4;
              s[t][0][i] = key <= limit ? s[t][0][i] : -INFINITY;
            }
            move_reference<HD, 1>(s[t], a.scale2, run[t]);
            float most;
            run[t].l += exponentiate<1>(s[t], a.scale2, shift_of(run[t].m), most);
          }
          page_values<HD, RT, 1>(stage + j * kBlock + kV, s, 0, run, lane);
        }
        if (++step < end)
        {
          stage = turn(step);
        }
      }

#pragma unroll
      for (int t = 0; t < RT; ++t)
      {
        const float sum = lane_sum32(run[t].l);
        if (!valid[t])
        {
          continue;
        }
        if (a.splits == 1)
        {
          const float inv = 1.0f / sum;
          std::uint16_t *out = a.out + static_cast<std::size_t>(row_at[t]) * HD + 4 * half;
#pragma unroll
          for (int dt = 0; dt < HD / 32; ++dt)
          {
#pragma unroll
            for (int b = 0; b < 4; ++b)
            {
              const f32x16 &o = run[t].o[dt];
              const half2v lo = {static_cast<_Float16>(o[4 * b] * inv),
                                 static_cast<_Float16>(o[4 * b + 1] * inv)};
              const half2v hi = {static_cast<_Float16>(o[4 * b + 2] * inv),
                                 static_cast<_Float16>(o[4 * b + 3] * inv)};
              *reinterpret_cast<u32x2 *>(out + 32 * dt + 8 * b) =
                  u32x2{__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi)};
            }
          }
          continue;
        }
        const std::size_t row =
            static_cast<std::size_t>(split) * a.seq_q * a.heads + row_at[t];
        if (half == 0)
        {
          *reinterpret_cast<f32x2 *>(a.part_ml + 2 * row) = f32x2{run[t].m, sum * kProbUnscale};
        }
        float *out = a.part_o + row * HD + 4 * half;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
        {
#pragma unroll
          for (int b = 0; b < 4; ++b)
          {
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
              v[i] = run[t].o[dt][4 * b + i] * kProbUnscale;
            }
            *reinterpret_cast<f32x4 *>(out + 32 * dt + 8 * b) = v;
          }
        }
      }
    }

    // Folds the splits of one (query, head) row: weights 2^(m_s - max m) (a
    // split that saw no key has m = -inf and weighs 0). A thread four
    // channels of a row, HD / 4 threads a row: at a dozen splits of a few
    // thousand rows it is bound by the partials' bytes.
    template <int HD>
    __global__ void __launch_bounds__(256) chunk_combine_kernel(ChunkArgs a, std::size_t rows)
    {
      constexpr int kLanes = HD / 4;
      const std::size_t i = static_cast<std::size_t>(blockIdx.x) * 256 + threadIdx.x;
      const std::size_t row = i / kLanes;
      const int d = 4 * static_cast<int>(i % kLanes);
      if (row >= rows)
      {
        return;
      }
      float top = -INFINITY;
      for (int s = 0; s < a.splits; ++s)
      {
        top = fmaxf(top, a.part_ml[2 * (s * rows + row)]);
      }
      float sum = 0.0f;
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
      for (int s = 0; s < a.splits; ++s)
      {
        const f32x2 ml = *reinterpret_cast<const f32x2 *>(a.part_ml + 2 * (s * rows + row));
        const f32x4 o = *reinterpret_cast<const f32x4 *>(a.part_o + (s * rows + row) * HD + d);
        const float w = __builtin_amdgcn_exp2f(ml[0] - top);
        sum += ml[1] * w;
        acc += o * w;
      }
      const half2v lo = {static_cast<_Float16>(acc[0] / sum), static_cast<_Float16>(acc[1] / sum)};
      const half2v hi = {static_cast<_Float16>(acc[2] / sum), static_cast<_Float16>(acc[3] / sum)};
      *reinterpret_cast<u32x2 *>(a.out + row * HD + d) =
          u32x2{__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi)};
    }

    // Rows a workgroup takes, RT row tiles a wave.
    constexpr int block_rows(int rt) { return kChunkWaves * rt * kTileRows; }

    std::size_t align_up(std::size_t n, std::size_t to) { return (n + to - 1) / to * to; }

    // The launches, or with a null workspace only the bytes it needs.
    template <int HD, int RT, int NP, bool kBias, int kWavesASimd>
    std::size_t run(ChunkArgs args, std::uint8_t *work, hipEvent_t done, hipStream_t stream)
    {
      args.qb = std::min(args.seq_q, block_rows(RT) / args.group);
      auto kernel = chunk_kernel<HD, RT, NP, kBias, kWavesASimd>;
      constexpr std::size_t kLds = 2 * NP * page_block<HD, kBias>() * sizeof(std::uint16_t);
      // Workgroups the device holds at once, and the LDS limit raised, once
      // (the stages of some shapes pass 64 KB only with the kernel's own LDS).
      static const long held = [&] {
        hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(kLds)),
                  "hipFuncSetAttribute chunk LDS");
        int per_cu = 0;
        hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kChunkThreads, kLds),
                  "hipOccupancyMaxActiveBlocksPerMultiprocessor chunk");
        return static_cast<long>(std::max(per_cu, 1)) * device_multiprocessors();
      }();
      const bool causal = args.kv.layout == Layout::kCausal;
      const int last = (args.seq_k - 1) / kP;
      const int first = causal ? (args.seq_k - args.seq_q) / kP : 0;
      args.sealed = causal ? last : 0;
      args.own_slot = static_cast<int>(align_up(args.sealed, NP));
      args.first_own = first;
      args.owned = last - first + 1;
      const int written = args.own_slot + args.owned;
      args.slots = written + NP; // a step's copies may reach past the last slot
      // Splits: as many runs of steps as make the rounds of workgroups, each
      // its steps and the fixed cost of a few, shortest.
      const long blocks = static_cast<long>((args.seq_q + args.qb - 1) / args.qb) * args.kv_heads;
      const int steps = (last + 1 + (causal ? 1 : 0)) / NP + 1;
      long best = 0;
      for (int s = 1; s <= std::min(kMaxSplits, std::max(1, steps / 4)); ++s)
      {
        const long rounds = (blocks * s + held - 1) / held;
        const long cost = rounds * ((steps + s - 1) / s + 6) + (s > 1 ? 8 : 0);
        if (best == 0 || cost < best)
        {
          best = cost;
          args.splits = s;
        }
      }
      const std::size_t rows = static_cast<std::size_t>(args.seq_q) * args.heads;
      const std::size_t pages_bytes = align_up(
          static_cast<std::size_t>(args.kv_heads) * args.slots * page_block<HD, kBias>() * 2, 256);
      const std::size_t live_bytes = align_up(args.slots, 256);
      const std::size_t ml_bytes = args.splits > 1 ? align_up(rows * args.splits * 8, 256) : 0;
      const std::size_t o_bytes = args.splits > 1 ? rows * args.splits * HD * 4 : 0;
      const std::size_t needed = pages_bytes + live_bytes + ml_bytes + o_bytes;
      if (work == nullptr)
      {
        return needed;
      }
      args.pages = reinterpret_cast<std::uint16_t *>(work);
      args.live = work + pages_bytes;
      args.part_ml = reinterpret_cast<float *>(work + pages_bytes + live_bytes);
      args.part_o = reinterpret_cast<float *>(work + pages_bytes + live_bytes + ml_bytes);
      hipLaunchKernelGGL((lay_out_kernel<HD, kBias>), dim3(written, args.kv_heads), dim3(256), 0,
                         stream, args);
      hip_check(hipGetLastError(), "chunk layout kernel launch");
      // The last launch signals `done` with its own completion: no packet of
      // its own on the stream (an event recorded after it takes 1 to 3 us).
      hipExtLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks * args.splits)),
                            dim3(kChunkThreads), kLds, stream, nullptr,
                            args.splits > 1 ? nullptr : done, 0, args);
      hip_check(hipGetLastError(), "chunk kernel launch");
      if (args.splits > 1)
      {
        const std::size_t threads = rows * (HD / 4);
        hipExtLaunchKernelGGL(chunk_combine_kernel<HD>,
                              dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0,
                              stream, nullptr, done, 0, args, rows);
        hip_check(hipGetLastError(), "chunk combine kernel launch");
      }
      return needed;
    }

    std::size_t dispatch(const KVSource &kv, const AttentionArgs &a, std::uint8_t *work,
                         hipEvent_t done, hipStream_t stream)
    {
      ChunkArgs args{};
      args.kv = kv;
      for (int t = kINT8; t <= kINT2; ++t)
      {
        if (kv.layout == Layout::kCausal && kv.may_be_at[t])
        {
          args.lay[t] = page_layout(t, kP, a.kv_heads, a.head_dim);
        }
      }
      args.q = a.q;
      args.out = a.out;
      args.k_bias = a.k_bias;
      args.rope = a.rope;
      args.seq_q = a.seq_q;
      args.seq_k = a.seq_k;
      args.heads = a.heads;
      args.kv_heads = a.kv_heads;
      args.group = a.heads / a.kv_heads;
      args.scale2 = 1.4426950408889634f / std::sqrt(static_cast<float>(a.head_dim));
      if (a.head_dim == 128)
      {
        return a.k_bias != nullptr ? run<128, 1, 1, true, 2>(args, work, done, stream)
                                   : run<128, 1, 2, false, 2>(args, work, done, stream);
      }
      return a.k_bias != nullptr ? run<64, 2, 2, true, 2>(args, work, done, stream)
                                 : run<64, 2, 2, false, 2>(args, work, done, stream);
    }

    // Whether the layout, a launch and the pages' bytes written and read as
    // FP16, costs less than dequantising and staging each page once a query
    // block. (Microseconds staged / laid out, mixed tiers, 8 to 64 heads in
    // groups of 1 to 16, heads / KV heads x queries after positions before.)
    bool laying_out_pays(const AttentionArgs &a)
    {
      // Fewer rows a KV head than a workgroup takes at head_dim 128: every
      // page is staged once either way (32/32 x 64 after 8,000 at head_dim
      // 128: 80 / 83).
      if (static_cast<long long>(a.seq_q) * (a.heads / a.kv_heads) < block_rows(1))
      {
        return false;
      }
      const long long rows = static_cast<long long>(a.seq_q) * a.heads;
      const bool wide = a.head_dim == 128;
      // Over many keys, once the rows keep the device busy: at head_dim 64
      // 8/8 x 128 after 8,000 33 / 38, x 256 60 / 43, 32/16 x 64 51 / 53, 14/2
      // x 160 after 2,000 with the key bias 32 / 29. At 128 8/8 x 128 after
      // 8,000 40 / 45, 8/1 x 192 after 3,000 35 / 31.
      if (a.seq_k > 2048)
      {
        return wide ? rows >= 1536 : rows > 2048;
      }
      // Over few, where the layout's and the splits' launches weigh more: at
      // head_dim 64 14/2 x 256 after 500 with the key bias 31 / 35, 8/8 x 513
      // after 100 with it 42 / 45, 32/16 x 160 after 500 39 / 35; at 128 8/1 x
      // 257 after 500 29 / 31, 14/2 x 160 28.2 / 28.6, 12/2 x 192 30.1 / 29.6.
      // Over fewer than 128 32/8 x 96 alone 11.8 / 13.3.
      return a.seq_k >= 128 && rows >= (wide ? 2304 : 4608);
    }

  } // namespace

  bool chunk_applies(const KVSource &kv, const AttentionArgs &a)
  {
    return kv.layout != Layout::kContiguous && a.kv_heads > 0 && a.heads % a.kv_heads == 0 &&
           a.heads / a.kv_heads <= block_rows(1) && laying_out_pays(a) && prefill_applies(kv, a);
  }

  std::size_t chunk_workspace_bytes(const KVSource &kv, const AttentionArgs &a)
  {
    return dispatch(kv, a, nullptr, nullptr, nullptr);
  }

  void launch_chunk(const KVSource &kv, const AttentionArgs &a, void *workspace, hipEvent_t done,
                    hipStream_t stream)
  {
    dispatch(kv, a, static_cast<std::uint8_t *>(workspace), done, stream);
  }

} // namespace mi
