// A page's keys and values as a chunk's attention reads them: a thread's eight
// channels of one key and its value from a page at its tier (or an FP16 row),
// dequantised in packed fp16, the key bias rotated and added. Shared by the
// kernel that stages pages as it goes (prefill.hip) and the one that lays
// them out once for every query block (chunk.hip).

#pragma once

#include "common.hpp"
#include "dequant.hpp"
#include "kernels.hpp"

namespace mi
{
  namespace
  {
    typedef _Float16 half8 __attribute__((ext_vector_type(8)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

    constexpr int kP = 32; // keys a page, and a key tile

    enum : int
    {
      kSealed = 0, // a page before the row's own, at its recorded tier
      kOwn = 1,    // the row's own page at FP16 (or any FP16/contiguous page)
    };

    // A load from device memory through a global-address-space pointer.
    // Pages are reached through addresses held as integers, which the
    // compiler would otherwise read with flat instructions; a flat load
    // counts against the LDS wait counter as well, so every LDS read of the
    // products would wait for the next step's page fetch.
    template <typename T>
    __device__ inline T load_global(const void *p)
    {
      return *((const __attribute__((address_space(1))) T *)(p));
    }

    // What one thread fetched for one (key, 8-channel chunk) of a page:
    // raw K and V (fp16 rows, or codes), and for a quantised page the key
    // channels' scales and zeros and the value row's scale and zero.
    struct Fetched
    {
      u32x4 k;
      u32x4 v;
      u32x4 ks;
      u32x4 kz;
      unsigned vsz; // value scale | value zero << 16
      int tier;     // kFP16, a quantised tier, or -1 for zeros
    };

    // The page-table entry of an item: the sealed page's address and tier
    // (or an FP16 page's address); loaded two items ahead of its data.
    struct Entry
    {
      unsigned long long page;
      int tier;
    };

    __device__ inline Entry entry_of(const KVSource &kv, int p, int version, int p_end)
    {
      Entry e{0, kFP16};
      if (p >= p_end)
      {
        return e;
      }
      if (kv.layout == Layout::kCausal && version == kSealed)
      {
        e.page = load_global<unsigned long long>(kv.pages + p);
        e.tier = load_global<std::uint8_t>(kv.tiers + p);
      }
      else if (kv.layout == Layout::kPaged)
      {
        e.page = load_global<unsigned long long>(kv.pages + p);
      }
      return e;
    }

    // Fetches one (key t, chunk c) of the item (page p, version) for KV head
    // kvh: global loads only; what it needs to dequantise comes with it.
    // Args: the launch's kv, lay, kv_heads and seq_k.
    template <int HD, typename Args>
    __device__ inline void fetch(const Args &a, int p, int version, const Entry &entry,
                                 int kvh, int t, int c, Fetched &f)
    {
      const KVSource &kv = a.kv;
      const std::size_t row = static_cast<std::size_t>(a.kv_heads) * HD;
      const std::size_t at = static_cast<std::size_t>(kvh) * HD + 8 * c;
      const int j = p * kP + t;
      f.tier = -1;
      const std::uint16_t *k_row = nullptr;
      const std::uint16_t *v_row = nullptr;
      if (kv.layout == Layout::kCausal && version == kSealed)
      {
        const int tier = entry.tier;
        const auto *page = reinterpret_cast<const std::uint8_t *>(entry.page);
        if (tier == kFP16)
        {
          const auto *h = reinterpret_cast<const std::uint16_t *>(page);
          k_row = h + t * row;
          v_row = h + (kP + t) * row;
        }
        else
        {
          const PageLayout &L = a.lay[tier];
          const int bits = tier == kINT8 ? 8 : tier == kINT4 ? 4 : 2;
          const std::size_t e = static_cast<std::size_t>(t) * row + at; // first element
          const std::uint8_t *kc = page + L.key_codes + e * bits / 8;
          const std::uint8_t *vc = page + L.value_codes + e * bits / 8;
          // 8 codes: 8 bytes at INT8, 4 at INT4, 2 at INT2.
          f.k = u32x4{0, 0, 0, 0};
          f.v = u32x4{0, 0, 0, 0};
          if (bits == 8)
          {
            f.k.x = load_global<unsigned>(kc);
            f.k.y = load_global<unsigned>(kc + 4);
            f.v.x = load_global<unsigned>(vc);
            f.v.y = load_global<unsigned>(vc + 4);
          }
          else if (bits == 4)
          {
            f.k.x = load_global<unsigned>(kc);
            f.v.x = load_global<unsigned>(vc);
          }
          else
          {
            f.k.x = load_global<unsigned short>(kc);
            f.v.x = load_global<unsigned short>(vc);
          }
          f.ks = load_global<u32x4>(page + L.key_scales + 2 * at);
          f.kz = load_global<u32x4>(page + L.key_zeros + 2 * at);
          const std::size_t group = static_cast<std::size_t>(t) * a.kv_heads + kvh;
          const auto *vs = reinterpret_cast<const std::uint16_t *>(page + L.value_scales);
          const auto *vz = reinterpret_cast<const std::uint16_t *>(page + L.value_zeros);
          f.vsz = static_cast<unsigned>(load_global<std::uint16_t>(vs + group)) |
                  (static_cast<unsigned>(load_global<std::uint16_t>(vz + group)) << 16);
          f.tier = tier;
          return;
        }
      }
      else if (j < a.seq_k)
      {
        switch (kv.layout)
        {
        case Layout::kContiguous:
          k_row = kv.k + static_cast<std::size_t>(j) * row;
          v_row = kv.v + static_cast<std::size_t>(j) * row;
          break;
        case Layout::kPaged:
        {
          const auto *h = reinterpret_cast<const std::uint16_t *>(entry.page);
          k_row = h + t * row;
          v_row = h + (kP + t) * row;
          break;
        }
        case Layout::kCausal:
          if (j >= kv.start)
          {
            k_row = kv.chunk_k + static_cast<std::size_t>(j - kv.start) * row;
            v_row = kv.chunk_v + static_cast<std::size_t>(j - kv.start) * row;
          }
          else
          {
            k_row = kv.open + t * row;
            v_row = kv.open + (kP + t) * row;
          }
          break;
        }
      }
      if (k_row != nullptr)
      {
        f.k = load_global<u32x4>(k_row + at);
        f.v = load_global<u32x4>(v_row + at);
        f.tier = kFP16;
      }
      else
      {
        f.k = u32x4{0, 0, 0, 0};
        f.v = u32x4{0, 0, 0, 0};
      }
    }

    __device__ inline std::uint16_t half_of(const u32x4 &w, int e)
    {
      const unsigned word = e < 2 ? w.x : e < 4 ? w.y : e < 6 ? w.z : w.w;
      return static_cast<std::uint16_t>(word >> (16 * (e & 1)));
    }

    // The 8 fp16 K and V values of a fetch, as words: FP16 rows as read,
    // zeros for nothing read, codes dequantised in packed fp16 (one rounding
    // of code * scale + zero). Every lane that reaches the quantised branch
    // holds the same tier (a sealed page's).
    __device__ inline void values_of(const Fetched &f, u32x4 &k, u32x4 &v)
    {
      if (f.tier == kFP16)
      {
        k = f.k;
        v = f.v;
        return;
      }
      if (f.tier < 0)
      {
        k = u32x4{0, 0, 0, 0};
        v = u32x4{0, 0, 0, 0};
        return;
      }
      const unsigned sp = (f.vsz & 0xFFFFu) * 0x10001u;
      const unsigned zp = (f.vsz >> 16) * 0x10001u;
      const u32x4 vs2 = {sp, sp, sp, sp};
      const u32x4 vz2 = {zp, zp, zp, zp};
      switch (__builtin_amdgcn_readfirstlane(f.tier))
      {
      case kINT8:
        k = __builtin_bit_cast(u32x4, dq::dequant_step<8>(f.k.x, f.k.y, f.ks, f.kz));
        v = __builtin_bit_cast(u32x4, dq::dequant_step<8>(f.v.x, f.v.y, vs2, vz2));
        break;
      case kINT4:
        k = __builtin_bit_cast(u32x4, dq::dequant_step<4>(f.k.x, 0u, f.ks, f.kz));
        v = __builtin_bit_cast(u32x4, dq::dequant_step<4>(f.v.x, 0u, vs2, vz2));
        break;
      default:
        k = __builtin_bit_cast(u32x4, dq::dequant_step<2>(f.k.x, 0u, f.ks, f.kz));
        v = __builtin_bit_cast(u32x4, dq::dequant_step<2>(f.v.x, 0u, vs2, vz2));
        break;
      }
    }

    // The cos/sin pairs of position j for channels d0..d0+7 (the rope table
    // holds {cos, sin} per (position, j < hd/2)).
    template <int HD>
    __device__ inline void fetch_rope(const float *rope, int j, int d0, f32x4 cs[4])
    {
      constexpr int half = HD / 2;
      const int j0 = d0 < half ? d0 : d0 - half;
      const float *src = rope + 2 * (static_cast<std::size_t>(j) * half + j0);
      for (int i = 0; i < 4; ++i)
      {
        cs[i] = load_global<f32x4>(src + 4 * i);
      }
    }

    // RoPE of the key bias at one position for channels d0..d0+7 (reference:
    // attention.cu:104-116): channel d < hd/2 pairs with d + hd/2. b_first
    // holds bias[j0 .. j0+7] and b_second bias[j0+hd/2 .. +7], j0 the pair index.
    __device__ inline void rotated_bias8(const u32x4 &b_first, const u32x4 &b_second,
                                         const f32x4 cs[4], bool first_half, float rb[8])
    {
      for (int e = 0; e < 8; ++e)
      {
        const float c = cs[e / 2][2 * (e % 2)];
        const float s = cs[e / 2][2 * (e % 2) + 1];
        const float b1 = h2f(half_of(b_first, e));
        const float b2 = h2f(half_of(b_second, e));
        rb[e] = first_half ? b1 * c - b2 * s : b2 * c + b1 * s;
      }
    }

    // Eight keys with the rotated bias added, k + RoPE(bias) formed in fp32
    // and split into fp16 high and low parts; zeros for nothing read.
    __device__ inline void biased_keys(int tier, const u32x4 &kw, const f32x4 cs[4],
                                       const u32x4 &b_first, const u32x4 &b_second,
                                       bool first_half, u32x4 &wh, u32x4 &wl)
    {
      std::uint16_t hi[8], lo[8];
      if (tier >= 0)
      {
        float rb[8];
        rotated_bias8(b_first, b_second, cs, first_half, rb);
        for (int e = 0; e < 8; ++e)
        {
          const float x = h2f(half_of(kw, e)) + rb[e];
          const __half h = __float2half_rn(x);
          hi[e] = __half_as_ushort(h);
          lo[e] = __half_as_ushort(__float2half_rn(x - __half2float(h)));
        }
      }
      else
      {
        for (int e = 0; e < 8; ++e)
        {
          hi[e] = 0;
          lo[e] = 0;
        }
      }
      wh.x = hi[0] | (unsigned(hi[1]) << 16);
      wh.y = hi[2] | (unsigned(hi[3]) << 16);
      wh.z = hi[4] | (unsigned(hi[5]) << 16);
      wh.w = hi[6] | (unsigned(hi[7]) << 16);
      wl.x = lo[0] | (unsigned(lo[1]) << 16);
      wl.y = lo[2] | (unsigned(lo[3]) << 16);
      wl.z = lo[4] | (unsigned(lo[5]) << 16);
      wl.w = lo[6] | (unsigned(lo[7]) << 16);
    }
  } // namespace
} // namespace mi
