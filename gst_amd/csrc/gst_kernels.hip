// gst_kernels.hip -- the five GST decode stages as gfx950 kernels (wave64, integer only).
//
// Every kernel is a grid-stride loop over "units" of its stage; a unit maps to
// (image, local unit) through the batch plan's per-stage prefix array, or to the
// single image passed by value.  Reference semantics are cited per kernel.
#include "gst_internal.h"

#include <mutex>

namespace gst {
namespace {

constexpr int32_t kBufferRsrcWord3 = 0x00020000;  // raw buffer, gfx9 family

// Pointers in the global address space.  Loads and stores through them compile to
// global_* instructions, which count in vmcnt only; through generic pointers they
// would be flat_* instructions, which also count in lgkmcnt, so every wait for an
// LDS access would wait for them as well (a sector store would stall the next
// rANS step until the store completes).  The host compilation pass only type-checks
// this code and has no address spaces for class-type copies, so there the aliases
// are plain pointers.
#if defined(__HIP_DEVICE_COMPILE__)
template <typename T>
using GPtr = __attribute__((address_space(1))) T *;
template <typename T>
using CPtr = __attribute__((address_space(4))) const T *;
#else
template <typename T>
using GPtr = T *;
template <typename T>
using CPtr = const T *;
#endif

template <typename T, typename U>
__device__ __forceinline__ GPtr<T> Gbl(U *p) {
  return (GPtr<T>)(reinterpret_cast<uintptr_t>(p));
}

// Element k of a 4-entry array without dynamic indexing (which would put the array
// in scratch memory).
template <typename T>
__device__ __forceinline__ T Pick4(const T (&v)[4], uint32_t k) {
  return k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
}

__device__ __forceinline__ uint32_t Popc64(uint64_t m) { return static_cast<uint32_t>(__popcll(m)); }

struct Located {
  uint32_t img;
  uint32_t local;
  bool valid;  // false: u is past the stage's last unit
};

// Locate among the up to 256 prefix entries a wave holds, entry lane + 64 k in v[k]
// (padding past the plan's).
constexpr uint32_t kPrefixInRegs = 256;
__device__ __forceinline__ Located LocateIn(const uint32_t (&v)[4], uint32_t u) {
  uint32_t cnt = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) cnt += Popc64(__builtin_amdgcn_ballot_w64(v[k] <= u));
  const uint32_t lo = cnt - 1;  // prefix[0] = 0 <= u
  // Reads of a lane and scalar selects, pinned so that the selects don't become branches.
  uint32_t at[4], after[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    at[k] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v[k]), static_cast<int>(lo & 63)));
    after[k] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v[k]), static_cast<int>(cnt & 63)));
  }
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(at[0]), "+s"(at[1]), "+s"(at[2]), "+s"(at[3]), "+s"(after[0]), "+s"(after[1]),
               "+s"(after[2]), "+s"(after[3]));
#endif
  const uint32_t next = cnt < kPrefixInRegs ? Pick4(after, cnt >> 6) : kPrefixPad;
  return {lo, u - Pick4(at, lo >> 6), next != kPrefixPad};
}

// Work unit u of `stage` as (image, unit within the image).  Called by a whole wave
// with u uniform.  The image is the last index i with prefix[i] <= u, found by
// counting over a ballot instead of a dependent binary search: for plans of up to 255
// images the wave loads all prefix entries in one round trip (a 64-way narrowing
// per round trip beyond).  Padding past n_images compares above every u, so a u past
// the last unit lands on i = n_images, whose successor entry is padding (or absent
// when n_images = cap): the unit is invalid.  The image count itself is not needed.
__device__ __forceinline__ Located Locate(const KernelArgs &a, uint32_t stage, uint32_t u,
                                          uint32_t groups_per_unit) {
  if (!a.plan) return {0u, u, u < StageUnitsOf(a.single, stage, groups_per_unit)};
  const uint32_t len = a.plan_cap + 1;
  const GPtr<const uint32_t> pre =
      Gbl<const uint32_t>(reinterpret_cast<const uint8_t *>(a.plan) + PlanPrefixOffset(a.plan_cap, stage));
  const uint32_t lane = __lane_id();
  uint32_t lo, start, next = kPrefixPad;
  if (len <= kPrefixInRegs) {
    uint32_t v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) v[k] = lane + 64 * k < len ? pre[lane + 64 * k] : kPrefixPad;
    return LocateIn(v, u);
  } else {
    lo = 0;
    uint32_t m = len;  // the answer lies in [lo, lo + m)
    while (m > 64) {
      const uint32_t step = (m + 63) / 64;
      const uint32_t v = lane * step < m ? pre[lo + lane * step] : kPrefixPad;
      const uint32_t c = Popc64(__builtin_amdgcn_ballot_w64(v <= u));  // >= 1: lane 0 reads prefix[lo]
      lo += (c - 1) * step;
      m = min(step, m - (c - 1) * step);
    }
    const uint32_t v = lane < m ? pre[lo + lane] : kPrefixPad;
    const uint32_t c = Popc64(__builtin_amdgcn_ballot_w64(v <= u));
    start = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(c - 1)));
    lo += c - 1;
    if (lo + 1 < len) next = pre[lo + 1];
  }
  return {lo, u - start, next != kPrefixPad};
}

// An image descriptor as the kernels use it: the same fields with global pointers.
struct DevDesc {
  uint32_t width, height, nv, bx;
  uint32_t palette_bytes;
  uint32_t groups[4];
  uint32_t stream_len[4];
  uint32_t table_base;
  const uint8_t *freqs;
  const uint8_t *streams[4];  // read through buffer resources
  GPtr<uint8_t> symbols;
  GPtr<int8_t> planes;
  GPtr<int32_t> indices;
  GPtr<int32_t> group_sums;
  GPtr<int32_t> lane_sums;  // may be null
  GPtr<uint8_t> out;
};

// The descriptor of image img: scalar loads (the plan is read-only while kernels run).
__device__ __forceinline__ DevDesc LoadDesc(const KernelArgs &a, uint32_t img) {
  ImageDesc s;
  if (a.plan) {
    const CPtr<ImageDesc> p = (CPtr<ImageDesc>)(reinterpret_cast<uintptr_t>(a.plan) + PlanImagesOffset(a.plan_cap));
    s = p[img];
  } else {
    s = a.single;
  }
  DevDesc d;
  d.width = s.width;
  d.height = s.height;
  d.nv = s.nv;
  d.bx = s.bx;
  d.palette_bytes = s.palette_bytes;
  for (int k = 0; k < 4; ++k) {
    d.groups[k] = s.groups[k];
    d.stream_len[k] = s.stream_len[k];
    d.streams[k] = s.streams[k];
  }
  d.table_base = s.table_base;
  d.freqs = s.freqs;
  d.symbols = Gbl<uint8_t>(s.symbols);
  d.planes = Gbl<int8_t>(s.planes);
  d.indices = Gbl<int32_t>(s.indices);
  d.group_sums = Gbl<int32_t>(s.group_sums);
  d.lane_sums = Gbl<int32_t>(s.lane_sums);
  d.out = Gbl<uint8_t>(s.out);
  return d;
}

// The descriptor of image img in constant memory, the plan's or the kernel argument's, for
// kernels that pick a stream's fields by index with scalar loads.
__device__ __forceinline__ CPtr<ImageDesc> DescAt(const KernelArgs &a, uint32_t img) {
  if (a.plan)
    return (CPtr<ImageDesc>)(reinterpret_cast<uintptr_t>(a.plan) + PlanImagesOffset(a.plan_cap)) + img;
#if defined(__HIP_DEVICE_COMPILE__)
  return (CPtr<ImageDesc>)((CPtr<uint8_t>)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(KernelArgs, single));
#else
  return &a.single;
#endif
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t MakeRsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(bytes),
                                           kBufferRsrcWord3);
}

// Inclusive prefix sum over a wave in six DPP adds (row shifts, then row broadcasts): no LDS
// round trip, where __shfl_up is a ds_bpermute each.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t DppAdd(uint32_t v) {
  return v + static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROWS, 0xF, false));
}
__device__ __forceinline__ uint32_t WaveInclusiveSum(uint32_t v) {
  v = DppAdd<0x111, 0xF>(v);  // row_shr:1
  v = DppAdd<0x112, 0xF>(v);  // row_shr:2
  v = DppAdd<0x114, 0xF>(v);  // row_shr:4
  v = DppAdd<0x118, 0xF>(v);  // row_shr:8
  v = DppAdd<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  return DppAdd<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
}

__device__ __forceinline__ uint32_t WaveTotal(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(WaveInclusiveSum(v)), 63));
}

// ---------------------------------------------------------------------------
// Stage 1: rANS slot tables (ans/build_table.cl:12-83).
//
// One work-group per table: a 256-entry scan of the frequencies, then every slot s
// takes the symbol x with cum[x] <= s < cum[x] + f[x].  The reference finds x with an
// 11-step branch-free search; for tables that sum to M its result is that closed
// form (the search path depends only on the target symbol, checked exhaustively
// against the oracle).  Entry packing, 4 bytes:
//   bits 0-11 f[x] (1..2048), bits 12-22 s - cum[x], bits 24-31 x.
// A table that does not sum to 2048 is flagged in table_status and replaced by the
// identity table (f = 2048, offset = slot, symbol 0), which never renormalises.
__global__ __launch_bounds__(256) void BuildTableKernel(KernelArgs a) {
  __shared__ uint32_t cum[256];
  __shared__ uint32_t freq[256];
  __shared__ uint32_t wsum[4];
  const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t total = a.plan ? a.plan->n_images * 4 : 4;
  for (uint32_t u = blockIdx.x; u < total; u += gridDim.x) {
    const uint32_t img = u >> 2, k = u & 3;
    const DevDesc d = LoadDesc(a, img);
    const uint32_t tix = d.table_base + k;
    const GPtr<const uint16_t> fr = Gbl<const uint16_t>(d.freqs + 512 * k);
    const uint32_t f = fr[t];
    uint32_t v = f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t n = __shfl_up(v, off);
      if (lane >= static_cast<uint32_t>(off)) v += n;
    }
    if (lane == 63) wsum[wave] = v;
    __syncthreads();
    uint32_t add = 0;
    for (uint32_t w = 0; w < wave; ++w) add += wsum[w];
    cum[t] = v + add - f;
    freq[t] = f;
    const uint32_t sum = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    const bool valid = sum == kTableSize;
    const GPtr<uint32_t> tab = Gbl<uint32_t>(a.tables + static_cast<size_t>(tix) * kTableSize);
    for (uint32_t slot = t; slot < kTableSize; slot += 256) {
      uint32_t e;
      if (valid) {
        uint32_t x;
        if (cum[255] <= slot) {
          x = 255;
        } else {
          uint32_t pos = 0;  // number of cum[0..254] <= slot
#pragma unroll
          for (uint32_t s = 128; s; s >>= 1)
            if (cum[pos + s - 1] <= slot) pos += s;
          x = pos - 1;
        }
        e = freq[x] | ((slot - cum[x]) << 12) | (x << 24);
      } else {
        e = kTableSize | (slot << 12);
      }
      tab[slot] = e;
    }
    if (t == 0) Gbl<uint32_t>(a.table_status)[tix] = valid ? 1u : 0u;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Stage 2: interleaved rANS decode (ans/ans_decode.cl:25-74,97-143).
//
// A work-group of WAVES wave64s decodes GPW*WAVES consecutive groups of one stream
// with that stream's table resident in LDS in the 4-byte packed form BuildTableKernel
// writes (one random LDS read per step: random table reads are where the LDS bank
// conflicts come from; 8 KiB per table, so a 4-wave work-group with its rings takes
// 18.5 KiB).  The state update is one v_mad_u32_u24 after two bit-field extracts.  With
// GPW = 2 a wave carries two 32-stream groups, one per half-wave; each lane holds
// one stream's state.  The reference's local-memory renormalisation mask
// (atomic_or / popcount / atomic_and between barriers) becomes one ballot: a lane
// that needs a word reads u16[p_half - total_in_half + rank_in_half], the rank
// coming from mbcnt over the 64-bit ballot, and each half-wave's pointer (a scalar)
// moves down by its total.
//
// The words are read from an LDS ring of two 256-word chunks per half-wave, so the
// serial chain of a step only touches LDS.  Chunk c covers stream words
// [256c, 256c + 256) and lives at ring slot c & 1.  With `top` the chunk holding the
// half's pointer - 1, chunks top and top-1 are resident and chunks top-2 and top-3
// are in flight in registers.  A step moves the pointer by at most 32 words, so 4
// steps read only chunks top and top-1; every 4 steps, if the pointer has dropped
// below 256*top, chunk top-2 is written over top's slot and top-4 is requested, which
// then has at least 16 steps to arrive.  Stream loads go through a
// buffer resource bounded by the stream length (corrupt offsets read zeros, never
// fault); a pointer that ends below the group's first byte raises kErrStreamOffsets.
// Each lane packs 64 symbols into 16 registers and writes them as one 64-byte sector,
// in the reference's output order (lane j, step i of the group at j*256 + 255 - i).
// Index-stream groups also emit
// the sum of (symbol - 128) per group and per lane, the totals the index scan
// starts from.
//
// VALU issue bounds it where every SIMD holds several waves: 128 images (11,040 groups, five
// or six waves a SIMD) spend 314 cycles a step and wave, 58 a wave's own VALU, after a
// prologue of 11,000 cycles (20,000 when the streams come from HBM).

// readfirstlane returns a signed int: every use converts through uint32_t so no
// 64-bit widening can sign-extend a value with bit 31 set.
__device__ __forceinline__ uint32_t Uniform(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

// LDS written by some lanes of a wave and read by others: the wave's LDS operations
// complete in order, so only the compiler needs a fence.
__device__ __forceinline__ void WaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr uint32_t kChunkWords = 256;
constexpr uint32_t kRingWords = 2 * kChunkWords;
constexpr uint32_t kRefillSteps = kChunkWords / kLanesPerGroup;  // 8
// The ring is checked every 4 steps, which read at most 128 words; below its first chunk
// stands a copy of the last 128 words of its second, so that they are consecutive downwards
// from any pointer and addresses need no wrap.
constexpr uint32_t kCheckSteps = 4;
constexpr uint32_t kRingBelow = kCheckSteps * kLanesPerGroup;
constexpr uint32_t kRingAlloc = kRingBelow + kRingWords;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Lane l's 8 bytes of chunk c (words 4l .. 4l+3): one wave moves a whole chunk, so a
// refill is never divergent.  A chunk wholly below the group's first chunk `clo` (the
// ring asks up to three chunks past the group's start near its end) reads nothing: its
// offset is moved past the stream (c * 512 wraps to 0xFFFFFE00), as are chunks below
// the stream start, which wrap by themselves.
constexpr uint32_t kNoChunk = 0xFFFFFFFFu >> 9;
__device__ __forceinline__ u32x2 LoadChunk(__amdgpu_buffer_rsrc_t rs, uint32_t c, uint32_t clo, uint32_t l) {
  c = c >= clo ? c : kNoChunk;
  return __builtin_amdgcn_raw_buffer_load_b64(rs, static_cast<int>((c * kChunkWords + 4 * l) * 2), 0, 0);
}

// (Odd chunks also leave their last 128 words below the ring: the upper lanes there, the
// others once more where they are.)
__device__ __forceinline__ void StoreChunk(uint16_t *ring, bool odd, uint32_t l, const u32x2 &a) {
  *reinterpret_cast<u32x2 *>(ring + kRingBelow + (odd ? kChunkWords : 0u) + 4 * l) = a;
  if (odd)
    *reinterpret_cast<u32x2 *>(ring + 4 * l + (4 * l >= kChunkWords - kRingBelow ? kRingBelow - kChunkWords
                                                                               : kRingBelow + kChunkWords)) = a;
}

// A local object's LDS address as the instructions take it.
template <typename T>
__device__ __forceinline__ uint32_t LdsAddress(T *p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)p));
}

// One step of a wave's two groups: the table read at slot x & 2047, the update, the
// pointers, and the next word for the lanes below their threshold.  Symbols are bits 24-31
// of the entry it returns; while the table read is in flight the step puts earlier ones
// into `acc`: the last two at once (kIns 1, `first` the earlier) or the last one (kIns 2).
//
// pA and pB are the halves' pointers as LDS word addresses.  An upper lane's word is at
// pB' plus its rank in its half, that is rank - tlo + pB', and pA' = pA - tlo, so the two
// halves' addresses are rank + pA' and rank + pA' + (pB' - pA): one v_mad with the half `h`.
//
// Written out because the loop is bound by issue (six waves a SIMD hide the latencies): the
// compare writes the lane mask, so the renormalisation is one v_lshl_or under it, and lanes
// that keep their state need no select.  12.75 VALU and 6 SALU a step, where the compiler's
// form, with selects, a wrap per lane and a masked add, had 15.6 and 5: the stage of 128
// images 64.8 -> 62.4 us with inputs from HBM (25.8 -> 21.0 M VALU).
template <int kIns>
__device__ __forceinline__ uint32_t AnsStep(uint32_t &x, uint32_t thr, uint32_t tab_at, uint32_t h, uint64_t lanes,
                                            uint32_t &pA, uint32_t &pB, uint32_t first, uint32_t last, uint32_t &acc,
                                            uint32_t sel) {
  uint32_t fs;
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t t, r, a, b;
#define GST_ANS_TABLE                               \
  "v_and_b32 %[t], 0x7ff, %[x]\n\t"                 \
  "v_lshl_add_u32 %[t], %[t], 2, %[tab]\n\t"        \
  "ds_read_b32 %[fs], %[t]\n\t"                     \
  "v_lshrrev_b32 %[x], 11, %[x]\n\t"
#define GST_ANS_UPDATE                              \
  "s_waitcnt lgkmcnt(0)\n\t"                        \
  "v_and_b32 %[t], 0xfff, %[fs]\n\t"                \
  "v_bfe_u32 %[r], %[fs], 12, 11\n\t"               \
  "v_mad_u32_u24 %[x], %[x], %[t], %[r]\n\t"        \
  "v_cmpx_lt_u32 vcc, %[x], %[thr]\n\t"             \
  "s_bcnt1_i32_b32 %[a], vcc_lo\n\t"                \
  "s_bcnt1_i32_b32 %[b], vcc_hi\n\t"                \
  "v_mbcnt_lo_u32_b32 %[t], vcc_lo, 0\n\t"           \
  "s_sub_u32 %[pB], %[pB], %[b]\n\t"                \
  "s_sub_u32 %[b], %[pB], %[pA]\n\t"                \
  "v_mbcnt_hi_u32_b32 %[t], vcc_hi, %[t]\n\t"       \
  "s_sub_u32 %[pA], %[pA], %[a]\n\t"                \
  "v_mad_i32_i24 %[t], %[h], %[b], %[t]\n\t"        \
  "v_add_lshl_u32 %[t], %[t], %[pA], 1\n\t"         \
  "ds_read_u16 %[t], %[t]\n\t"                      \
  "s_waitcnt lgkmcnt(0)\n\t"                        \
  "v_lshl_or_b32 %[x], %[x], 16, %[t]\n\t"          \
  "s_mov_b64 exec, %[lanes]"
#define GST_ANS_OUT                                                                                           \
  [x] "+v"(x), [fs] "=&v"(fs), [t] "=&v"(t), [r] "=&v"(r), [a] "=&s"(a), [b] "=&s"(b), [pA] "+s"(pA), [pB] "+s"(pB)
#define GST_ANS_IN                                                                                             \
  [thr] "v"(thr), [tab] "s"(tab_at), [h] "v"(h), [lanes] "s"(lanes)
  if constexpr (kIns == 0)
    asm volatile(GST_ANS_TABLE GST_ANS_UPDATE : GST_ANS_OUT : GST_ANS_IN : "vcc", "scc", "memory");
  else if constexpr (kIns == 1)
    asm volatile(GST_ANS_TABLE "v_perm_b32 %[acc], %[first], %[last], %[sel]\n\t" GST_ANS_UPDATE
                 : GST_ANS_OUT, [acc] "=&v"(acc)
                 : GST_ANS_IN, [first] "v"(first), [last] "v"(last), [sel] "s"(sel)
                 : "vcc", "scc", "memory");
  else
    asm volatile(GST_ANS_TABLE "v_perm_b32 %[acc], %[last], %[acc], %[sel]\n\t" GST_ANS_UPDATE
                 : GST_ANS_OUT, [acc] "+v"(acc)
                 : GST_ANS_IN, [last] "v"(last), [sel] "s"(sel)
                 : "vcc", "scc", "memory");
#undef GST_ANS_TABLE
#undef GST_ANS_UPDATE
#undef GST_ANS_OUT
#undef GST_ANS_IN
#endif
  return fs;
}

// The first two chunks of each half's ring (top and top-1, top = the chunk holding
// the half's word pointer - 1), requested before the table is built and written to
// LDS after it.
struct AnsRing {
  u32x2 rA0, rA1, rB0, rB1;
  uint32_t topA, topB;
};

template <uint32_t GPW>
__device__ __forceinline__ AnsRing RequestRing(__amdgpu_buffer_rsrc_t rs, uint32_t pA, uint32_t pB,
                                               uint32_t loA, uint32_t loB, uint32_t lane) {
  AnsRing r;
  r.topA = pA ? (pA - 1) / kChunkWords : 0;
  r.topB = pB ? (pB - 1) / kChunkWords : 0;
  const uint32_t cloA = loA / kChunkWords, cloB = loB / kChunkWords;
  r.rA0 = LoadChunk(rs, r.topA, cloA, lane);
  r.rA1 = LoadChunk(rs, r.topA - 1, cloA, lane);
  r.rB0 = r.rB1 = u32x2{0u, 0u};
  if (GPW == 2) {
    r.rB0 = LoadChunk(rs, r.topB, cloB, lane);
    r.rB1 = LoadChunk(rs, r.topB - 1, cloB, lane);
  }
  return r;
}

// Stream-tail touch.  Every refill waits for all loads in flight, so a refill whose
// chunk is still on its way from HBM stalls the wave for the whole round trip, a dozen
// times per group when the compressed streams are not in any cache (the usual case in a
// decode pipeline, whose other kernel moves a few hundred MB between two rANS passes).
// One pass of 4-byte LDS-DMA loads, a lane per 64 bytes, pulls the rest of the half's
// stream (bytes [lo, 512 (top - 3)), below the four chunks already requested) into L2
// and the memory-side cache at the start; the refills then find their chunks there.
// The loads write a 256-byte LDS sink that nothing reads and hold no VGPR; offsets
// past the stream (and halves with nothing left) read nothing through the buffer's
// range check.  A group's stream is at most 2 * kGroupSyms bytes, so at most
// kTouchPasses passes of 32 lanes x 64 bytes.
constexpr uint32_t kTouchStride = 64;
constexpr uint32_t kTouchPasses = 2 * kGroupSyms / (kLanesPerGroup * kTouchStride);

__device__ __forceinline__ void TouchStreamTail(__amdgpu_buffer_rsrc_t rs, uint32_t top, uint32_t lo_byte,
                                                uint32_t j, uint32_t *sink) {
  const uint32_t hi = top >= 3 ? 2 * kChunkWords * (top - 3) : 0u;
  const uint32_t span = kLanesPerGroup * kTouchStride;
  const uint32_t need = hi > lo_byte ? (hi - lo_byte + span - 1) / span : 0u;
  const uint32_t n0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(need, 0));
  const uint32_t n1 = static_cast<uint32_t>(__builtin_amdgcn_readlane(need, 32));
  const uint32_t n = min(n0 > n1 ? n0 : n1, kTouchPasses);
  for (uint32_t i = 0; i < n; ++i) {
    const uint32_t back = kTouchStride * (j + 1) + span * i;
    const bool in = hi >= back && hi - back + kTouchStride > lo_byte;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)sink, 4,
                                             static_cast<int>(in ? hi - back : 0x7FFFFFF0u), 0, 0, 0);
  }
}

template <bool kSum, uint32_t GPW>
__device__ __forceinline__ void DecodeHalfGroups(const uint32_t *tab, uint16_t *ring_wave, uint32_t *sink,
                                                 __amdgpu_buffer_rsrc_t rs, AnsRing ring, uint32_t lane, bool active, uint32_t x, uint32_t pA, uint32_t pB,
                                                 uint32_t loA, uint32_t loB, GPtr<uint8_t> outp,
                                                 GPtr<int32_t> group_sum, GPtr<int32_t> lane_sum,
                                                 GPtr<int32_t> lane_suffix, uint32_t *err) {
  const uint32_t j = lane & 31;
  // Renormalisation threshold per lane: L for a lane with a stream, 0 (never) for one
  // without, so the compare's mask is already the renormalising lanes.
  uint32_t thr = active ? kStateL : 0u;
  asm volatile("" : "+v"(thr));
  uint16_t *const ringA = ring_wave;
  uint16_t *const ringB = ring_wave + kRingAlloc;
  const uint32_t tab_at = Uniform(LdsAddress(tab));
  // Word addresses of the two rings' first chunks, and from here on the pointers and the
  // start of the chunk each is in.
  const uint32_t slotA = Uniform(LdsAddress(ringA)) / 2 + kRingBelow, slotB = slotA + kRingAlloc;
  const uint32_t mostA = pA - loA, mostB = pB - loB;
  uint32_t topA = ring.topA, topB = ring.topB;
  uint32_t limA = slotA + (topA & 1u) * kChunkWords, limB = slotB + (topB & 1u) * kChunkWords;
  const uint32_t startA = pA, startB = pB;
  pA += limA - topA * kChunkWords;
  pB += limB - topB * kChunkWords;
  uint32_t h = lane >> 5;
  asm volatile("" : "+v"(h));
  const uint64_t lanes = __builtin_amdgcn_read_exec();
  // Chunks top-2 and top-3 go in flight in two fixed registers by chunk parity (even
  // chunks in pXE, odd in pXO): a load lands in the register its chunk is later
  // stored from, so no register moves sit between in-flight loads.  The wait before a
  // refill's store is still vmcnt(0) (the number of refill loads between two crossings
  // is data-dependent and output stores are in flight), which TouchStreamTail makes
  // cheap.
  const uint32_t cloA = loA / kChunkWords, cloB = loB / kChunkWords;
  u32x2 pAE = LoadChunk(rs, (topA & 1u) ? topA - 3 : topA - 2, cloA, lane);
  u32x2 pAO = LoadChunk(rs, (topA & 1u) ? topA - 2 : topA - 3, cloA, lane);
  u32x2 pBE = {0u, 0u}, pBO = {0u, 0u};
  if (GPW == 2) {
    pBE = LoadChunk(rs, (topB & 1u) ? topB - 3 : topB - 2, cloB, lane);
    pBO = LoadChunk(rs, (topB & 1u) ? topB - 2 : topB - 3, cloB, lane);
  }
  TouchStreamTail(rs, lane < 32 ? topA : topB, 2u * (lane < 32 ? loA : loB), j, sink);
  StoreChunk(ringA, (topA & 1u) != 0, lane, ring.rA0);
  StoreChunk(ringA, (topA & 1u) == 0, lane, ring.rA1);
  if (GPW == 2) {
    StoreChunk(ringB, (topB & 1u) != 0, lane, ring.rB0);
    StoreChunk(ringB, (topB & 1u) == 0, lane, ring.rB1);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  int32_t sum = 0;
  // 64 steps fill one 64-byte sector of the lane's output; whole sectors leave in four
  // back-to-back 16-byte stores (smaller pieces of a lane's segment, 256 B apart
  // across lanes, are evicted half-written and written back several times).
  for (uint32_t sector = 0; sector < kSymsPerLane / 64; ++sector) {
    // A SIMD's waves compete for issue slots and the oldest win, so young waves
    // would be left with most of their steps for the end, when too few waves remain
    // to keep the SIMD busy.  Priority falls as a wave gets further ahead, which
    // keeps the waves of a SIMD within about a sector of each other.
    switch (sector) {
      case 0: __builtin_amdgcn_s_setprio(3); break;
      case 1: __builtin_amdgcn_s_setprio(2); break;
      case 2: __builtin_amdgcn_s_setprio(1); break;
      default: __builtin_amdgcn_s_setprio(0); break;
    }
    uint32_t acc[16], first = 0, last = 0, none = 0;
#pragma unroll
    for (uint32_t blk = 0; blk < 64 / kRefillSteps; ++blk) {
#pragma unroll
      for (uint32_t s = 0; s < kRefillSteps; ++s) {
        // Step 8*blk + s decodes byte 63 - 8*blk - s of the sector, the last first; byte
        // `at` is the step before's.  v_perm: selector codes 4-7 take bytes of the first
        // operand, 0-3 bytes of the second, 0x0c is zero.
        const uint32_t at = 64 - kRefillSteps * blk - s;
        uint32_t fs;
        if (at == 64 || (at & 3) == 3)
          fs = AnsStep<0>(x, thr, tab_at, h, lanes, pA, pB, 0u, 0u, none, 0u);
        else if ((at & 3) == 2)
          fs = AnsStep<1>(x, thr, tab_at, h, lanes, pA, pB, first, last, acc[at >> 2], 0x07030C0Cu);
        else
          fs = AnsStep<2>(x, thr, tab_at, h, lanes, pA, pB, 0u, last, acc[at >> 2],
                          (at & 3) == 1 ? 0x0302070Cu : 0x03020107u);
        first = last;
        last = fs;
        // The pointers moved at most 128 words since the last check, so each crossed at most
        // one chunk's start, and the next 4 steps read only chunks top and top-1 (top =
        // chunk of pointer - 1).  Per crossed half (uniform branches, all 64 lanes): store
        // chunk top-2 from the register of its parity, request chunk top-4 (same parity)
        // into it, and from the first chunk's copy below move on to the second.
        if ((s + 1) % kCheckSteps == 0 && static_cast<int32_t>((pA - limA) | (pB - limB)) < 0) {
          const bool crossA = pA < limA, crossB = pB < limB;
          const bool oddA = (topA & 1u) != 0, oddB = (topB & 1u) != 0;
          if (crossA && oddA) {
            StoreChunk(ringA, true, lane, pAO);
            asm volatile("" ::: "memory");
            pAO = LoadChunk(rs, topA - 4, cloA, lane);
          }
          if (crossA && !oddA) {
            StoreChunk(ringA, false, lane, pAE);
            asm volatile("" ::: "memory");
            pAE = LoadChunk(rs, topA - 4, cloA, lane);
          }
          if (GPW == 2 && crossB && oddB) {
            StoreChunk(ringB, true, lane, pBO);
            asm volatile("" ::: "memory");
            pBO = LoadChunk(rs, topB - 4, cloB, lane);
          }
          if (GPW == 2 && crossB && !oddB) {
            StoreChunk(ringB, false, lane, pBE);
            asm volatile("" ::: "memory");
            pBE = LoadChunk(rs, topB - 4, cloB, lane);
          }
          pA += crossA && !oddA ? kRingWords : 0u;
          pB += crossB && !oddB ? kRingWords : 0u;
          limA = crossA ? slotA + (oddA ? 0u : kChunkWords) : limA;
          limB = crossB ? slotB + (oddB ? 0u : kChunkWords) : limB;
          topA -= crossA ? 1u : 0u;
          topB -= crossB ? 1u : 0u;
          WaveSync();
        }
      }
    }
    acc[0] = __builtin_amdgcn_perm(last, acc[0], 0x03020107u);
    if (kSum) {
      // Byte sums of the sector's two 32-symbol halves (v_sad_u8 against zero), less
      // the biases.  The sector covers lane positions 192 - 64 sector + [0, 64), so
      // its halves are sub-segments k = 6 - 2 sector and 7 - 2 sector, and the running
      // total from the top gives the suffix sums R[k] and R[k + 1].
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) lo = __builtin_amdgcn_sad_u8(acc[i], 0u, lo);
#pragma unroll
      for (uint32_t i = 8; i < 16; ++i) hi = __builtin_amdgcn_sad_u8(acc[i], 0u, hi);
      const int32_t r_hi = sum + static_cast<int32_t>(hi) - 32 * 128;
      const int32_t r_lo = r_hi + static_cast<int32_t>(lo) - 32 * 128;
      sum = r_lo;
      if (active && lane_suffix)
        *(GPtr<int2>)(lane_suffix + 8 * j + 6 - 2 * sector) = make_int2(r_lo, r_hi);
    }
    if (active) {
      const GPtr<uint4> dst = (GPtr<uint4>)(outp + (kSymsPerLane - 64) - 64 * sector);
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        dst[i] = make_uint4(acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]);
    }
  }
  // Words each group consumed (modulo 2^32: at most 2^13), against those it has.
  const uint32_t usedA = startA - (topA * kChunkWords + (pA - limA));
  const uint32_t usedB = startB - (topB * kChunkWords + (pB - limB));
  const bool under = lane < 32 ? usedA > mostA : usedB > mostB;
  if (active && under && j == 0) atomicOr(err, kErrStreamOffsets);
  if (kSum) {
    // Inclusive prefix of the lane totals over the half-wave's 32 lanes.
    int32_t incl = sum;
#pragma unroll
    for (uint32_t off = 1; off < 32; off <<= 1) {
      const int32_t n = __shfl_up(incl, off, 32);
      if (j >= off) incl += n;
    }
    if (active && lane_sum) lane_sum[j] = incl;
    const int32_t total = __shfl(incl, 31, 32);
    if (active && j == 0) *group_sum = total;
  }
}

// Work-groups are dispatched to the 8 XCDs round robin (group b on XCD b % 8), each XCD
// with its own L2.  This maps group b to a unit so that every XCD takes one contiguous
// range of the grid's first pass: neighbouring units, which share cache lines and an
// image's palette and sums, then meet in one L2.  A bijection on [0, n) for any n.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t XcdContiguous(uint32_t b, uint32_t n) {
  const uint32_t q = n / kXcds, r = n % kXcds, xcd = b % kXcds, idx = b / kXcds;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
}

// The same split by the stage's actual unit count, for grids of any size (persistent
// grids below it, plan grids above it): XCD x owns the x-th of 8 contiguous ranges of
// [0, units) and its work-groups stride through that range, so every XCD gets an equal
// share whatever the grid (a split by the grid's size would leave whole XCDs idle when
// the grid exceeds the units, and one XCD with the last round when it falls short).
// Grids under 8 work-groups leave XCDs without work-groups: they stride over all units.
struct XcdSpan {
  uint32_t first, end, stride;
};
__device__ __forceinline__ XcdSpan XcdBalanced(uint32_t b, uint32_t grid, uint32_t units) {
  if (grid < kXcds) return {b, units, grid};
  const uint32_t q = units / kXcds, r = units % kXcds, xcd = b % kXcds, idx = b / kXcds;
  const uint32_t lo = xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
  const uint32_t n = q + (xcd < r ? 1u : 0u);
  const uint32_t groups_here = (grid - xcd + kXcds - 1) / kXcds;  // work-groups with b % 8 == xcd
  return {lo + idx, lo + n, groups_here};
}

__device__ __forceinline__ const uint8_t *Uniform(const uint8_t *p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint64_t lo = Uniform(static_cast<uint32_t>(v));
  const uint64_t hi = Uniform(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const uint8_t *>(lo | (hi << 32));
}

// Work-group barrier that orders LDS only: waits for the wave's own LDS operations,
// not for its global loads in flight (a __syncthreads fence would wait for those too).
__device__ __forceinline__ void LdsBarrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The work of BuildTableKernel for one table, straight into a rANS kernel's LDS (256 <=
// THREADS): thread t < 256 brings frequency f[t].  The slot -> symbol map is a count, not a
// search:
//   A. the marks are cleared (a bit a slot); the first four waves scan f + (f != 0) << 24,
//      giving every symbol its cum (low 24 bits: 256 u16 sum below 2^24) and its rank
//      among the nonzero symbols (high bits);
//   B. every nonzero symbol x writes {f | x << 24, cum} at its rank and sets the mark of
//      slot cum;
//   C. each wave counts the marks before its 64-slot chunks (a lane per chunk and one DPP
//      scan), and mbcnt over a chunk's marks, in scalar registers, gives each slot the
//      rank of its symbol: one gather a slot, all of a wave's in flight together.
// A table that does not sum to 2048 becomes the identity table.  `put(slot, {f | symbol
// << 24, slot - cum})` stores an entry.  Returns whether the table is valid; ends with a
// work-group barrier.  One round trip of gathers where a first version had three a chunk
// (marks, rank to symbol, symbol to frequency), with ds_bpermute scans: 4,300 -> 2,060
// cycles for a work-group alone on its CU.
constexpr uint32_t kBuildScratchWords = 2 * 256 + kTableSize / 32 + 4;

template <uint32_t THREADS, typename Put>
__device__ __forceinline__ bool BuildTableInLds(uint32_t f, uint32_t *scratch, Put put) {
  constexpr uint32_t kWaves = THREADS / 64, kSlotsPerWave = kTableSize / kWaves, kChunks = kSlotsPerWave / 64;
  static_assert(THREADS >= 256 && kChunks * 64 * kWaves == kTableSize, "launch shape");
  u32x2 *const ent = reinterpret_cast<u32x2 *>(scratch);   // [256], by rank
  uint32_t *const marks = scratch + 512;                   // a bit per slot
  uint32_t *const wsum = scratch + 512 + kTableSize / 32;  // [4]
  const uint32_t t = threadIdx.x, lane = t & 63, wave = Uniform(t >> 6);
  if (t < kTableSize / 32) marks[t] = 0;
  const uint32_t pk = f + (static_cast<uint32_t>(f != 0) << 24);
  const uint32_t v = WaveInclusiveSum(pk);
  if (lane == 63 && t < 256) wsum[wave] = v;
  LdsBarrier();
  const u32x4 ws = *reinterpret_cast<const u32x4 *>(wsum);
  const bool valid = Uniform((ws.x + ws.y + ws.z + ws.w) & 0xFFFFFFu) == kTableSize;
  if (valid && t < 256) {
    const uint32_t add = (wave > 0 ? ws.x : 0u) + (wave > 1 ? ws.y : 0u) + (wave > 2 ? ws.z : 0u);
    const uint32_t excl = add + v - pk, cum = excl & 0xFFFFFFu;
    if (f != 0) {  // the table sums to 2048, so cum + f <= 2048: the mark is inside it
      ent[excl >> 24] = u32x2{f | (t << 24), cum};
      atomicOr(&marks[cum >> 5], 1u << (cum & 31));
    }
  }
  LdsBarrier();
  const uint32_t slot0 = wave * kSlotsPerWave + lane;
  if (valid) {
    const u32x2 m = reinterpret_cast<const u32x2 *>(marks)[lane & 31];  // lane c: chunk c's marks
    const uint32_t n = lane < 32 ? static_cast<uint32_t>(__popc(m.x) + __popc(m.y)) : 0u;
    // Rank of a slot's symbol: marks at slots up to it, less 1 = those of earlier chunks and
    // of the chunk's first slot, then mbcnt (lanes below) over the marks moved down a slot.
    const uint32_t first = WaveInclusiveSum(n) - n + (m.x & 1u) - 1u;
    u32x2 e[kChunks];
#pragma unroll
    for (uint32_t j = 0; j < kChunks; ++j) {
      const int c = static_cast<int>(wave * kChunks + j);
      const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m.x), c));
      const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m.y), c));
      const uint64_t up = ((static_cast<uint64_t>(hi) << 32) | lo) >> 1;
      const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
          static_cast<uint32_t>(up >> 32),
          __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(up),
                                    static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(first), c))));
      e[j] = ent[rank & 255];
    }
#pragma unroll
    for (uint32_t j = 0; j < kChunks; ++j) put(slot0 + 64 * j, u32x2{e[j].x, slot0 + 64 * j - e[j].y});
  } else {
#pragma unroll
    for (uint32_t j = 0; j < kChunks; ++j) put(slot0 + 64 * j, u32x2{kTableSize, slot0 + 64 * j});
  }
  LdsBarrier();
  return valid;
}

// kBuild: build the stream's table from its frequencies in LDS instead of loading
// the one BuildTableKernel wrote (the decode pipeline then skips that launch).
// kPair: units are numbered with short remainders paired (AnsUnitAt); a pair's two
// streams each get half of the waves and a table of their own, built one after the
// other.  The second table takes 8 KiB of LDS, which caps the kernel at 6 work-groups
// per CU: that is the point, a SIMD then never holds more than 6 decoding waves.
// A work-unit starts with a chain of dependent loads (plan -> descriptor -> group
// offsets -> lane states and ring chunks), all from HBM in a full pipeline; the
// frequencies go out with the offsets and the states and chunks before the table is
// built, so the LDS build overlaps their latency.
// LDS of the rANS kernels beside their tables and rings.
struct AnsLdsSmall {
  uint32_t touch_sink[64];
};

// The LDS of AnsDecodeUnits: tables (one, two with kPair) and the half-waves' rings.
// The table build's scratch lives in the rings: every wave has left the previous
// unit's ring (barrier) before the build, and the rings are filled after it.
template <uint32_t WAVES, bool kPair>
struct AnsLds {
  uint32_t tab[kPair ? 2 : 1][kTableSize];
  uint16_t ring[WAVES][2][kRingAlloc];
};

template <uint32_t WAVES, uint32_t GPW, bool kBuild, bool kPair>
__device__ __forceinline__ void AnsDecodeUnits(const KernelArgs &a, AnsLds<WAVES, kPair> &L,
                                               AnsLdsSmall &S) {
  static_assert(!kPair || (kBuild && WAVES % 2 == 0), "paired units build their tables in LDS");
  static_assert(!kBuild || WAVES * 2 * kRingAlloc * 2 >= 4 * kBuildScratchWords, "build scratch fits the rings");
  auto &tab = L.tab;
  auto &ring = L.ring;
  uint32_t *const build_scratch = reinterpret_cast<uint32_t *>(&ring[0][0][0]);
  uint32_t *const touch_sink = S.touch_sink;
  constexpr uint32_t kGroupsPerUnit = WAVES * GPW;
  constexpr uint32_t kUnitCode = kGroupsPerUnit | (kPair ? kAnsPairShort : 0u);
  const uint32_t lane = threadIdx.x & 63, wave = Uniform(threadIdx.x >> 6);
  const uint32_t half = GPW == 2 ? (lane >> 5) : 0;
  const uint32_t j = lane & 31;
  for (uint32_t u = blockIdx.x;; u += gridDim.x) {
    const Located loc = Locate(a, kStageAns, u, kUnitCode);
    if (!loc.valid) break;
    // Scalar loads by index in two trips, the group counts and then the fields of the
    // unit's stream: no selects over a descriptor in registers.
    const CPtr<ImageDesc> d = DescAt(a, loc.img);
    const AnsGroupCounts counts = {{d->groups[0], d->groups[1], d->groups[2], d->groups[3]}};
    uint32_t k, first, count, k2 = 0, gi = wave * GPW + half, seg = 0;
    bool second = false;
    uint32_t k_first;
    if constexpr (kPair) {
      const AnsUnit unit = AnsUnitAt(counts, kUnitCode, Uniform(loc.local));
      // This wave's segment: the unit's only one, or its half of a pair.
      seg = unit.pair && wave >= WAVES / 2 ? 1u : 0u;
      k = Uniform(seg ? unit.k[1] : unit.k[0]);
      first = Uniform(seg ? unit.first[1] : unit.first[0]);
      count = Uniform(seg ? unit.count[1] : unit.count[0]);
      if (unit.pair) gi = (wave % (WAVES / 2)) * GPW + half;
      second = unit.pair && unit.count[1] != 0;
      k_first = unit.k[0];
      k2 = unit.k[1];
    } else {
      const StreamUnit unit =
          StreamUnitAt(kGroupsPerUnit, counts.groups[0], counts.groups[1], counts.groups[2], counts.groups[3], loc.local);
      k = k_first = unit.k;
      first = unit.first;
      count = unit.count;
    }
    const uint32_t G = d->groups[k], slen = d->stream_len[k];
    const uint32_t g = first + gi;
    const __amdgpu_buffer_rsrc_t rs = MakeRsrc(d->streams[k], slen);
    // Straight-line loads (out-of-range offsets read zeros): a load under a branch
    // makes the wait for it land at the join, after later loads have gone out.
    const uint32_t end = __builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(4 * g), 0, 0);
    const uint32_t lo_word = __builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(4 * (g - 1)), 0, 0);
    // Frequencies of the unit's table(s): thread t brings symbol t's.
    uint32_t f = 0, f2 = 0;
    if constexpr (kBuild) {
      const GPtr<const uint16_t> fr = Gbl<const uint16_t>(d->freqs);
      f = fr[256 * k_first + (threadIdx.x & 255)];
      if (kPair && second) f2 = fr[256 * k2 + (threadIdx.x & 255)];
    }
    const uint32_t lo = g == 0 ? 4 * G : lo_word;
    const bool ok = ((end | lo) & 3) == 0 && end <= slen && lo >= 4 * G && lo <= end &&
                    end - lo >= 4 * kLanesPerGroup;
    const bool in_stream = (GPW == 2 || lane < 32) && gi < count;
    if (in_stream && !ok && j == 0) atomicOr(a.err, kErrStreamOffsets);
    const bool active = in_stream && ok;
    const uint32_t x_word =
        __builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(end - 4 * kLanesPerGroup + 4 * j), 0, 0);
    const uint32_t x = active ? x_word : 0u;
    const uint32_t p = active ? (end - 4 * kLanesPerGroup) >> 1 : 0u;
    const uint32_t plo = active ? lo >> 1 : 0u;
    const uint32_t pA = __builtin_amdgcn_readlane(p, 0);
    const uint32_t loA = __builtin_amdgcn_readlane(plo, 0);
    const uint32_t pB = __builtin_amdgcn_readlane(p, 32);  // 0 with one group a wave
    const uint32_t loB = __builtin_amdgcn_readlane(plo, 32);
    const AnsRing chunks = RequestRing<GPW>(rs, pA, pB, loA, loB, lane);

    LdsBarrier();  // every wave is done with the previous unit's tables and rings
    bool table_ok;
    if constexpr (kBuild) {
      // Entries packed as in the kernel's header comment: the slot's offset is below 2^11.
      const auto put = [](uint32_t *t) {
        return [t](uint32_t slot, const u32x2 &e) { t[slot] = e.x | (e.y << 12); };
      };
      table_ok = BuildTableInLds<WAVES * 64>(f, build_scratch, put(tab[0]));
      if (kPair && second)
        table_ok = BuildTableInLds<WAVES * 64>(f2, build_scratch, put(tab[kPair ? 1 : 0])) && table_ok;
    } else {
      const uint32_t tix = d->table_base + k;
      const GPtr<const uint32_t> src = Gbl<const uint32_t>(a.tables + static_cast<size_t>(tix) * kTableSize);
      for (uint32_t i = threadIdx.x; i < kTableSize; i += WAVES * 64) tab[0][i] = src[i];
      table_ok = Gbl<const uint32_t>(a.table_status)[tix] != 0;
      LdsBarrier();
    }
    if (!table_ok && threadIdx.x == 0) atomicOr(a.err, kErrFrequencies);

    // A wave past its stream's last group (the stream's group count is not a multiple
    // of the unit) has nothing to decode: it would only take issue slots from the waves
    // that do.  It goes straight to the next unit's barrier.
    if (__builtin_amdgcn_ballot_w64(active) == 0) continue;
    const uint32_t *const tw = tab[kPair ? seg : 0];
    const GPtr<uint8_t> outp = Gbl<uint8_t>(d->symbols + SymbolOffset(d->nv, d->palette_bytes, k)) +
                               static_cast<size_t>(g) * kGroupSyms + j * kSymsPerLane;
    if (k == 3) {
      const GPtr<int32_t> sums = Gbl<int32_t>(d->lane_sums);
      DecodeHalfGroups<true, GPW>(tw, ring[wave][0], touch_sink, rs, chunks, lane, active, x, pA, pB, loA, loB, outp,
                                  Gbl<int32_t>(d->group_sums) + g, sums ? sums + g * kLanesPerGroup : nullptr,
                                  sums ? sums + LaneSuffixBase(d->nv) + g * kLanesPerGroup * 8 : nullptr, a.err);
    } else {
      DecodeHalfGroups<false, GPW>(tw, ring[wave][0], touch_sink, rs, chunks, lane, active, x, pA, pB, loA, loB, outp,
                                   nullptr, nullptr, nullptr, a.err);
    }
  }
}

template <uint32_t WAVES, uint32_t GPW, bool kBuild>
// With 4 or 8 waves LDS allows 7 waves per SIMD; hold the VGPRs to that (at most 72).
__global__ __launch_bounds__(WAVES * 64, WAVES >= 4 ? 7 : 1)
void AnsDecodeKernel(KernelArgs a) {
  __shared__ __align__(16) AnsLds<WAVES, false> lds;
  __shared__ AnsLdsSmall small;
  AnsDecodeUnits<WAVES, GPW, kBuild, false>(a, lds, small);
}

// The rANS stage whose work-unit form is data: the plan's unit code (or, for a single
// image, the one in the arguments) selects units of 8 groups of one stream or the
// paired form (short remainders share a work-group), both AnsDecodeUnits<4, 2> with
// tables built in LDS.  The two share the LDS of the larger, the paired form's two
// tables (6 work-groups per CU), and a captured graph of this launch replays either,
// so a batch can change forms from bind to bind.
constexpr uint32_t kAutoWaves = 4;
union AnsAutoLds {
  AnsLds<kAutoWaves, false> single;
  AnsLds<kAutoWaves, true> paired;
};

__global__ __launch_bounds__(kAutoWaves * 64, 6) void AnsAutoKernel(KernelArgs a) {
  __shared__ __align__(16) AnsAutoLds lds;
  __shared__ AnsLdsSmall small;
  const uint32_t code = a.plan ? Uniform(Gbl<const uint32_t>(&a.plan->ans_unit_code)[0]) : a.ans_unit_code;
  if (code & kAnsPairShort)
    AnsDecodeUnits<kAutoWaves, 2, true, true>(a, lds.paired, small);
  else
    AnsDecodeUnits<kAutoWaves, 2, true, false>(a, lds.single, small);
}

// ---------------------------------------------------------------------------
// The rANS stage where latency bounds it: few groups, so that every SIMD holds at most a
// handful of decoding waves and a step costs its dependency chain, not its issue slots.
//
// A wave decodes one group (32 lanes), and a step has one LDS round trip.  The lane's
// state y is kept as it comes out of the update, before renormalisation:
//   keep   (y >= L): next y = (y >> 11) f + off, {f, off} the table entry of slot y & 2047
//   renorm (y <  L): x = y << 16 | w, so (x >> 11) f + off = y (32 f) + ((w >> 11) f + off)
// with the entry of slot w & 2047: everything but y is known from the word alone.  So the
// table holds {f | symbol << 24, off} and the ring, next to it in LDS, the renormalising
// entry {32 f | symbol << 24, (w >> 11) f + off} of every word, made when its chunk comes
// in (64 words' gathers in parallel, off the chain).  A step selects one of two LDS
// addresses and one of two multiplicands, reads 8 bytes and does one v_mad_u32_u24 (which
// takes the low 24 bits of both factors, so the symbol rides along): mad, compare, mbcnt,
// address, select, read.
//
// Lane l decodes stream 31 - l and the ring is stored in reading order (descending word
// index), so a lane's word is `q` + the renormalising lanes below it: mbcnt gives it
// without waiting for the total.  The ring has two 256-word chunks and a copy of the
// first behind the second: the 256 words that 8 steps can read at most are consecutive
// from any q < 512, and addresses need no wrap.  q (a scalar byte address) moves by 8
// times the popcount while the read is in flight; each 8 steps it is compared with the
// chunk's end, and a crossing writes the chunk requested two crossings earlier.
//
// A step is bound by that chain: 101 cycles, about 52 of them the LDS read, and 440 a refill
// (133 a step with an index stream's 13 refills), against some 280 in AnsAutoKernel (two LDS
// round trips, 12 dependent VALU, two scalar hops).  Stage times by events, which add 1.5 us,
// this kernel / AnsAutoKernel: one 512x512 image 18.6 / 33.6 us, 1024x1024 images by the dozen:
// 8 (480 groups) 20.9 / 36.0, 34 (2,040) 27.8 / 39.8, 68 (4,080, four waves a SIMD) 35.7 / 43.2.
// LDS holds four work-groups a CU; a second pass loses the gain (4,620 groups: 43.6 / 44.2;
// 7,200: 53.7 / 47.4).
//
// With the four steps of a symbol word in one block and one test a ring check: one 4096x4096
// image 21.8 -> 21.0 us, 24 images 24.3 -> 23.1, 16 512x512 images 20.3 -> 19.4, 24 groups of
// AnsGroupsKernel 20.8 -> 19.4 (three sets of inputs in turn).  16 steps a loop iteration
// instead of 64, for a quarter of the code, was slower: 27,900 -> 29,200 cycles a group.
constexpr uint32_t kChainWaves = kChainGroups;
constexpr uint32_t kChainRing = 3 * kChunkWords;  // entries per wave

struct AnsChainLds {
  u32x2 tab[kTableSize];
  u32x2 ring[kChainWaves][kChainRing];
};
static_assert(sizeof(AnsChainLds) == 40960, "four work-groups per CU");

// The renormalising entries of lane l's four words of a chunk, in reading order, at entry
// `at` of the ring (and again at `copy`, for the chunk the ring holds twice).
__device__ __forceinline__ void StoreChainChunk(const u32x2 *tab, u32x2 *ring, uint32_t at, bool twice, uint32_t l,
                                                const u32x2 &w) {
  u32x4 o[2];
  uint32_t word[4] = {w.x & 0xFFFFu, w.x >> 16, w.y & 0xFFFFu, w.y >> 16};
  u32x2 e[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) e[k] = tab[word[k] & (kTableSize - 1)];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t lo = __builtin_amdgcn_perm(e[k].x, e[k].x << 5, 0x07020100u);  // 32 f, the symbol on top
    const uint32_t hi = __umul24(word[k] >> kTableLog, e[k].x) + e[k].y;
    const uint32_t pos = 3 - k;
    o[pos >> 1][(pos & 1) * 2] = lo;
    o[pos >> 1][(pos & 1) * 2 + 1] = hi;
  }
  u32x4 *const d = reinterpret_cast<u32x4 *>(ring + at + kChunkWords - 4 - 4 * l);
  d[0] = o[0];
  d[1] = o[1];
  if (twice) {
    d[kChunkWords] = o[0];
    d[kChunkWords + 1] = o[1];
  }
}

// Four steps, whose symbols are the returned word (the first in byte 3): moves the state y,
// and q past the words the wave's lanes take.  `thr0` is the first step's threshold.
//
// One block in a fixed order: the address chain first, what fits behind it while the read is
// in flight, the wait, the update, and the symbol's insertion where the update's latency
// would idle.  (A step left to the compiler took 135 cycles, a block a step 123, of which a
// wait state that the compiler puts behind every block and the 18 scalar instructions of a
// ring check; see DecodeGroupChain.  A read of either entry under its own exec mask, without
// the address select, also took 135.)  Two instructions stand between the compare and the
// first vector read of its vcc_lo, the wait states that this chip asks for and that the
// compiler does not add inside the block.  tab_at is the table's LDS address, q the next
// word's entry's; the entry is in fixed registers because its halves have no name otherwise.
__device__ __forceinline__ uint32_t ChainSteps(uint32_t &y, uint32_t thr0, uint32_t thr, uint32_t tab_at, uint32_t &q) {
  uint32_t word = 0;
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t slot, rank, mul, moved;
#define GST_CHAIN_STEP(THR, INSERT)                    \
  "v_cmp_lt_u32 vcc, %[y], " THR "\n\t"                \
  "v_and_b32 %[slot], 0x7ff, %[y]\n\t"                 \
  "v_lshl_add_u32 %[slot], %[slot], 3, %[tab]\n\t"     \
  "v_mbcnt_lo_u32_b32 %[rank], vcc_lo, 0\n\t"          \
  "v_lshl_add_u32 %[rank], %[rank], 3, %[q]\n\t"       \
  "v_cndmask_b32 %[slot], %[slot], %[rank], vcc\n\t"   \
  "ds_read_b64 v[120:121], %[slot]\n\t"                \
  "v_lshrrev_b32 %[mul], 11, %[y]\n\t"                 \
  "s_bcnt1_i32_b32 %[moved], vcc_lo\n\t"               \
  "v_cndmask_b32 %[mul], %[mul], %[y], vcc\n\t"        \
  "s_lshl3_add_u32 %[q], %[moved], %[q]\n\t"           \
  "s_waitcnt lgkmcnt(0)\n\t"                           \
  "v_mad_u32_u24 %[y], %[mul], v120, v121\n\t" INSERT "\n\t"
  asm volatile(GST_CHAIN_STEP("%[thr0]", "v_mov_b32 %[word], v120")
               GST_CHAIN_STEP("%[thr]", "v_perm_b32 %[word], v120, %[word], %[s2]")
               GST_CHAIN_STEP("%[thr]", "v_perm_b32 %[word], v120, %[word], %[s1]")
               GST_CHAIN_STEP("%[thr]", "v_perm_b32 %[word], v120, %[word], %[s0]")
               : [y] "+v"(y), [q] "+s"(q), [word] "=&v"(word), [slot] "=&v"(slot), [rank] "=&v"(rank),
                 [mul] "=&v"(mul), [moved] "=&s"(moved)
               : [thr0] "v"(thr0), [thr] "v"(thr), [tab] "s"(tab_at), [s2] "s"(0x03070100u), [s1] "s"(0x03020700u),
                 [s0] "s"(0x03020107u)
               : "vcc", "scc", "memory", "v120", "v121");
#undef GST_CHAIN_STEP
#endif
  return word;
}

// One group of n <= 32 streams: lanes 0 .. n - 1 decode streams n - 1 .. 0 from state y,
// their words below word p (chunk top first, chunks below clo read zeros), with E and O
// the chunks top - 2 and top - 3 in flight.  Leaves the state before its last
// renormalisation in y and the ring address of the next word in q; returns how many words
// the group consumed before that renormalisation.
template <bool kSum>
__device__ __forceinline__ uint32_t DecodeGroupChain(const AnsChainLds &lds, u32x2 *ring,
                                                     __amdgpu_buffer_rsrc_t rs, uint32_t lane, uint32_t n,
                                                     uint32_t &y, uint32_t &q, uint32_t p, uint32_t clo, u32x2 pE,
                                                     u32x2 pO, GPtr<uint8_t> outp, GPtr<int32_t> group_sum,
                                                     GPtr<int32_t> lane_sum, GPtr<int32_t> lane_suffix) {
  const bool active = lane < n;
  const uint32_t j = active ? n - 1 - lane : 0u;
  const uint32_t full = active ? kStateL : 0u;
  uint32_t thr = 0;  // a group's first step never renormalises: its states come as stored
  asm volatile("" : "+v"(thr));
  uint32_t top = p ? (p - 1) / kChunkWords : 0u;
  const uint32_t tab_at = Uniform(LdsAddress(&lds.tab[0])), ring_at = Uniform(LdsAddress(ring));
  const uint32_t q0 = ring_at + 8 * (kChunkWords - 1 - ((p - 1) & (kChunkWords - 1)));
  q = Uniform(q0);
  const uint32_t end0 = ring_at + 8 * kChunkWords, end1 = ring_at + 16 * kChunkWords;
  uint32_t limit = end0, wraps = 0;
  int32_t sum = 0;
  for (uint32_t sector = 0; sector < kSymsPerLane / 64; ++sector) {
    uint32_t acc[16];
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
      acc[15 - w] = ChainSteps(y, thr, full, tab_at, q);
      thr = full;
      // 8 steps read at most 256 words, so at most one chunk's end was crossed.  One test
      // on the way past (two scalar instructions; both cases' tests there took 18, 100
      // cycles of each 8 steps), and behind it two uniform branches, not an if/else, so that
      // each request stays in its register.
      if (w % 2 == 1 && __builtin_expect(q >= limit, 0)) {
        const bool first = limit == end0, second = limit == end1;
        if (first) {
          StoreChainChunk(lds.tab, ring, 0, true, lane, pE);
          asm volatile("" ::: "memory");
          pE = LoadChunk(rs, top - 4, clo, lane);
        }
        if (second) {
          StoreChainChunk(lds.tab, ring, kChunkWords, false, lane, pO);
          asm volatile("" ::: "memory");
          pO = LoadChunk(rs, top - 4, clo, lane);
          q -= 16 * kChunkWords;
          ++wraps;
        }
        limit = first ? end1 : end0;
        --top;
        WaveSync();
      }
    }
    if (kSum) {
      // As in DecodeHalfGroups: the sector's suffix sums from 32-symbol steps.
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) lo = __builtin_amdgcn_sad_u8(acc[i], 0u, lo);
#pragma unroll
      for (uint32_t i = 8; i < 16; ++i) hi = __builtin_amdgcn_sad_u8(acc[i], 0u, hi);
      const int32_t r_hi = sum + static_cast<int32_t>(hi) - 32 * 128;
      const int32_t r_lo = r_hi + static_cast<int32_t>(lo) - 32 * 128;
      sum = r_lo;
      if (active && lane_suffix)
        *(GPtr<int2>)(lane_suffix + 8 * j + 6 - 2 * sector) = make_int2(r_lo, r_hi);
    }
    if (active) {
      const GPtr<uint4> dst = (GPtr<uint4>)(outp + j * kSymsPerLane + (kSymsPerLane - 64) - 64 * sector);
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        dst[i] = make_uint4(acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]);
    }
  }
  if (kSum) {
    // Inclusive prefix over the 32 streams, which run down the lanes: within each row of 16
    // by DPP row shifts, then the upper row's total to the lower.
    uint32_t v = static_cast<uint32_t>(sum);
    v = DppAdd<0x101, 0xF>(v);  // row_shl:1, 2, 4, 8
    v = DppAdd<0x102, 0xF>(v);
    v = DppAdd<0x104, 0xF>(v);
    v = DppAdd<0x108, 0xF>(v);
    const uint32_t upper = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 16));
    const int32_t incl = static_cast<int32_t>(lane < 16 ? v + upper : v);
    if (active && lane_sum) lane_sum[j] = incl;
    if (lane == 0) *group_sum = incl;
  }
  return (q + 16 * kChunkWords * wraps - q0) / 8;
}

// A work-group takes four consecutive groups of one stream, a wave each; the waves past
// the stream's last group only help with the table.
__global__ __launch_bounds__(kChainWaves * 64, 4) void AnsChainKernel(KernelArgs a) {
  __shared__ __align__(16) AnsChainLds lds;
  const uint32_t lane = threadIdx.x & 63, wave = Uniform(threadIdx.x >> 6);
  const uint32_t lane_stream = 31 - (lane & 31);
  for (uint32_t w = blockIdx.x;; w += gridDim.x) {
    const Located loc = Locate(a, kStageChain, w, 0);
    if (!loc.valid) break;
    const CPtr<ImageDesc> d = DescAt(a, loc.img);
    const StreamUnit unit = StreamUnitAt(kChainGroups, d->groups[0], d->groups[1], d->groups[2], d->groups[3], loc.local);
    const uint32_t k = unit.k, g = unit.first + wave;
    const uint32_t G = d->groups[k], slen = d->stream_len[k], nv = d->nv;
    const __amdgpu_buffer_rsrc_t rs = MakeRsrc(d->streams[k], slen);
    uint32_t end_v = __builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(4 * g), 0, 0);
    uint32_t lo_v = __builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(4 * (g - 1)), 0, 0);
    const GPtr<const uint16_t> fr = Gbl<const uint16_t>(d->freqs + 512 * k);
    const uint32_t f = fr[threadIdx.x];
    asm volatile("" : "+v"(end_v), "+v"(lo_v));  // one wait for both: else the second load waits for g != 0
    const uint32_t end = Uniform(end_v), lo = g == 0 ? 4 * G : Uniform(lo_v);
    const bool ok = ((end | lo) & 3) == 0 && end <= slen && lo >= 4 * G && lo <= end &&
                    end - lo >= 4 * kLanesPerGroup;
    const bool in_stream = wave < unit.count;
    if (in_stream && !ok && lane == 0) atomicOr(a.err, kErrStreamOffsets);
    const bool active = in_stream && ok;
    const uint32_t x_word = __builtin_amdgcn_raw_buffer_load_b32(
        rs, static_cast<int>(end - 4 * kLanesPerGroup + 4 * lane_stream), 0, 0);
    const uint32_t x = active && lane < kLanesPerGroup ? x_word : 0u;
    const uint32_t p = active ? (end - 4 * kLanesPerGroup) >> 1 : 0u;
    const uint32_t plo = active ? lo >> 1 : 0u;
    const uint32_t top = p ? (p - 1) / kChunkWords : 0u, clo = plo / kChunkWords;
    const u32x2 c0 = LoadChunk(rs, top, clo, lane), c1 = LoadChunk(rs, top - 1, clo, lane);
    const u32x2 pE = LoadChunk(rs, top - 2, clo, lane), pO = LoadChunk(rs, top - 3, clo, lane);

    LdsBarrier();  // every wave is done with the previous unit's table and rings
    const bool table_ok = BuildTableInLds<kChainWaves * 64>(
        f, reinterpret_cast<uint32_t *>(&lds.ring[0][0]),
        [tab = &lds.tab[0]](uint32_t slot, const u32x2 &e) { tab[slot] = e; });
    if (!table_ok && threadIdx.x == 0) atomicOr(a.err, kErrFrequencies);
    if (!active) continue;
    u32x2 *const ring = lds.ring[wave];
    StoreChainChunk(lds.tab, ring, 0, false, lane, c0);
    StoreChainChunk(lds.tab, ring, kChunkWords, false, lane, c1);
    WaveSync();
    const GPtr<uint8_t> outp = Gbl<uint8_t>(d->symbols + SymbolOffset(nv, d->palette_bytes, k)) + static_cast<size_t>(g) * kGroupSyms;
    uint32_t y = x, q, used;
    if (k == 3) {
      const GPtr<int32_t> sums = Gbl<int32_t>(d->lane_sums);
      used = DecodeGroupChain<true>(lds, ring, rs, lane, kLanesPerGroup, y, q, p, clo, pE, pO, outp,
                                    Gbl<int32_t>(d->group_sums) + g, sums ? sums + g * kLanesPerGroup : nullptr,
                                    sums ? sums + LaneSuffixBase(nv) + g * kLanesPerGroup * 8 : nullptr);
    } else {
      used = DecodeGroupChain<false>(lds, ring, rs, lane, kLanesPerGroup, y, q, p, clo, pE, pO, outp,
                                     nullptr, nullptr, nullptr);
    }
    used += Popc64(__builtin_amdgcn_ballot_w64(lane < kLanesPerGroup && y < kStateL));  // the last renormalisation's
    if (used > p - plo && lane == 0) atomicOr(a.err, kErrStreamOffsets);
  }
}

// ---------------------------------------------------------------------------
// Stand-alone interleaved rANS groups of 1..32 streams, in the layout the reference's
// ANS decoder object packs (ans/ans_ocl.cpp:154-427) and its kernel reads
// (ans/ans_decode.cl:25-95): `groups` u32 end offsets, then per group its 16-bit
// renormalisation words in emission order followed by its n final states.  Same
// step as the texture path: slot = x & 2047, x = (x >> 11) f + slot - cum, and lanes
// with x < 2^15 take the next words in lane order.
//
// A wave per group, four to a work-group, decoding as AnsChainKernel does from the given
// table; lanes >= n never renormalise.  Words come from anywhere below the group's states
// (a pointer that runs below the data reads zeros); every global read is range-checked
// through a buffer resource.  Stream j of group g leaves its 256 symbols at
// out[(g n + j) 256 ..], the last decoded first.  status[g] is 1 for a malformed end
// offset or a group that does not end in the encoder's initial state 2^15, else 0; the
// output of a group with a malformed end offset is zeros.  data, out and status may be
// pinned host memory: every chunk is read once, two chunks ahead.
//
// 24 groups of 32 streams: 19.0 us with data, output and status in pinned memory, 16.4 with all
// of them in device memory, where a wave per group with two LDS round trips a step and the words
// copied to LDS two bytes a lane took 87 us.
__global__ __launch_bounds__(kChainWaves * 64, 4) void AnsGroupsKernel(const uint32_t *table, const uint8_t *data,
                                                                       uint32_t data_len, uint32_t groups,
                                                                       uint32_t n, uint8_t *out, uint32_t *status) {
  __shared__ __align__(16) AnsChainLds lds;
  const uint32_t lane = threadIdx.x & 63, wave = Uniform(threadIdx.x >> 6);
  const uint32_t g = blockIdx.x * kChainWaves + wave;
  const __amdgpu_buffer_rsrc_t rs = MakeRsrc(data, data_len);
  const uint32_t end = Uniform(__builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(4 * g), 0, 0));
  // The packed table, 8 entries a thread.
  const GPtr<const uint4> t = Gbl<const uint4>(table);
  const uint4 t0 = t[2 * threadIdx.x], t1 = t[2 * threadIdx.x + 1];
  const bool in = g < groups;
  const bool ok = in && (end & 3) == 0 && end <= data_len && end >= 4 * n;
  const uint32_t p = ok ? (end - 4 * n) / 2 : 0u;
  const uint32_t top = p ? (p - 1) / kChunkWords : 0u;
  const uint32_t x = __builtin_amdgcn_raw_buffer_load_b32(
      rs, static_cast<int>(ok && lane < n ? end - 4 * (lane + 1) : 0u), 0, 0);  // stream n - 1 - lane
  const u32x2 c0 = LoadChunk(rs, top, 0, lane), c1 = LoadChunk(rs, top - 1, 0, lane);
  const u32x2 pE = LoadChunk(rs, top - 2, 0, lane), pO = LoadChunk(rs, top - 3, 0, lane);
  const uint32_t packed[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i)
    lds.tab[8 * threadIdx.x + i] = u32x2{packed[i] & 0xFF000FFFu, (packed[i] >> 12) & (kTableSize - 1)};
  LdsBarrier();
  if (!in) return;
  GPtr<uint8_t> dst = Gbl<uint8_t>(out) + static_cast<size_t>(g) * n * kSymsPerLane;
  if (!ok) {
    for (uint32_t i = 4 * lane; i < n * kSymsPerLane; i += 256) *(GPtr<uint32_t>)(dst + i) = 0;
    if (lane == 0) Gbl<uint32_t>(status)[g] = 1;
    return;
  }
  u32x2 *const ring = lds.ring[wave];
  StoreChainChunk(lds.tab, ring, 0, false, lane, c0);
  StoreChainChunk(lds.tab, ring, kChunkWords, false, lane, c1);
  WaveSync();
  const bool active = lane < n;
  uint32_t y = active ? x : 0u, q;
  DecodeGroupChain<false>(lds, ring, rs, lane, n, y, q, p, 0, pE, pO, dst, nullptr, nullptr, nullptr);
  // The final state is 2^15: y itself, or y = 0 renormalised with the word 2^15, which its
  // ring entry tells from every other word (slot 0, 16 above it: an rANS step is one to one).
  const uint64_t ends = __builtin_amdgcn_ballot_w64(active && y < kStateL);
  const u32x2 e = ring[(q - LdsAddress(ring)) / 8 + __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(ends), 0u)];
  const uint32_t f = lds.tab[0].x & 0xFFFFFFu;
  const bool last = y >= kStateL ? y == kStateL
                                 : y == 0 && e.x == ((f << 5) | (lds.tab[0].x & 0xFF000000u)) && e.y == 16 * f;
  const uint64_t wrong = __builtin_amdgcn_ballot_w64(active && !last);
  if (lane == 0) Gbl<uint32_t>(status)[g] = wrong != 0 ? 1u : 0u;
}

// ---------------------------------------------------------------------------
// Stage 3: palette indices (codec/decode_indices.cl:6-84 composed by
// codec/decoder.cpp:304-393): idx[i] = sum_{j<=i} (diff[j] - 128), int32.
//
// One work-group per 8192-entry index group.  The group's starting value is the
// sum of the preceding groups' totals, which the rANS stage already produced, so
// the whole scan is one launch with no inter-work-group traffic.  Each thread
// scans 32 entries in registers, then wave and work-group scans join them.
__global__ __launch_bounds__(256) void DecodeIndicesKernel(KernelArgs a) {
  __shared__ uint32_t wtot[4];
  __shared__ uint32_t gprefix;
  const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (uint32_t u = blockIdx.x;; u += gridDim.x) {
    const Located loc = Locate(a, kStageIndices, u, 1);
    if (!loc.valid) break;
    const DevDesc d = LoadDesc(a, loc.img);
    const uint32_t g = loc.local;
    if (wave == 0) {
      uint32_t s = 0;
      for (uint32_t i = lane; i < g; i += 64) s += static_cast<uint32_t>(d.group_sums[i]);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
      if (lane == 0) gprefix = s;
    }
    const GPtr<const uint4> diffs =
        (GPtr<const uint4>)(d.symbols + SymbolOffset(d.nv, d.palette_bytes, 3) + static_cast<size_t>(g) * kGroupSyms + 32 * t);
    const uint4 q0 = diffs[0];
    const uint4 q1 = diffs[1];
    const uint32_t words[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    uint32_t run[32];
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      acc += ((words[i >> 2] >> (8 * (i & 3))) & 0xFFu) - 128u;
      run[i] = acc;
    }
    uint32_t incl = acc;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t n = __shfl_up(incl, off);
      if (lane >= static_cast<uint32_t>(off)) incl += n;
    }
    if (lane == 63) wtot[wave] = incl;
    __syncthreads();
    uint32_t offset = gprefix + incl - acc;
    for (uint32_t w = 0; w < wave; ++w) offset += wtot[w];
    const GPtr<uint4> dst = (GPtr<uint4>)(d.indices + static_cast<size_t>(g) * kGroupSyms + 32 * t);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      dst[i] = make_uint4(run[4 * i] + offset, run[4 * i + 1] + offset, run[4 * i + 2] + offset,
                          run[4 * i + 3] + offset);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Stage 4: inverse 5/3 wavelet (codec/inverse_wavelet.cl:14-192).
//
// A wave64 transforms four 32x32 tiles (two work units) at once: lane r of half-wave
// h holds row r of tile h of the first unit in the low 16 bits and row r of tile h
// of the second unit in the high 16 bits of 32 registers, so every add and shift is
// a packed 16-bit op over two tiles.  16 bits reproduce the reference's int32
// arithmetic exactly: inputs are symbol - 128 in [-128, 127]; a 1-D pass maps
// low-band bound Lo and high-band bound Hi to at most Lo + 1.5 Hi + 0.5 (the 5/3
// synthesis taps sum to 1 on the low band and 1.5 on the high band, truncation adds
// under 1), so a level (rows, then columns) adds at most 674 to the bound, every
// value after 5 levels stays within 128 + 5 * 674 = 3498 and every sum formed on the
// way within 2 * 3498 + 2.
//
// The row pass of each level is straight-line code with compile-time mirror
// indices; the column pass runs after a transpose through LDS (row stride 33
// words: conflict-free in both directions).  Levels len = 2..32 each transform rows
// y < len over x < len, then columns x < len over y < len, exactly the reference's
// transposed ping-pong.  A last transpose returns rows, whose low bytes leave as
// int8 in two 16-byte stores per tile row.
typedef int16_t s16x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ s16x2 AsPair(uint32_t w) { return __builtin_bit_cast(s16x2, w); }
__device__ __forceinline__ uint32_t Bits(s16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// C's truncating division of each half: negative values take divisor - 1 first.  Every
// sum divided here is within 2 * 3498 + 2 < 2^14 in magnitude (bound above), so bits
// 14 and 15 agree and the top two bits are the divisor - 1 (3) exactly when negative.
__device__ __forceinline__ s16x2 TruncDiv4(s16x2 s) {
  const u16x2 fix = __builtin_bit_cast(u16x2, s) >> static_cast<u16x2>(14);  // 0 or 3
  return (s + __builtin_bit_cast(s16x2, fix)) >> static_cast<s16x2>(2);
}
__device__ __forceinline__ s16x2 TruncDiv2(s16x2 s) {
  const u16x2 sign = __builtin_bit_cast(u16x2, s) >> static_cast<u16x2>(15);  // 0 or 1
  return (s + __builtin_bit_cast(s16x2, sign)) >> static_cast<s16x2>(1);
}

__host__ __device__ constexpr int Mirror(int idx, int range) {
  return (idx - static_cast<int>(idx >= range) * (idx - range + 2)) < 0
             ? -(idx - static_cast<int>(idx >= range) * (idx - range + 2))
             : (idx - static_cast<int>(idx >= range) * (idx - range + 2));
}

template <int LEN>
__device__ __forceinline__ void Inverse1D(s16x2 (&v)[kTileDim]) {
  constexpr int MID = LEN / 2;
  s16x2 e[LEN];
#pragma unroll
  for (int k = 0; k < MID; ++k) {
    const int p = MID + Mirror(2 * k - 1, LEN) / 2;
    const int n = MID + Mirror(2 * k + 1, LEN) / 2;
    e[2 * k] = v[k] - TruncDiv4(v[p] + v[n] + static_cast<s16x2>(2));
  }
#pragma unroll
  for (int k = 0; k < MID; ++k) {
    const int p = Mirror(2 * k, LEN);
    const int n = Mirror(2 * k + 2, LEN);
    e[2 * k + 1] = v[MID + k] + TruncDiv2(e[p] + e[n]);
  }
#pragma unroll
  for (int i = 0; i < LEN; ++i) v[i] = e[i];
}

constexpr int kLdsStride = kTileDim + 1;

// One level on the half-wave's tile pair; lanes r >= LEN sit out (their rows and
// columns are outside this level's square).  Each half-wave owns its LDS tile, so
// wave-level ordering is all the transposes need.  The level's result is left in L, row y
// at L[33 y], and with kReadBack in the rows again.
template <int LEN, bool kReadBack = true>
__device__ __forceinline__ void WaveletLevel(s16x2 (&v)[kTileDim], uint32_t *L, int r) {
  if (r < LEN) {
    Inverse1D<LEN>(v);
#pragma unroll
    for (int c = 0; c < LEN; ++c) L[r * kLdsStride + c] = Bits(v[c]);
  }
  WaveSync();
  if (r < LEN) {
#pragma unroll
    for (int c = 0; c < LEN; ++c) v[c] = AsPair(L[c * kLdsStride + r]);
  }
  WaveSync();
  if (r < LEN) {
    Inverse1D<LEN>(v);
#pragma unroll
    for (int c = 0; c < LEN; ++c) L[c * kLdsStride + r] = Bits(v[c]);
  }
  WaveSync();
  if (kReadBack) {
    if (r < LEN) {
#pragma unroll
      for (int c = 0; c < LEN; ++c) v[c] = AsPair(L[r * kLdsStride + c]);
    }
    WaveSync();
  }
}

// One pass of level LEN = 8 or 16 in L, by all 32 lanes of the half-wave: 32 / LEN lanes a
// line, each the outputs of N = LEN * LEN / 64 consecutive k.  `step` is the distance of a
// line's elements, `line` its start, `part` the lane's place in it.  The mirrored ends
// are other addresses for the first and last part: the neighbour before is lo and hi 0 of
// the line itself, the one after the last is the last again (its even output, recomputed
// from hi[k - 1] and hi[k]).
template <int LEN>
__device__ __forceinline__ void SplitPass(uint32_t *L, uint32_t line, uint32_t step, uint32_t part) {
  constexpr int MID = LEN / 2, N = LEN * LEN / 64;
  constexpr uint32_t kParts = MID / N;
  const uint32_t *const own = L + line + part * N * step;
  const uint32_t *const prev = part == 0 ? own : own - step;
  const bool end = part == kParts - 1;
  const uint32_t *const next = own + (end ? N - 1 : N) * step;
  s16x2 lo[N + 1], hi[N + 2];  // hi[j + 1] is hi of the lane's j-th k
#pragma unroll
  for (int j = 0; j < N; ++j) {
    lo[j] = AsPair(own[j * step]);
    hi[j + 1] = AsPair(own[(MID + j) * step]);
  }
  hi[0] = AsPair(prev[MID * step]);
  lo[N] = AsPair(next[0]);
  hi[N + 1] = AsPair(next[MID * step]);
  WaveSync();
  s16x2 even[N + 1];
#pragma unroll
  for (int j = 0; j < N; ++j) even[j] = lo[j] - TruncDiv4(hi[j] + hi[j + 1] + static_cast<s16x2>(2));
  const s16x2 before = end ? hi[N - 1] : hi[N];
  even[N] = lo[N] - TruncDiv4(before + hi[N + 1] + static_cast<s16x2>(2));
  uint32_t *const out = L + line + 2 * part * N * step;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    out[2 * j * step] = Bits(even[j]);
    out[(2 * j + 1) * step] = Bits(hi[j + 1] + TruncDiv2(even[j] + even[j + 1]));
  }
  WaveSync();
}

template <int LEN>
__device__ __forceinline__ void SplitLevel(uint32_t *L, uint32_t r) {
  constexpr uint32_t kParts = 32 / LEN;
  const uint32_t i = r / kParts, part = r % kParts;
  SplitPass<LEN>(L, i * kLdsStride, 1, part);
  SplitPass<LEN>(L, i, kLdsStride, part);
}

// Levels 2 to 16.  They touch the tile's first 16 rows and columns only, so a lane a row
// would leave half the lanes idle at level 16 and three quarters at level 8: those two run
// from L, with 2 and 4 lanes a line (140 fewer vector instructions a wave of some 1,090).
__device__ __forceinline__ void CoarseLevels(s16x2 (&v)[kTileDim], uint32_t *L, uint32_t r) {
  if (r < 16) {
#pragma unroll
    for (uint32_t c = 0; c < 16; ++c) L[r * kLdsStride + c] = Bits(v[c]);
  }
  WaveletLevel<2>(v, L, static_cast<int>(r));
  WaveletLevel<4, false>(v, L, static_cast<int>(r));
  uint32_t lane = r;
  asm volatile("" : "+v"(lane));  // addresses made here, not kept in registers between units
  SplitLevel<8>(L, lane);
  SplitLevel<16>(L, lane);
  if (r < 16) {
#pragma unroll
    for (uint32_t c = 0; c < 16; ++c) v[c] = AsPair(L[r * kLdsStride + c]);
  }
  WaveSync();
}

struct TileRef {
  GPtr<const uint8_t> src;  // tile-linear symbols (1024 bytes)
  GPtr<int8_t> dst;         // top-left of the tile in the raster plane
  uint32_t pitch;           // plane row length (blocks)
};

__device__ __forceinline__ TileRef TileAt(const DevDesc &d, uint32_t tile) {
  const uint32_t per_plane = d.nv / kTileSyms, tiles_x = d.bx / kTileDim;
  const uint32_t plane = tile / per_plane, t = tile - plane * per_plane;
  const uint32_t ty = t / tiles_x, tx = t - ty * tiles_x;
  const size_t base = static_cast<size_t>(plane) * d.nv;
  return {d.symbols + base + static_cast<size_t>(t) * kTileSyms,
          d.planes + base + static_cast<size_t>(ty) * kTileDim * d.bx + tx * kTileDim, d.bx};
}

// Tile `half` of wavelet unit `u`, if the unit exists (uniform address math, one
// select per lane; whole-wave call).
__device__ __forceinline__ bool WaveletTile(const KernelArgs &a, uint32_t u, uint32_t half, TileRef *t) {
  const Located loc = Locate(a, kStageWavelet, u, 1);
  if (!loc.valid) return false;
  const DevDesc d = LoadDesc(a, loc.img);
  const TileRef t0 = TileAt(d, loc.local * kWaveletTilesPerUnit);
  const TileRef t1 = TileAt(d, loc.local * kWaveletTilesPerUnit + 1);
  *t = half ? t1 : t0;
  return true;
}

// Row r of two tiles (a: 32 symbols of the first, b: of the second) as 16-bit pairs.
__device__ __forceinline__ void UnpackRowPair(const uint4 &a0, const uint4 &a1, const uint4 &b0, const uint4 &b1,
                                              s16x2 (&v)[kTileDim]) {
  const uint32_t wa[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
  const uint32_t wb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
  for (int i = 0; i < static_cast<int>(kTileDim); ++i) {
    // Byte i&3 of the first tile's word to bits 0-7, of the second's to bits
    // 16-23 (selector 0x0c is a zero byte), then remove the +128 bias.
    const uint32_t q = static_cast<uint32_t>(i & 3);
    const uint32_t sel = 0x0C000C00u | q | ((4u + q) << 16);
    v[i] = AsPair(__builtin_amdgcn_perm(wb[i >> 2], wa[i >> 2], sel)) - static_cast<s16x2>(128);
  }
}

// The pair's rows through the five levels, with this half-wave's transpose tile L;
// returns the rows' int8 results, 32 bytes each.
__device__ __forceinline__ void TransformRowPair(const uint4 &a0, const uint4 &a1, const uint4 &b0,
                                                 const uint4 &b1, uint32_t *L, uint32_t r, uint32_t (&oa)[8],
                                                 uint32_t (&ob)[8]) {
  s16x2 v[kTileDim];
  UnpackRowPair(a0, a1, b0, b1, v);
  CoarseLevels(v, L, r);
  WaveletLevel<32>(v, L, static_cast<int>(r));
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    // Low bytes of four pairs: t01 = (A0, A1, B0, B1), t23 = (A2, A3, B2, B3).
    const uint32_t t01 = __builtin_amdgcn_perm(Bits(v[4 * w + 1]), Bits(v[4 * w]), 0x06020400u);
    const uint32_t t23 = __builtin_amdgcn_perm(Bits(v[4 * w + 3]), Bits(v[4 * w + 2]), 0x06020400u);
    oa[w] = __builtin_amdgcn_perm(t23, t01, 0x05040100u);
    ob[w] = __builtin_amdgcn_perm(t23, t01, 0x07060302u);
  }
}

// The same, with the results left in L instead: the pair of row y, column x at L[33 y + x],
// each value wrapped to a signed byte as the reference's int8 planes hold it.  The column
// pass of the last level writes them there, so the rows are not read back.
__device__ __forceinline__ void TransformToLds(const uint4 &a0, const uint4 &a1, const uint4 &b0, const uint4 &b1,
                                               uint32_t *L, uint32_t r) {
  s16x2 v[kTileDim];
  UnpackRowPair(a0, a1, b0, b1, v);
  CoarseLevels(v, L, r);
  Inverse1D<kTileDim>(v);
#pragma unroll
  for (uint32_t c = 0; c < kTileDim; ++c) L[r * kLdsStride + c] = Bits(v[c]);
  WaveSync();
#pragma unroll
  for (uint32_t c = 0; c < kTileDim; ++c) v[c] = AsPair(L[c * kLdsStride + r]);
  WaveSync();
  Inverse1D<kTileDim>(v);
#pragma unroll
  for (uint32_t c = 0; c < kTileDim; ++c)
    L[c * kLdsStride + r] = Bits((v[c] << static_cast<s16x2>(8)) >> static_cast<s16x2>(8));
}

template <uint32_t WAVES>
__global__ __launch_bounds__(WAVES * 64) void InvWaveletKernel(KernelArgs a) {
  __shared__ uint32_t lds[WAVES][2][kTileDim * kLdsStride];
  const uint32_t lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
  const uint32_t wave = Uniform(threadIdx.x >> 6);
  uint32_t *L = lds[wave][half];
  const uint32_t stride = gridDim.x * WAVES;
  // The rows of the next pair are requested before the current pair is transformed,
  // so a wave's loads overlap its own lifting when it takes more than one pair.
  uint32_t pair = blockIdx.x * WAVES + wave;
  TileRef nlo{}, nhi{};
  uint4 na0{}, na1{}, nb0{}, nb1{};
  bool nhas_lo = WaveletTile(a, 2 * pair, half, &nlo);
  bool nhas_hi = nhas_lo && WaveletTile(a, 2 * pair + 1, half, &nhi);
  if (nhas_lo) {
    na0 = ((GPtr<const uint4>)(nlo.src + r * kTileDim))[0];
    na1 = ((GPtr<const uint4>)(nlo.src + r * kTileDim))[1];
    if (nhas_hi) {
      nb0 = ((GPtr<const uint4>)(nhi.src + r * kTileDim))[0];
      nb1 = ((GPtr<const uint4>)(nhi.src + r * kTileDim))[1];
    }
  }
  for (; nhas_lo; pair += stride) {
    const TileRef lo = nlo, hi = nhi;
    const bool has_hi = nhas_hi;
    const uint4 a0 = na0, a1 = na1;
    const uint4 b0 = nhas_hi ? nb0 : make_uint4(0, 0, 0, 0), b1 = nhas_hi ? nb1 : make_uint4(0, 0, 0, 0);
    const uint32_t next = pair + stride;
    nhas_lo = WaveletTile(a, 2 * next, half, &nlo);
    nhas_hi = nhas_lo && WaveletTile(a, 2 * next + 1, half, &nhi);
    if (nhas_lo) {
      na0 = ((GPtr<const uint4>)(nlo.src + r * kTileDim))[0];
      na1 = ((GPtr<const uint4>)(nlo.src + r * kTileDim))[1];
      if (nhas_hi) {
        nb0 = ((GPtr<const uint4>)(nhi.src + r * kTileDim))[0];
        nb1 = ((GPtr<const uint4>)(nhi.src + r * kTileDim))[1];
      }
    }
    uint32_t oa[8], ob[8];
    TransformRowPair(a0, a1, b0, b1, L, r, oa, ob);
    const GPtr<uint4> da = (GPtr<uint4>)(lo.dst + static_cast<size_t>(r) * lo.pitch);
    da[0] = make_uint4(oa[0], oa[1], oa[2], oa[3]);
    da[1] = make_uint4(oa[4], oa[5], oa[6], oa[7]);
    if (has_hi) {
      const GPtr<uint4> db = (GPtr<uint4>)(hi.dst + static_cast<size_t>(r) * hi.pitch);
      db[0] = make_uint4(ob[0], ob[1], ob[2], ob[3]);
      db[1] = make_uint4(ob[4], ob[5], ob[6], ob[7]);
    }
  }
}

// ---------------------------------------------------------------------------
// Stage 5: DXT1 assembly (codec/assemble.cl:14-81) and RGB8 assembly (:83-130).
//
// A thread assembles 4 consecutive blocks: one 4-byte load per plane, one 16-byte
// index load, 4 palette gathers and two 16-byte stores.  YCoCg -> RGB565 uses C
// truncating division; the pack keeps the low 16 bits of the int shifts.  A palette
// index outside the palette (corrupt input only) yields a zero word and raises
// kErrPaletteIndex instead of reading out of bounds.
__device__ __forceinline__ uint32_t Rgb565(int y, int co, int cg) {
  const int t = y - cg / 2;
  const int g = cg + t;
  const int b = (t - co) / 2;
  const int r = b + co;
  return ((static_cast<uint32_t>(r) << 11) | (static_cast<uint32_t>(g) << 5) |
          static_cast<uint32_t>(b)) & 0xFFFFu;
}

__device__ __forceinline__ int SByte(uint32_t w, int q) {
  return static_cast<int>(static_cast<int8_t>((w >> (8 * q)) & 0xFFu));
}

__global__ __launch_bounds__(256) void AssembleDxtKernel(KernelArgs a) {
  for (uint32_t u = blockIdx.x;; u += gridDim.x) {
    const Located loc = Locate(a, kStageAssemble, u, 1);
    if (!loc.valid) break;
    const DevDesc d = LoadDesc(a, loc.img);
    const uint32_t nv = d.nv;
    const size_t b0 = static_cast<size_t>(loc.local) * kAssembleBlocksPerUnit + 4 * threadIdx.x;
    uint32_t pw[6];
#pragma unroll
    for (int p = 0; p < 6; ++p)
      pw[p] = *(GPtr<const uint32_t>)(d.planes + static_cast<size_t>(p) * nv + b0);
    const int4 ix = *(GPtr<const int4>)(d.indices + b0);
    const GPtr<const uint32_t> pal = (GPtr<const uint32_t>)(d.symbols + SymbolOffset(d.nv, d.palette_bytes, 2));
    const uint32_t words = d.palette_bytes / 4;
    const int idx[4] = {ix.x, ix.y, ix.z, ix.w};
    uint32_t o[8];
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t ep1 = Rgb565(SByte(pw[0], q), SByte(pw[2], q), SByte(pw[3], q));
      const uint32_t ep2 = Rgb565(SByte(pw[1], q), SByte(pw[4], q), SByte(pw[5], q));
      const uint32_t pi = static_cast<uint32_t>(idx[q]);
      uint32_t word = 0;
      if (pi < words) word = pal[pi]; else bad = true;
      o[2 * q] = ep1 | (ep2 << 16);
      o[2 * q + 1] = word;
    }
    const GPtr<uint4> dst = (GPtr<uint4>)(d.out + 8 * b0);
    dst[0] = make_uint4(o[0], o[1], o[2], o[3]);
    dst[1] = make_uint4(o[4], o[5], o[6], o[7]);
    if (bad) atomicOr(a.err, kErrPaletteIndex);
  }
}

// Index scan fused into DXT1 assembly: one wave per 1024-block unit, which covers
// four 256-block segments of the index stream (one rANS lane each).  The value
// before the unit is the sum of the earlier groups' totals plus the sum before it
// within its group, both from the partial sums the rANS stage wrote; a segment is a
// 4-per-lane register prefix plus a wave scan.  The palette indices never go to
// memory, so a block costs 1 diff byte instead of 1 + 4 + 4 bytes of index traffic.
// Results are those of DecodeIndicesKernel followed by AssembleDxtKernel.
__device__ __forceinline__ int32_t WaveSum64(int32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Sum of (diff - 128) over the blocks of b's rANS group that come before block b
// (b a multiple of 32): the lane's inclusive prefix less the lane's suffix from b.
template <typename Desc>
__device__ __forceinline__ int32_t GroupLocalPrefix(const Desc &d, uint32_t b) {
  const uint32_t lane_ix = b / kSymsPerLane;  // group * 32 + lane
  const uint32_t k = (b % kSymsPerLane) / kRowBlocks;
  return d.lane_sums[lane_ix] - d.lane_sums[LaneSuffixBase(d.nv) + lane_ix * 8 + k];
}

template <uint32_t WAVES>
__global__ __launch_bounds__(WAVES * 64) void AssembleFusedKernel(KernelArgs a) {
  constexpr uint32_t kSegments = kAssembleBlocksPerUnit / kSymsPerLane;  // 4
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = Uniform(threadIdx.x >> 6);
  for (uint32_t u = blockIdx.x * WAVES + wave;; u += gridDim.x * WAVES) {
    const Located loc = Locate(a, kStageAssemble, u, 1);
    if (!loc.valid) break;
    const DevDesc d = LoadDesc(a, loc.img);
    const uint32_t nv = d.nv;
    const uint32_t b0 = loc.local * kAssembleBlocksPerUnit;
    const uint32_t g = b0 / kGroupSyms;
    int32_t base = 0;
    for (uint32_t i = lane; i < g; i += 64) base += d.group_sums[i];
    base = WaveSum64(base) + GroupLocalPrefix(d, b0);
    const GPtr<const uint8_t> diffs = d.symbols + SymbolOffset(d.nv, d.palette_bytes, 3);
    const GPtr<const uint32_t> pal = (GPtr<const uint32_t>)(d.symbols + SymbolOffset(d.nv, d.palette_bytes, 2));
    const uint32_t words = d.palette_bytes / 4;
    bool bad = false;
#pragma unroll
    for (uint32_t seg = 0; seg < kSegments; ++seg) {
      const uint32_t blk = b0 + seg * kSymsPerLane + 4 * lane;
      const uint32_t dw = *(GPtr<const uint32_t>)(diffs + blk);
      uint32_t pw[6];
#pragma unroll
      for (int p = 0; p < 6; ++p)
        pw[p] = *(GPtr<const uint32_t>)(d.planes + static_cast<size_t>(p) * nv + blk);
      int32_t run[4];
      int32_t acc = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc += static_cast<int32_t>((dw >> (8 * q)) & 0xFFu) - 128;
        run[q] = acc;
      }
      int32_t incl = acc;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int32_t n = __shfl_up(incl, off);
        if (lane >= static_cast<uint32_t>(off)) incl += n;
      }
      const int32_t before = base + incl - acc;
      base += __shfl(incl, 63);
      uint32_t o[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t ep1 = Rgb565(SByte(pw[0], q), SByte(pw[2], q), SByte(pw[3], q));
        const uint32_t ep2 = Rgb565(SByte(pw[1], q), SByte(pw[4], q), SByte(pw[5], q));
        const uint32_t pi = static_cast<uint32_t>(before + run[q]);
        uint32_t word = 0;
        if (pi < words) word = pal[pi]; else bad = true;
        o[2 * q] = ep1 | (ep2 << 16);
        o[2 * q + 1] = word;
      }
      const GPtr<uint4> dst = (GPtr<uint4>)(d.out + 8 * static_cast<size_t>(blk));
      dst[0] = make_uint4(o[0], o[1], o[2], o[3]);
      dst[1] = make_uint4(o[4], o[5], o[6], o[7]);
    }
    if (bad) atomicOr(a.err, kErrPaletteIndex);
  }
}

// The same unit with 16 consecutive blocks per lane: 16-byte loads of the diffs and
// of each plane, one wave scan per unit, 128 contiguous output bytes per lane.
__device__ __forceinline__ uint32_t ByteOf(const uint4 &v, int q) {
  const uint32_t w = q < 4 ? v.x : q < 8 ? v.y : q < 12 ? v.z : v.w;
  return (w >> (8 * (q & 3))) & 0xFFu;
}

template <uint32_t WAVES>
__global__ __launch_bounds__(WAVES * 64) void AssembleFusedWideKernel(KernelArgs a) {
  constexpr uint32_t kPerLane = kAssembleBlocksPerUnit / 64;  // 16
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = Uniform(threadIdx.x >> 6);
  for (uint32_t u = blockIdx.x * WAVES + wave;; u += gridDim.x * WAVES) {
    const Located loc = Locate(a, kStageAssemble, u, 1);
    if (!loc.valid) break;
    const DevDesc d = LoadDesc(a, loc.img);
    const uint32_t nv = d.nv;
    const uint32_t b0 = loc.local * kAssembleBlocksPerUnit;
    const uint32_t blk = b0 + kPerLane * lane;
    const uint4 dv = *(GPtr<const uint4>)(d.symbols + SymbolOffset(d.nv, d.palette_bytes, 3) + blk);
    uint4 pv[6];
#pragma unroll
    for (int p = 0; p < 6; ++p)
      pv[p] = *(GPtr<const uint4>)(d.planes + static_cast<size_t>(p) * nv + blk);
    const uint32_t g = b0 / kGroupSyms;
    int32_t base = 0;
    for (uint32_t i = lane; i < g; i += 64) base += d.group_sums[i];
    base = WaveSum64(base) + GroupLocalPrefix(d, b0);
    int32_t run[kPerLane];
    int32_t acc = 0;
#pragma unroll
    for (int q = 0; q < static_cast<int>(kPerLane); ++q) {
      acc += static_cast<int32_t>(ByteOf(dv, q)) - 128;
      run[q] = acc;
    }
    int32_t incl = acc;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t n = __shfl_up(incl, off);
      if (lane >= static_cast<uint32_t>(off)) incl += n;
    }
    const int32_t before = base + incl - acc;
    const GPtr<const uint32_t> pal = (GPtr<const uint32_t>)(d.symbols + SymbolOffset(d.nv, d.palette_bytes, 2));
    const uint32_t words = d.palette_bytes / 4;
    bool bad = false;
    const GPtr<uint4> dst = (GPtr<uint4>)(d.out + 8 * static_cast<size_t>(blk));
#pragma unroll
    for (int i = 0; i < static_cast<int>(kPerLane) / 2; ++i) {
      uint32_t o[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int q = 2 * i + h;
        const int32_t y1 = static_cast<int8_t>(ByteOf(pv[0], q)), y2 = static_cast<int8_t>(ByteOf(pv[1], q));
        const int32_t co1 = static_cast<int8_t>(ByteOf(pv[2], q)), cg1 = static_cast<int8_t>(ByteOf(pv[3], q));
        const int32_t co2 = static_cast<int8_t>(ByteOf(pv[4], q)), cg2 = static_cast<int8_t>(ByteOf(pv[5], q));
        const uint32_t pi = static_cast<uint32_t>(before + run[q]);
        uint32_t word = 0;
        if (pi < words) word = pal[pi]; else bad = true;
        o[2 * h] = Rgb565(y1, co1, cg1) | (Rgb565(y2, co2, cg2) << 16);
        o[2 * h + 1] = word;
      }
      dst[i] = make_uint4(o[0], o[1], o[2], o[3]);
    }
    if (bad) atomicOr(a.err, kErrPaletteIndex);
  }
}

// Rgb565 of both endpoints of a block at once, endpoint 1 in the low and endpoint 2 in
// the high half: the same truncating divisions and the same low 16 bits of the shifts
// (|y|, |co|, |cg| <= 128, so every intermediate fits 16 bits).
struct EndPair {
  s16x2 r, g, b;
};
__device__ __forceinline__ EndPair EndpointPair(uint32_t y, uint32_t co, uint32_t cg) {
  asm volatile("" : "+v"(cg));  // else cg / 2 is split into two 16-bit halves and re-packed
  const s16x2 t = AsPair(y) - TruncDiv2(AsPair(cg));
  EndPair e;
  e.g = AsPair(cg) + t;
  e.b = TruncDiv2(t - AsPair(co));
  e.r = e.b + AsPair(co);
  return e;
}
__device__ __forceinline__ uint32_t Rgb565Pair(uint32_t y, uint32_t co, uint32_t cg) {
  const EndPair e = EndpointPair(y, co, cg);
  return Bits(e.r << static_cast<s16x2>(11)) | Bits(e.g << static_cast<s16x2>(5)) | Bits(e.b);
}

// The four colours of a block (codec/assemble.cl:83-130) as three words, one a channel: byte
// i of rgb[c] is channel c of colour i.  Both endpoints go through the 16-bit halves of a
// register (|r|, |b| <= 288 and |g| <= 319 before the shifts, so every 16-bit result is the
// int32 one); the two between are thirds in C's truncating division: for |s| < 2^15,
// s * 21846 >> 16 is the floor of s / 3, off from it by under a third of a step, and 1 less
// than the truncation when s is negative.
__device__ __forceinline__ uint32_t Third(int32_t s) {
  return static_cast<uint32_t>((__mul24(s, 21846) >> 16) + static_cast<int32_t>(static_cast<uint32_t>(s) >> 31));
}

__device__ __forceinline__ uint32_t FourColours(s16x2 ends) {
  const uint32_t e = Bits(ends);
  const int32_t a = static_cast<int16_t>(e & 0xFFFFu), b = static_cast<int32_t>(e) >> 16;
  const uint32_t between = __builtin_amdgcn_perm(Third(a + 2 * b), Third(2 * a + b), 0x0C0C0400u);
  return __builtin_amdgcn_perm(between, e, 0x05040200u);
}

__device__ __forceinline__ void BlockColours(uint32_t y, uint32_t co, uint32_t cg, uint32_t (&rgb)[3]) {
  const EndPair e = EndpointPair(y, co, cg);
  rgb[0] = FourColours((e.r << static_cast<s16x2>(3)) | (e.r >> static_cast<s16x2>(2)));
  rgb[1] = FourColours((e.g << static_cast<s16x2>(2)) | (e.g >> static_cast<s16x2>(4)));
  rgb[2] = FourColours((e.b << static_cast<s16x2>(3)) | (e.b >> static_cast<s16x2>(2)));
}

// One texel row of a block, 4 texels of RGB8 in three words: the row's four 2-bit indices
// become the byte selectors of v_perm, which picks four texels of a channel at once.
__device__ __forceinline__ void BlockRow(const uint32_t (&rgb)[3], uint32_t word, uint32_t row, uint32_t *out) {
  const uint32_t idx = (word >> (8 * row)) & 0xFFu, pairs = idx | (idx << 6);
  const uint32_t sel = (pairs | (pairs << 12)) & 0x03030303u;
  const uint32_t r = __builtin_amdgcn_perm(0u, rgb[0], sel);
  const uint32_t g = __builtin_amdgcn_perm(0u, rgb[1], sel);
  const uint32_t b = __builtin_amdgcn_perm(0u, rgb[2], sel);
  // r0 g0 b0 r1 | g1 b1 r2 g2 | b2 r3 g3 b3: selector codes 0-3 are bytes of the second
  // operand, 4-7 of the first.
  const uint32_t rg01 = __builtin_amdgcn_perm(g, r, 0x05010400u);  // r0 g0 r1 g1
  const uint32_t rg23 = __builtin_amdgcn_perm(g, r, 0x07030602u);  // r2 g2 r3 g3
  out[0] = __builtin_amdgcn_perm(b, rg01, 0x02040100u);
  out[1] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(b, rg01, 0x0C0C0503u), rg23, 0x01000504u);
  out[2] = __builtin_amdgcn_perm(b, rg23, 0x07030206u);
}

// 16 bytes to an address that is a multiple of 4 (RGB8 output has no wider guarantee).
typedef uint32_t u32x4Words __attribute__((ext_vector_type(4), aligned(4)));

// Stages 4 and 5 in one kernel: inverse wavelet, index scan and assembly of two
// tile positions per work-group, so the int8 planes never leave LDS (the planes
// buffer's write and read, 12 bytes a block, are the traffic this saves).
//
// A work unit is two consecutive assembly units of one image, i.e. tile positions
// t0 and t0 + 1 of the per-plane raster tile order (every plane has a multiple of 8
// tiles, so pairs never straddle images).  Wave 0 transforms the Y planes, wave 1 the Co
// and wave 2 the Cg planes, endpoint 1's in the low and endpoint 2's in the high 16 bits,
// position t0 in the lower and t0 + 1 in the upper half-wave, with the arithmetic of
// InvWaveletKernel, and leaves the values in its transpose space.  A block's three words
// there are then what the endpoint conversion takes for both endpoints at once, with
// nothing packed or unpacked in between.  After a work-group barrier the waves assemble
// the tile rows: a lane takes four blocks, whose palette indices are the row's base plus
// a scan of the diffs over 8 lanes.  A row's base is the earlier groups' totals (one
// 64-lane scan of the group sums of the groups the unit's rows touch, when at most 64;
// else a per-row reduction) plus the sum before the row within its group.
constexpr uint32_t kTileFusedWaves = 3;

// Tile positions t0 and t0 + 1 of an image: what the fused kernel needs of its descriptor,
// the first position's tile row and column, and the index-stream groups its rows touch,
// g_min .. g_min + g_span.
struct TilePair {
  uint32_t nv, bx, tiles_x, palette_bytes;
  uint32_t t0, ty0, tx0, g_min, g_span;
  GPtr<uint8_t> symbols;
  GPtr<int32_t> group_sums;
  GPtr<int32_t> lane_sums;
  GPtr<uint8_t> out;
};

__device__ __forceinline__ TilePair PairAt(CPtr<ImageDesc> d, uint32_t t0) {
  TilePair p;
  p.nv = d->nv;
  p.bx = d->bx;
  p.tiles_x = p.bx / kTileDim;
  p.palette_bytes = d->palette_bytes;
  p.t0 = t0;
  p.ty0 = TileRowOf(t0, d->tile_mul);
  p.tx0 = t0 - p.ty0 * p.tiles_x;
  const bool wraps = p.tx0 + 1 == p.tiles_x;
  const uint32_t ty1 = wraps ? p.ty0 + 1 : p.ty0, tx1 = wraps ? 0 : p.tx0 + 1;
  p.g_min = (p.ty0 * kTileDim * p.bx + p.tx0 * kTileDim) / kGroupSyms;
  p.g_span = ((ty1 * kTileDim + kTileDim - 1) * p.bx + tx1 * kTileDim) / kGroupSyms - p.g_min;
  p.symbols = Gbl<uint8_t>(d->symbols);
  p.group_sums = Gbl<int32_t>(d->group_sums);
  p.lane_sums = Gbl<int32_t>(d->lane_sums);
  p.out = Gbl<uint8_t>(d->out);
  return p;
}

// kRgb writes RGB8 instead of DXT1 blocks: the same planes, indices and palette words, a
// lane's four blocks being 48 bytes of four texel rows each.  Bound by its writes (48 bytes
// a block of 55): 32 2048x2048 textures in 115.8 us (4.0 TB/s), where the index scan, the
// wavelet and AssembleRgbKernel took 17.3 + 38.3 + 370.1 us, the last one a texel's byte
// at a time in the vector unit; six mixed textures (5.2 Mtexel) 14.4 us against 4.9 + 6.9
// + 23.8.
//
// A unit starts with three dependent trips to memory (plan, descriptor, rows and sums), two
// thirds of the transform's own time.  So the plan's prefix is in LDS, the next unit's
// descriptor and loads go out while this one is assembled, where the transform's registers
// are free, and all sums over lanes are DPP: the batch of 128 textures 55.1 -> 53.0 us, 24
// textures 15.6 -> 14.4.  From there on the vector unit bounds it (22.1 M instructions, 42
// of the 53 us at 4.5 waves a SIMD): pairs of planes that the conversion takes as they lie,
// no read back of the last level's rows, addresses with a scalar base, signed dot products
// for the running indices and the palette's range check in the buffer: 20.8 M, 49.6 us (24
// textures 13.4, one 512x512 image 7.6 -> 7.0, 4096x4096 11.4 -> 10.3); with the coarse
// levels by all lanes (SplitPass) 19.2 M, 47.2 us (12.8, 6.7, 10.1).
//
// At most 96 VGPRs: 5 waves per SIMD, about what the 26 KiB of LDS allows.
template <bool kRgb>
__global__ __launch_bounds__(kTileFusedWaves * 64, 5) void WaveletAssembleKernel(KernelArgs a) {
  __shared__ uint32_t lds[kTileFusedWaves][2][kTileDim * kLdsStride];
  __shared__ uint32_t prefix[kPrefixInRegs];
  const uint32_t lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
  const uint32_t wave = Uniform(threadIdx.x >> 6);
  uint32_t *const L = lds[wave][half];
  // The plan's prefix once per work-group, so that finding a unit costs no round trip to
  // memory; requested together with the unit count.
  const bool in_lds = a.plan != nullptr && a.plan_cap + 1 <= kPrefixInRegs;
  if (in_lds) {
    const GPtr<const uint32_t> pre =
        Gbl<const uint32_t>(reinterpret_cast<const uint8_t *>(a.plan) + PlanPrefixOffset(a.plan_cap, kStageAssemble));
    for (uint32_t i = threadIdx.x; i < kPrefixInRegs; i += kTileFusedWaves * 64)
      prefix[i] = i <= a.plan_cap ? pre[i] : kPrefixPad;
  }
  // Work units are pairs of assembly units (every image has an even number of them).
  const uint32_t pairs = (a.plan ? ((CPtr<PlanHeader>)(reinterpret_cast<uintptr_t>(a.plan)))->units[kStageAssemble]
                                 : StageUnitsOf(a.single, kStageAssemble, 1)) / 2;
  const XcdSpan span = XcdBalanced(blockIdx.x, gridDim.x, pairs);
  if (in_lds) LdsBarrier();
  uint32_t img = 0, t0 = 0;  // of the unit requested last
  uint4 a0, a1, b0, b1;
  int32_t gs = 0, gb = 0;
  // The unit's descriptor, and its loads that do not depend on anything else: row r of the
  // wave's two planes (Y1, Y2; Co1, Co2; Cg1, Cg2) for the half's position, the group totals
  // from g_min on and those before it.
  const uint32_t plane1 = wave == 0 ? 0u : wave + 1, planes_apart = wave == 0 ? 1u : 2u;
  const auto request = [&](uint32_t u) {
    Located loc;
    if (in_lds) {
      const uint32_t v[4] = {prefix[lane], prefix[lane + 64], prefix[lane + 128], prefix[lane + 192]};
      loc = LocateIn(v, 2 * u);
    } else {
      loc = Locate(a, kStageAssemble, 2 * u, 1);
    }
    img = Uniform(loc.img);
    t0 = Uniform(loc.local);
    const TilePair nxt = PairAt(DescAt(a, img), t0);
    const GPtr<const uint8_t> src = nxt.symbols + static_cast<size_t>(plane1) * nxt.nv + nxt.t0 * kTileSyms;
    const GPtr<const uint8_t> src2 = src + static_cast<size_t>(planes_apart) * nxt.nv;
    const uint32_t at = half * kTileSyms + r * kTileDim;
    a0 = ((GPtr<const uint4>)(src + at))[0], a1 = ((GPtr<const uint4>)(src + at))[1];
    b0 = ((GPtr<const uint4>)(src2 + at))[0], b1 = ((GPtr<const uint4>)(src2 + at))[1];
    if (nxt.g_span < 64) {
      gs = lane <= nxt.g_span ? nxt.group_sums[nxt.g_min + lane] : 0;
      gb = lane < nxt.g_min ? nxt.group_sums[lane] : 0;
    }
  };
  if (span.first < span.end) request(span.first);
  for (uint32_t u = span.first; u < span.end; u += span.stride) {
    // Read again from the scalar cache rather than carried: two units' descriptors would not
    // fit the scalar registers.
    const TilePair cur = PairAt(DescAt(a, Uniform(img)), Uniform(t0));
    const uint32_t nv = cur.nv, bx = cur.bx;
    const uint32_t ty0 = cur.ty0, tx0 = cur.tx0;
    const bool wraps = tx0 + 1 == cur.tiles_x;
    const uint32_t ty1 = wraps ? ty0 + 1 : ty0, tx1 = wraps ? 0 : tx0 + 1;
    const uint32_t g_min = cur.g_min;
    const bool few_groups = cur.g_span < 64;
    // Totals of the groups before each of the (at most 64) groups the rows touch: lane i
    // holds the sum over groups < g_min + i.
    int32_t gpre = 0;
    if (few_groups) {
      int32_t before = gb;
      if (g_min > 64) {
        uint32_t i = lane + 64;
        asm volatile("" : "+v"(i));  // made here: kept through the unit loop, it was spilled
        for (; i < g_min; i += 64) before += cur.group_sums[i];
      }
      before = static_cast<int32_t>(WaveTotal(static_cast<uint32_t>(before)));
      gpre = before + static_cast<int32_t>(WaveInclusiveSum(static_cast<uint32_t>(gs))) - gs;
    }

    TransformToLds(a0, a1, b0, b1, L, r);
    LdsBarrier();
    // The next unit's loads are in flight while this one is assembled (the registers of the
    // transform are free now).
    if (u + span.stride < span.end) request(u + span.stride);

    const GPtr<const uint8_t> diffs = cur.symbols + 6 * static_cast<size_t>(nv) + cur.palette_bytes;
    const GPtr<const uint8_t> lane_sums = (GPtr<const uint8_t>)cur.lane_sums;
    const GPtr<const uint8_t> suffixes = lane_sums + 4 * static_cast<size_t>(LaneSuffixBase(nv));
    const __amdgpu_buffer_rsrc_t pal =
        MakeRsrc(reinterpret_cast<const void *>((uintptr_t)(cur.symbols + 6 * static_cast<size_t>(nv))), cur.palette_bytes);
    const uint32_t words = cur.palette_bytes / 4;
    uint32_t worst = 0;  // the largest palette index
    // 64 tile rows (2 positions x 32) in row groups of 8: lane l takes blocks
    // 4 (l % 8) .. +3 of row l / 8 of its group, and wave w groups w, w + 3, w + 6
    // (< 8).  Each phase runs over all of a wave's groups, so their loads are in
    // flight together: diffs and row bases, then palette words, then the stores.  What
    // depends on the group alone is scalar, so that a load takes its address from a
    // scalar base and one 32-bit offset.
    constexpr uint32_t kGroupsOfRows = 2 * kTileDim / 8;
    constexpr uint32_t kSteps = (kGroupsOfRows + kTileFusedWaves - 1) / kTileFusedWaves;  // 3
    const uint32_t sub = lane >> 3, xb = 4 * (lane & 7);
    const int32_t from1 = (lane & 7) >= 1 ? -1 : 0, from2 = (lane & 7) >= 2 ? -1 : 0;
    const uint32_t row_off = sub * bx, blk_off = row_off + xb;
    uint32_t group0[kSteps], dw[kSteps];  // first block of the row group; the lane's four diffs
    int32_t base[kSteps];
#pragma unroll
    for (uint32_t i = 0; i < kSteps; ++i) {
      const uint32_t grp0 = wave + kTileFusedWaves * i;
      const uint32_t grp = grp0 < kGroupsOfRows ? grp0 : wave;  // a spare step repeats group `wave`
      const uint32_t P = grp / 4, ty = P ? ty1 : ty0, tx = P ? tx1 : tx0;
      group0[i] = (ty * kTileDim + 8 * (grp & 3)) * bx + tx * kTileDim;
      dw[i] = *(GPtr<const uint32_t>)(diffs + group0[i] + blk_off) ^ 0x80808080u;  // signed bytes: diff - 128
      const uint32_t row0 = group0[i] + row_off;
      const uint32_t g = row0 / kGroupSyms;
      int32_t before;
      if (few_groups) {
        before = __shfl(gpre, static_cast<int>(g - g_min));
      } else {
        before = 0;
        for (uint32_t k = xb / 4; k < g; k += 8) before += cur.group_sums[k];
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) before += __shfl_xor(before, off, 8);
      }
      // GroupLocalPrefix: entries row0 / 256 and row0 / 32 (row0 is a multiple of 32).
      base[i] = before + *(GPtr<const int32_t>)(lane_sums + row0 / kSymsPerLane * 4) -
                *(GPtr<const int32_t>)(suffixes + row0 / kRowBlocks * 4);
    }
    uint32_t word[kSteps][4];
#pragma unroll
    for (uint32_t i = 0; i < kSteps; ++i) {
      // Inclusive sum over 8 lanes: row shifts, with a lane's reach past its 8 masked off.
      const int32_t total = __builtin_amdgcn_sdot4(static_cast<int>(dw[i]), 0x01010101, 0, false);
      int32_t incl = total;
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xF, 0xF, true) & from1;
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xF, 0xF, true) & from2;
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xF, 0xA, true);  // into lanes 4-7 of each 8
      const int32_t start = base[i] + incl - total;
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        // The sum of the first k + 1 diffs on top of `start`.
        const uint32_t pi = static_cast<uint32_t>(
            __builtin_amdgcn_sdot4(static_cast<int>(dw[i]), static_cast<int>(0x01010101u >> (24 - 8 * k)), start, false));
        worst = max(worst, pi);
        // An index outside the palette reads a zero word through the buffer's range check.
        word[i][k] = __builtin_amdgcn_raw_buffer_load_b32(pal, static_cast<int>(min(pi, words) * 4), 0, 0);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < kSteps; ++i) {
      const uint32_t grp = wave + kTileFusedWaves * i;
      if (grp >= kGroupsOfRows) continue;
      const uint32_t P = grp / 4;
      const uint32_t at = (8 * (grp & 3) + sub) * kLdsStride + xb;
      uint32_t pw[3][4];
#pragma unroll
      for (uint32_t p = 0; p < 3; ++p)
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) pw[p][k] = lds[p][P][at + k];
      if constexpr (kRgb) {
        uint32_t rgb[4][3];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) BlockColours(pw[0][k], pw[1][k], pw[2][k], rgb[k]);
        // Byte 48 of a block, 12 of it a texel row; a texel row of the image is 12 bx bytes.
        const uint32_t tx = P ? tx1 : tx0, ty = P ? ty1 : ty0;
        GPtr<uint8_t> row = cur.out + 48 * static_cast<size_t>(ty * kTileDim + 8 * (grp & 3)) * bx + 12 * tx * kTileDim;
        const uint32_t off = 48 * row_off + 12 * xb;
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
          uint32_t o[12];
#pragma unroll
          for (uint32_t k = 0; k < 4; ++k) BlockRow(rgb[k], word[i][k], t, o + 3 * k);
          const GPtr<u32x4Words> dst = (GPtr<u32x4Words>)(row + off);
#pragma unroll
          for (uint32_t k = 0; k < 3; ++k) dst[k] = u32x4Words{o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]};
          row += 12 * static_cast<size_t>(bx);
        }
      } else {
        uint32_t o[8];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          o[2 * k] = Rgb565Pair(pw[0][k], pw[1][k], pw[2][k]);
          o[2 * k + 1] = word[i][k];
        }
        const GPtr<uint4> dst = (GPtr<uint4>)(cur.out + 8 * static_cast<size_t>(group0[i]) + 8 * blk_off);
        dst[0] = make_uint4(o[0], o[1], o[2], o[3]);
        dst[1] = make_uint4(o[4], o[5], o[6], o[7]);
      }
    }
    const bool bad = worst >= words;
    if (bad) atomicOr(a.err, kErrPaletteIndex);
    LdsBarrier();  // the next unit's transposes reuse the tiles' space
  }
}

__global__ __launch_bounds__(256) void AssembleRgbKernel(KernelArgs a) {
  for (uint32_t u = blockIdx.x;; u += gridDim.x) {
    const Located loc = Locate(a, kStageAssemble, u, 1);
    if (!loc.valid) break;
    const DevDesc d = LoadDesc(a, loc.img);
    const uint32_t nv = d.nv;
    const size_t b0 = static_cast<size_t>(loc.local) * kAssembleBlocksPerUnit + 4 * threadIdx.x;
    uint32_t pw[6];
#pragma unroll
    for (int p = 0; p < 6; ++p)
      pw[p] = *(GPtr<const uint32_t>)(d.planes + static_cast<size_t>(p) * nv + b0);
    const int4 ix = *(GPtr<const int4>)(d.indices + b0);
    const GPtr<const uint32_t> pal = (GPtr<const uint32_t>)(d.symbols + SymbolOffset(d.nv, d.palette_bytes, 2));
    const uint32_t words = d.palette_bytes / 4;
    const int idx[4] = {ix.x, ix.y, ix.z, ix.w};
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int pal8[4][3];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int y = SByte(pw[e], q), co = SByte(pw[2 + 2 * e], q), cg = SByte(pw[3 + 2 * e], q);
        const int t = y - cg / 2;
        const int g = cg + t;
        const int b = (t - co) / 2;
        const int r = b + co;
        pal8[e][0] = static_cast<int>((static_cast<uint32_t>(r) << 3) | static_cast<uint32_t>(r >> 2));
        pal8[e][1] = static_cast<int>((static_cast<uint32_t>(g) << 2) | static_cast<uint32_t>(g >> 4));
        pal8[e][2] = static_cast<int>((static_cast<uint32_t>(b) << 3) | static_cast<uint32_t>(b >> 2));
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        pal8[2][c] = (2 * pal8[0][c] + pal8[1][c]) / 3;
        pal8[3][c] = (pal8[0][c] + 2 * pal8[1][c]) / 3;
      }
      const uint32_t pi = static_cast<uint32_t>(idx[q]);
      uint32_t word = 0;
      if (pi < words) word = pal[pi]; else bad = true;
      const size_t blk = b0 + q;
      const uint32_t bxi = static_cast<uint32_t>(blk % d.bx), byi = static_cast<uint32_t>(blk / d.bx);
#pragma unroll
      for (int row = 0; row < 4; ++row) {
        uint32_t bytes[12];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int sel = (word >> (2 * (4 * row + c))) & 3;
          bytes[3 * c + 0] = static_cast<uint32_t>(pal8[sel][0]) & 0xFFu;
          bytes[3 * c + 1] = static_cast<uint32_t>(pal8[sel][1]) & 0xFFu;
          bytes[3 * c + 2] = static_cast<uint32_t>(pal8[sel][2]) & 0xFFu;
        }
        const GPtr<uint32_t> dst =
            (GPtr<uint32_t>)(d.out + 3 * (static_cast<size_t>(d.width) * (4 * byi + row) + 4 * bxi));
#pragma unroll
        for (int w = 0; w < 3; ++w)
          dst[w] = bytes[4 * w] | (bytes[4 * w + 1] << 8) | (bytes[4 * w + 2] << 16) |
                   (bytes[4 * w + 3] << 24);
      }
    }
    if (bad) atomicOr(a.err, kErrPaletteIndex);
  }
}

template <uint32_t WAVES, uint32_t GPW, bool kBuild = false>
hipError_t LaunchAns(const KernelArgs &args, uint32_t grid, hipStream_t stream) {
  hipLaunchKernelGGL((AnsDecodeKernel<WAVES, GPW, kBuild>), dim3(grid), dim3(WAVES * 64), 0, stream, args);
  return hipGetLastError();
}

}  // namespace

hipError_t LaunchStage(uint32_t stage, const KernelArgs &args, uint32_t grid,
                       const StageConfig &cfg, hipStream_t stream) {
  if (grid == 0) return hipSuccess;
  switch (stage) {
    case kStageTables:
      if (cfg.ans_build_tables) return hipSuccess;  // the rANS kernel builds them in LDS
      hipLaunchKernelGGL(BuildTableKernel, dim3(grid), dim3(256), 0, stream, args);
      return hipGetLastError();
    case kStageAns: {
      const uint32_t w = cfg.ans_waves, g = cfg.ans_groups_per_wave;
      if (cfg.ans_auto) {
        // The form travels in the plan (or in args.ans_unit_code for a single image).
        if (!cfg.ans_build_tables || g != 2 || w != kAutoWaves) return hipErrorInvalidValue;
        if (cfg.ans_chain)
          hipLaunchKernelGGL(AnsChainKernel, dim3(grid), dim3(kChainWaves * 64), 0, stream, args);
        else
          hipLaunchKernelGGL(AnsAutoKernel, dim3(grid), dim3(kAutoWaves * 64), 0, stream, args);
        return hipGetLastError();
      }
      if (cfg.ans_pair_short) return hipErrorInvalidValue;  // paired units run in AnsAutoKernel
      if (cfg.ans_build_tables) {
        if (g == 2 && w == 4) return LaunchAns<4, 2, true>(args, grid, stream);
        if (g == 2 && w == 8) return LaunchAns<8, 2, true>(args, grid, stream);
        if (g == 1 && w == 4) return LaunchAns<4, 1, true>(args, grid, stream);
        if (g == 1 && w == 8) return LaunchAns<8, 1, true>(args, grid, stream);
        return hipErrorInvalidValue;
      }
      if (g == 2 && w == 1) return LaunchAns<1, 2>(args, grid, stream);
      if (g == 2 && w == 2) return LaunchAns<2, 2>(args, grid, stream);
      if (g == 2 && w == 4) return LaunchAns<4, 2>(args, grid, stream);
      if (g == 2 && w == 8) return LaunchAns<8, 2>(args, grid, stream);
      if (g == 1 && w == 2) return LaunchAns<2, 1>(args, grid, stream);
      if (g == 1 && w == 4) return LaunchAns<4, 1>(args, grid, stream);
      if (g == 1 && w == 8) return LaunchAns<8, 1>(args, grid, stream);
      return hipErrorInvalidValue;
    }
    case kStageIndices:
      if (cfg.fused_waves || cfg.tile_fused) return hipSuccess;  // the assembly scans them itself
      hipLaunchKernelGGL(DecodeIndicesKernel, dim3(grid), dim3(256), 0, stream, args);
      return hipGetLastError();
    case kStageWavelet:
      if (cfg.tile_fused) return hipSuccess;  // inside the assembly
      if (cfg.wavelet_waves == 1)
        hipLaunchKernelGGL(InvWaveletKernel<1>, dim3(grid), dim3(64), 0, stream, args);
      else if (cfg.wavelet_waves == 2)
        hipLaunchKernelGGL(InvWaveletKernel<2>, dim3(grid), dim3(128), 0, stream, args);
      else if (cfg.wavelet_waves == 4)
        hipLaunchKernelGGL(InvWaveletKernel<4>, dim3(grid), dim3(256), 0, stream, args);
      else
        return hipErrorInvalidValue;
      return hipGetLastError();
    case kStageAssemble:
      if (cfg.tile_fused) {
        if (cfg.rgb)
          hipLaunchKernelGGL(WaveletAssembleKernel<true>, dim3(grid), dim3(kTileFusedWaves * 64), 0, stream, args);
        else
          hipLaunchKernelGGL(WaveletAssembleKernel<false>, dim3(grid), dim3(kTileFusedWaves * 64), 0, stream, args);
      } else if (cfg.rgb) {
        if (cfg.fused_waves) return hipErrorInvalidValue;  // the fused scan writes DXT1 only
        hipLaunchKernelGGL(AssembleRgbKernel, dim3(grid), dim3(256), 0, stream, args);
      } else if (cfg.fused_waves && cfg.fused_wide) {
        if (cfg.fused_waves == 1)
          hipLaunchKernelGGL(AssembleFusedWideKernel<1>, dim3(grid), dim3(64), 0, stream, args);
        else if (cfg.fused_waves == 2)
          hipLaunchKernelGGL(AssembleFusedWideKernel<2>, dim3(grid), dim3(128), 0, stream, args);
        else if (cfg.fused_waves == 4)
          hipLaunchKernelGGL(AssembleFusedWideKernel<4>, dim3(grid), dim3(256), 0, stream, args);
        else
          return hipErrorInvalidValue;
      } else if (cfg.fused_waves == 1) {
        hipLaunchKernelGGL(AssembleFusedKernel<1>, dim3(grid), dim3(64), 0, stream, args);
      } else if (cfg.fused_waves == 2) {
        hipLaunchKernelGGL(AssembleFusedKernel<2>, dim3(grid), dim3(128), 0, stream, args);
      } else if (cfg.fused_waves == 4) {
        hipLaunchKernelGGL(AssembleFusedKernel<4>, dim3(grid), dim3(256), 0, stream, args);
      } else if (cfg.fused_waves == 0) {
        hipLaunchKernelGGL(AssembleDxtKernel, dim3(grid), dim3(256), 0, stream, args);
      } else {
        return hipErrorInvalidValue;
      }
      return hipGetLastError();
    default:
      return hipErrorInvalidValue;
  }
}

// One work-group row per job: 16-byte loads grid-stride over the job's bytes (four
// pairs in flight per lane, so a large output is not one load round trip per 256 KiB),
// one ballot per wave, and a flag store only where a difference was seen.
__global__ __launch_bounds__(256) void CompareKernel(CompareArgs a) {
  const CompareJob j = a.job[blockIdx.y];
  const GPtr<const uint4> x = Gbl<const uint4>(j.out);
  const GPtr<const uint4> y = Gbl<const uint4>(j.expected);
  const uint64_t words = j.bytes / 16;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  bool diff = false;
  uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i + 3 * stride < words; i += 4 * stride) {
    uint4 p[4], q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      p[k] = x[i + k * stride];
      q[k] = y[i + k * stride];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      diff |= ((p[k].x ^ q[k].x) | (p[k].y ^ q[k].y) | (p[k].z ^ q[k].z) | (p[k].w ^ q[k].w)) != 0;
  }
  for (; i < words; i += stride) {
    const uint4 p = x[i], q = y[i];
    diff |= ((p.x ^ q.x) | (p.y ^ q.y) | (p.z ^ q.z) | (p.w ^ q.w)) != 0;
  }
  if (__builtin_amdgcn_ballot_w64(diff) != 0 && __lane_id() == 0) Gbl<uint32_t>(a.flags)[j.flag] = 1u;
}

hipError_t LaunchCompare(const CompareArgs &a, hipStream_t stream) {
  if (a.n == 0) return hipSuccess;
  if (a.n > kCompareJobs) return hipErrorInvalidValue;
  hipLaunchKernelGGL(CompareKernel, dim3(64, a.n), dim3(256), 0, stream, a);
  return hipGetLastError();
}

// Work-group row per job, 16-byte words grid-stride with four loads in flight per
// lane before their stores (reads cross PCIe: latency wants many requests out); the
// job's last bytes past a whole word go one at a time.
__global__ __launch_bounds__(256) void GatherKernel(GatherArgs a) {
  const GatherJob j = a.job[blockIdx.y];
  const GPtr<const uint4> src = Gbl<const uint4>(j.src);
  const GPtr<uint4> dst = Gbl<uint4>(j.dst);
  const uint64_t words = j.bytes / 16;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i + 3 * stride < words; i += 4 * stride) {
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[i + k * stride];
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[i + k * stride] = v[k];
  }
  for (; i < words; i += stride) dst[i] = src[i];
  if (blockIdx.x == 0 && threadIdx.x < (j.bytes & 15)) {
    const uint64_t b = words * 16 + threadIdx.x;
    Gbl<uint8_t>(j.dst)[b] = Gbl<const uint8_t>(j.src)[b];
  }
}

hipError_t LaunchGather(const GatherArgs &a, hipStream_t stream) {
  if (a.n == 0) return hipSuccess;
  if (a.n > kGatherJobs) return hipErrorInvalidValue;
  uint64_t most = 0;
  for (uint32_t i = 0; i < a.n; ++i) {
    if ((reinterpret_cast<uintptr_t>(a.job[i].src) | reinterpret_cast<uintptr_t>(a.job[i].dst)) & 15)
      return hipErrorInvalidValue;
    most = std::max(most, a.job[i].bytes);
  }
  // A few work-groups keep the link busy (each has 16 KiB of loads in flight; about
  // 2 us x 55 GB/s is needed), so the gather takes at most 128 work-groups in all and
  // leaves the CUs to the decodes it runs beside: at most 128 / n a job.  A small job gets
  // one work-group per 4 KiB (a word a lane), so all its loads go out at once: one link
  // round trip, shorter than a DMA copy's fixed cost.
  const uint64_t per_group = 4 << 10;
  const uint32_t gx = static_cast<uint32_t>(
      std::max<uint64_t>(1, std::min<uint64_t>(128 / a.n, (most + per_group - 1) / per_group)));
  hipLaunchKernelGGL(GatherKernel, dim3(gx, a.n), dim3(256), 0, stream, a);
  return hipGetLastError();
}

namespace {

// The no-allocation entry point's scratch.  In host code `scratch` names a host-side
// stand-in, not device memory: host code uses only the address ResolveNoAllocScratch
// obtained for each device.
__device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint8_t *g_scratch_ptr[kMaxDevices] = {};

}  // namespace

hipError_t ResolveNoAllocScratch(int device) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return hipSuccess;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  if (!p) return hipErrorInvalidSymbol;
  g_scratch_ptr[device] = static_cast<uint8_t *>(p);
  return hipSuccess;
}

uint8_t *NoAllocScratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch_ptr[device];
}

__global__ __launch_bounds__(64) void ExportBitsKernel(uint32_t *bits, uint32_t *host) {
  if (threadIdx.x != 0) return;
  Gbl<uint32_t>(host)[0] = Gbl<uint32_t>(bits)[0];
  Gbl<uint32_t>(bits)[0] = 0;
}

__global__ __launch_bounds__(64) void ClearWordKernel(uint32_t *word) {
  if (threadIdx.x == 0) Gbl<uint32_t>(word)[0] = 0;
}

hipError_t LaunchClearWord(uint32_t *word, hipStream_t stream) {
  hipLaunchKernelGGL(ClearWordKernel, dim3(1), dim3(64), 0, stream, word);
  return hipGetLastError();
}

hipError_t LaunchExportBits(uint32_t *bits, uint32_t *host, hipStream_t stream) {
  hipLaunchKernelGGL(ExportBitsKernel, dim3(1), dim3(64), 0, stream, bits, host);
  return hipGetLastError();
}

hipError_t LaunchAnsGroups(const uint32_t *table, const uint8_t *data, uint32_t data_len, uint32_t groups,
                           uint32_t n, uint8_t *out, uint32_t *status, hipStream_t stream) {
  if (groups == 0) return hipSuccess;
  if (n == 0 || n > kLanesPerGroup) return hipErrorInvalidValue;
  hipLaunchKernelGGL(AnsGroupsKernel, dim3((groups + kChainWaves - 1) / kChainWaves), dim3(kChainWaves * 64), 0,
                     stream, table, data, data_len, groups, n, out, status);
  return hipGetLastError();
}

}  // namespace gst
