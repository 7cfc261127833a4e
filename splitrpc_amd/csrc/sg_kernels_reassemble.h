// sg_kernels_reassemble.h -- sorting a burst of arrivals into requests on the
// device (k_ra_*).  A part of sg_hip.hip's translation unit, included there,
// after sg_kernels_prep.h, and nowhere else.
#pragma once

#include "sg_device.h"

#include "sg_kernels_prep.h"

namespace {

// ---------------------------------------------------------------------------
// request reassembly on the device
// ---------------------------------------------------------------------------
// What the receive thread of the reference does per packet -- look the request
// up by token (get_rr), file the fragment at its sequence number
// (rr_emplace_mbuf), hand the request over once complete (is_rr_ready,
// mark_rx_ready_rr) -- done for a whole burst of arrivals at once, with the
// requests that are still incomplete kept on the device from call to call, as
// rr_cache keeps them (src/p2p_rpc_rr_pool_ng.h:97-119):
//   request table   token -> cell, open addressing in buckets of kRaBucket
//                   cells: a lookup reads the whole bucket, so emptying a cell
//                   (a completed request) never hides another request, and a
//                   new token claims an empty cell by atomicCAS.  Four cells per
//                   request that may be in flight, and a token belongs to one
//                   bucket; or, to save memory, two or one (SPILL), and a full
//                   bucket sends its tokens on to others and keeps count of how
//                   far (`reach`)
//   records         every cell has a record of its own: SG_MAX_BI_SIZE entries
//                   {slot, length} indexed by sequence number (p2p_bufs of the
//                   reference's rr).  The cell a token is found in says where
//                   its fragments are filed; a record is neither taken nor
//                   given back.
//   k_ra_insert  one thread per arrival.  The workgroup first sorts its
//                arrivals by token in LDS; one thread per DISTINCT token finds
//                or claims the request's cell and adds the workgroup's share
//                to its fragment count, byte total and last position; then
//                every arrival files its entry in the request's record
//   k_ra_flag    the thread of a complete request's LAST arrival flags that
//                position with the request's fragment count; workgroup-local
//                scan of the packed (requests, fragments) flags
//   k_ra_emit    batch index of a request = number of requests completed before
//                it in this call (completion order, the order of the rx-ready
//                ring); a wavefront in which requests complete adds up the
//                totals of the workgroups before its own (where they are many,
//                k_ra_scan has), copies the records
//                into the output tables, empties them and their cells; the
//                first wavefront closes the call: counts, epoch
// Nothing waits on another thread: every probe makes progress by itself.
//
// What bounds it: dependent round trips (arrival -> header -> bucket -> claim -> entry), not bytes.
// So each is made once, for all of a workgroup's tokens side by side, and nothing is added to a word
// that other workgroups add to as well except the request's own totals.  Kernel trace, us:
//                                          220672 arrivals of        65536 interleaved arrivals of
//                                          512 requests (431 each)   32768 requests (2 each)
//   a group of lanes after the other goes
//   to the table, records from a ring:
//     insert / flag / scan / emit          23.2 / 5.5 / 4.9 / 8.4    30.1 / 9.7 / 4.7 / 13.0
//   this form: insert / flag / emit        11.5 / 4.9 / 6.3          14.0 / 4.9 / 6.5
//   64 arrivals in one launch              8.6 -> 5.4, and 3.8 where the counts stay on the device
// (a launch that does nothing shows as 2 to 4 us there).  Workgroups of 512 threads: 11.9 / 5.2 / 6.0
// and 14.0 / 5.1 / 9.4; of 1024: 12.2 / 5.2 / 5.8 and 20.5 / 6.8 / 10.8.  The ring of free records
// cost a returning addition per workgroup to one word, 35 to 70 ns each and one after the other, and
// two dependent reads per new request.  With all entries of a record in one place (ra_entry) the second
// column was 14.7 / 4.9 / 7.5.

constexpr uint32_t kRaBucket = 32;
static_assert(kRaBucket == 32, "ra_look keeps one bit per cell; a token's first cell is the top five bits of its hash");
constexpr uint32_t kRaNoCell = 0x7fffffffu;
// beside the cell of an arrival: its thread is the one that went to the table for the token
constexpr uint32_t kRaOwner = 0x80000000u;
constexpr int kRaBlock = 256;       // workgroup of the three kernels
constexpr int kRaBurst = 1024;      // most arrivals that one workgroup takes in one launch
constexpr int kRaSmallBurst = 256;  // most that a smaller one takes
constexpr int kRaScan = 1024;       // workgroup of k_ra_scan
// Most workgroups whose totals every wavefront of k_ra_emit that hands something over adds up by itself
// (which grows with the square of the burst); those of more are scanned by a launch in between.  A call,
// us, added up / scanned:  220672 arrivals  17.8 / 20.5   524288  118.7 / 119.1   1000000  657 / 640
//                          1024000 of 512 each  46.3 / 43.1      4000000  1200 / 1215
constexpr uint32_t kRaSumBlocks = 3072;
// device words of the reassembly state
enum { kRaEpoch = 0, kRaInFlight, kRaEvicted, kRaWords = 16 };

struct RaArgs {
  const uint8_t *ring;
  uint32_t n_slots, slot_size, ref64;
  uint32_t n;             // arrivals of this call, or their upper bound with n_dev
  const uint32_t *n_dev;  // device-resident arrival count, or nullptr
  const uint32_t *arrivals;
  const uint32_t *len_nic;
  uint64_t req_size;  // REF64 readiness: bytes == req_size; BL58: fragments == num_frags
  uint32_t cells, bmask;  // cells; buckets - 1
  uint32_t pool;      // requests that may be in flight
  uint32_t max_req, max_frag;  // room in the output tables
  // request table: cells
  unsigned long long *keys;
  uint32_t *reach;           // per bucket: how many buckets further a token whose first bucket it is may sit
  unsigned long long *acc;   // fragments so far << 40 | payload bytes so far: one atomic addition per workgroup and token
  uint32_t *last;            // position in this call of the token's latest arrival; zero between calls
  uint32_t *want, *seen;     // fragments of the request; epoch of the latest call that brought one
  unsigned long long *tab;   // a record per cell: SG_MAX_BI_SIZE entries slot | length << 32 ...
  unsigned long long *head;  // ... of which the first kRaHead lie here, a cell's beside the next one's
  uint32_t *words;           // kRa* above
  // per arrival of this call
  uint32_t *arr_cell;            // | kRaOwner
  unsigned long long *arr_pack;  // RaPack at the completing arrival, else 0
  // per workgroup of k_ra_insert / k_ra_flag
  unsigned long long *blk;       // packed (requests, fragments) completed in it
  unsigned long long *blk_new;   // cells claimed << 32 | arrivals dropped
  // outputs
  uint32_t *frag_slot, *frag_len, *req_first, *req_hdr_slot;
  uint64_t *req_token;
  uint32_t *counts_out;            // device: requests, fragments, arrivals dropped, requests in flight
  volatile uint32_t *counts_host;  // the same four, pinned host memory; nullptr: the host does not ask
  uint32_t *status;
  volatile uint32_t *status_flag;  // pinned host word: non-zero once any kernel refused something
};

// Entry j of a cell's record.  The first few lie apart, 32 bytes a cell: all that a request of a few
// fragments has, where 65536 such requests spread over records of 8 KB each would have their entries
// in gigabytes.  (Four bursts of 65536 arrivals, two fragments a request, filed, gathered and answered:
// 407 us with records in one piece, 397 with eight entries apart; in another process 398.6 with eight
// and 397.6 with four, one burst of 220672, 431 fragments a request, 123.9 and 123.3: four are no
// worse and half the memory.)
constexpr uint32_t kRaHead = 4;
__device__ __forceinline__ unsigned long long *ra_entry(const RaArgs &a, uint32_t cell, uint32_t j)
{
  const bool h = j < kRaHead;
  return (h ? a.head : a.tab) + ((size_t)cell * (h ? kRaHead : SG_MAX_BI_SIZE) + j);
}

__device__ __forceinline__ uint32_t ra_n(const RaArgs &a)
{
  return dev_count(a.n_dev, 0, a.n);
}

// A cell's fragment count and byte total in one word (a request has at most SG_MAX_BI_SIZE
// fragments and far fewer than 2^40 bytes): device-scope atomics are what a burst of many small
// requests pays for, one per addition instead of two.
constexpr int kRaCntShift = 40;
__device__ __forceinline__ unsigned long long ra_pack(uint32_t n, unsigned long long bytes)
{
  return ((unsigned long long)n << kRaCntShift) + bytes;
}
__device__ __forceinline__ uint32_t ra_cnt(unsigned long long acc) { return (uint32_t)(acc >> kRaCntShift); }
__device__ __forceinline__ unsigned long long ra_bytes(unsigned long long acc)
{
  return acc & ((1ull << kRaCntShift) - 1ull);
}

// What k_ra_flag leaves at a completing arrival: top bit set, the request's fragment count (at most
// 1024: 11 bits), the requests (11 bits) and fragments (21 bits) completed before it in its workgroup.
static_assert(SG_MAX_BI_SIZE <= 1024, "eleven bits for a fragment count");
__device__ __forceinline__ unsigned long long ra_done(uint32_t cnt, uint64_t before)
{
  return 1ull << 63 | (unsigned long long)cnt << 48 | (before >> 32) << 32 | (uint32_t)before;
}
__device__ __forceinline__ uint32_t ra_done_cnt(unsigned long long d) { return (uint32_t)(d >> 48) & 0x7fffu; }
__device__ __forceinline__ uint64_t ra_done_before(unsigned long long d)
{
  return d & 0x0000ffffffffffffull;
}

__device__ __forceinline__ uint32_t ra_hash(unsigned long long k)
{
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  return (uint32_t)k;
}

__device__ __forceinline__ unsigned long long ra_key(const unsigned long long *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The cells of a bucket that hold `token`, and those that are empty, a bit each.
struct RaSeen {
  uint32_t found, empty;
};
__device__ __forceinline__ RaSeen ra_look(const RaArgs &a, uint32_t b, unsigned long long token)
{
  // Ordinary 16-byte loads, two keys each, all of them asked for at once.  While arrivals are being
  // filed a key only ever goes from empty to a token, so all a load that is behind the times can show
  // is an empty cell that has just been taken -- and a claim goes through atomicCAS, which then
  // returns the taker (this thread's own token included).
  const ulonglong2 *kp = reinterpret_cast<const ulonglong2 *>(a.keys + b);
  ulonglong2 v[kRaBucket / 2];
#pragma unroll
  for (uint32_t j = 0; j < kRaBucket / 2; j++) v[j] = kp[j];
  RaSeen s = {0u, 0u};
#pragma unroll
  for (uint32_t j = 0; j < kRaBucket / 2; j++) {
    s.found |= (v[j].x == token ? 1u << (2 * j) : 0u) | (v[j].y == token ? 2u << (2 * j) : 0u);
    s.empty |= (v[j].x == 0ull ? 1u << (2 * j) : 0u) | (v[j].y == 0ull ? 2u << (2 * j) : 0u);
  }
  return s;
}

// Claims a cell of a bucket that showed empty ones.  Every token walks a bucket in an order of its
// own -- cyclically from a cell its hash picks -- starting at the first cell of
// that order it has seen empty and trying every empty cell on the way; cells
// before that one in the order were taken when they were read and stay taken
// while arrivals are being filed, so two threads that bring the same new token
// end up in the same cell whatever else is claimed around them.  (With one
// order for all tokens -- lowest cell first -- the new requests of a burst that
// share a bucket queued up on its lowest empty cells, one failed
// compare-and-swap round trip after the other.)
__device__ __forceinline__ uint32_t ra_claim(const RaArgs &a, uint32_t b, unsigned long long token, uint32_t start, uint32_t empty,
                                             bool *claimed)
{
  // place in this token's order of the first cell seen empty
  const uint32_t turned = start ? (empty >> start) | (empty << (32u - start)) : empty;
  const uint32_t first_rank = (uint32_t)__ffs((int)turned) - 1;
#pragma unroll 1
  for (uint32_t rank = first_rank; rank < kRaBucket; rank++) {
    const uint32_t j = (start + rank) & (kRaBucket - 1);
    unsigned long long k = rank == first_rank ? 0ull : ra_key(a.keys + b + j);
    if (k == 0ull) {
      k = atomicCAS(&a.keys[b + j], 0ull, token);
      if (k == 0ull) {
        *claimed = true;
        return b + j;
      }
    }
    if (k == token) return b + j;
  }
  return kRaNoCell;  // taken by others meanwhile
}

// Find or claim the cell of `token`.
//
// SPILL: every token has an order of buckets -- its first, then on by an odd stride of its own, which
// comes past all of them -- and sits in the first of them that was not full when it came.  It is looked
// for as far as any token has gone from its first bucket (mostly nowhere: `reach`), and only then
// claimed, in the first bucket that shows an empty cell.  Buckets before that one were full when they
// were read and stay so while arrivals are being filed, so here too all who bring the same new token
// meet.  `full`: every cell was taken before this call, nothing is to be claimed.  65536 interleaved
// requests of two fragments into 131072 cells take 56 us (43 us with four cells each), 98304 take 107
// (57); the last per mille of a table looks through many buckets, at most kRaFar.  Bursts of 64 take
// 8.1 us (6.8): a table that need not does without.
constexpr uint32_t kRaFar = 1023;
template <bool SPILL>
__device__ __forceinline__ uint32_t ra_find_cell(const RaArgs &a, unsigned long long token, uint32_t hash, bool full, bool *claimed)
{
  const uint32_t first = hash & a.bmask;
  const uint32_t start = hash >> 27;  // the top five bits: the bucket takes the low ones
  *claimed = false;
  if (!SPILL) {
    const uint32_t b = first * kRaBucket;
    const RaSeen s = ra_look(a, b, token);
    if (s.found) return b + (uint32_t)__ffs((int)s.found) - 1;
    return s.empty ? ra_claim(a, b, token, start, s.empty, claimed) : kRaNoCell;
  }
  const uint32_t stride = (hash >> 13) | 1u;
  const uint32_t reach = a.reach[first];
  const uint32_t far = a.bmask < kRaFar ? a.bmask : kRaFar;
  uint32_t at = ~0u, empty = 0;  // the first bucket of the order with empty cells
  uint32_t k = 0;
#pragma unroll 1
  for (;;) {
    const uint32_t b = ((first + k * stride) & a.bmask) * kRaBucket;
    const RaSeen s = ra_look(a, b, token);
    if (s.found) return b + (uint32_t)__ffs((int)s.found) - 1;
    if (at == ~0u && s.empty) {
      at = k;
      empty = s.empty;
    }
    if (k < far && (k < reach || (at == ~0u && !full))) {
      k++;
      continue;
    }
    if (at == ~0u) return kRaNoCell;
    const uint32_t c = ra_claim(a, ((first + at * stride) & a.bmask) * kRaBucket, token, start, empty, claimed);
    if (c != kRaNoCell) {
      if (*claimed && at) atomicMax(&a.reach[first], at);  // for later calls
      return c;
    }
    k = at + 1;  // its empty cells went to others meanwhile: on to the next
    at = ~0u;
    if (k > far) return kRaNoCell;
  }
}

// The distinct tokens among a workgroup's arrivals, open addressing in LDS, twice as many entries
// as arrivals: what the workgroup brings of each -- fragments and bytes, last position -- and, once
// the thread that put the token in has been to the table, its cell.
template <int B>
struct RaLds {
  static constexpr uint32_t kEntries = 2 * B;
  unsigned long long key[kEntries];
  unsigned long long acc[kEntries];
  uint32_t last[kEntries];  // thread index
  uint32_t cell[kEntries];
};

template <int B>
__device__ __forceinline__ void ra_lds_clear(RaLds<B> &l)
{
#pragma unroll
  for (uint32_t k = 0; k < RaLds<B>::kEntries / B; k++) {
    l.key[k * B + threadIdx.x] = 0;
    l.acc[k * B + threadIdx.x] = 0;
    l.last[k * B + threadIdx.x] = 0;
  }
}

// The entry of `token`; *owner: this thread has put it in.
template <int B>
__device__ __forceinline__ uint32_t ra_lds_entry(RaLds<B> &l, unsigned long long token, uint32_t hash, bool *owner)
{
  constexpr uint32_t kMask = RaLds<B>::kEntries - 1;
  uint32_t e = (hash >> 7) & kMask;
  for (;;) {  // at most B distinct tokens: an empty entry is always found
    unsigned long long k = __hip_atomic_load(&l.key[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (k == 0ull) {
      k = atomicCAS(&l.key[e], 0ull, token);
      if (k == 0ull) {
        *owner = true;
        return e;
      }
    }
    if (k == token) return e;
    e = (e + 1) & kMask;
  }
}

struct __attribute__((packed, aligned(1))) u32x4_unaligned { u32x4 v; };
__device__ __forceinline__ u32x4 load128_any(const uint8_t *p)
{
  return reinterpret_cast<const u32x4_unaligned *>(p)->v;
}

// An arrival as its thread knows it.
struct RaMine {
  uint32_t slot = 0, len = 0, fidx = 0, want = 0;
  unsigned long long token = 0;  // 0: not to be filed (no such arrival, token 0, refused)
};

__device__ __forceinline__ RaMine ra_read(const RaArgs &a, uint32_t i, bool in_range)
{
  RaMine m;
  if (!in_range) return m;
  m.slot = a.arrivals[i];
  if (m.slot >= a.n_slots) {
    refuse(a.status, a.status_flag, kStBadSlot);
    return m;
  }
  const uint8_t *h = a.ring + (size_t)m.slot * a.slot_size;
  // token and, with the 58-byte header, everything else as well: bytes 42..57 in one load (every
  // lane has a cache line of its own, so what counts is the number of loads)
  const u32x4 w = load128_any(h + 42);
  if (a.ref64) {
    m.fidx = load32_any(h + 58) & 0xffffu;
    m.len = a.len_nic[m.slot];
  } else {
    m.fidx = w[2] & 0xffffu;
    m.want = w[2] >> 16;
    m.len = a.len_nic ? a.len_nic[m.slot] : w[3];
  }
  const uint32_t hl = a.ref64 ? 64u : 58u;
  if (m.len > a.slot_size - hl) {
    refuse(a.status, a.status_flag, kStBadLen);
    m.len = 0;
  } else {
    m.token = ((unsigned long long)w[1] << 32) | w[0];  // token 0: dropped (src/transport/dpdk_transport_ng.h:231)
  }
  return m;
}

// Enters the workgroup's arrivals into the LDS table.  Fragments of one request tend to arrive
// together: where the first waiting lane's token is that of many lanes, they go in with one
// addition (LDS atomics of a wavefront on one word take a turn per lane).
template <int B>
__device__ __forceinline__ uint32_t ra_group(RaLds<B> &l, const RaMine &m, uint32_t hash, uint32_t lane, bool *owner)
{
  uint32_t e = 0;
  bool waiting = m.token != 0;
  const unsigned long long all = __ballot(waiting);
  *owner = false;
  if (!all) return 0;
  const int first = __ffsll((long long)all) - 1;
  const unsigned long long t = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(m.token >> 32), first) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)m.token, first);
  const bool same = waiting && m.token == t;
  const unsigned long long group = __ballot(same);
  if (__popcll(group) >= 8) {
    const uint32_t bytes = wave_sum_uniform(same ? m.len : 0u);
    if ((int)lane == first) {
      e = ra_lds_entry<B>(l, t, hash, owner);
      atomicAdd(&l.acc[e], ra_pack((uint32_t)__popcll(group), bytes));
      atomicMax(&l.last[e], threadIdx.x - lane + (63u - (uint32_t)__clzll((long long)group)));
    }
    const uint32_t eg = (uint32_t)__builtin_amdgcn_readlane((int)e, first);
    if (same) {
      e = eg;
      waiting = false;
    }
  }
  if (waiting) {
    e = ra_lds_entry<B>(l, m.token, hash, owner);
    atomicAdd(&l.acc[e], ra_pack(1u, m.len));
    atomicMax(&l.last[e], threadIdx.x);
  }
  return e;
}

// rr_emplace_mbuf: the entry goes where its sequence number says.
__device__ __forceinline__ void ra_file(const RaArgs &a, uint32_t cell, const RaMine &m)
{
  if (m.fidx < SG_MAX_BI_SIZE)
    *ra_entry(a, cell, m.fidx) = (unsigned long long)m.slot | ((unsigned long long)m.len << 32);
  else
    refuse(a.status, a.status_flag, kStBadTable);  // beyond what a request's tables hold (src/p2p_bufs.h:10)
}

// Arrivals that belong to no request (token 0, refused, no room) and cells claimed, counted over
// the workgroup.  Every thread calls this; the totals are thread 0's.
template <int B>
__device__ __forceinline__ unsigned long long ra_count_new(bool claimed, bool lost, uint32_t lane, unsigned long long *lds)
{
  const unsigned long long c = __ballot(claimed), d = __ballot(lost);
  if (lane == 0) lds[threadIdx.x / kWave] = (unsigned long long)__popcll(c) << 32 | (uint32_t)__popcll(d);
  __syncthreads();
  unsigned long long t = 0;
  if (threadIdx.x == 0)
    for (uint32_t w = 0; w < B / kWave; w++) t += lds[w];
  return t;
}

template <int B, bool SPILL>
__global__ __launch_bounds__(B) void k_ra_insert(RaArgs a)
{
  __shared__ RaLds<B> l;
  __shared__ unsigned long long wave_new[B / kWave];
  const uint32_t i0 = blockIdx.x * B, i = i0 + threadIdx.x;
  const uint32_t n = ra_n(a);
  if (i0 >= n) return;  // the whole workgroup
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const bool in_range = i < n;
  const uint32_t epoch = sload(a.words + kRaEpoch);  // advanced by k_ra_emit, two kernels behind
  const bool full = SPILL && sload(a.words + kRaInFlight) >= a.cells;
  const RaMine m = ra_read(a, i, in_range);
  ra_lds_clear(l);
  __syncthreads();
  const uint32_t hash = ra_hash(m.token);
  bool owner, claimed = false;
  const uint32_t e = ra_group<B>(l, m, hash, lane, &owner);
  __syncthreads();
  if (owner) {
    const uint32_t c = ra_find_cell<SPILL>(a, m.token, hash, full, &claimed);
    l.cell[e] = c;
    if (c != kRaNoCell) {
      atomicAdd(&a.acc[c], l.acc[e]);
      atomicMax(&a.last[c], i0 + l.last[e]);
      a.seen[c] = epoch;
      if (!a.ref64) a.want[c] = m.want;  // every fragment of a request says the same
    } else {
      refuse(a.status, a.status_flag, kStPoolFull);
    }
  }
  __syncthreads();
  const uint32_t cell = m.token ? l.cell[e] : kRaNoCell;
  if (cell != kRaNoCell) ra_file(a, cell, m);
  if (in_range) a.arr_cell[i] = cell | (owner ? kRaOwner : 0u);
  const unsigned long long t = ra_count_new<B>(claimed, in_range && cell == kRaNoCell, lane, wave_new);
  if (threadIdx.x == 0) a.blk_new[blockIdx.x] = t;
}

__device__ __forceinline__ bool ra_complete(const RaArgs &a, uint32_t want, unsigned long long acc)
{
  return a.ref64 ? ra_bytes(acc) == a.req_size : ra_cnt(acc) == want;
}

// Whether a complete request of this many fragments can be handed over.
__device__ __forceinline__ bool ra_fits(const RaArgs &a, uint32_t cnt)
{
  if (cnt <= SG_MAX_BI_SIZE) return true;
  refuse(a.status, a.status_flag, kStBadTable);
  return false;
}

template <int B>
__global__ __launch_bounds__(B) void k_ra_flag(RaArgs a)
{
  __shared__ uint64_t wave_tot[B / kWave];
  const uint32_t i = blockIdx.x * B + threadIdx.x;
  const uint32_t n = ra_n(a);
  if (blockIdx.x * B >= n) return;  // the whole workgroup
  uint64_t mine = 0;
  if (i < n) {
    const uint32_t cell = a.arr_cell[i] & ~kRaOwner;
    if (cell != kRaNoCell) {
      const unsigned long long acc = a.acc[cell];
      const uint32_t last = a.last[cell], want = a.want[cell];
      if (last == i && ra_complete(a, want, acc) && ra_fits(a, ra_cnt(acc)))
        mine = 1ull << 32 | ra_cnt(acc);
    }
  }
  uint64_t tot;
  const uint64_t before = block_exclusive_scan<B>(mine, wave_tot, &tot);
  if (i < n) a.arr_pack[i] = mine ? ra_done((uint32_t)mine, before) : 0ull;
  if (threadIdx.x == 0) a.blk[blockIdx.x] = tot;
}

// Closes the call (one wavefront's lane 0): counts and epoch.  `tot` is the packed (requests,
// fragments) total of the call, `fresh` the cells claimed << 32 | arrivals dropped.  The kernel's
// other wavefronts read none of the words written here.
__device__ __forceinline__ void ra_close(const RaArgs &a, uint64_t tot, unsigned long long fresh, bool overflow)
{
  const uint32_t n_req = overflow ? 0u : (uint32_t)(tot >> 32), n_frag = overflow ? 0u : (uint32_t)tot;
  const uint32_t claims = (uint32_t)(fresh >> 32), before = a.words[kRaInFlight];
  const uint32_t in_flight = before + claims - n_req;
  // more than the context was made for are left (not dropped: every one has its cell)
  if (claims && in_flight > a.pool) refuse(a.status, a.status_flag, kStPoolFull);
  // the output tables cannot take what completed: nothing is emitted, the requests stay parked
  if (overflow) refuse(a.status, a.status_flag, kStBadTable);
  a.req_first[n_req] = n_frag;
  a.words[kRaInFlight] = in_flight;
  a.words[kRaEpoch] += 1;
  const uint32_t c[4] = {n_req, n_frag, (uint32_t)fresh, in_flight};
  for (int k = 0; k < 4; k++) {
    if (a.counts_out) a.counts_out[k] = c[k];
    if (a.counts_host) a.counts_host[k] = c[k];  // straight into pinned host memory: nothing to copy back
  }
}

// Empties the cell of a request that has been handed over (its record is empty already).
__device__ __forceinline__ void ra_free_cell(const RaArgs &a, uint32_t cell)
{
  a.acc[cell] = 0;
  __hip_atomic_store(&a.keys[cell], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Hands over the requests that complete on this wavefront's lanes: `done` what k_ra_flag left
// there (0 on the other lanes).  `base` gives the packed (requests, fragments) completed before
// the wavefront's workgroup, or returns false where nothing is to be handed over after all; it is
// asked once the first records are on their way.  Every lane of the wavefront calls this.
template <class Base>
__device__ __forceinline__ void ra_emit(const RaArgs &a, uint32_t cell, unsigned long long done, uint32_t lane, Base base)
{
  // requests of a few fragments are handed over by the completing lane itself, all such lanes
  // at once; the wavefront then walks the larger ones together, eight entries per lane asked for
  // before the first is stored
  constexpr uint32_t kOwn = 8, kAhead = 8;
  const uint32_t cnt = ra_done_cnt(done);
  const bool own = done && cnt <= kOwn;
  unsigned long long todo = __ballot(done && !own);
  unsigned long long e[kOwn], f[kAhead];
  if (own) {
#pragma unroll
    for (uint32_t j = 0; j < kOwn; j++) e[j] = j < cnt ? *ra_entry(a, cell, j) : 0ull;
  }
  auto ask = [&](uint32_t c, uint32_t k, uint32_t j0) {
#pragma unroll
    for (uint32_t q = 0; q < kAhead; q++) {
      const uint32_t j = j0 + q * kWave + lane;
      f[q] = j < k ? *(q ? a.tab + (size_t)c * SG_MAX_BI_SIZE + j : ra_entry(a, c, j)) : 0ull;
    }
  };
  if (todo) {
    const int l = __ffsll((long long)todo) - 1;
    ask((uint32_t)__builtin_amdgcn_readlane((int)cell, l), (uint32_t)__builtin_amdgcn_readlane((int)cnt, l), 0);
  }
  uint64_t before;
  if (!base(&before)) return;
  const uint64_t at = before + ra_done_before(done);
  if (own) {
    const uint32_t r = (uint32_t)(at >> 32), first = (uint32_t)at;
#pragma unroll
    for (uint32_t j = 0; j < kOwn; j++) {
      if (j < cnt) {
        a.frag_slot[first + j] = (uint32_t)e[j];
        a.frag_len[first + j] = (uint32_t)(e[j] >> 32);
        *ra_entry(a, cell, j) = 0;  // a fresh request finds an empty record
      }
    }
    a.req_first[r] = first;
    if (a.req_token) a.req_token[r] = ra_key(a.keys + cell);
    if (a.req_hdr_slot) a.req_hdr_slot[r] = (uint32_t)e[0];  // the slot whose header the responses answer
    ra_free_cell(a, cell);
  }
  bool asked = true;
  while (todo) {
    const int l = __ffsll((long long)todo) - 1;
    todo &= todo - 1;
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cell, l);
    const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)cnt, l);
    const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(at >> 32), l);
    const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)at, l);
    for (uint32_t j0 = 0; j0 < k; j0 += kAhead * kWave) {
      if (!asked) ask(c, k, j0);
      asked = false;
#pragma unroll
      for (uint32_t q = 0; q < kAhead; q++) {
        const uint32_t j = j0 + q * kWave + lane;
        if (j < k) {
          a.frag_slot[first + j] = (uint32_t)f[q];
          a.frag_len[first + j] = (uint32_t)(f[q] >> 32);
          *(q ? a.tab + (size_t)c * SG_MAX_BI_SIZE + j : ra_entry(a, c, j)) = 0;
        }
      }
      if (j0 == 0 && lane == 0) {
        a.req_first[r] = first;
        if (a.req_token) a.req_token[r] = ra_key(a.keys + c);
        if (a.req_hdr_slot) a.req_hdr_slot[r] = (uint32_t)f[0];
        ra_free_cell(a, c);
      }
    }
  }
}

// Sum over the wavefront of words that hold two counts of 32 bits each (neither sum leaves its half).
__device__ __forceinline__ uint64_t wave_sum_pairs(uint64_t v)
{
  return (uint64_t)wave_sum_uniform((uint32_t)(v >> 32)) << 32 | wave_sum_uniform((uint32_t)v);
}

// A word per workgroup, `n` of them, added up over the wavefront: all of them, and those before
// number `upto`.  Eight per lane are asked for before the first is added.
__device__ __forceinline__ void ra_sum_blocks(const unsigned long long *p, uint32_t n, uint32_t upto, uint32_t lane,
                                              uint64_t *all, uint64_t *before)
{
  uint64_t t = 0, b = 0;
  for (uint32_t q0 = lane; q0 < n; q0 += 8 * kWave) {
    uint64_t v[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; k++) v[k] = q0 + k * kWave < n ? p[q0 + k * kWave] : 0ull;
#pragma unroll
    for (uint32_t k = 0; k < 8; k++) {
      t += v[k];
      b += q0 + k * kWave < upto ? v[k] : 0ull;
    }
  }
  *all = wave_sum_pairs(t);
  *before = wave_sum_pairs(b);
}

// The totals of more workgroups than that are scanned once, by one workgroup of T threads: in place,
// with the sums of all behind them.  (B: as for k_ra_emit.)
template <int T, int B>
__global__ __launch_bounds__(T) void k_ra_scan(RaArgs a)
{
  __shared__ uint64_t wave_tot[T / kWave];
  constexpr uint32_t kEach = 4;
  const uint32_t n_blocks = (ra_n(a) + B - 1) / B;
  uint64_t run = 0, fresh = 0;
  for (uint32_t b0 = 0; b0 < n_blocks; b0 += kEach * T) {
    const uint32_t b = b0 + kEach * threadIdx.x;
    uint64_t v[kEach], mine = 0, tot;
#pragma unroll
    for (uint32_t k = 0; k < kEach; k++) {
      v[k] = b + k < n_blocks ? a.blk[b + k] : 0ull;
      fresh += b + k < n_blocks ? a.blk_new[b + k] : 0ull;
      mine += v[k];
    }
    uint64_t at = run + block_exclusive_scan<T>(mine, wave_tot, &tot);
#pragma unroll
    for (uint32_t k = 0; k < kEach; k++) {
      if (b + k < n_blocks) a.blk[b + k] = at;
      at += v[k];
    }
    run += tot;
  }
  uint64_t all;
  (void)block_exclusive_scan<T>(fresh, wave_tot, &all);
  if (threadIdx.x == 0) {
    a.blk[n_blocks] = run;
    a.blk_new[n_blocks] = all;
  }
}

// B: the workgroup size of this kernel and of the two before it (a total per workgroup).  SCANNED:
// k_ra_scan has been over the totals.
template <int B, bool SCANNED>
__global__ __launch_bounds__(B) void k_ra_emit(RaArgs a)
{
  const uint32_t n = ra_n(a);
  const uint32_t i = blockIdx.x * B + threadIdx.x;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const bool closer = __builtin_amdgcn_readfirstlane(i / kWave) == 0;
  unsigned long long done = 0;
  uint32_t cell = kRaNoCell;
  if (i < n) {
    done = a.arr_pack[i];
    const uint32_t oc = a.arr_cell[i];
    cell = oc & ~kRaOwner;
    if ((oc & kRaOwner) && cell != kRaNoCell) a.last[cell] = 0;  // the position counts per call
  }
  if (!__any(done != 0) && !closer) return;
  // What completed in the workgroups before this one, and in all of them: every wavefront that
  // has something to hand over adds the totals up by itself where they are few.
  const uint32_t n_blocks = (n + B - 1) / B;
  ra_emit(a, cell, done, lane, [&](uint64_t *base) {
    uint64_t tot;
    if (SCANNED) {
      *base = sload(a.blk + blockIdx.x);
      tot = sload(a.blk + n_blocks);
    } else {
      ra_sum_blocks(a.blk, n_blocks, blockIdx.x, lane, &tot, base);
    }
    const bool overflow = (uint32_t)(tot >> 32) > a.max_req || (uint32_t)tot > a.max_frag;
    if (closer) {
      uint64_t fresh, none;
      if (SCANNED) fresh = sload(a.blk_new + n_blocks);
      else ra_sum_blocks(a.blk_new, n_blocks, 0, lane, &fresh, &none);
      if (lane == 0) ra_close(a, tot, fresh, overflow);
    }
    return !overflow;
  });
}

// A burst that one workgroup takes, which is what a NIC delivers: the three steps in ONE kernel.
// Nothing else touches the table meanwhile, so the owner of a token works on its cell with
// ordinary loads and stores and hands the new total to the token's other arrivals through LDS.
template <int B, bool SPILL>
__global__ __launch_bounds__(B) void k_ra_burst(RaArgs a)
{
  __shared__ RaLds<B> l;
  __shared__ unsigned long long wave_new[B / kWave];
  __shared__ uint64_t wave_tot[B / kWave];
  const uint32_t i = threadIdx.x;
  const uint32_t n = ra_n(a);
  const uint32_t lane = i & (kWave - 1);
  const bool in_range = i < n;
  const uint32_t epoch = a.words[kRaEpoch];
  const bool full = SPILL && a.words[kRaInFlight] >= a.cells;
  const RaMine m = ra_read(a, i, in_range);
  ra_lds_clear(l);
  __syncthreads();
  const uint32_t hash = ra_hash(m.token);
  bool owner, claimed = false;
  const uint32_t e = ra_group<B>(l, m, hash, lane, &owner);
  __syncthreads();
  if (owner) {
    const uint32_t c = ra_find_cell<SPILL>(a, m.token, hash, full, &claimed);
    l.cell[e] = c;
    if (c != kRaNoCell) {
      const unsigned long long acc = (claimed ? 0ull : a.acc[c]) + l.acc[e];  // an empty cell's total is zero
      a.acc[c] = acc;
      l.acc[e] = acc;
      a.seen[c] = epoch;
    } else {
      refuse(a.status, a.status_flag, kStPoolFull);
    }
  }
  __syncthreads();
  const uint32_t cell = m.token ? l.cell[e] : kRaNoCell;
  uint64_t mine = 0;
  if (cell != kRaNoCell) {
    ra_file(a, cell, m);
    const unsigned long long acc = l.acc[e];
    if (l.last[e] == i && ra_complete(a, m.want, acc) && ra_fits(a, ra_cnt(acc))) mine = 1ull << 32 | ra_cnt(acc);
  }
  uint64_t tot;
  const uint64_t before = block_exclusive_scan<B>(mine, wave_tot, &tot);
  // (its barriers also stand between the entries filed above and the records read below)
  const bool overflow = (uint32_t)(tot >> 32) > a.max_req || (uint32_t)tot > a.max_frag;
  const unsigned long long fresh = ra_count_new<B>(claimed, in_range && cell == kRaNoCell, lane, wave_new);
  if (i == 0) ra_close(a, tot, fresh, overflow);
  ra_emit(a, cell, mine ? ra_done((uint32_t)mine, before) : 0ull, lane, [&](uint64_t *base) {
    *base = 0;
    return !overflow;
  });
}

// Empties the table: every cell, every record.  Any grid: the records of millions of requests are
// more than a launch has threads for.
__global__ __launch_bounds__(256) void k_ra_reset(RaArgs a)
{
  const size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
  for (size_t i = i0; i < a.cells; i += step) {
    a.keys[i] = 0;
    a.acc[i] = 0;
    a.last[i] = a.want[i] = a.seen[i] = 0;
    if (i <= a.bmask) a.reach[i] = 0;
  }
  // two entries at a time
  for (size_t i = i0; 2 * i < (size_t)a.cells * SG_MAX_BI_SIZE; i += step) reinterpret_cast<u32x4 *>(a.tab)[i] = (u32x4){0u, 0u, 0u, 0u};
  for (size_t i = i0; 2 * i < (size_t)a.cells * kRaHead; i += step) reinterpret_cast<u32x4 *>(a.head)[i] = (u32x4){0u, 0u, 0u, 0u};
  if (i0 < kRaWords) a.words[i0] = 0;
}

// Drops the requests no fragment has come in for during the last max_age calls
// (a lost fragment parks its request for good in the reference,
// src/p2p_rpc_rr_pool_ng.h:57-64; here the caller can clear such requests out).
// One wavefront per cell.
__global__ __launch_bounds__(256) void k_ra_evict(RaArgs a, uint32_t max_age)
{
  const uint32_t c = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  if (c >= a.cells) return;
  if (a.keys[c] == 0ull) return;
  if (a.words[kRaEpoch] - a.seen[c] <= max_age) return;
  for (uint32_t j = lane; j < SG_MAX_BI_SIZE; j += kWave) *ra_entry(a, c, j) = 0;
  if (lane == 0) {
    a.acc[c] = 0;
    a.keys[c] = 0;
    atomicSub(&a.words[kRaInFlight], 1u);
    atomicAdd(&a.words[kRaEvicted], 1u);
  }
}

}  // namespace
