// iamx_decode.hip -- Blosc2 block decode (LZ4 + un-shuffle / bit-un-shuffle)
// and the dense transpose, for gfx950.
//
// Decode is two launches:
//   k_lz4_streams   one workgroup per LZ4 stream, of 8, 4 or 1 wavefronts by
//                   the number of streams.  Input positions are decoded as
//                   sequence headers all at once, the sequences really there
//                   are picked out by following them from every start, and
//                   output bytes are produced one a lane, whatever sequences
//                   they belong to.
//   k_unfilter      (iamx_unfilter.hip) gathers each element's bytes from its
//                   byte or bit planes and writes it into its tile of the dense
//                   destination.
// Stream sources are either the compressed chunk arena (raw streams, read in
// place), the LZ4 scratch, or a constant byte (zero / run streams, special
// chunks).
#include "iamx_internal.h"

namespace {

using iamx::u32x4;
using iamx::u32x4_any;

__device__ __forceinline__ uint32_t rdlane(uint32_t v, int32_t l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

// lane l of v
__device__ __forceinline__ void set_lane(uint32_t &v, int l, uint32_t x) {
  asm("v_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(x), "n"(l));
}

// bit i of m
__device__ __forceinline__ void bit_on(uint64_t &m, int32_t i) { asm("s_bitset1_b64 %0, %1" : "+s"(m) : "s"(i)); }
__device__ __forceinline__ void bit_off(uint64_t &m, int32_t i) { asm("s_bitset0_b64 %0, %1" : "+s"(m) : "s"(i)); }

__device__ __forceinline__ uint64_t ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }

// 4 bytes at any offset, by two aligned reads
__device__ __forceinline__ uint32_t lds_u32(const uint8_t *lds, int32_t at) {
  const uint32_t *w = reinterpret_cast<const uint32_t *>(lds + (at & ~3));
  return __builtin_amdgcn_alignbyte(w[1], w[0], (uint32_t)at);
}

__device__ __forceinline__ int32_t bperm(int32_t l, int32_t v) {  // v of lane l & 63
  return __builtin_amdgcn_ds_bpermute(l << 2, v);
}

// bits of m below this lane, added to v
__device__ __forceinline__ int32_t bits_below(uint64_t m, int32_t v) {
  return (int32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)v));
}

// Inclusive prefix sum over the 64 lanes (DPP row shifts, then row broadcasts).
__device__ __forceinline__ int32_t wave_inclusive_sum(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// Workgroup barrier that orders LDS only: global loads and stores in flight
// stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A sequence that rounds decode has at most one literal and one match length
// byte: 269 literals and a match of 273 bytes, in kSeqIn input bytes.
constexpr int kSeqIn = 1 + 1 + 269 + 2 + 1;
constexpr int kSeqOut = 269 + 273;

// Sizes of a stream decoder of NW wavefronts (NW > 1: one window of 64 input
// positions per wavefront and round).
template <int NW>
struct Lz4Geom {
  static constexpr int kThreads = 64 * NW;
  static constexpr int kRing = 4096 * NW;         // output history, bytes
  static constexpr int kOut = 512 * NW;           // most output bytes of a round
  static constexpr int kStep = 256 * NW;          // output bytes of a step of the general path
  static constexpr int kStageWords = 16 * NW + 72;  // input of a round: 64 NW positions and what the last ones reach
  static constexpr int kStage = 4 * kStageWords;
  static constexpr int kSeqs = (64 * NW + 2) / 3;   // a sequence takes at least 3 input bytes
  // LDS: ring, two stages, sequence table, first-output-byte bits, source
  // records of an output step, window exits, the cut
  static constexpr int kTabAt = kRing + 2 * kStage;
  static constexpr int kBitsAt = kTabAt + 8 * kSeqs;
  static constexpr int kRecAt = kBitsAt + kOut / 8;
  static constexpr int kExitAt = kRecAt + 4 * kThreads;
  static constexpr int kCutAt = kExitAt + 4 * kThreads;
  static constexpr int kLds = kCutAt + 8;
  static_assert(kOut >= kSeqOut, "a round holds any one sequence");
  static_assert(kStage >= 3 + 64 * NW + kSeqIn + 8, "and the stage its input");
};

// One wavefront: up to three windows of 63 positions a round, at most 64
// sequences.
template <>
struct Lz4Geom<1> {
  static constexpr int kThreads = 64;
  static constexpr int kRing = 4096;
  static constexpr int kOut = 1024;
  static constexpr int kStep = 256;
  static constexpr int kStage = 1024;  // a ring, its first bytes repeated after its end
  static constexpr int kSeqs = 64;
  static constexpr int kTabAt = kRing + kStage + 16;
  static constexpr int kBitsAt = kTabAt + 8 * kSeqs;
  static constexpr int kListAt = kBitsAt + kOut / 8;
  static constexpr int kLds = kListAt + 2 * kSeqs;
  static_assert(kOut >= kSeqOut, "a round holds any one sequence");
};

// One LZ4 stream by one workgroup of NW wavefronts.  The state (input and
// output position, what is flushed) is uniform over the workgroup: every
// wavefront derives it from the same LDS words.
//
// Rounds.  A round takes the 64 NW input positions from `base`, whatever the
// sequences in them, so its input is staged in LDS one round ahead.
//   headers  thread t decodes the sequence that would start at position base
//            + t.  Sequences of at most 269 literals and 273 match bytes (one
//            length byte each) inside the stream are decoded by rounds (`ok`).
//   reach    each wavefront follows the sequences of its 64-position window
//            from all 64 starts at once, by pointer doubling (at most 22
//            hops, at 0, 3, .. 63): where the chain leaves the window or stops at a sequence
//            that is not ok, and how many sequences and output bytes it
//            passes.  None of this needs to know where the window is entered.
//   chain    the windows' exits are then followed from the round's entry, one
//            lookup per window, which gives each wavefront its first start, the
//            sequences and the output bytes before it.
//   walk     from there each wavefront collects its starts, eight hops a step.
//   scan     a prefix sum of their output lengths over the lanes gives every
//            sequence's first output byte; the round is cut before the first
//            one that does not fit.
//   table    the starts store their fields in LDS in sequence order and set
//            the bit of their first output byte.
//   output   one byte a thread, two at a time, whatever sequences they belong
//            to: a thread finds its sequence by counting the bits up to its
//            byte and takes a literal from the stage or a match byte from the
//            ring (from the flushed output when the offset passes it).  A
//            match that overlaps itself reads from the bytes before it.  A
//            source written in the same step is a lower byte: the threads
//            leave their byte, or the number of their source byte, in LDS and
//            follow the numbers until they find a byte.
// What bounds it where streams are few is the chain from round to round (header
// reads, 5 hops of pointer doubling, the exits, the scans, the table, the
// sources), so its time falls with the windows a round takes: a 250 KB
// bitshuffled float32 stream takes 451 us with one wavefront, 205 with 4, 134
// with 8; one sequence after the other, with 64 lanes copying each, took 783.
// With four streams of 8 wavefronts a CU it is vector issue: the vector
// instructions of 1024 exponent planes fill 91% of their wavefronts' life at four
// cycles each.  With 25 of one wavefront (6400 bitshuffled streams) a wavefront
// waits 65% of its life, for LDS and for HBM, and issues 23%.  So a round's cost
// is its instructions and its waits:
//  - LDS words at any byte offset are two aligned reads and a byte align; one
//    misaligned read a lane took 522 us where this takes 424 (1024 exponent
//    planes of 64 KB of float32).
//  - The records are read and written as LDS; through a volatile pointer they
//    were flat accesses that waited for every global load and store in flight
//    (561 against 531 us), as a byte from the slot did where its path met the
//    others', and a flush before the staged input had arrived.
//  - The chain has no branch and selects nothing: what a window's wavefront
//    needs is left in the lane of its number (645 to 561 us).
// Of a launch of 6400 bitshuffled streams, 0.35 ms are their literal runs
// crossing HBM at 4.8 TB/s.
//
// A round's output is cut at 8 bytes an input position (1024 bytes with one
// wavefront); several wavefronts then take the rest of the same positions.  At 4
// bytes a position, with the input staged anew, streams of sparse rows were cut
// in every round: 1024 byte planes of 700 bytes for 15625 took 63 us, now 51.
//
// What a round cannot hold (long literal runs, matches of more than 273
// bytes, the stream's end) is decoded one sequence at a time by the general
// path, with all threads copying.  Where the next sequence is seen to be long as
// well, several wavefronts stay there (a bitshuffled float32 stream 136 to 133
// us, one of a matrix's last rows 102 to 94; nothing with one wavefront).
//
// Many streams of one kind are all in the same place at once: bitshuffled ones
// begin with their lowest planes, a literal run of half the stream, and wait for
// HBM together, and then leave it idle while they decode rounds.  So with one
// wavefront a stream that begins with a run of 8 KB or more, or is of 64 KB or
// more compressed (SIDEWAYS), copies only what the ring has to hold of such a
// run and moves the rest a little in every round: 4096 streams of an 8000^2
// float64 matrix 320 to 303 us, 9216 of a 12000^2 float32 one 422 to 385, 10800
// of normal float32 values in blocks of 100^2 275 to 221; nothing where streams
// differ and overlap by themselves (20000^2 float32, 1290).  By the first run
// alone the float64 ones took 342: some moved, some not.  In a body of its own:
// other streams took 2 to 4% longer in one for both.
//
// Output bytes go to an LDS ring and reach the stream's scratch slot in
// 16-byte stores whenever a quarter of the ring (FLUSH_AT) is pending.  An offset
// of more than NEAR reads the slot back from global memory.  With several
// wavefronts such a source must lie before the last flush, whose stores alone may
// still be on their way: those of the flush before it were waited for by every
// wavefront before a barrier that precedes the read.  It does: a round begins
// with less than FLUSH_AT bytes pending, the last flush wrote at most FLUSH_AT +
// kOut, and the byte that reads is at most kOut past the round's first, so NEAR
// has to be twice FLUSH_AT + kOut or more (15/16 of the ring against 12/16).
template <int NW, bool SIDEWAYS = false>
__device__ __forceinline__ void lz4_stream(const iamx_lz4_job_t job, uint8_t *__restrict__ scratch, int *status,
                                           uint8_t *lds, int32_t ahead_at) {
  using G = Lz4Geom<NW>;
  constexpr int32_t NT = G::kThreads;
  constexpr int32_t RING = G::kRing, RM = RING - 1;
  constexpr int32_t NEAR = RING - G::kStep;
  constexpr int32_t FLUSH_AT = RING / 4;
  static_assert(NW == 1 || NEAR >= 2 * (FLUSH_AT + G::kOut), "a far source was stored before the last flush");
  static_assert(G::kStep <= G::kOut, "and by the general path");
  uint8_t *ring = lds;
  uint8_t *stage = lds + RING;
  uint64_t *tab = reinterpret_cast<uint64_t *>(lds + G::kTabAt);
  uint32_t *obits = reinterpret_cast<uint32_t *>(lds + G::kBitsAt);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint64_t abase = job.src & ~3ull;  // input positions are relative to this aligned address
  const IAMX_GLOBAL uint32_t *__restrict__ sw = iamx::gptr<const uint32_t>(abase);
  const IAMX_GLOBAL uint8_t *__restrict__ sb = iamx::gptr<const uint8_t>(abase);
  IAMX_GLOBAL uint8_t *dst = iamx::gptr<uint8_t>((uint64_t)(scratch + job.dst_off));
  IAMX_GLOBAL uint32_t *dstw = iamx::gptr<uint32_t>((uint64_t)(scratch + job.dst_off));
  const bool wide = ((uint64_t)(scratch + job.dst_off) & 15) == 0;  // 16-byte stores of the slot
  const int32_t iend = (int32_t)(job.src & 3) + job.csize;
  const int32_t oend = job.nbytes;
  const int32_t lastw = (iend - 1) >> 2;  // last word holding stream bytes

  // word i of the input from pos; words past the stream repeat its last word
  // (never parsed)
  auto ld_word = [&](int32_t pos, int32_t i) -> uint32_t { return sw[min((pos >> 2) + i, lastw)]; };
  int32_t ip = (int32_t)(job.src & 3), op = 0, flushed = 0, flush_at = FLUSH_AT;
  // this wavefront's memory operations so far are complete
  auto drain = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
  };
  // store the whole 16-byte groups (as dwords where the slot is not 16-byte
  // aligned) of ring bytes [flushed, cur) to the slot; flushed stays a
  // multiple of 16
  auto flush = [&](int32_t cur) {
    if (NW > 1) drain();  // the stores of the flush before this one
    if (wide) {
      for (int32_t p = flushed + 16 * tid; p + 16 <= cur; p += 16 * NT)
        *iamx::gptr<u32x4>((uint64_t)(dst + p)) = *reinterpret_cast<const u32x4 *>(ring + (p & RM));
    } else {
      for (int32_t p = flushed + 4 * tid; p + 4 <= (cur & ~15); p += 4 * NT)
        dstw[p >> 2] = *reinterpret_cast<const uint32_t *>(ring + (p & RM));
    }
    flushed = __builtin_amdgcn_readfirstlane(cur & ~15);
    flush_at = flushed + FLUSH_AT;
  };

  // SIDEWAYS: what is left of a long literal run is moved by the rounds after it,
  // SIDE bytes each.  Bytes of the run, moved or not, are read from the input.
  constexpr int32_t SIDE = 1024;
  int32_t side_n = 0, side_src = 0, side_dst = 0;  // bytes left, from where, to where
  int32_t run_at = 0, run_n = 0, run_in = 0;       // the run's output bytes, and input less output position
  auto side_load = [&](int32_t i) -> u32x4 { return *(const IAMX_GLOBAL u32x4_any *)(sb + side_src + i); };
  auto side_store = [&](int32_t i, u32x4 w) { *iamx::gptr<u32x4>((uint64_t)(dst + side_dst + i)) = w; };
  auto side_finish = [&]() {
    for (int32_t i = 16 * lane; i < side_n; i += 2 * SIDE) {
      const bool two = i + SIDE < side_n;
      const u32x4 a = side_load(i);
      u32x4 b;
      if (two) b = side_load(i + SIDE);
      side_store(i, a);
      if (two) side_store(i + SIDE, b);
    }
    side_n = 0;
  };
  // a byte that a flush wrote, or of the run; it has arrived
  auto slot_byte = [&](int32_t at) -> uint32_t {
    uint32_t v;
    if (SIDEWAYS && run_n > 0) {
      const bool in_run = (uint32_t)(at - run_at) < (uint32_t)run_n;
      v = *(in_run ? sb + at + run_in : (const IAMX_GLOBAL uint8_t *)dst + at);
      asm volatile("" : "+v"(v));
    } else {
      v = dst[at];
      asm volatile("" : "+v"(v));
    }
    return v;
  };

  // Wavefronts with more input left go first.  Streams that share a CU then end
  // together, the long ones of unlike streams and all of equal ones, and none
  // is left to decode with the CU to itself: 1024 exponent planes 426 to 366 us,
  // 6400 of them 1733 to 1540; 1024 bitshuffled streams of 33 to 85 rounds 396
  // to 340.
  auto rank = [&](int32_t at) {
    const int32_t left = iend - at;
    if (left > ahead_at) __builtin_amdgcn_s_setprio(3);
    else if (left > ahead_at >> 1) __builtin_amdgcn_s_setprio(2);
    else if (left > ahead_at >> 2) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
  };
  rank(ip);

  int bad = 0;
  bool general = false;
  for (;;) {
    // ---- rounds
    if (!general) {
      if constexpr (NW == 1) {
        constexpr int32_t SM = G::kStage - 1, WIN = 63, NEAR1 = RING - 64;
        uint16_t *list = reinterpret_cast<uint16_t *>(lds + G::kListAt);
        uint32_t *stage32 = reinterpret_cast<uint32_t *>(stage);
        // 256 input bytes from pos, a multiple of 256, into the stage
        auto put_stage = [&](int32_t pos, uint32_t w) {
          const int32_t at = (pos & SM) >> 2;
          stage32[at + lane] = w;
          if (at == 0 && lane < 4) stage32[G::kStage / 4 + lane] = w;
          __builtin_amdgcn_wave_barrier();
        };
        int32_t have = (ip & ~255) + 768;  // the stage holds the input from ip up to here
        {
          const uint32_t a = ld_word(have - 768, lane), b = ld_word(have - 512, lane), c = ld_word(have - 256, lane);
          put_stage(have - 768, a);
          put_stage(have - 512, b);
          put_stage(have - 256, c);
        }
        for (;;) {
          // no window of a round starts 189 bytes from ip or more, and its last
          // sequence starts within 62
          while (have < ip + 3 * WIN + 62 + kSeqIn + 8) {
            put_stage(have, ld_word(have, lane));
            have += 256;
          }
          const bool more = have - ip < 768;
          uint32_t ahead = 0;
          if (more) ahead = ld_word(have, lane);
          u32x4 side;
          if (SIDEWAYS && side_n > 0) side = side_load(16 * lane);
          if (lane < G::kOut / 32) obits[lane] = 0;
          // walk: the starts of up to three windows, listed by position
          int32_t n = 0, at = ip;  // sequences so far, the next one's position
          bool stopped = false;
          do {
            const uint32_t h = lds_u32(stage, (at + lane) & SM);
            const uint32_t hl = (h >> 4) & 15u, lb = (h >> 8) & 255u;
            const int32_t adv = 3 + (int32_t)hl + (hl == 15 ? (int32_t)lb + 1 : 0) + ((h & 15u) == 15 ? 1 : 0);
            const bool ok = (!((hl == 15) & (lb == 255)) & (adv <= iend - at - lane) & (lane < WIN)) != 0;
            const int32_t to = ok ? min(lane + adv, WIN) : lane;
            const int32_t to2 = bperm(to, to);
            uint64_t starts = 0;
            int32_t l = 0, t1;
            do {
              t1 = (int32_t)rdlane((uint32_t)to, l);
              bit_on(starts, l);
              bit_on(starts, t1);
              l = (int32_t)rdlane((uint32_t)to2, l);
            } while (l != t1);
            bit_off(starts, l);  // where it ends is no start: a stop, or past the window
            stopped = l < WIN;
            if (starts == 0) break;
            const int32_t k = bits_below(starts, n);
            if ((starts >> lane) & 1ull) list[k] = (uint16_t)(at - ip + lane);
            n += __builtin_popcountll(starts);
            const int32_t last = 63 - __builtin_clzll(starts);
            at += last + (int32_t)rdlane((uint32_t)adv, last);
          } while (!stopped && at - ip < 3 * WIN);  // a window leads past its 63 positions
          if (n == 0) {
            general = true;
            break;
          }
          __builtin_amdgcn_wave_barrier();
          // lane k takes sequence k
          const int32_t pos = ip + (int32_t)list[lane];
          const uint32_t h = lds_u32(stage, pos & SM);
          const uint32_t hl = (h >> 4) & 15u, hm = h & 15u, lb = (h >> 8) & 255u;
          const uint32_t lext = hl == 15 ? 1u : 0u;  // one literal length byte
          const int32_t lit = (int32_t)(hl + (lext ? lb : 0u));
          const int32_t src = pos + 1 + (int32_t)lext;  // first literal
          const uint32_t h2 = lds_u32(stage, (src + lit) & SM);
          const int32_t hoff = (int32_t)(h2 & 0xffffu);
          const uint32_t he = (h2 >> 16) & 255u;
          const uint32_t ext = hm == 15 ? 1u : 0u;  // one match length byte
          const int32_t len = lit + (int32_t)(hm + 4 + (ext ? he : 0u));
          const bool mine = lane < n;
          const int32_t oinc = wave_inclusive_sum(mine ? len : 0);
          const int32_t os = oinc - len;  // this sequence's first output byte, from op
          // the first sequence that does not fit, or ends in a second length byte
          const bool hard =
              (((ext != 0) & (he == 255)) | (hoff < 1) | (hoff > op + os + lit) | (oinc > oend - op)) != 0;
          const uint64_t cutm = ballot(mine & (hard | (oinc > G::kOut)));
          const uint64_t hardm = ballot(hard);
          int32_t nseq = n;
          if (cutm) {
            nseq = __builtin_ctzll(cutm);
            stopped = ((hardm >> nseq) & 1ull) != 0;
            at = (int32_t)rdlane((uint32_t)pos, nseq);
            if (nseq == 0) {
              general = true;
              break;
            }
          }
          const int32_t total = (int32_t)rdlane((uint32_t)oinc, nseq - 1);
          if (lane < nseq) {
            // byte x of the output is a literal below `os + lit`
            tab[lane] =
                (uint64_t)((uint32_t)(os + lit) | ((uint32_t)hoff << 16)) | ((uint64_t)(uint32_t)(src - os) << 32);
            const int32_t ob = (os - 1) & (G::kOut - 1);
            atomicOr(obits + (ob >> 5), 1u << (ob & 31));
          }
          __builtin_amdgcn_wave_barrier();
          const uint64_t *words = reinterpret_cast<const uint64_t *>(obits);
          const uint64_t ob = lane < G::kOut / 64 ? words[lane & (G::kOut / 64 - 1)] : 0ull;
          int32_t before = 0;  // sequences that start in earlier steps, or with this one, less one
          auto entry_of = [&](int32_t x0) -> uint64_t {
            const uint64_t m = ((uint64_t)rdlane((uint32_t)(ob >> 32), x0 >> 6) << 32) | rdlane((uint32_t)ob, x0 >> 6);
            const int32_t k = bits_below(m, before);  // the last start at or before its byte
            before += __builtin_popcountll(m);
            return tab[k];
          };
          uint64_t e = entry_of(0);
          for (int32_t x0 = 0;;) {
            const int32_t x = x0 + lane;
            const uint32_t elo = (uint32_t)e;
            const int32_t im = x - (int32_t)(elo & 0xffffu);  // byte of the match, negative in the literals
            int32_t off = (int32_t)(elo >> 16);
            const int32_t lat = RING + ((x + (int32_t)(uint32_t)(e >> 32)) & SM);
            int32_t sp = op + x - off;
            // a source past the ring, inside the match itself or inside this step
            const bool odd = (im >= 0) & (x < total) & ((off > NEAR1) | (off <= max(im, lane)));
            const int32_t x1 = x0 + 64;
            uint32_t v;
            if (ballot(odd)) {
              if (odd & (im >= off)) {
                // (im + 1/2) / off is at least 1/546 away from a whole number
                const int32_t turn = (int32_t)(((float)im + 0.5f) * __builtin_amdgcn_rcpf((float)off));
                off = (int32_t)__umul24((uint32_t)off, (uint32_t)(turn + 1));
              }
              sp = op + x - off;
              v = lds[im < 0 ? lat : sp & RM];
              if (x1 < total) e = entry_of(x1);
              // at most FLUSH_AT + kOut bytes are pending, so a far source was
              // flushed, by this wavefront's own stores
              if (odd & (off > NEAR1)) v = slot_byte(sp);  // arrived, here and not where the paths meet
              const bool dep = odd & (off <= lane);
              if (ballot(dep)) {
                // bit 6: the lane has its own byte
                int32_t code = dep ? lane - off : lane | 64;
                do {
                  code = bperm(code, code);
                } while (ballot(code < 64));
                v = (uint32_t)bperm(code, (int32_t)v);
              }
            } else {
              v = lds[im < 0 ? lat : sp & RM];
              if (x1 < total) e = entry_of(x1);
            }
            __builtin_amdgcn_wave_barrier();
            ring[(op + x) & RM] = (uint8_t)v;
            __builtin_amdgcn_wave_barrier();
            if (x1 >= total) break;
            x0 = x1;
          }
          op += total;
          ip = at;
          asm volatile("" : "+v"(ahead));  // arrived; what follows is stored without a wait
          if (more) {
            put_stage(have, ahead);
            have += 256;
          }
          if (SIDEWAYS && side_n > 0) {
            side_store(16 * lane, side);
            side_src += SIDE;
            side_dst += SIDE;
            side_n -= SIDE;
          }
          if (op >= flush_at) {
            flush(op);
            rank(ip);
          }
          if (stopped) {
            general = true;
            break;
          }
        }
      } else {
        uint16_t *rec = reinterpret_cast<uint16_t *>(lds + G::kRecAt);
        uint32_t *exits = reinterpret_cast<uint32_t *>(lds + G::kExitAt);
        unsigned long long *cut = reinterpret_cast<unsigned long long *>(lds + G::kCutAt);
        int32_t base = ip, entry = 0, buf = 0;
        if (tid < G::kStageWords) reinterpret_cast<uint32_t *>(stage)[tid] = ld_word(base, tid);
        lds_barrier();
        for (;;) {
          const int32_t nbase = base + 64 * NW;
          uint32_t ahead = 0;  // the next round's input, on its way until the end of this one
          if (tid < G::kStageWords) ahead = ld_word(nbase, tid);
          if (tid < G::kOut / 32) obits[tid] = 0;
          if (tid == 0) *cut = ~0ull;
          // headers
          const int32_t st = RING + buf * G::kStage + (base & 3);
          const uint32_t h = lds_u32(lds, st + tid);
          const uint32_t hl = (h >> 4) & 15u, hm = h & 15u, lb = (h >> 8) & 255u;
          const uint32_t lext = hl == 15 ? 1u : 0u;  // one literal length byte
          const int32_t lit = (int32_t)(hl + (lext ? lb : 0u));
          const int32_t src = tid + 1 + (int32_t)lext;  // first literal, from base
          const uint32_t h2 = lds_u32(lds, st + min(src + lit, G::kStage - 8));
          const int32_t hoff = (int32_t)(h2 & 0xffffu);
          const uint32_t he = (h2 >> 16) & 255u;
          const uint32_t ext = hm == 15 ? 1u : 0u;  // one match length byte
          const int32_t len = lit + (int32_t)(hm + 4 + (ext ? he : 0u));
          const int32_t adv = 3 + lit + (int32_t)(lext + ext);
          // (bitwise: one vector compare chain, no branches)
          const bool ok = (!(lext & (lb == 255)) & !(ext & (he == 255)) & (hoff >= 1) &
                           (adv <= iend - base - tid)) != 0;
          const uint64_t okm = ballot(ok);
          // reach: bits 0..9 the lane the chain from here has got to (64 and more
          // is a position of a later window; a start that is not ok leads to
          // itself), bits 10..26 the output bytes and bits 27..31 the sequences on
          // the way (at most 22 of 542 bytes; over all windows kSeqs of them)
          static_assert((64 + 2) / 3 < 32 && G::kSeqs * kSeqOut < 1 << 17, "they fit their fields");
          static_assert(63 + kSeqIn + 64 * (NW - 1) < 1024, "and the position");
          uint32_t way = ok ? (uint32_t)(lane + adv) | ((uint32_t)len << 10) | (1u << 27) : (uint32_t)lane;
          auto hop = [&]() {
            const uint32_t f = (uint32_t)bperm((int32_t)way, (int32_t)way);
            if ((way & 1023u) < 64) way = f + (way & ~1023u);
          };
          uint64_t pass = 1ull << lane;  // the starts of the next eight hops
          auto join = [&]() {
            const uint32_t lo = (uint32_t)bperm((int32_t)way, (int32_t)(uint32_t)pass);
            const uint32_t hi = (uint32_t)bperm((int32_t)way, (int32_t)(uint32_t)(pass >> 32));
            if ((way & 1023u) < 64) pass |= ((uint64_t)hi << 32) | lo;
          };
          {
            const uint32_t to = way & 1023u;
            if (to < 64) pass |= 1ull << to;
          }
          hop();
          join();
          hop();
          join();
          hop();
          const uint32_t to8 = way & 1023u;
          const uint32_t way8 = to8 == (uint32_t)lane ? 64u : to8;  // below 64: go on from there
          hop();
          hop();
          exits[tid] = way + 64 * wave;  // positions from base
          lds_barrier();
          // chain: a stop stays in its window, where no later step takes it up.
          // Lane v of `at` and `past` is where window v is entered, and the bytes
          // (17 bits) and sequences before it.
          uint32_t ex[NW];
#pragma unroll
          for (int v = 0; v < NW; v++) ex[v] = exits[64 * v + lane];
          uint32_t e = (uint32_t)entry, sum = 0;
          uint32_t at = 0, past = 0;
#pragma unroll
          for (int v = 0; v < NW; v++) {
            const uint32_t x = rdlane(ex[v], (int32_t)(e & 63u));
            set_lane(at, v, e);
            set_lane(past, v, sum);
            const uint32_t y = (e >> 6) == (uint32_t)v ? x : e;
            sum += y >> 10;
            e = y & 1023u;
          }
          asm("s_nop 1" : "+v"(at), "+v"(past));  // before lanes written in asm are read
          const int32_t mine_at = (int32_t)rdlane(at, wave);
          const uint32_t before_me = rdlane(past, wave);
          const int32_t obase = (int32_t)(before_me & 0x1ffffu), kbase = (int32_t)(before_me >> 17);
          int32_t total = (int32_t)(sum & 0x1ffffu);
          int32_t stop = e < 64 * NW ? (int32_t)e : -1;
          if (stop == entry) {  // the first sequence is not one for a round
            ip = base + entry;
            general = true;
            break;
          }
          // walk
          uint64_t starts = 0;
          if (mine_at >> 6 == wave) {
            int32_t l = mine_at & 63;
            do {
              starts |= ((uint64_t)rdlane((uint32_t)(pass >> 32), l) << 32) | rdlane((uint32_t)pass, l);
              l = (int32_t)rdlane(way8, l);
            } while (l < 64);
            starts &= okm;
          }
          // scan
          const bool mine = ((starts >> lane) & 1ull) != 0;
          const int32_t oinc = obase + wave_inclusive_sum(mine ? len : 0);
          const int32_t os = oinc - len;  // this sequence's first output byte, from op
          if (mine) {
            const bool hard = (oinc > oend - op) | (hoff > op + os + lit);
            if (hard | (oinc > G::kOut)) {
              atomicMin(cut, ((unsigned long long)tid << 32) | ((uint32_t)os << 1) | (hard ? 1u : 0u));
            } else {
              // table: byte x of the output is a literal below `os + lit`
              tab[bits_below(starts, kbase)] =
                  (uint64_t)((uint32_t)(os + lit) | ((uint32_t)hoff << 16)) | ((uint64_t)(uint32_t)(src - os) << 32);
              const int32_t ob = (os - 1) & (G::kOut - 1);
              atomicOr(obits + (ob >> 5), 1u << (ob & 31));
            }
          }
          lds_barrier();
          // output: lane q of a wavefront holds the bits of bytes 64 q .. 64 q + 63
          // and the number of sequences that start before them
          const uint64_t ob = reinterpret_cast<const uint64_t *>(obits)[lane & (G::kOut / 64 - 1)];
          const uint64_t c = *cut;
          const uint32_t clo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)c),
                         chi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(c >> 32));
          const bool is_cut = chi != ~0u;
          if (is_cut) {
            total = (int32_t)(clo >> 1);
            stop = (int32_t)chi;
            general = (clo & 1u) != 0;
            if (total == 0) {  // the first sequence itself (never for its length alone)
              ip = base + stop;
              general = true;
              break;
            }
          } else {
            general = stop >= 0;
          }
          const int32_t own = __builtin_popcountll(ob);
          const int32_t before = wave_inclusive_sum(own) - own;
          for (int32_t x0 = 0; x0 < total; x0 += 2 * NT) {
            // bit 15 and the byte, or the number of the source byte
            uint32_t w[2] = {0x8000u, 0x8000u};
            auto entry_of = [&](int32_t xw) -> uint64_t {  // the last sequence that starts at or before the byte
              const int32_t q = xw >> 6;
              const uint64_t m = ((uint64_t)rdlane((uint32_t)(ob >> 32), q) << 32) | rdlane((uint32_t)ob, q);
              return tab[bits_below(m, (int32_t)rdlane((uint32_t)before, q))];
            };
            auto source_of = [&](int32_t x, uint64_t en) -> uint32_t {
              const uint32_t elo = (uint32_t)en;
              const int32_t im = x - (int32_t)(elo & 0xffffu);  // byte of the match, negative in the literals
              int32_t off = (int32_t)(elo >> 16);
              const bool live = (im >= 0) & (x < total);
              const bool far = live & (off > NEAR);
              if (live & (im >= off)) {
                // (im + 1/2) / off is at least 1/546 away from a whole number
                const int32_t turn = (int32_t)(((float)im + 0.5f) * __builtin_amdgcn_rcpf((float)off));
                off = (int32_t)__umul24((uint32_t)off, (uint32_t)(turn + 1));
              }
              const int32_t sp = x - off;  // source byte of a match, from op
              const int32_t lat = st + x + (int32_t)(uint32_t)(en >> 32);
              const int32_t rat = (op + sp) & RM, lm = im >> 31;
              uint32_t v = lds[(lat & lm) | (rat & ~lm)];
              if (far) {
                v = dst[op + sp];
                asm volatile("" : "+v"(v));  // arrived, here and not where the paths meet
              }
              return (live & (sp >= x0)) ? (uint32_t)(sp - x0) : 0x8000u | v;
            };
            const int32_t xw = x0 + 64 * wave;
            if (xw + NT < total) {
              const uint64_t e0 = entry_of(xw), e1 = entry_of(xw + NT);
              w[0] = source_of(xw + lane, e0);
              w[1] = source_of(xw + NT + lane, e1);
              rec[tid] = (uint16_t)w[0];
              rec[NT + tid] = (uint16_t)w[1];
            } else if (xw < total) {
              w[0] = source_of(xw + lane, entry_of(xw));
              rec[tid] = (uint16_t)w[0];
            }
            lds_barrier();
#pragma unroll
            for (int u = 0; u < 2; u++) {
              uint16_t *mine = rec + NT * u + tid;
              while (ballot(w[u] < 0x8000u)) {
                // (one that has its byte reads it again)
                const uint16_t *at = w[u] < 0x8000u ? rec + w[u] : mine;
                w[u] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_store(mine, (uint16_t)w[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              }
              const int32_t x = x0 + NT * u + tid;
              if (x < total) ring[(op + x) & RM] = (uint8_t)w[u];
            }
            if (x0 + 2 * NT >= total) {
              asm volatile("" : "+v"(ahead));  // arrived, in every wavefront
              if (tid < G::kStageWords) reinterpret_cast<uint32_t *>(stage + (buf ^ 1) * G::kStage)[tid] = ahead;
            }
            lds_barrier();
          }
          op += total;
          if (op >= flush_at) {
            flush(op);
            rank(base);
          }
          if (stop >= 0) {
            ip = base + stop;
            if (general) break;
            entry = stop;  // cut: the rest of the same positions
            continue;
          }
          if (e >= 128 * NW) {  // past all of the next round
            ip = base + (int32_t)e;
            break;
          }
          base = nbase;
          entry = (int32_t)e - 64 * NW;
          buf ^= 1;
        }
      }
    }
    if (!general) continue;  // cut where the round's output was full
    // ---- general path: one sequence.  Every wavefront keeps the 256 input
    // bytes from gb in a register and parses them alike.
    int32_t gb = 0;
    uint32_t gw = 0;
    auto look = [&](int32_t pos) {
      gb = pos & ~3;
      gw = ld_word(gb, lane);
    };
    auto rbyte = [&](int32_t pos) -> uint32_t {  // gb <= pos < gb + 256
      const int32_t q = pos - gb;
      return (rdlane(gw, q >> 2) >> ((q & 3) << 3)) & 0xffu;
    };
    // Adds the length continuation bytes from ip on (255s, then one below 255)
    // to v, 64 input bytes a step (a ballot finds the last one); false when the
    // stream ends first or the length exceeds the block.
    auto read_len = [&](int32_t &v) -> bool {
      for (;;) {
        if (ip + 64 > gb + 256) look(ip);
        const int32_t q = ip - gb + lane;
        const uint32_t b = ((uint32_t)bperm(q >> 2, (int32_t)gw) >> ((q & 3) << 3)) & 255u;
        const uint64_t stop = ballot(ip + lane < iend && b != 255u);
        if (stop) {
          const int32_t t = (int32_t)__builtin_ctzll(stop);
          v += 255 * t + (int32_t)rdlane(b, t);
          ip += t + 1;
          return true;
        }
        if (iend - ip < 64) return false;
        v += 255 * 64;
        ip += 64;
        if (v > oend) return false;
      }
    };
    // Writes n output bytes at op without the ring in between: what is pending
    // goes out first, then whole 16-byte groups are stored to the slot, the
    // next groups' bytes asked for before the last ones are stored; the last
    // RING bytes also go to the ring.  byte_of and group_of give byte i and
    // bytes i .. i + 15 of the n; groups before g0 are left out.
    auto bulk = [&](int32_t n, int32_t g0, auto byte_of, auto group_of) {
      flush(op);
      if (tid < op - flushed) dst[flushed + tid] = ring[(flushed + tid) & RM];
      lds_barrier();  // the ring is written below
      const int32_t keep = op + n - RING;                   // the ring holds positions from here
      const int32_t head = min((16 - (op & 15)) & 15, n);  // bytes up to the first whole group
      const int32_t ng = (n - head) >> 4;                   // whole groups after the head
      const int32_t bend = head + (ng << 4);
      uint8_t hb = 0, tb = 0;
      if (tid < head) hb = byte_of(tid);
      if (tid < n - bend) tb = byte_of(bend + tid);
      auto group_store = [&](int32_t g, u32x4 w) {
        const int32_t d = op + head + 16 * g;  // a multiple of 16
        if (wide) {
          *iamx::gptr<u32x4>((uint64_t)(dst + d)) = w;
        } else {
          dstw[d >> 2] = w.x;
          dstw[(d >> 2) + 1] = w.y;
          dstw[(d >> 2) + 2] = w.z;
          dstw[(d >> 2) + 3] = w.w;
        }
        if (d >= keep) {
          *reinterpret_cast<u32x4 *>(ring + (d & RM)) = w;
        } else if (d + 16 > keep) {  // the group the ring starts in
          for (int t = 0; t < 16; t++)
            if (d + t >= keep) ring[(d + t) & RM] = (uint8_t)(w[t >> 2] >> (8 * (t & 3)));
        }
      };
      u32x4 wa, wb;
      if (g0 + tid < ng) wa = group_of(head + 16 * (g0 + tid));
      for (int32_t g = g0 + tid; g < ng; g += 2 * NT) {
        if (g + NT < ng) wb = group_of(head + 16 * (g + NT));
        group_store(g, wa);
        if (g + 2 * NT < ng) wa = group_of(head + 16 * (g + 2 * NT));
        if (g + NT < ng) group_store(g + NT, wb);
      }
      auto put_byte = [&](int32_t i, uint8_t v) {
        dst[op + i] = v;
        if (op + i >= keep) ring[(op + i) & RM] = v;
      };
      if (tid < head) put_byte(tid, hb);
      if (tid < n - bend) put_byte(bend + tid, tb);
      op += n;
      flushed = __builtin_amdgcn_readfirstlane(op & ~15);
      flush_at = flushed + FLUSH_AT;
      if (NW > 1) drain();
      lds_barrier();
    };
    // the next sequence has a second length byte: its literals', or its match's
    // after literals without one (a round would stop at it at once)
    auto long_next = [&]() -> bool {
      if (ip + 20 > gb + 256) return false;
      const uint32_t t = rbyte(ip), l = t >> 4;
      return l == 15 ? rbyte(ip + 1) == 255u : (t & 15u) == 15 && rbyte(ip + 3 + (int32_t)l) == 255u;
    };
    if (ip >= iend) { bad = 1; break; }
    look(ip);
    const uint32_t token = rbyte(ip);
    ++ip;
    int32_t lit = (int32_t)(token >> 4);
    if (lit == 15 && !read_len(lit)) { bad = 2; break; }
    if (lit > iend - ip || lit > oend - op) { bad = 3; break; }
    lds_barrier();  // no wavefront still reads the LDS of the last round
    if (lit > 0) {
      if (lit <= NT) {
        if (ip - gb + lit <= 256) {
          const int32_t q = ip - gb + tid;
          const uint32_t b = (uint32_t)bperm(q >> 2, (int32_t)gw) >> ((q & 3) << 3);
          if (tid < lit) ring[(op + tid) & RM] = (uint8_t)b;
        } else if (tid < lit) {
          ring[(op + tid) & RM] = sb[ip + tid];
        }
        lds_barrier();
        ip += lit;
        op += lit;
        if (op >= flush_at) flush(op);
      } else {
        look(ip + lit);  // for what follows the run
        const IAMX_GLOBAL uint8_t *from = sb + ip;
        int32_t g0 = 0;
        if (SIDEWAYS && wide) {
          const int32_t head = (16 - (op & 15)) & 15, before = (lit - RING - head) & ~(SIDE - 1);
          if (before >= 4 * SIDE) {
            side_finish();
            side_n = run_n = before;
            side_src = ip + head;
            side_dst = run_at = op + head;
            run_in = ip - op;
            g0 = before >> 4;
          }
        }
        bulk(
            lit, g0, [&](int32_t i) -> uint8_t { return from[i]; },
            [&](int32_t i) -> u32x4 { return *(const IAMX_GLOBAL u32x4_any *)(from + i); });
        ip += lit;
      }
    }
    if (ip == iend) break;  // last sequence: literals only
    if (iend - ip < 2) { bad = 4; break; }
    if (ip + 2 > gb + 256) look(ip);
    const int32_t off = (int32_t)(rbyte(ip) | (rbyte(ip + 1) << 8));
    ip += 2;
    int32_t ml = (int32_t)(token & 15u);
    if (ml == 15 && !read_len(ml)) { bad = 5; break; }
    ml += 4;
    if (off == 0 || off > op || ml > oend - op) { bad = 6; break; }
    if (ml >= 512 && off <= 16 && (off & (off - 1)) == 0) {
      // the match repeats 1, 2, 4, 8 or 16 bytes: every whole 16-byte group of
      // the output is the same one
      const int32_t m0 = op - off;  // byte i of the output is byte m0 + (i - op) mod off
      const uint32_t b = ring[(m0 + ((lane - op) & (off - 1))) & RM];  // of an i that is lane mod 16
      u32x4 w;
#pragma unroll
      for (int t = 0; t < 4; t++)
        w[t] = rdlane(b, 4 * t) | (rdlane(b, 4 * t + 1) << 8) | (rdlane(b, 4 * t + 2) << 16) | (rdlane(b, 4 * t + 3) << 24);
      const int32_t op0 = op;
      bulk(
          ml, 0,
          [&](int32_t i) -> uint8_t {
            const int32_t j = (op0 + i) & 15;
            const uint32_t lo = j & 4 ? w.y : w.x, hi = j & 4 ? w.w : w.z;
            return (uint8_t)((j & 8 ? hi : lo) >> (8 * (j & 3)));
          },
          [&](int32_t) -> u32x4 { return w; });
      general = NW > 1 && long_next();
      continue;
    }
    if (SIDEWAYS && off > NEAR) side_finish();
    // kStep bytes a step: byte i of a step is byte (i mod off) of the `off`
    // bytes before the step
    {
      constexpr int U = G::kStep / NT;
      int32_t at[U];  // source of this thread's bytes, from the step's first byte less off
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int32_t i = NT * u + tid;
        // i < 4096: (i + 1/2) / off is at least 1/8192 of a turn from a whole number
        const int32_t turn = off > i ? 0 : (int32_t)(((float)i + 0.5f) / (float)off);
        at[u] = i - turn * off;
      }
      for (int32_t k = 0; k < ml; k += G::kStep) {
        uint8_t v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int32_t s = op + k - off + at[u];
          v[u] = 0;
          if (k + NT * u + tid < ml) v[u] = off > NEAR ? dst[s] : ring[s & RM];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
          if (k + NT * u + tid < ml) ring[(op + k + NT * u + tid) & RM] = v[u];
        lds_barrier();
        const int32_t cur = op + min(ml, k + G::kStep);
        if (cur >= flush_at) flush(cur);
      }
      op += ml;
    }
    general = NW > 1 && long_next();
  }
  if (!bad && op != oend) bad = 7;
  if (!bad) {  // the slot is padded to 4 bytes at least
    if (SIDEWAYS) side_finish();
    flush(oend);
    const int32_t p = flushed + 4 * tid;
    if (p < oend) dstw[p >> 2] = *reinterpret_cast<const uint32_t *>(ring + (p & RM));
  }
  if (bad && tid == 0) atomicOr(status, 1 << bad);
}

// One BloscLZ stream by one wavefront (the stream format is restated in the
// oracle, oracle/blosclz_block.c, from c-blosc's compressor output): a
// control byte per token, literal runs of up to 32 bytes, matches of 3 or
// more bytes at distances up to 8191 + 1, or 8192 + 65535 through the
// far-distance escape.  The parse is uniform (a 256-byte register window of
// the input, bytes taken with readlane); every output byte is written to the
// scratch slot and to the LDS history ring.  Matches within RING - 64 bytes
// copy ring to ring in steps of min(distance, 64) bytes; farther ones read
// the slot in global memory after a release/acquire fence (again before
// every step that reads bytes of the same match).
template <int RING>
__device__ __forceinline__ void blosclz_stream(const iamx_lz4_job_t job, uint8_t *__restrict__ scratch,
                                               int *status, uint8_t *ring) {
  constexpr int32_t RM = RING - 1;
  const int lane = threadIdx.x;
  const uint64_t abase = job.src & ~3ull;
  const IAMX_GLOBAL uint32_t *__restrict__ sw = iamx::gptr<const uint32_t>(abase);
  const IAMX_GLOBAL uint8_t *__restrict__ sb = iamx::gptr<const uint8_t>(abase);
  IAMX_GLOBAL uint8_t *dst = iamx::gptr<uint8_t>((uint64_t)(scratch + job.dst_off));
  int32_t ip = (int32_t)(job.src & 3);
  const int32_t iend = ip + job.csize, oend = job.nbytes;
  const int32_t lastw = (iend - 1) >> 2;
  int32_t wb = 0;
  uint32_t w = sw[min(lane, lastw)];
  auto byte_at = [&](int32_t pos) -> uint32_t {  // pos uniform, pos < iend
    if (pos - wb >= 256) {
      wb = pos & ~3;
      w = sw[min((wb >> 2) + lane, lastw)];
    }
    const int32_t q = pos - wb;
    return (rdlane(w, q >> 2) >> ((q & 3) << 3)) & 0xffu;
  };
  auto fence = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  int32_t op = 0;
  int bad = 0;
  uint32_t ctrl = byte_at(ip++) & 31u;
  for (;;) {
    if (ctrl >= 32) {
      int32_t len = (int32_t)(ctrl >> 5) - 1;
      int32_t dist = (int32_t)(ctrl & 31) << 8;
      if (len == 6) {
        uint32_t code;
        do {
          if (ip >= iend || len > oend) { bad = 1; break; }
          code = byte_at(ip++);
          len += (int32_t)code;
        } while (code == 255);
        if (bad) break;
      }
      if (ip >= iend) { bad = 1; break; }
      const uint32_t code = byte_at(ip++);
      len += 3;
      if (code == 255 && dist == (31 << 8)) {
        if (iend - ip < 2) { bad = 1; break; }
        dist = (int32_t)((byte_at(ip) << 8) | byte_at(ip + 1)) + 8192;
        ip += 2;
      } else {
        dist += (int32_t)code + 1;
      }
      if (dist > op || len > oend - op) { bad = 1; break; }
      if (dist <= RING - 64) {
        const int32_t step = min(dist, 64);
        for (int32_t k = 0; k < len; k += step) {
          const int32_t j = k + lane;
          const bool on = lane < step && j < len;
          uint8_t v = 0;
          if (on) v = ring[(op + j - dist) & RM];
          __builtin_amdgcn_wave_barrier();
          if (on) {
            ring[(op + j) & RM] = v;
            dst[op + j] = v;
          }
          __builtin_amdgcn_wave_barrier();
        }
      } else {
        fence();
        for (int32_t k = 0; k < len; k += 64) {
          if (k + 64 > dist) fence();  // this step reads bytes of this match
          const int32_t j = k + lane;
          if (j < len) {
            const uint8_t v = dst[op + j - dist];
            ring[(op + j) & RM] = v;
            dst[op + j] = v;
          }
          __builtin_amdgcn_wave_barrier();
        }
      }
      op += len;
    } else {
      const int32_t len = (int32_t)ctrl + 1;
      if (len > iend - ip || len > oend - op) { bad = 1; break; }
      if (lane < len) {
        const uint8_t v = sb[ip + lane];
        ring[(op + lane) & RM] = v;
        dst[op + lane] = v;
      }
      __builtin_amdgcn_wave_barrier();
      ip += len;
      op += len;
    }
    if (ip >= iend) break;
    ctrl = byte_at(ip++);
  }
  if (!bad && op != oend) bad = 1;
  if (bad && lane == 0) atomicOr(status, IAMX_STATUS_BLOSCLZ);
}

constexpr int kBloscRing = 4096;

// the decoded stream, padded to 16 bytes, must lie inside the scratch
__device__ __forceinline__ bool in_scratch(const iamx_lz4_job_t &job, int64_t cap) {
  return job.dst_off >= 0 && job.nbytes >= 0 && job.dst_off <= cap - (((int64_t)job.nbytes + 15) & ~(int64_t)15);
}

template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 1 ? 7 : 8, 8))) void k_lz4_streams(
    const iamx_lz4_job_t *__restrict__ jobs, int njobs, uint8_t *__restrict__ scratch, int64_t cap, int *status,
    int zstd_on) {
  __shared__ __align__(16) uint8_t lds[Lz4Geom<NW>::kLds];
  const int j = blockIdx.x;
  if (j >= njobs) return;
  const iamx_lz4_job_t job = jobs[j];
  if (!in_scratch(job, cap)) {
    if (threadIdx.x == 0) atomicOr(status, IAMX_STATUS_RANGE);
    return;
  }
  if (job.codec == IAMX_CODEC_BLOSCLZ) {
    if (threadIdx.x < 64) blosclz_stream<kBloscRing>(job, scratch, status, lds);
    return;
  }
  if (job.codec == IAMX_CODEC_ZSTD) {  // decoded by a pass of its own
    if (!zstd_on && threadIdx.x == 0) atomicOr(status, IAMX_STATUS_CODEC);
    return;
  }
  if (job.codec != IAMX_CODEC_LZ4) {  // no decoder for this codec
    if (threadIdx.x == 0) atomicOr(status, IAMX_STATUS_CODEC);
    return;
  }
  if (job.csize <= 0) {  // nothing to read: ends before its first token
    if (threadIdx.x == 0) atomicOr(status, 1 << 1);
    return;
  }
  // half the first job's input (the longest where they are sorted), or of a typical long one
  const int32_t ahead_at = min(jobs[0].csize / 2, 24576);
  if constexpr (NW == 1) {  // long, or a literal run of 8 KB or more to begin with (32 length bytes of 255)
    const uint8_t *in = reinterpret_cast<const uint8_t *>(job.src);
    const int i = min((int)threadIdx.x, 32);
    if (job.csize >= 65536 || (job.csize > 8192 && ballot(in[i] < (i ? 255 : 0xf0)) == 0)) {
      lz4_stream<1, true>(job, scratch, status, lds, ahead_at);
      return;
    }
  }
  lz4_stream<NW>(job, scratch, status, lds, ahead_at);
}

// BloscLZ streams alone, 32 a CU.  Beside LZ4 streams (above) each holds that
// kernel's LDS, which lets 25 of one wavefront into a CU; a stream is bound by
// its own chain of tokens, so the time goes with how many are there.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_blosclz_streams(
    const iamx_lz4_job_t *__restrict__ jobs, int njobs, uint8_t *__restrict__ scratch, int64_t cap, int *status) {
  __shared__ __align__(16) uint8_t ring[kBloscRing];
  const int j = blockIdx.x;
  if (j >= njobs) return;
  const iamx_lz4_job_t job = jobs[j];
  if (!in_scratch(job, cap)) {
    if (threadIdx.x == 0) atomicOr(status, IAMX_STATUS_RANGE);
  } else if (job.codec != IAMX_CODEC_BLOSCLZ) {
    if (threadIdx.x == 0) atomicOr(status, IAMX_STATUS_CODEC);
  } else {
    blosclz_stream<kBloscRing>(job, scratch, status, ring);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_transpose(int64_t rows, int64_t cols, const T *__restrict__ src,
                                                   T *__restrict__ dst) {
  __shared__ T tile[32][33];
  const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;  // 32 x 8
  for (int i = ty; i < 32; i += 8) {
    const int64_t r = r0 + i, c = c0 + tx;
    if (r < rows && c < cols) tile[i][tx] = src[r * cols + c];
  }
  __syncthreads();
  for (int i = ty; i < 32; i += 8) {
    const int64_t c = c0 + i, r = r0 + tx;  // dst is cols x rows
    if (r < rows && c < cols) dst[c * rows + r] = tile[tx][i];
  }
}

}  // namespace

namespace iamx {

// Wavefronts per stream, by how many streams a CU gets.  A stream's time is set
// by its own chain of rounds, so few streams are spread over many wavefronts
// each; many streams hide each other's waits, and one wavefront decodes a
// sequence with the fewest instructions.  The first line is where a CU still
// holds all of its streams at once with 8 wavefronts (4 x 8), the second where
// 4 wavefronts, in one and a half loads of a CU (8 x 4), are overtaken.
// Measured in us with 8 / 4 / 1 wavefronts on bitshuffled float32 streams of 250
// KB: 4 streams 134 / 205 / 451, 1024 streams 290 / 332 / 606, 1280 streams 392
// / 366, 2048 streams 521 / 471 / 675, 3072 streams - / 745 / 743, 4096 streams
// - / 852 / 828, 6400 streams - / 1381 / 1076; exponent planes of float32 (64
// KB): 4 streams 222 / 387 / 891, 1024 streams 371 / 500 / 1038, 1280 streams
// 556 / 540, 2048 streams 706 / 658 / 1116, 3072 streams - / 1090 / 1194, 4096
// streams - / 1267 / 1273, 6400 streams - / 2101 / 1550; a ragged matrix's
// bitshuffled float64 streams: 3072 streams - / 510 / 1011, equal ones - / 282 /
// 232; byte planes of 16 KB of float64: 3072 streams - / 244 / 255, 4096 streams
// - / 292 / 275.  So around the second line the count alone does not decide:
// streams of unlike length want more wavefronts than equal ones, by up to twice
// the time, and the jobs' sizes do not tell the two apart (lines at 24 streams a
// CU, or four wavefronts for the longest 12 a CU, won 10 to 40% on the one and
// lost as much on the other).
int launch_lz4(const char *name, const iamx_lz4_job_t *d_lz4, int n_lz4, void *d_scratch, int64_t cap) {
  const int z = zstd_enabled() ? 1 : 0;
  if (n_lz4 <= 4 * g_num_cus)
    IAMX_LAUNCH(name, k_lz4_streams<8>, dim3(n_lz4), dim3(512), 0, d_lz4, n_lz4, (uint8_t *)d_scratch, cap,
                status_word(), z);
  else if (n_lz4 <= 12 * g_num_cus)
    IAMX_LAUNCH(name, k_lz4_streams<4>, dim3(n_lz4), dim3(256), 0, d_lz4, n_lz4, (uint8_t *)d_scratch, cap,
                status_word(), z);
  else
    IAMX_LAUNCH(name, k_lz4_streams<1>, dim3(n_lz4), dim3(64), 0, d_lz4, n_lz4, (uint8_t *)d_scratch, cap,
                status_word(), z);
  if (z) return launch_zstd("zstd_streams", d_lz4, n_lz4, d_scratch, cap);
  return IAMX_OK;
}

}  // namespace iamx

extern "C" {

IAMX_API int iamx_decode(const iamx_lz4_job_t *d_lz4, int n_lz4, const iamx_block_job_t *d_blocks, int n_blocks,
                         void *d_scratch, void *d_dst) {
  int rc = iamx::ensure_init();
  if (rc) return rc;
  if (n_lz4 < 0 || n_blocks < 0) return iamx::set_error(IAMX_EINVAL, "iamx_decode: negative job count");
  if (n_lz4 > 0)
    rc = iamx::launch_lz4("lz4_streams", d_lz4, n_lz4, d_scratch);
  if (rc) return rc;
  if (n_blocks > 0)
    rc = iamx::launch_unfilter(d_blocks, n_blocks, d_scratch, d_dst);
  return rc;
}

// The line is launch_lz4's to one wavefront a stream.  Measured in us, this
// kernel / beside LZ4, bit-shuffled float32 streams of up to 64 KB in split
// blocks: 2544 streams 1129 / 1083, 5724 1175 / 1268, 10176 1237 / 1331, 15900
// 1589 / 1822, 30528 2820 / 3290.
IAMX_API int iamx_decode_blosclz(const iamx_lz4_job_t *d_jobs, int n_jobs, void *d_scratch) {
  int rc = iamx::ensure_init();
  if (rc) return rc;
  if (n_jobs < 0) return iamx::set_error(IAMX_EINVAL, "iamx_decode_blosclz: negative job count");
  if (n_jobs == 0) return IAMX_OK;
  if (n_jobs <= 12 * iamx::g_num_cus) return iamx::launch_lz4("lz4_streams", d_jobs, n_jobs, d_scratch);
  IAMX_LAUNCH("blosclz_streams", k_blosclz_streams, dim3(n_jobs), dim3(64), 0, d_jobs, n_jobs, (uint8_t *)d_scratch,
              INT64_MAX, iamx::status_word());
  return IAMX_OK;
}

IAMX_API int iamx_transpose(int typesize, int64_t rows, int64_t cols, const void *d_src, void *d_dst) {
  int rc = iamx::ensure_init();
  if (rc) return rc;
  dim3 grid((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32));
  if (typesize == 8)
    IAMX_LAUNCH("transpose", k_transpose<uint64_t>, grid, dim3(256), 0, rows, cols, (const uint64_t *)d_src,
                (uint64_t *)d_dst);
  else if (typesize == 4)
    IAMX_LAUNCH("transpose", k_transpose<uint32_t>, grid, dim3(256), 0, rows, cols, (const uint32_t *)d_src,
                (uint32_t *)d_dst);
  else
    return iamx::set_error(IAMX_EINVAL, "iamx_transpose: typesize %d", typesize);
  return IAMX_OK;
}

}  // extern "C"
