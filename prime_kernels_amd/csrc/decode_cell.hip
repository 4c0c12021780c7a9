// SmolLM2-135M batched decode step (3..16 sequences) on cells of XCDs, one persistent kernel per step for
// gfx950 (MI355X).
//
// The 8 XCDs are grouped into cells of PX neighbouring XCDs (workgroup wg runs on XCD wg % 8 under
// round-robin dispatch; nothing below depends on that for correctness).  The sequences are dealt to
// the cells by context length, and a cell decodes its own sequences through every layer alone: its
// 32 PX workgroups hold all rows of every projection between them, so each weight matrix is read
// once per cell and an exchange reaches 32 PX workgroups and carries the cell's few sequences,
// instead of reaching all 256 with all of them.  Only the final hidden states cross cells, before
// the LM head, whose rows are split over all 256 workgroups.
//
// What bounds it: a step is a chain of seven exchanges per layer (x, qkv, softmax statistics, P.V
// partials, attention vector, h1, act).  Each is about 1 us from store to last arrival, and more
// when the poll queues behind the workgroup's own weight stream or brings in many sequences, so
// fewer sequences per poll and one round trip per exchange (payload and tag in one 16-byte unit, no
// store acknowledgement and no flag) are what the split buys, for (8 / PX) times the weight traffic (seven
// sequences of 2157..4002 tokens: 1,511 MB a step behind the L2s, 835 MB of them needed; 2.5 TB/s).
//
// Waves 0..3 of a workgroup are producers (LDS-DMA of every byte the workgroup reads, in order, into
// a ring), waves 4..7 consumers, as in the other decode kernels.  Ring packets are 1 KB: 8 rows x
// 128 bytes, row r's 16-byte piece c in slot (c + r) mod 8, for weight rows and cached tokens alike,
// so that an MFMA operand read touches 8 different bank groups with each 8 lanes.  A projection's
// packets run k-step by k-step over all of the workgroup's rows; consumer wave w takes its quarter of the k-steps
// into registers before the phase's input is waited for, and one LDS reduction, (w0 + w1) + (w2 + w3), ends the
// phase (deterministic).
//
// Exchange format: 16-byte units {two 32-bit words of payload (four bf16, the four consecutive rows
// a lane holds after v_mfma_f32_16x16x32_bf16) or three fp32 words, 32-bit tag}, one store and one
// load each (never seen torn: test_gpu_safety.py::test_exchange_units_are_never_torn).  The buffers
// are reused by every layer, which is safe because a buffer can only be written for layer l + 1 after
// every workgroup of the cell has read it for layer l (each exchange waits for units that depend on all
// of the previous exchange's readers).  A unit of two payload words says its layer and step epoch; one
// of three has a single word for both (CC::tag).
//
// Rounding points are those of HF eager Llama (modeling_llama.py), as in the other kernels.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

#include "pk_common.h"

namespace pk {
namespace cell {

constexpr int BMAX = 16;                   // sequences per step
constexpr uint32_t LDS_CU = 160u * 1024u;  // LDS of a CU (one workgroup each)
#ifndef PK_CELL_DEPTH
#define PK_CELL_DEPTH 4
#endif
#ifndef PK_CELL_TMIN
#define PK_CELL_TMIN 8
#endif
constexpr int DEPTH_C = PK_CELL_DEPTH;     // packets in flight per producer wave
constexpr int GRP = 32;                    // 6-value groups of a head group's 192 attention outputs

// How a cell splits its (sequence, KV head) pairs over its workgroups: in whole workgroups (geometry G itself), or
// end to end on a line of tiles that the workgroups share evenly (EndToEnd<G>).
template <class G>
struct EndToEnd : G {};
template <class G> constexpr bool end_to_end = false;
template <class G> constexpr bool end_to_end<EndToEnd<G>> = true;
constexpr int IPW_MAX = 8;                 // attention items per workgroup, at most (end to end)

// Geometry of a cell: PX XCDs, R workgroups, at most NS sequences.
template <class G, int PX>
struct CG {
  static constexpr int NC = 8 / PX;                      // cells
  static constexpr int R = 32 * PX;                      // workgroups per cell
  static constexpr int NS = BMAX / NC;                   // most sequences per cell
  static constexpr int HU = G::H / 4, IU = G::I / 4, QU = G::QKV / 4;  // units of a vector
  static constexpr int UQ = (QU + R - 1) / R, UO = (HU + R - 1) / R, UA = (IU + R - 1) / R;  // per workgroup
  static constexpr int TQ = (4 * UQ + 15) / 16, TO = (4 * UO + 15) / 16, TA = (UA + 1) / 2;  // MFMA tiles
  static constexpr int LMROWS = G::V / NWG, TL = LMROWS / 16;
  static constexpr bool E2E = end_to_end<G>;
  static constexpr int IPC = E2E ? IPW_MAX : 1;          // attention items per workgroup
  static constexpr int TM = E2E && TA < 6 ? 6 : TA;      // tiles of the LDS reduction (6: the items' P.V sums)
  static constexpr int KSH = G::H / 64, KSI = G::I / 64; // 64-wide k-steps
  static constexpr int XH = G::H + 8, XI = G::I + 8;     // staged row strides (bank spread)
  static constexpr uint32_t NSEG = 2 * PKT;              // ring bytes of a norm weight vector
  static constexpr int LU = (HU + 63) / 64;              // units of an H-vector per lane
  static constexpr int LA = (IU + NCT - 1) / NCT;        // act units per thread and sequence
  // Most tiles of a workgroup.  Whole workgroups: with T tiles a chunk, n pairs of together N tiles take at most
  // N / T + n workgroups.  End to end: its share of every sequence at the longest context, plus the padding of
  // short pairs (1/4 of a share each).  Items start at whole quads of tiles.
  static constexpr int NP = NS * G::KVH, NT_MAX = NP * ((kMaxSeq + 15) / 16);
  static constexpr int TILES = E2E ? NT_MAX / R + IPC : (NT_MAX + R - NP - 1) / (R - NP);
  static constexpr int SCT = E2E ? TILES * 16 + IPC * 64 : (TILES * 16 + 63) / 64 * 64;
  static_assert(NP < R && NP <= 64, "a workgroup for every pair, a lane for every pair");
  static_assert(NS <= NCW, "a wave for every sequence of the cell");
  static_assert(HU >= R && QU >= R && IU >= R, "rows of every projection for each workgroup (the producer divides by them)");
  static_assert(G::H % 64 == 0 && G::I % 64 == 0 && G::H % 4 == 0 && HU <= NCT, "whole k-steps and units");
  static_assert(G::V % (NWG * 16) == 0 && TL % NCW == 0, "LM-head tiles");
  static_assert(G::H * 2 <= int(NSEG) && HU <= NCT, "two packets of norm weights, one unit per thread");
  static_assert(TM * NCW * 256 >= IPC * NCW * 192 && TO <= TM && TQ <= TM, "the reduction buffer");
  static_assert(TQ <= NCW && NS * LA <= 32, "one QKV tile per wave; pending bits of the act poll");
  static_assert(R / G::KVH + 2 <= 64, "a lane for every chunk of a pair: a sequence's heads have equally many");
};

// Exchange region (units of 16 bytes from its base; one layout for both splits of the pairs, so that no unit is
// read in a format it was not written in): the workgroups' end records per sequence (tag: epoch), the
// vectors per sequence (tag: epoch, and the layer in the word before it; the attention vector: CC::tag), the
// attention records of each workgroup's items (statistics, 2 units; partial sums, 64 units; CC::tag).
enum CKind { C_X, C_ATT, C_H1, C_QKV, C_ACT };
template <class G>
struct CW {
  static constexpr int HU = G::H / 4, IU = G::I / 4, QU = G::QKV / 4;
  static constexpr uint32_t V0 = BMAX * NWG;
  // UPL units of a vector per 64-byte line; consecutive lines of a vector lie SLOTS lines apart, so
  // that its lines spread over the memory channels
  static constexpr uint32_t UPL = 4, LINES = (640 + UPL - 1) / UPL, SLOTS = BMAX * 5 + 1;
  static_assert(HU <= 640 && QU <= 640 && IU <= 640, "a vector's lines");
  static constexpr uint32_t REC0 = V0 + LINES * SLOTS * 4;
  static constexpr uint32_t REC = 66;
  static constexpr uint32_t TOTAL = REC0 + uint32_t(NWG) * IPW_MAX * REC;
  __device__ static uint32_t end(int b, int wg) { return (uint32_t(b) * NWG + uint32_t(wg)) * 16u; }
  // unit u of vector `kind` of sequence slot cs (cell * NS + slot): lane part and uniform part
  __device__ static uint32_t vec_u(int u) { return (V0 + uint32_t(u) / UPL * SLOTS * 4u + uint32_t(u) % UPL) * 16u; }
  static_assert(64 % UPL == 0, "units 64 apart lie a constant apart");
  static constexpr uint32_t STRIDE64 = 64 / UPL * SLOTS * 64u;
  __device__ static uint32_t vec_s(int kind, int cs) { return (uint32_t(cs) * 5u + uint32_t(kind)) * 64u; }
  __device__ static uint32_t rec(int wgkey, int k, int unit) {
    const uint32_t at = end_to_end<G> ? uint32_t(wgkey) * IPW_MAX + uint32_t(k) : uint32_t(wgkey);
    return (REC0 + at * REC + uint32_t(unit)) * 16u;
  }
};

// An attention item: a chunk (a run of 16-token tiles) of a (sequence, KV head) pair.
struct Item {
  int slot, b, g;        // sequence slot in the cell, global sequence, KV head
  int t0, n, ntile;      // first cached token, cached tokens and tiles of the chunk
  int tile0, quad0;      // tiles and quads (of 4 tiles) of the workgroup's items before this one
  int sc0;               // first score slot
  int r0, C, c, k0;      // first workgroup of the pair, its chunks, this one's index, item index in r0
  int leader;            // holds the pair's end: the new token
};

template <class G, int PX>
struct SmemRest {
  using S = CG<G, PX>;
  struct One {
    float wml[NCW][6];                    // per-wave softmax max / sum of the three heads
    alignas(16) uint16_t sc[3][S::SCT];   // bf16 scores, then probabilities, per head
  };
  struct Many {
    uint16_t q[S::IPC][5][64];            // roped q heads, new k (leaders), new v (leaders)
    float wml[S::IPC][NCW][6];
    float gml[S::IPC][6];                 // the pair's max and 1 / sum
    float snew[S::IPC][4];                // leaders: the new token's scores
    uint16_t sc[3][S::SCT];
  };
  using Attn = std::conditional_t<S::E2E, Many, One>;
  static constexpr int XN = S::NS * S::XI > BMAX * S::XH ? S::NS * S::XI : BMAX * S::XH;
  union {
    alignas(16) uint16_t xs[XN];          // staged activations [sequence][K + 8]
    Attn at;
  };
  alignas(16) float red[S::TM][NCW][256];  // per-wave MFMA partial tiles; attention: per-wave P.V sums [item][wave][192]
  uint2 res[S::NS][S::UO];                // residual rows of this workgroup (x, then h1)
  float sums[NCW][BMAX];
  LayerW lw[G::L];
  const void* kvp[G::L];
  Item it[S::IPC];
  int32_t blk[S::TILES + S::IPC];
  int32_t sid[BMAX];                      // the cell's sequences by slot
  int32_t cs[BMAX];                       // every sequence's exchange slot
  int32_t ns, ni, ntile;
  int32_t sS[BMAX], sPos[BMAX], sId[BMAX];
  long long sSlot[BMAX];
  float lm_val[NCW][BMAX];
  int32_t lm_idx[NCW][BMAX];
  alignas(16) uint32_t front[NPW];
  alignas(16) uint32_t consumed[NCW];
  uint32_t cbar;
};
// The ring takes what the rest and the diagnostic timestamps leave of the LDS, in whole packets: the
// further the stream runs ahead, the less of a phase's weights is still to come when its turn is there.
template <class G, int PX>
struct SmemC : SmemRest<G, PX> {
  static constexpr uint32_t RING_BYTES =
      (LDS_CU - TRACE_LDS_BYTES - uint32_t(sizeof(SmemRest<G, PX>)) - 64u) / PKT * PKT;
  alignas(16) uint8_t ring[RING_BYTES];
};

template <class G, int PX>
struct PlanC {
  using S = CG<G, PX>;
  int wg, cell, r;
  int q0, q1, o0, o1, a0, a1, v0, v1;  // units of QKV, O / down, act; LM-head rows
  __device__ __forceinline__ PlanC(const Params& p, int wg_) {
    wg = wg_;
    const int x = wg & 7;
    cell = x / PX;
    r = (wg >> 3) * PX + x % PX;
    q0 = split_lo(S::QU, S::R, r); q1 = split_lo(S::QU, S::R, r + 1);
    o0 = split_lo(S::HU, S::R, r); o1 = split_lo(S::HU, S::R, r + 1);
    a0 = split_lo(S::IU, S::R, r); a1 = split_lo(S::IU, S::R, r + 1);
    v0 = p.lm_head ? S::LMROWS * wg : 0;
    v1 = p.lm_head ? v0 + S::LMROWS : 0;
  }
};

// ------------------------------------------------------------------------------------------------
// Set-up by one wave: the cell's sequences and the workgroup's attention items.
// Sequences are dealt to the cells in order of falling context length, back and forth.
// Whole workgroups: a pair of n tiles takes ceil(n / T) workgroups in equal chunks, T the least that all pairs'
// chunks need no more than R for, and at least TMIN: shorter chunks leave waves idle and widen the pair's exchanges.
// End to end: the pairs lie on a line of tiles, a short one padded to a quarter of a workgroup's share (so that a
// workgroup never holds more than IPC pairs); workgroup r takes tiles [NT r / R, NT (r + 1) / R).
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ int wave_scan_incl(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o);
    if (lane >= o) v += u;
  }
  return v;
}

template <class G, int PX>
__device__ __forceinline__ void setup(const Params& p, const PlanC<G, PX>& P, SmemC<G, PX>& sm) {
  using S = CG<G, PX>;
  const int lane = threadIdx.x & 63;
  const int B = p.B;
  {
    const int mine = lane < B ? sm.sS[lane] : -1;
    int rank = 0;
    for (int j = 0; j < B; ++j) {
      const int o = __shfl(mine, j);
      rank += (o > mine || (o == mine && j < lane)) ? 1 : 0;
    }
    const int round = rank / S::NC, at = rank % S::NC;
    const int cl = (round & 1) ? S::NC - 1 - at : at;
    const bool here = lane < B && cl == P.cell;
    if (here) sm.sid[round] = lane;
    if (lane < B) sm.cs[lane] = cl * S::NS + round;
    const uint64_t m = __ballot(here);
    if (lane == 0) sm.ns = __popcll(m);
  }
  wait_lgkm0();
  const int ns = __builtin_amdgcn_readfirstlane(*(volatile int*)&sm.ns);
  const int np = ns * G::KVH;
  const bool on = lane < np;
  const int slot = on ? lane / G::KVH : 0, g = lane - slot * G::KVH;
  const int b = on ? *(volatile int*)&sm.sid[slot] : 0;
  const int old = on ? sm.sS[b] - 1 : 0;
  const int tiles = (old + 15) / 16;
  if constexpr (S::E2E) {
    const int nt0 = __shfl(wave_scan_incl(on ? tiles : 0, lane), 63);
    const int least = max(1, (nt0 + 4 * S::R - 1) / (4 * S::R));
    const int nt = on ? max(tiles, least) : 0;
    const int incl = wave_scan_incl(nt, lane);
    const int NT = __shfl(incl, 63);
    const int base = incl - nt;
    // workgroups that take a share: at least TMIN tiles each while the line is short
    const int RE = min(S::R, (NT + PK_CELL_TMIN - 1) / PK_CELL_TMIN);
    auto wg_of = [&](int tile) { return ((tile + 1) * RE - 1) / max(NT, 1); };  // workgroup of a tile of the line
    const int r0 = wg_of(base), r1 = wg_of(base + max(nt, 1) - 1);
    int k0 = -1;  // pairs that start at or before r0's first tile
    const int first = NT > 0 ? split_lo(NT, RE, r0) : 0;
    for (int j = 0; j < np; ++j) k0 += __shfl(base, j) <= first ? 1 : 0;
    k0 = lane - k0;
    const int w0 = P.r < RE ? split_lo(NT, RE, P.r) : NT, w1 = P.r < RE ? split_lo(NT, RE, P.r + 1) : NT;
    const int a = max(base, w0) - base, e = min(base + nt, w1) - base;  // tiles of the pair in this workgroup
    const bool have = on && a < e;
    const uint64_t m = __ballot(have);
    const int k = __popcll(m & ((uint64_t(1) << lane) - 1u));
    const int re = min(e, tiles), n = have && re > a ? min(re * 16, old) - a * 16 : 0;
    const int ntile = (n + 15) / 16, nquad = (ntile + 3) / 4;
    const int ts = wave_scan_incl(have ? ntile : 0, lane), qs = wave_scan_incl(have ? nquad : 0, lane);
    if (have && k < S::IPC) {
      Item it;
      it.slot = slot; it.b = b; it.g = g;
      it.t0 = a * 16; it.n = n;
      it.tile0 = ts - ntile; it.ntile = ntile;
      it.quad0 = qs - nquad;
      it.sc0 = (qs - nquad) * 64;
      it.r0 = r0; it.C = r1 - r0 + 1; it.c = P.r - r0; it.k0 = k0;
      it.leader = e == nt;
      sm.it[k] = it;
    }
    if (lane == 63) {
      sm.ni = min(__popcll(m), S::IPC);
      sm.ntile = ts;
    }
  } else {
    const int nt = on ? max(tiles, 1) : 0;
    const int NT = __shfl(wave_scan_incl(nt, lane), 63);
    int t = max(PK_CELL_TMIN, (NT + S::R - 1) / S::R);
    for (int hi = max(t, (NT + S::R - np - 1) / (S::R - np)); t < hi;) {  // hi is always enough
      const int mid = (t + hi) / 2;
      float s[1] = {float((nt + mid - 1) / mid)};
      wave_sum_n<1>(s);
      if (s[0] <= float(S::R)) hi = mid;
      else t = mid + 1;
    }
    const int C = (nt + t - 1) / t;
    const int r0 = wave_scan_incl(C, lane) - C, c = P.r - r0;
    const bool have = on && c >= 0 && c < C;  // in one lane at most
    if (have) {
      const int a = nt * c / C, e = min(nt * (c + 1) / C, tiles);
      Item it;
      it.slot = slot; it.b = b; it.g = g;
      it.t0 = a * 16;
      it.n = e > a ? min(e * 16, old) - a * 16 : 0;
      it.tile0 = 0; it.ntile = max(e - a, 0); it.quad0 = 0; it.sc0 = 0;
      it.r0 = r0; it.C = C; it.c = c; it.k0 = 0;
      it.leader = c == C - 1;
      sm.it[0] = it;
      sm.ntile = it.ntile;
    }
    const uint64_t m = __ballot(have);
    if (lane == 0) {
      sm.ni = m ? 1 : 0;
      if (!m) sm.ntile = 0;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Producer
// ------------------------------------------------------------------------------------------------
// A pointer that is the same in every lane, as a scalar.
__device__ __forceinline__ const uint8_t* uni(const uint8_t* q) {
  const uint64_t v = reinterpret_cast<uint64_t>(q);
  return reinterpret_cast<const uint8_t*>(uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))))) |
                                          (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))))) << 32));
}
// One LDS-DMA packet from a uniform base and a 32-bit lane offset (dma16 with the address arithmetic
// left to the instruction).
__device__ __forceinline__ void dma16s(const uint8_t* base, uint32_t lane_off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)),
               "v"(lane_off), "s"(uni(base))
               : "memory", "m0");
}
template <class G, int PX>
__device__ __forceinline__ void producer(const Params& p, const PlanC<G, PX>& P, SmemC<G, PX>& sm, uint32_t epoch) {
  using S = CG<G, PX>;
  constexpr uint32_t CRING = SmemC<G, PX>::RING_BYTES;
  const int pw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int prow = lane >> 3;                                           // row of the packet
  const uint32_t col = uint32_t((lane - (lane >> 3)) & 7) * 16u;        // source byte of its 128
  const uint32_t ring_base = uint32_t(reinterpret_cast<uintptr_t>(sm.ring));
  uint32_t n = 0;
  uint32_t avail = 0;  // packets ending at or below it may be issued (consumer positions only grow)
  Spin spin(p.ws, epoch, 41);
  bool dead = false;
  auto cmin = [&]() -> uint32_t {
    typedef __attribute__((address_space(3))) const volatile u32x4 lds_u32x4;
    const u32x4 c = *(lds_u32x4*)(sm.consumed);
    return __builtin_amdgcn_readfirstlane(min(min(c.x, c.y), min(c.z, c.w)));
  };
  auto publish = [&](uint32_t first_pending_packet) {
    if (lane == 0) st_lds(&sm.front[pw], first_pending_packet * PKT);
  };
  // room for packet gn in the ring; when there is none the queue drains, so that everything issued
  // so far is visible to the consumers
  auto room = [&](uint32_t gn) {
    if ((gn + 1) * PKT <= avail || (gn + 1) * PKT <= (avail = cmin() + CRING)) return;
    wait_vmcnt<0>();
    publish(gn);
    while ((gn + 1) * PKT > (avail = cmin() + CRING))
      if (!spin.again()) { dead = true; return; }
  };
  auto issued = [&](uint32_t gn) {
    wait_vmcnt<DEPTH_C - 1>();
    if (gn >= uint32_t(DEPTH_C - 1) * NPW) publish(gn - uint32_t(DEPTH_C - 1) * NPW);
  };
  // Weight rows as ks k-steps x `groups` packets.  The issue loop runs on the scalar unit: a packet's
  // address is a uniform base (matrix, group, k-step) plus this lane's offset within 8 rows, which is
  // the same in every layer.  base(g): byte offset of group g; lane_off(g): this lane's.
  auto weights = [&](const uint8_t* w, int ks, int groups, auto base, auto lane_off) {
    const uint32_t npk = uint32_t(ks) * uint32_t(groups);
    uint32_t i = (uint32_t(pw) + NPW - n % NPW) % NPW;
    int s = 0, g = int(i);
    while (g >= groups) { g -= groups; ++s; }
    for (; i < npk && !dead; i += NPW) {
      const uint32_t gn = n + i;
      room(gn);
      if (dead) break;
      dma16s(w + base(g) + uint32_t(s) * 128u, lane_off(g), ring_base + gn % (CRING / PKT) * PKT);
      issued(gn);
      g += NPW;
      while (g >= groups) { g -= groups; ++s; }
    }
    n += npk;
  };
  const int nq = 4 * (P.q1 - P.q0), no = 4 * (P.o1 - P.o0);
  const int gq = (nq + 7) / 8, go = (no + 7) / 8;
  // rows past the last one read it again
  const uint32_t hb = G::H * 2, ib = G::I * 2;
  uint32_t vq[S::TQ * 2];  // QKV: slots in qkv_row order
#pragma unroll
  for (int g = 0; g < S::TQ * 2; ++g) vq[g] = uint32_t(qkv_row<G>(4 * P.q0 + min(8 * g + prow, nq - 1))) * hb + col;
  const uint32_t vh = uint32_t(prow) * hb + col, vi = uint32_t(prow) * ib + col;
  const uint32_t lo = uint32_t(min(prow, no - 1 - 8 * (go - 1)));
  const uint32_t vho = lo * hb + col, vio = lo * ib + col;
  // gate/up: 4 gate rows, then the up rows of the same act unit
  const uint32_t vg = uint32_t(prow < 4 ? prow : G::I + prow - 4) * hb + col;
  const int ntile = __builtin_amdgcn_readfirstlane(sm.ntile), ni = __builtin_amdgcn_readfirstlane(sm.ni);
  constexpr int BV = (S::TILES + 63) / 64;
  int blkv[BV];  // lane i: block ids of tiles i, i + 64, ...
#pragma unroll
  for (int k = 0; k < BV; ++k) blkv[k] = 64 * k + lane < ntile ? sm.blk[64 * k + lane] : 0;
  auto kv = [&](int l, long long off) {
    const uint8_t* cache = reinterpret_cast<const uint8_t*>(sm.kvp[l]);
    const uint32_t npk = uint32_t(ntile) * 2u;
    int k = -1, tile0 = 0, end = 0, last = 0;
    long long head = 0;
    for (uint32_t i = (uint32_t(pw) + NPW - n % NPW) % NPW; i < npk && !dead; i += NPW) {
      const uint32_t gn = n + i;
      room(gn);
      if (dead) break;
      const int tile = int(i >> 1);
      while (tile >= end && k + 1 < ni) {
        const Item& it = sm.it[++k];
        tile0 = __builtin_amdgcn_readfirstlane(it.tile0);
        end = tile0 + __builtin_amdgcn_readfirstlane(it.ntile);
        last = __builtin_amdgcn_readfirstlane(it.n) - 1;
        head = (long long)__builtin_amdgcn_readfirstlane(it.g) * p.head_stride + off;
      }
      int blk = 0;
#pragma unroll
      for (int v = 0; v < BV; ++v)
        if (tile >> 6 == v) blk = __builtin_amdgcn_readlane(blkv[v], tile & 63);
      // token of this lane's row; rows past the run's end read its last token again
      const int j = min(int(i & 1u) * 8 + prow, last - (tile - tile0) * 16);
      const uint8_t* src = cache + ((long long)blk * p.block_stride + head) * 2 + (long long)j * (p.token_stride * 2) + col;
      dma16(src, __builtin_amdgcn_readfirstlane(ring_base + gn % (CRING / PKT) * PKT));
      issued(gn);
    }
    n += npk;
  };
  auto u8 = [](const void* q) { return reinterpret_cast<const uint8_t*>(q); };
  auto norm = [&](const uint8_t* w) {  // a norm weight vector: two packets
    for (uint32_t i = (uint32_t(pw) + NPW - n % NPW) % NPW; i < 2u && !dead; i += NPW) {
      const uint32_t gn = n + i;
      room(gn);
      if (dead) break;
      const uint32_t o = i * PKT + uint32_t(lane) * 16u;
      if (o < hb) dma16(w + o, __builtin_amdgcn_readfirstlane(ring_base + gn % (CRING / PKT) * PKT));
      issued(gn);
    }
    n += 2u;
  };
  if (__builtin_amdgcn_readfirstlane(sm.ns) > 0)
    for (int l = 0; l < p.n_layers && !dead; ++l) {
      const LayerW& Lw = sm.lw[l];
      norm(uni(u8(Lw.norm1)));
      const uint8_t *wq = uni(u8(Lw.qkv)), *wo = uni(u8(Lw.o)), *wg = uni(u8(Lw.gate_up)), *wd = uni(u8(Lw.down));
      weights(wq, S::KSH, gq, [&](int) { return 0u; }, [&](int g) {
        uint32_t v = vq[0];
#pragma unroll
        for (int k = 1; k < S::TQ * 2; ++k) v = g == k ? vq[k] : v;
        return v;
      });
      if (!dead) kv(l, p.k_off);
      if (!dead) kv(l, p.v_off);
      if (!dead)
        weights(wo, S::KSH, go, [&](int g) { return uint32_t(4 * P.o0 + 8 * g) * hb; },
                [&](int g) { return g == go - 1 ? vho : vh; });
      if (!dead) norm(uni(u8(Lw.norm2)));
      if (!dead)
        weights(wg, S::KSH, P.a1 - P.a0, [&](int g) { return uint32_t(4 * (P.a0 + g)) * hb; }, [&](int) { return vg; });
      if (!dead)
        weights(wd, S::KSI, go, [&](int g) { return uint32_t(4 * P.o0 + 8 * g) * ib; },
                [&](int g) { return g == go - 1 ? vio : vi; });
    }
  if (!dead) norm(u8(p.final_norm));
  if (!dead && P.v1 > P.v0)
    weights(u8(p.embed), S::KSH, 2 * S::TL, [&](int g) { return uint32_t(P.v0 + 8 * g) * hb; }, [&](int) { return vh; });
  wait_vmcnt<0>();
  publish(dead ? 0x3fffffu : n);
}

// ------------------------------------------------------------------------------------------------
// Consumer
// ------------------------------------------------------------------------------------------------
template <class G, int PX>
struct CC {
  using S = CG<G, PX>;
  using W = CW<G>;
  using SM = SmemC<G, PX>;
  const Params& p;
  const PlanC<G, PX>& P;
  SM& sm;
  int cw, lane, ct, ns;
  uint32_t pos = 0, bar_gen = 0, seen = 0;
  uint32_t epoch;
  bool dead = false;
  __amdgpu_buffer_rsrc_t rx;

  __device__ __forceinline__ CC(const Params& p_, const PlanC<G, PX>& P_, SM& sm_, uint32_t ep, const void* region)
      : p(p_), P(P_), sm(sm_), epoch(ep), rx(rsrc(region)) {
    // on the scalar unit: a branch on the wave must not leave an MFMA to the lane mask, which it ignores
    cw = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6) - NPW);
    lane = threadIdx.x & 63;
    ct = cw * 64 + lane;
    ns = __builtin_amdgcn_readfirstlane(sm.ns);
  }
  __device__ __forceinline__ void refresh() { asm volatile("" : "+v"(lane), "+v"(ct)); }
  // The attention's units hold three payload words and one for the epoch and the layer.  Every unit that a step uses
  // is written and read by the same waves in each of its layers, so from a step's second layer on only the layer
  // before it has to be told apart: the top bits of the epoch, flipped in turn, do that.  At its first use in a step a
  // unit may be as old as the program, so the first and the last layer have the epoch as it is, and a first use finds
  // whole epochs of other steps, as with the units that hold both words.  (A step of two layers, or one that gave up,
  // leaves flipped ones, which pass as another step's after 2^30 steps at the earliest.)
  uint32_t tag = 0;
  __device__ __forceinline__ void begin_layer(int l) {
    const bool whole = l == 0 || (l == p.n_layers - 1 && l > 1);
    tag = epoch ^ (whole ? 0u : l & 1 ? 1u << 31 : 1u << 30);
  }
  __device__ __forceinline__ uint32_t filled() const {
    typedef __attribute__((address_space(3))) const volatile u32x4 lds_u32x4;
    const u32x4 f = *(lds_u32x4*)(sm.front);
    return min(min(f.x, f.y), min(f.z, f.w));
  }
  __device__ __forceinline__ void wait_filled(uint32_t end) {
    if (dead || end <= seen) return;
    Spin spin(p.ws, epoch, 42);
    while ((seen = filled()) < end)
      if (!spin.again()) { dead = true; return; }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);  // the ring reads that follow stay after the wait
  }
  __device__ __forceinline__ void release(uint32_t end) {
    wait_lgkm0();  // ring reads of this wave have returned
    if (lane == 0) st_lds(&sm.consumed[cw], end);
  }
  __device__ __forceinline__ void cbar() {
    bar_gen += NCW;
    if (lane == 0) __hip_atomic_fetch_add(&sm.cbar, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    Spin spin(p.ws, epoch, 43);
    while (ld_lds(&sm.cbar) < bar_gen)
      if (!spin.again()) { dead = true; break; }
  }
  // Ring bytes at stream position at + lo: `at` uniform, `lo` this lane's part (less than a ring).
  static constexpr uint32_t CRING = SM::RING_BYTES;
  __device__ __forceinline__ uint32_t ring_at(uint32_t at, uint32_t lo) const {
    const uint32_t o = at % CRING + lo;
    return min(o, o - CRING);  // unsigned: below the ring's end the difference wraps to a large value
  }
  __device__ __forceinline__ uint4 ring16(uint32_t at, uint32_t lo) const {
    return *reinterpret_cast<const uint4*>(sm.ring + ring_at(at, lo));
  }
  // ds_read_b64_tr_b16: of 16 lanes, lane 4 j + q gives the address of 4 values, lane i gets value i % 4 of lanes i / 4,
  // 4 + i / 4, 8 + i / 4 and 12 + i / 4
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  __device__ __forceinline__ uint2 ring_tr(uint32_t at, uint32_t lo) const {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(sm.ring + ring_at(at, lo))));
  }
  __device__ __forceinline__ uint2 ring8(uint32_t at, uint32_t lo) const {
    return *reinterpret_cast<const uint2*>(sm.ring + ring_at(at, lo));
  }
  __device__ __forceinline__ u32x4 ld(uint32_t off, uint32_t soff = 0) const {
    return __builtin_amdgcn_raw_buffer_load_b128(rx, int(off), int(soff), 16);
  }
  __device__ __forceinline__ void st(uint32_t off, u32x4 v, uint32_t soff = 0) const {
    __builtin_amdgcn_raw_buffer_store_b128(v, rx, int(off), int(soff), 16);
  }
  __device__ __forceinline__ u32x4 vec_unit(uint32_t lo, uint32_t hi, int l) const {
    return u32x4{lo, hi, uint32_t(l), epoch};
  }
  __device__ __forceinline__ bool vec_ok(const u32x4& v, int l) const { return v.w == epoch && v.z == uint32_t(l); }
  __device__ __forceinline__ int slot0() const { return P.cell * S::NS; }
  // Poll N units per thread: off(i) is unit i's byte offset, soff(i) a uniform part, `live` the uniform mask
  // of the i in use.  Every lane polls something that arrives (a lane without a unit of its own repeats
  // another's), so readiness is a wave's and the loop runs on scalar branches: per-lane masks around
  // every load cost more instructions on the chain than the repeated loads.  Units some lane still
  // waits for are loaded again.
  template <int N, class Ok, class Off, class SOff>
  __device__ __forceinline__ void poll(int site, uint32_t live, Ok ok, Off off, SOff soff, u32x4 (&v)[N]) {
    Spin spin(p.ws, epoch, site);
    uint32_t pend = live;
    while (true) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        if ((pend >> i) & 1u) v[i] = ld(off(i), soff(i));
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (((pend >> i) & 1u) && __builtin_amdgcn_ballot_w64(!ok(v[i])) == 0ull) pend &= ~(1u << i);
      if (!pend) break;
      if (dead || !spin.again()) { dead = true; break; }
    }
  }
};

// rsqrt(mean + eps): the hardware estimate (1 ulp) and one Newton step, a third of the instructions of rms_scale's
// square root and divide on a chain that runs 61 times a step (seven sequences: 566 us, 577 with rms_scale).  Over 2^26 sums
// from 1e-6 to 1e9 it is nearer to 64 bits: mean error 0.43 to 0.47, worst 1.70 (times 2^-24); rms_scale 0.53 to
// 0.55 and 2.36.
template <int N>
__device__ __forceinline__ float rms_rs(float sumsq) {
  const float m = fmaf(sumsq, 1.0f / float(N), 1e-5f);
  const float r = __builtin_amdgcn_rsqf(m);
  return fmaf(0.5f * r, fmaf(-m * r, r, 1.0f), r);
}
__device__ __forceinline__ float sumsq4(uint2 v) {
  const float a = bf_lo(v.x), b = bf_hi(v.x), c = bf_lo(v.y), d = bf_hi(v.y);
  return a * a + b * b + c * c + d * d;
}
// LlamaRMSNorm rounding of four values: bf16(w * bf16(x * rs)) (modeling_llama.py:62-67).
__device__ __forceinline__ uint2 norm4(uint2 x, uint2 w, float rs) {
  const uint32_t t0 = pack2(bf_lo(x.x) * rs, bf_hi(x.x) * rs), t1 = pack2(bf_lo(x.y) * rs, bf_hi(x.y) * rs);
  return make_uint2(pack2(bf_lo(w.x) * bf_lo(t0), bf_hi(w.x) * bf_hi(t0)),
                    pack2(bf_lo(w.y) * bf_lo(t1), bf_hi(w.y) * bf_hi(t1)));
}

// A norm's weights in registers, read from the ring before the vector they scale is waited for: units
// lane + 64 j of a wave-held sequence, and unit t of a thread-held one.
template <class G, int PX>
struct NormW {
  uint2 w[CG<G, PX>::LU], t;
  __device__ __forceinline__ explicit NormW(CC<G, PX>& C) {
    const uint32_t at = C.pos;
    C.pos += CG<G, PX>::NSEG;
    C.wait_filled(C.pos);
#pragma unroll
    for (int j = 0; j < CG<G, PX>::LU; ++j) w[j] = C.ring8(at, uint32_t(C.lane + 64 * j) * 8u);
    t = C.ring8(at, uint32_t(C.ct) * 8u);
  }
};
// RMS-normalise one sequence held by a wave (lane: units lane + 64 j) into staged row q: its sum needs no
// other wave.
template <class G, int PX>
__device__ __forceinline__ void norm_row(CC<G, PX>& C, const uint2 (&v)[CG<G, PX>::LU], int q, const NormW<G, PX>& nw) {
  using S = CG<G, PX>;
  float s[1] = {0.f};
#pragma unroll
  for (int j = 0; j < S::LU; ++j) s[0] += C.lane + 64 * j < S::HU ? sumsq4(v[j]) : 0.f;
  wave_sum_n<1>(s);
  const float rs = rms_rs<G::H>(s[0]);
#pragma unroll
  for (int j = 0; j < S::LU; ++j) {
    const int u = C.lane + 64 * j;
    if (u < S::HU) *reinterpret_cast<uint2*>(C.sm.xs + q * S::XH + 4 * u) = norm4(v[j], nw.w[j], rs);
  }
}
// This workgroup's residual rows of the wave's sequence, from the units as norm_row takes them.
template <class G, int PX>
__device__ __forceinline__ void keep_rows(CC<G, PX>& C, const uint2 (&v)[CG<G, PX>::LU]) {
#pragma unroll
  for (int j = 0; j < CG<G, PX>::LU; ++j) {
    const int u = C.lane + 64 * j;
    if (u >= C.P.o0 && u < C.P.o1) C.sm.res[C.cw][u - C.P.o0] = v[j];
  }
}

// Wait for the cell's x or h1 vectors (wave w: sequence w), keep this workgroup's residual rows, normalise.
template <class G, int PX>
__device__ __forceinline__ void stage_norm(CC<G, PX>& C, int kind, int l, const NormW<G, PX>& nw) {
  using S = CG<G, PX>;
  const bool mine = C.cw < C.ns;
  u32x4 x[S::LU];
  uint2 v[S::LU];
  const uint32_t o = CW<G>::vec_u(C.lane), oe = CW<G>::vec_u(min(C.lane, S::HU - 1 - 64 * (S::LU - 1)));
  C.template poll<S::LU>(44 + kind, mine ? (1u << S::LU) - 1u : 0u, [&](const u32x4& u) { return C.vec_ok(u, l); },
                         [&](int j) { return j == S::LU - 1 ? oe : o; },
                         [&](int j) { return CW<G>::vec_s(kind, C.slot0() + C.cw) + uint32_t(j) * CW<G>::STRIDE64; }, x);
#pragma unroll
  for (int j = 0; j < S::LU; ++j) v[j] = make_uint2(x[j].x, x[j].y);
  if (mine) {
    keep_rows(C, v);
    norm_row(C, v, C.cw, nw);
  }
  C.cbar();
}
// The same for at most N sequences with thread t holding unit t of each: one load a sequence instead of
// LU, against a second barrier for the sums.
template <int N, class G, int PX>
__device__ __forceinline__ void stage_norm_t(CC<G, PX>& C, int kind, int l, const NormW<G, PX>& nw) {
  using S = CG<G, PX>;
  u32x4 x[N];
  uint2 v[N];
  const uint32_t o = CW<G>::vec_u(min(C.ct, S::HU - 1));
  C.template poll<N>(44 + kind, (1u << C.ns) - 1u, [&](const u32x4& u) { return C.vec_ok(u, l); }, [&](int) { return o; },
                     [&](int i) { return CW<G>::vec_s(kind, C.slot0() + i); }, x);
  float s[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = make_uint2(x[i].x, x[i].y);
    s[i] = C.ct < S::HU ? sumsq4(v[i]) : 0.f;
  }
  if (C.ct >= C.P.o0 && C.ct < C.P.o1)
#pragma unroll
    for (int i = 0; i < N; ++i) C.sm.res[i][C.ct - C.P.o0] = v[i];
  wave_sum_n<N>(s);
  float mine = s[0];
#pragma unroll
  for (int i = 1; i < N; ++i) mine = C.lane == i ? s[i] : mine;
  if (C.lane < N) C.sm.sums[C.cw][C.lane] = mine;
  C.cbar();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (i >= C.ns) continue;
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < NCW; ++k) t += C.sm.sums[k][i];
    const float rs = rms_rs<G::H>(t);
    if (C.ct < S::HU) *reinterpret_cast<uint2*>(C.sm.xs + i * S::XH + 4 * C.ct) = norm4(v[i], nw.t, rs);
  }
  C.cbar();
}
template <class G, int PX>
__device__ __forceinline__ void stage_x(CC<G, PX>& C, int kind, int l, const NormW<G, PX>& nw) {
  if (C.ns <= 2) stage_norm_t<2>(C, kind, l, nw);
  else stage_norm(C, kind, l, nw);
}

// Wait for the cell's attention vectors and stage them as rows of xs.
template <class G, int PX>
__device__ __forceinline__ void stage_att(CC<G, PX>& C) {
  using S = CG<G, PX>;
  constexpr int N = S::NS, AU = G::H / 6;
  u32x4 x[N];
  const uint32_t o = CW<G>::vec_u(min(C.ct, AU - 1)), tg = C.tag;
  C.template poll<N>(44 + C_ATT, (1u << C.ns) - 1u, [&](const u32x4& u) { return u.w == tg; }, [&](int) { return o; },
                     [&](int i) { return CW<G>::vec_s(C_ATT, C.slot0() + i); }, x);
  if (C.ct < AU)
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (i < C.ns) {
        uint32_t* d = reinterpret_cast<uint32_t*>(C.sm.xs + i * S::XH + 6 * C.ct);
        d[0] = x[i].x; d[1] = x[i].y; d[2] = x[i].z;
      }
  C.cbar();
}

template <int N, class G, int PX>
__device__ __forceinline__ void stage_act_n(CC<G, PX>& C, int l) {
  using S = CG<G, PX>;
  u32x4 x[N * S::LA];
  uint32_t live = 0;
#pragma unroll
  for (int i = 0; i < N * S::LA; ++i)  // whole waves past the vector's end have nothing to wait for
    if (i / S::LA < C.ns && C.cw * 64 + (i % S::LA) * NCT < S::IU) live |= 1u << i;
  static_assert(S::IU % 64 == 0, "a vector's units fill whole waves");
  const uint32_t o = CW<G>::vec_u(C.ct);
  C.template poll<N * S::LA>(44 + C_ACT, live, [&](const u32x4& u) { return C.vec_ok(u, l); }, [&](int) { return o; },
                             [&](int i) {
                               return CW<G>::vec_s(C_ACT, C.slot0() + i / S::LA) +
                                      uint32_t(i % S::LA) * (NCT / 64) * CW<G>::STRIDE64;
                             }, x);
#pragma unroll
  for (int i = 0; i < N * S::LA; ++i) {
    const int u = C.ct + (i % S::LA) * NCT;
    if ((live >> i) & 1u)
      *reinterpret_cast<uint2*>(C.sm.xs + (i / S::LA) * S::XI + 4 * u) = make_uint2(x[i].x, x[i].y);
  }
  C.cbar();
}
template <class G, int PX>
__device__ __forceinline__ void stage_act(CC<G, PX>& C, int l) {
  if (C.ns <= 2) stage_act_n<2>(C, l);
  else stage_act_n<CG<G, PX>::NS>(C, l);
}

// One projection phase: D[row][sequence] = W x over this workgroup's `groups` 8-row groups (NT 16-row
// tiles).  The four waves are KW ways over k times TW = 4 / KW ways over tiles: wave w takes tiles
// w / KW, w / KW + TW, ... and k-steps w % KW, w % KW + KW, ..., U of them at a time: every operand of
// a batch is read from LDS before its MFMAs, so the reads overlap, and the ring space is given back
// before them.  A batch over all waves spans KW U k-steps of the stream, which the ring must hold.
template <int KW, int NT>
constexpr int tiles_per_wave() { return (NT + NCW / KW - 1) / (NCW / KW); }
template <int KS, int NT, int KW, int U, int GMAX, class G, int PX>
__device__ __forceinline__ void project(CC<G, PX>& C, int groups, int xstride,
                                        floatx4 (&acc)[tiles_per_wave<KW, NT>()], int nseq) {
  constexpr int TW = NCW / KW, NTW = tiles_per_wave<KW, NT>();
  constexpr int SPAN = KW * U < KS ? KW * U : KS;
  static_assert(uint32_t(SPAN * GMAX) * PKT <= SmemC<G, PX>::RING_BYTES, "a batch fits the ring");
  const uint32_t pos0 = C.pos;
  const uint32_t step = uint32_t(groups) * PKT;
  C.pos += uint32_t(KS) * step;
  const int kw = C.cw % KW, tw = C.cw / KW;
  const int row = C.lane & 15, q = C.lane >> 4;
  const uint16_t* xr = C.sm.xs + (row < nseq ? row : 0) * xstride + q * 8;
#pragma unroll
  for (int t = 0; t < NTW; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  C.release(pos0 + uint32_t(kw) * step);
#pragma unroll 1
  for (int s0 = 0; s0 < KS; s0 += KW * U) {
    uint4 x[U][2], a[U][NTW][2];
    const int last = min(s0 + kw + (U - 1) * KW, KS - 1);  // waiting for a step past this wave's last is harmless
    C.wait_filled(pos0 + uint32_t(last + 1) * step);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = min(s0 + kw + u * KW, KS - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) x[u][h] = *reinterpret_cast<const uint4*>(xr + s * 64 + h * 32);
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        const int grp = min(2 * (tw + t * TW) + (row >> 3), groups - 1);
        const uint32_t lo = uint32_t(grp) * PKT + uint32_t(row & 7) * 128u;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          a[u][t][h] = C.ring16(pos0 + uint32_t(s) * step, lo + uint32_t((4 * h + q + row) & 7) * 16u);
      }
    }
    const int next = s0 + KW * U + kw;
    C.release(next < KS ? pos0 + uint32_t(next) * step : C.pos);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s0 + kw + u * KW >= KS) continue;
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u][t][h]),
                                                          __builtin_bit_cast(bf16x8, x[u][h]), acc[t], 0, 0, 0);
    }
  }
}
// A phase's MFMA weight operands in registers: this wave's quarter of the k-steps of all NT tiles, read from the
// ring (and its space given back) before the phase's input is waited for.  The registers of the four
// waves are another buffer as large as the ring, so the stream runs on through the exchange, and after it
// only the input's own operands are to be read.
template <int KS, int NT, class G, int PX>
struct Weights {
  static constexpr int NU = (KS + NCW - 1) / NCW;
  uint4 a[NU][NT][2];
  __device__ __forceinline__ Weights(CC<G, PX>& C, int groups) {
    const uint32_t pos0 = C.pos;
    const uint32_t step = uint32_t(groups) * PKT;
    C.pos += uint32_t(KS) * step;
    const int row = C.lane & 15, q = C.lane >> 4;
    uint32_t lo[NT], sl[2];
#pragma unroll
    for (int t = 0; t < NT; ++t) lo[t] = uint32_t(min(2 * t + (row >> 3), groups - 1)) * PKT + uint32_t(row & 7) * 128u;
#pragma unroll
    for (int h = 0; h < 2; ++h) sl[h] = uint32_t((4 * h + q + row) & 7) * 16u;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int s = KS * C.cw / NCW + u;
      if (s < KS * (C.cw + 1) / NCW) {
        const uint32_t at = pos0 + uint32_t(s) * step;
        C.release(at);
        C.wait_filled(at + step);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int h = 0; h < 2; ++h) a[u][t][h] = C.ring16(at, lo[t] + sl[h]);
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int h = 0; h < 2; ++h) a[u][t][h] = make_uint4(0u, 0u, 0u, 0u);
      }
    }
    C.release(C.pos);
  }
  // D[row][sequence] over this wave's k-steps; the staged rows are zero-padded to whole batches by the
  // zero weights above (the operand read stays inside the row).
  __device__ __forceinline__ void apply(CC<G, PX>& C, int xstride, floatx4 (&acc)[NT], int nseq) const {
    const int row = C.lane & 15, q = C.lane >> 4;
    const uint16_t* xr = C.sm.xs + (row < nseq ? row : 0) * xstride + q * 8;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int s = KS * C.cw / NCW + u;
      if (s >= KS * (C.cw + 1) / NCW) continue;
      uint4 x[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) x[h] = *reinterpret_cast<const uint4*>(xr + s * 64 + h * 32);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u][t][h]),
                                                          __builtin_bit_cast(bf16x8, x[h]), acc[t], 0, 0, 0);
    }
  }
};
// The waves' partial tiles to LDS (valid after the barrier), and a tile's sum over its KW partials.
template <int KW, int NT, class G, int PX>
__device__ __forceinline__ void to_red(CC<G, PX>& C, const floatx4 (&acc)[tiles_per_wave<KW, NT>()]) {
  constexpr int TW = NCW / KW;
#pragma unroll
  for (int t = 0; t < tiles_per_wave<KW, NT>(); ++t) {
    const int tile = C.cw / KW + t * TW;
    if (tile < NT) *reinterpret_cast<floatx4*>(&C.sm.red[tile][C.cw % KW][C.lane * 4]) = acc[t];
  }
  C.cbar();
}
template <int KW, class G, int PX>
__device__ __forceinline__ floatx4 red_sum(const CC<G, PX>& C, int t, int lane) {
  static_assert(KW == NCW, "four partials");
  floatx4 u[KW], v;
#pragma unroll
  for (int k = 0; k < KW; ++k) u[k] = *reinterpret_cast<const floatx4*>(&C.sm.red[t][k][lane * 4]);
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = (u[0][j] + u[1][j]) + (u[2][j] + u[3][j]);
  return v;
}

// ------------------------------------------------------------------------------------------------
// Attention over this workgroup's one chunk (of four waves, two barriers).
// ------------------------------------------------------------------------------------------------
template <class G, int PX>
__device__ __forceinline__ void attention_one(CC<G, PX>& C, int l) {
  using S = CG<G, PX>;
  using W = CW<G>;
  const Params& p = C.p;
  SmemC<G, PX>& sm = C.sm;
  const int lane = C.lane, w = C.cw;
  auto tr = [&](int ev) { if (C.ct == 0) trace_at(p, l, ev, p.n_layers); };
  auto one = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  if (one(sm.ni) == 0) return;
  const Item& it = sm.it[0];
  const int g = one(it.g), n = one(it.n), nt = one(it.ntile), Cc = one(it.C), ci = one(it.c);
  const int r0 = C.P.cell * S::R + one(it.r0);  // record key of the pair's first chunk
  const int slot = C.slot0() + one(it.slot);
  const int nquad = (nt + 3) / 4;
  const int me = C.P.cell * S::R + C.P.r;
  const uint32_t tg = C.tag;
  const uint32_t kpos = C.pos, vpos = kpos + uint32_t(nt) * 2u * PKT;
  C.pos = vpos + uint32_t(nt) * 2u * PKT;
  const bool has_new = w == NCW - 1 && one(it.leader);  // the new token is wave 3's, in the chunk with the pair's end
  // ---- q straight into MFMA operands: lane (head lane % 4, piece j = lane / 16) takes dims 8j .. 8j + 7 and 32 + 8j
  // .. of its head, which are the two halves of four units (two RoPE pairs each) of one 64-byte line; the new
  // token's k alike, for every column of an operand, and v unit lane / 4 (4 dims): one round trip ----
  const int hr = (lane & 3) < 3 ? (lane & 3) : 0, pj = lane >> 4;
  static_assert(W::UPL == 4, "a lane's four units share a line");
  u32x4 x[9];
  {
    const uint32_t oq = W::vec_u(g * 48 + hr * 16 + 4 * pj), ok = W::vec_u((G::NH + g) * 16 + 4 * pj);
    const uint32_t ov = W::vec_u((G::NH + G::KVH + g) * 16 + (lane >> 2)), sq = W::vec_s(C_QKV, slot);
    C.template poll<9>(50, has_new ? 0x1ffu : 0xfu, [&](const u32x4& u) { return C.vec_ok(u, l); },
                       [&](int i) { return i < 8 ? (i < 4 ? oq : ok) + 16u * uint32_t(i % 4) : ov; }, [&](int) { return sq; }, x);
  }
  auto half = [&](int i, int h) {
    return h == 0 ? make_uint4(x[i].x, x[i + 1].x, x[i + 2].x, x[i + 3].x)
                  : make_uint4(x[i].y, x[i + 1].y, x[i + 2].y, x[i + 3].y);
  };
  const uint4 k0 = half(4, 0), k1 = half(4, 1);
  const uint2 vnew = make_uint2(x[8].x, x[8].y);
  tr(4);
  float vn[3] = {-INFINITY, -INFINITY, -INFINITY};
  const bf16x8 qa0 = __builtin_bit_cast(bf16x8, half(0, 0)), qa1 = __builtin_bit_cast(bf16x8, half(0, 1));
  // ---- scores: quads of 4 tiles (64 tokens), dealt round-robin to the waves.  D = Q K^T on the matrix
  // cores with the three q heads in rows 4i .. 4i + 2 of every row block i, so lane l takes its token's
  // three scores from tile l / 16's accumulator: token l of the quad ----
  float m[3] = {-INFINITY, -INFINITY, -INFINITY};
  uint16_t* sc = &sm.at.sc[0][lane];
  for (int j = w; j < nquad; j += NCW) {
    const int tl = min(4, nt - 4 * j);
    const uint32_t at = kpos + uint32_t(4 * j) * 2u * PKT;
    C.release(at);
    C.wait_filled(at + uint32_t(tl) * 2u * PKT);
    const uint32_t lo = uint32_t((lane & 15) >> 3) * PKT + uint32_t(lane & 7) * 128u;
    uint4 ka[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        ka[t][h] = C.ring16(at + uint32_t(min(t, tl - 1)) * 2u * PKT, lo + uint32_t((4 * h + pj + (lane & 7)) & 7) * 16u);
    floatx4 d[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa0, __builtin_bit_cast(bf16x8, ka[t][0]),
                                                    floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa1, __builtin_bit_cast(bf16x8, ka[t][1]), d[t], 0, 0, 0);
    const bool in = j * 64 + lane < n;
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      const float y = lane < 32 ? (lane < 16 ? d[0][h] : d[1][h]) : (lane < 48 ? d[2][h] : d[3][h]);
      const float v = in ? rnd(y) * 0.125f : -INFINITY;  // bf16(q.k) / 8 (HF)
      sc[h * S::SCT + j * 64] = uint16_t(f2bf(v));
      m[h] = fmaxf(m[h], v);
    }
  }
  if (has_new) {
    floatx4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa0, __builtin_bit_cast(bf16x8, k0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa1, __builtin_bit_cast(bf16x8, k1), d, 0, 0, 0);
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      vn[h] = rnd(d[h]) * 0.125f;
      m[h] = fmaxf(m[h], vn[h]);
    }
  }
  // ---- the wave's statistics ----
  wave_max_n<3>(m);
  float ls[3] = {0.f, 0.f, 0.f};
  wait_lgkm0();
  for (int j = w; j < nquad; j += NCW)
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      const float v = bf2f(sc[h * S::SCT + j * 64]);
      ls[h] += v == -INFINITY ? 0.f : __expf(v - m[h]);
    }
  wave_sum_n<3>(ls);
  if (has_new)
#pragma unroll
    for (int h = 0; h < 3; ++h) ls[h] += __expf(vn[h] - m[h]);
  if (lane < 6) {
    const int h = lane < 3 ? lane : lane - 3;
    const float a = h == 0 ? m[0] : h == 1 ? m[1] : m[2], b = h == 0 ? ls[0] : h == 1 ? ls[1] : ls[2];
    sm.at.wml[w][lane] = lane < 3 ? a : b;
  }
  C.release(vpos);
  C.cbar();
  // ---- the chunk's statistics: the waves' merged by every wave (lanes 0-11: wave lane % 4, head lane / 4) and
  // published by wave 0 where the pair has other chunks; then the pair's (lane i: chunk i) ----
  auto rl = [](float v, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
  };
  float M[3], inv[3];
  {
    float mq = -INFINITY, lq = 0.f;
    if (lane < 12) { mq = sm.at.wml[lane & 3][lane >> 2]; lq = sm.at.wml[lane & 3][3 + (lane >> 2)]; }
    float mx = fmaxf(mq, dpp<0xb1>(mq, mq));
    mx = fmaxf(mx, dpp<0x4e>(mx, mx));
    float ex = mq == -INFINITY ? 0.f : lq * __expf(mq - mx);
    ex += dpp<0xb1>(0.f, ex);
    ex += dpp<0x4e>(0.f, ex);
#pragma unroll
    for (int h = 0; h < 3; ++h) { M[h] = rl(mx, 4 * h); inv[h] = rl(ex, 4 * h); }
  }
  if (Cc > 1) {
    if (w == 0) {
      skew_delay(p.skew, C.P.wg, l, 14);
      if (lane < 2)
        C.st(W::rec(me, 0, lane),
             lane == 0 ? u32x4{__float_as_uint(M[0]), __float_as_uint(M[1]), __float_as_uint(M[2]), tg}
                       : u32x4{__float_as_uint(inv[0]), __float_as_uint(inv[1]), __float_as_uint(inv[2]), tg});
    }
    tr(5);
    u32x4 y[2];
    const uint32_t o = W::rec(r0 + min(lane, Cc - 1), 0, 0);
    C.template poll<2>(51, 3u, [&](const u32x4& u) { return u.w == tg; }, [&](int i) { return o + 16u * uint32_t(i); },
                       [&](int) { return 0u; }, y);
    const bool mine = lane < Cc;
    float mk[3];
#pragma unroll
    for (int h = 0; h < 3; ++h) M[h] = mk[h] = mine ? __uint_as_float(h == 0 ? y[0].x : h == 1 ? y[0].y : y[0].z) : -INFINITY;
    wave_max_n<3>(M);
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      const float lk = __uint_as_float(h == 0 ? y[1].x : h == 1 ? y[1].y : y[1].z);
      inv[h] = mk[h] == -INFINITY ? 0.f : lk * __expf(mk[h] - M[h]);
    }
    wave_sum_n<3>(inv);
  }
  // ---- KV append of the new token (block360_kernel.inc:124-135), where no load follows for 1 us and more
  // (a wave's loads wait for its earlier stores): k unit u
  // (k0, k1 word u % 4 of piece u / 4) holds dims 2u, 2u + 1 and 32 + 2u, 33 + 2u, v unit u dims 4u .. 4u + 3 ----
  if (has_new) {
    const long long ns = sm.sSlot[one(it.b)];
    if (ns >= 0) {
      uint16_t* cache = reinterpret_cast<uint16_t*>(const_cast<void*>(sm.kvp[l]));
      const long long e = (ns / 16) * p.block_stride + (ns % 16) * p.token_stride + (long long)g * p.head_stride;
      uint16_t *kd = cache + e + p.k_off + 8 * pj, *vd = cache + e + p.v_off + lane;  // v: lanes 0, 4, ...
      if (((reinterpret_cast<uintptr_t>(kd) | reinterpret_cast<uintptr_t>(vd - lane)) & 15u) == 0) {
        if ((lane & 15) == 0) {
          st_global16(kd, k0.x, k0.y, k0.z, k0.w);
          st_global16(kd + 32, k1.x, k1.y, k1.z, k1.w);
        }
        typedef __attribute__((address_space(1))) uint64_t g_u64;
        if ((lane & 3) == 0) *(g_u64*)(vd) = uint64_t(vnew.x) | (uint64_t(vnew.y) << 32);
      } else {
        const uint32_t a[4] = {k0.x, k0.y, k0.z, k0.w}, b[4] = {k1.x, k1.y, k1.z, k1.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if ((lane & 15) == 0) {
            st_global2(kd + 2 * i, uint16_t(a[i] & 0xffffu));
            st_global2(kd + 2 * i + 1, uint16_t(a[i] >> 16));
            st_global2(kd + 32 + 2 * i, uint16_t(b[i] & 0xffffu));
            st_global2(kd + 32 + 2 * i + 1, uint16_t(b[i] >> 16));
          }
        if ((lane & 3) == 0) {
          st_global2(vd, uint16_t(vnew.x & 0xffffu));
          st_global2(vd + 1, uint16_t(vnew.x >> 16));
          st_global2(vd + 2, uint16_t(vnew.y & 0xffffu));
          st_global2(vd + 3, uint16_t(vnew.y >> 16));
        }
      }
    }
  }
  tr(6);
  // ---- p = bf16(exp(s - M) / L) with the pair's M and L (HF); P.V on the matrix cores, p of the heads in the
  // rows as q above, 32 tokens a step: lane l's tokens are packet l / 16 of the step's four, its dims l % 16 of each
  // block of 16.  A lane's eight tokens of one dim come from two transposing reads, four lanes to a row's 32 bytes.
  // (In fp32 dot products on the vector unit this took 0.84 us a quad.) ----
  float* wo = &sm.red[0][0][0];  // [wave][192]
  const int tr_row = (lane & 15) >> 2;
#pragma unroll
  for (int h = 0; h < 3; ++h) inv[h] = 1.0f / inv[h];
  floatx4 acc[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) acc[d] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int j = w; j < nquad; j += NCW) {
    const int tl = min(4, nt - 4 * j);
    const uint32_t at = vpos + uint32_t(4 * j) * 2u * PKT;
    C.release(at);
    uint16_t* pq = &sm.at.sc[0][j * 64];
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      uint16_t* s = pq + h * S::SCT + lane;
      *s = uint16_t(f2bf(__expf(bf2f(*s) - M[h]) * inv[h]));
    }
    C.wait_filled(at + uint32_t(tl) * 2u * PKT);
    wait_lgkm0();
    asm volatile("" ::: "memory");  // the operands read below are these stores, of another type
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // tiles past the run read its last one again, with probability 0
      const uint4 pa = *reinterpret_cast<const uint4*>(pq + hr * S::SCT + 32 * i + 8 * pj);
      uint4 vb[4];
      const uint32_t pk = uint32_t(2 * min(2 * i + (pj >> 1), tl - 1) + (pj & 1)) * PKT + uint32_t(lane & 1) * 8u;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const int c = 2 * d + ((lane >> 1) & 1);  // 16-byte piece of the row
        const uint2 lo = C.ring_tr(at, pk + uint32_t(tr_row) * 128u + uint32_t((c + tr_row) & 7) * 16u);
        const uint2 hi = C.ring_tr(at, pk + uint32_t(tr_row + 4) * 128u + uint32_t((c + tr_row + 4) & 7) * 16u);
        vb[d] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
#pragma unroll
      for (int d = 0; d < 4; ++d)
        acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pa), __builtin_bit_cast(bf16x8, vb[d]),
                                                        acc[d], 0, 0, 0);
    }
  }
  const float vf = (lane & 1) ? bf_hi((lane & 2) ? vnew.y : vnew.x) : bf_lo((lane & 2) ? vnew.y : vnew.x);
#pragma unroll
  for (int h = 0; h < 3; ++h) {  // lane: dim
    float v = lane < 32 ? (lane < 16 ? acc[0][h] : acc[1][h]) : (lane < 48 ? acc[2][h] : acc[3][h]);
    if (has_new) v = fmaf(rnd(__expf(vn[h] - M[h]) * inv[h]), vf, v);
    wo[w * 192 + h * 64 + lane] = v;
  }
  C.release(C.pos);
  C.cbar();
  // ---- publish (wave 0): a pair in one chunk gives its attention values, others their fp32 partial sums ----
  const uint32_t att = W::vec_s(C_ATT, slot);
  if (w == 0) {
    skew_delay(p.skew, C.P.wg, l, 15);
    if (Cc > 1) {
      float v[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NCW; ++j) v[i] += wo[j * 192 + 3 * lane + i];
      }
      C.st(W::rec(me, 0, 2 + lane), u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), tg});
    } else if (lane < GRP) {
      float v[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NCW; ++j) v[i] += wo[j * 192 + 6 * lane + i];
      }
      C.st(W::vec_u(g * GRP + lane), u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), tg}, att);
    }
    tr(7);
  }
  // ---- combine (wave 2): chunk c of a pair adds groups [32 c / C, 32 (c + 1) / C) of 6 values over the C chunks, in
  // chunk order, two lanes a group, and publishes them ----
  const int g0 = GRP * ci / Cc, ng = GRP * (ci + 1) / Cc - g0;
  if (w == 2 && Cc > 1 && ng > 0) {
    const uint32_t ou = uint32_t(2 + 2 * g0 + min(lane, 2 * ng - 1)) * 16u;
    float v[3] = {0.f, 0.f, 0.f};
    constexpr int N = 13;  // a sequence alone in its cell has up to 21 chunks a head
    for (int c0 = 0; c0 < Cc; c0 += N) {
      u32x4 y[N];
      const int nc = min(N, Cc - c0);
      C.template poll<N>(52, (1u << nc) - 1u, [&](const u32x4& u) { return u.w == tg; }, [&](int) { return ou; },
                         [&](int i) { return W::rec(r0 + c0 + i, 0, 0); }, y);
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (i < nc) {
          v[0] += __uint_as_float(y[i].x);
          v[1] += __uint_as_float(y[i].y);
          v[2] += __uint_as_float(y[i].z);
        }
    }
    float y[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) y[i] = dpp<0xb1>(0.f, v[i]);  // the pair's other lane
    if ((lane & 1) == 0 && lane < 2 * ng)
      C.st(W::vec_u(g * GRP + g0 + (lane >> 1)), u32x4{pack2(v[0], v[1]), pack2(v[2], y[0]), pack2(y[1], y[2]), tg}, att);
  }
  tr(8);
}
// ------------------------------------------------------------------------------------------------
// Attention over this workgroup's items, end to end.
// ------------------------------------------------------------------------------------------------
template <class G, int PX>
__device__ __forceinline__ void attention_many(CC<G, PX>& C, int l) {
  using S = CG<G, PX>;
  using W = CW<G>;
  const Params& p = C.p;
  SmemC<G, PX>& sm = C.sm;
  const int lane = C.lane, w = C.cw;
  const int ni = __builtin_amdgcn_readfirstlane(sm.ni), ntile = __builtin_amdgcn_readfirstlane(sm.ntile);
  const uint32_t tg = C.tag;
  const int wgkey = C.P.cell * S::R;
  const uint32_t kpos = C.pos, vpos = kpos + uint32_t(ntile) * 2u * PKT;
  C.pos = vpos + uint32_t(ntile) * 2u * PKT;
  auto tr = [&](int ev) { if (C.ct == 0) trace_at(p, l, ev, p.n_layers); };
  const int slot0 = C.slot0();
  // ---- q (and leaders' new k, v): 48 + 32 units per item ----
  auto q_units = [&](auto nn, int id0) {
    constexpr int UPI = 80, N = decltype(nn)::value;
    int off[N], at[N];
    u32x4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int id = min(id0 + C.ct + i * NCT, ni * UPI - 1), k = id / UPI;
      const int e0 = id - k * UPI, e = e0 < 48 || sm.it[k].leader ? e0 : e0 - 32;  // no k, v: a q unit again
      const int g = sm.it[k].g;
      const int u = e < 48 ? g * 48 + e : e < 64 ? G::NH * 16 + g * 16 + e - 48 : (G::NH + G::KVH) * 16 + g * 16 + e - 64;
      off[i] = int(W::vec_u(u) + W::vec_s(C_QKV, slot0 + sm.it[k].slot));
      // q and k units: two RoPE pairs, dims 2d, 2d + 1 and 2d + 32, 2d + 33 (d = e % 16); v: dims 4d ..
      at[i] = (k * 5 + (e >> 4)) * 64 + (e & 15) * (e < 64 ? 2 : 4) + (e < 64 ? 0 : 1 << 16);
    }
    C.template poll<N>(50, ni > 0 ? (1u << N) - 1u : 0u, [&](const u32x4& u) { return C.vec_ok(u, l); },
                       [&](int i) { return uint32_t(off[i]); }, [&](int) { return 0u; }, x);
    uint16_t* q = &sm.at.q[0][0][0];
    if (ni > 0)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int a = at[i] & 0xffff;
        *reinterpret_cast<uint32_t*>(q + a) = x[i].x;
        *reinterpret_cast<uint32_t*>(q + a + (at[i] >> 16 ? 2 : 32)) = x[i].y;
      }
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (ni <= 3) q_units(One{}, 0);
  else { q_units(Two{}, 0); if (ni > 6) q_units(One{}, 2 * NCT); }
  C.cbar();
  tr(4);
  // ---- scores: quads of 4 tiles (64 tokens), dealt round-robin to the waves.  D = Q K^T on the matrix
  // cores with the three q heads in rows 4i .. 4i + 2 of every row block i, so lane l takes its token's
  // three scores from tile l / 16's accumulator: token l of the quad ----
  const int hr = (lane & 3) < 3 ? (lane & 3) : 0, q8 = (lane >> 4) * 8;
  for (int k = 0; k < ni; ++k) {
    const int n = __builtin_amdgcn_readfirstlane(sm.it[k].n), nt = __builtin_amdgcn_readfirstlane(sm.it[k].ntile);
    const int tile0 = __builtin_amdgcn_readfirstlane(sm.it[k].tile0), quad0 = __builtin_amdgcn_readfirstlane(sm.it[k].quad0);
    const int sc0 = __builtin_amdgcn_readfirstlane(sm.it[k].sc0);
    const int nquad = (nt + 3) / 4;
    const bf16x8 qa0 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&sm.at.q[k][hr][q8]));
    const bf16x8 qa1 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&sm.at.q[k][hr][32 + q8]));
    float m[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int j = (w - quad0) & 3; j < nquad; j += NCW) {
      const int tl = min(4, nt - 4 * j);
      const uint32_t at = kpos + uint32_t(tile0 + 4 * j) * 2u * PKT;
      C.release(at);
      C.wait_filled(at + uint32_t(tl) * 2u * PKT);
      const uint32_t lo = uint32_t((lane & 15) >> 3) * PKT + uint32_t(lane & 7) * 128u;
      uint4 ka[4][2];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          ka[t][h] = C.ring16(at + uint32_t(min(t, tl - 1)) * 2u * PKT, lo + uint32_t((4 * h + (lane >> 4) + (lane & 7)) & 7) * 16u);
      floatx4 d[4];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa0, __builtin_bit_cast(bf16x8, ka[t][0]),
                                                      floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa1, __builtin_bit_cast(bf16x8, ka[t][1]), d[t], 0, 0, 0);
      const bool in = j * 64 + lane < n;
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        const float x = lane < 32 ? (lane < 16 ? d[0][h] : d[1][h]) : (lane < 48 ? d[2][h] : d[3][h]);
        const float v = in ? rnd(x) * 0.125f : -INFINITY;  // bf16(q.k) / 8 (HF)
        sm.at.sc[h][sc0 + j * 64 + lane] = uint16_t(f2bf(v));
        m[h] = fmaxf(m[h], v);
      }
    }
    // the new token, by the wave after the one that has the item's last quad
    const bool has_new = sm.it[k].leader && ((quad0 + nquad) & 3) == w;
    float vn[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (has_new) {
      const float kd = bf2f(sm.at.q[k][3][lane]);
#pragma unroll
      for (int h = 0; h < 3; ++h) vn[h] = bf2f(sm.at.q[k][h][lane]) * kd;
      wave_sum_n<3>(vn);
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        vn[h] = rnd(vn[h]) * 0.125f;
        if (lane == 0) sm.at.snew[k][h] = vn[h];
        m[h] = fmaxf(m[h], vn[h]);
      }
    }
    wave_max_n<3>(m);
    float ls[3] = {0.f, 0.f, 0.f};
    wait_lgkm0();
    for (int j = (w - quad0) & 3; j < nquad; j += NCW)
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        const float v = bf2f(sm.at.sc[h][sc0 + j * 64 + lane]);
        ls[h] += v == -INFINITY ? 0.f : __expf(v - m[h]);
      }
    wave_sum_n<3>(ls);
    if (has_new)
#pragma unroll
      for (int h = 0; h < 3; ++h) ls[h] += __expf(vn[h] - m[h]);
    if (lane < 6) {
      const int h = lane < 3 ? lane : lane - 3;
      const float a = h == 0 ? m[0] : h == 1 ? m[1] : m[2], b = h == 0 ? ls[0] : h == 1 ? ls[1] : ls[2];
      sm.at.wml[k][w][lane] = lane < 3 ? a : b;
    }
  }
  C.release(vpos);
  C.cbar();
  // ---- the waves' statistics merged (lanes 0-11: wave lane % 4, head lane / 4); only a workgroup's first
  // and last item can belong to a pair with other chunks, whose statistics are exchanged ----
  skew_delay(p.skew, C.P.wg, l, 14);
  auto rl = [](float v, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
  };
  for (int k = w; k < ni; k += NCW) {
    float mq = -INFINITY, lq = 0.f;
    if (lane < 12) { mq = sm.at.wml[k][lane & 3][lane >> 2]; lq = sm.at.wml[k][lane & 3][3 + (lane >> 2)]; }
    float mx = fmaxf(mq, dpp<0xb1>(mq, mq));
    mx = fmaxf(mx, dpp<0x4e>(mx, mx));
    float ex = mq == -INFINITY ? 0.f : lq * __expf(mq - mx);
    ex += dpp<0xb1>(0.f, ex);
    ex += dpp<0x4e>(0.f, ex);
    if (sm.it[k].C > 1) {
      const u32x4 um = {__float_as_uint(rl(mx, 0)), __float_as_uint(rl(mx, 4)), __float_as_uint(rl(mx, 8)), tg};
      const u32x4 ul = {__float_as_uint(rl(ex, 0)), __float_as_uint(rl(ex, 4)), __float_as_uint(rl(ex, 8)), tg};
      if (lane < 2) C.st(W::rec(wgkey + C.P.r, k, lane), lane == 0 ? um : ul);
    } else if (lane < 12 && (lane & 3) == 0) {
      sm.at.gml[k][lane >> 2] = mx;
      sm.at.gml[k][3 + (lane >> 2)] = 1.0f / ex;
    }
  }
  tr(5);
  if (w < 2) {  // wave 0: the first item; wave 1: the last, when there are two or more
    const int k = w == 0 ? 0 : ni - 1;
    if (ni > w && sm.it[k].C > 1) {
      const int Cc = sm.it[k].C, r0 = sm.it[k].r0, k0 = sm.it[k].k0;
      int off[2];
      u32x4 x[2];
      const int c = min(lane, Cc - 1);
#pragma unroll
      for (int i = 0; i < 2; ++i) off[i] = int(W::rec(wgkey + r0 + c, c == 0 ? k0 : 0, i));
      C.template poll<2>(51, 3u, [&](const u32x4& u) { return u.w == tg; }, [&](int i) { return uint32_t(off[i]); },
                         [&](int) { return 0u; }, x);
      const bool mine = lane < Cc;
      float M[3], mk[3], lk[3];
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        mk[h] = M[h] = mine ? __uint_as_float(h == 0 ? x[0].x : h == 1 ? x[0].y : x[0].z) : -INFINITY;
        lk[h] = __uint_as_float(h == 0 ? x[1].x : h == 1 ? x[1].y : x[1].z);
      }
      wave_max_n<3>(M);
#pragma unroll
      for (int h = 0; h < 3; ++h) lk[h] = mk[h] == -INFINITY ? 0.f : lk[h] * __expf(mk[h] - M[h]);
      wave_sum_n<3>(lk);
      if (lane < 3) {
        sm.at.gml[k][lane] = lane == 0 ? M[0] : lane == 1 ? M[1] : M[2];
        sm.at.gml[k][3 + lane] = 1.0f / (lane == 0 ? lk[0] : lane == 1 ? lk[1] : lk[2]);
      }
    }
  }
  if (w == 2)  // KV append of the leaders' new tokens (block360_kernel.inc:124-135)
    for (int k = 0; k < ni; ++k) {
      if (!sm.it[k].leader || lane >= 16) continue;
      const long long slot = sm.sSlot[sm.it[k].b];
      if (slot < 0) continue;
      uint16_t* cache = reinterpret_cast<uint16_t*>(const_cast<void*>(sm.kvp[l]));
      const int part = lane >> 3, piece = lane & 7;
      const long long e = (slot / 16) * p.block_stride + (slot % 16) * p.token_stride +
                          (long long)sm.it[k].g * p.head_stride + (part ? p.v_off : p.k_off);
      const uint4 x = *reinterpret_cast<const uint4*>(&sm.at.q[k][3 + part][piece * 8]);
      uint16_t* dst = cache + e + piece * 8;
      if ((reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
        st_global16(dst, x.x, x.y, x.z, x.w);
      } else {
        const uint32_t val[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          st_global2(dst + 2 * i, uint16_t(val[i] & 0xffffu));
          st_global2(dst + 2 * i + 1, uint16_t(val[i] >> 16));
        }
      }
    }
  C.cbar();
  tr(6);
  // ---- p = bf16(exp(s - M) / L) with the pair's M and L (HF), P.V: lane (quarter, d4) owns dims
  // 4 d4 .. 4 d4 + 3; the token pairs of a tile go round-robin to the four 16-lane quarters ----
  const int qv = lane >> 4, d4 = lane & 15;
  const uint32_t voff = uint32_t(d4 & 1) * 8u;
  float* wo = &sm.red[0][0][0];  // [item][wave][192]
  for (int k = 0; k < ni; ++k) {
    const int nt = __builtin_amdgcn_readfirstlane(sm.it[k].ntile);
    const int tile0 = __builtin_amdgcn_readfirstlane(sm.it[k].tile0), quad0 = __builtin_amdgcn_readfirstlane(sm.it[k].quad0);
    const int sc0 = __builtin_amdgcn_readfirstlane(sm.it[k].sc0);
    const int nquad = (nt + 3) / 4;
    float M[3], inv[3];
#pragma unroll
    for (int h = 0; h < 3; ++h) { M[h] = sm.at.gml[k][h]; inv[h] = sm.at.gml[k][3 + h]; }
    float acc[3][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int j = (w - quad0) & 3; j < nquad; j += NCW) {
      const int tl = min(4, nt - 4 * j);
      const uint32_t at = vpos + uint32_t(tile0 + 4 * j) * 2u * PKT;
      C.release(at);
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        uint16_t* s = &sm.at.sc[h][sc0 + j * 64 + lane];
        *s = uint16_t(f2bf(__expf(bf2f(*s) - M[h]) * inv[h]));
      }
      wait_lgkm0();
      asm volatile("" ::: "memory");  // the pairs read below are these stores, of another type
      C.wait_filled(at + uint32_t(tl) * 2u * PKT);
      const uint16_t* pb = &sm.at.sc[0][sc0 + j * 64];
      // tiles past the run read its last one again, with probability 0; two tiles' operands at a time
#pragma unroll
      for (int t0 = 0; t0 < 4; t0 += 2) {
        uint2 va[4], vb[4];
        uint32_t pp[4][3];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int t = t0 + (x >> 1), jt = 2 * (qv + 4 * (x & 1));  // token pair jt, jt + 1 of tile t
          const uint32_t pk = at + uint32_t(2 * min(t, tl - 1) + (x & 1)) * PKT;
          const int r = jt & 7;
          va[x] = C.ring8(pk, uint32_t(r) * 128u + uint32_t(((d4 >> 1) + r) & 7) * 16u + voff);
          vb[x] = C.ring8(pk, uint32_t(r + 1) * 128u + uint32_t(((d4 >> 1) + r + 1) & 7) * 16u + voff);
#pragma unroll
          for (int h = 0; h < 3; ++h) pp[x][h] = *reinterpret_cast<const uint32_t*>(pb + h * S::SCT + t * 16 + jt);
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const uint32_t v0 = __builtin_amdgcn_perm(vb[x].x, va[x].x, 0x05040100u), v1 = __builtin_amdgcn_perm(vb[x].x, va[x].x, 0x07060302u);
          const uint32_t v2 = __builtin_amdgcn_perm(vb[x].y, va[x].y, 0x05040100u), v3 = __builtin_amdgcn_perm(vb[x].y, va[x].y, 0x07060302u);
#pragma unroll
          for (int h = 0; h < 3; ++h) {
            acc[h][0] = dot2(pp[x][h], v0, acc[h][0]);
            acc[h][1] = dot2(pp[x][h], v1, acc[h][1]);
            acc[h][2] = dot2(pp[x][h], v2, acc[h][2]);
            acc[h][3] = dot2(pp[x][h], v3, acc[h][3]);
          }
        }
      }
    }
    if (sm.it[k].leader && ((quad0 + nquad) & 3) == w && qv == 0)
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        const float pj = rnd(__expf(sm.at.snew[k][h] - M[h]) * inv[h]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[h][i] = fmaf(pj, bf2f(sm.at.q[k][4][4 * d4 + i]), acc[h][i]);
      }
#pragma unroll
    for (int h = 0; h < 3; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[h][i] = column_total<false>(acc[h][i]);
    if (lane < 16)
#pragma unroll
      for (int h = 0; h < 3; ++h)
        *reinterpret_cast<floatx4*>(wo + (k * NCW + w) * 192 + h * 64 + 4 * d4) =
            floatx4{acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
  }
  C.release(C.pos);
  C.cbar();
  // ---- publish: a pair in one chunk gives its attention values, others their fp32 partial sums ----
  skew_delay(p.skew, C.P.wg, l, 15);
  for (int k = w; k < ni; k += NCW) {
    const float* o = wo + k * NCW * 192;
    if (sm.it[k].C > 1) {
      float v[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int x = 0; x < NCW; ++x) v[i] += o[x * 192 + 3 * lane + i];
      }
      C.st(W::rec(wgkey + C.P.r, k, 2 + lane), u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), tg});
    } else if (lane < 32) {
      float v[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int x = 0; x < NCW; ++x) v[i] += o[x * 192 + 6 * lane + i];
      }
      C.st(W::vec_u(sm.it[k].g * 32 + lane) + W::vec_s(C_ATT, slot0 + sm.it[k].slot),
           u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), tg});
    }
  }
  tr(7);
  // ---- combine: chunk c of a pair adds groups [32 c / C, 32 (c + 1) / C) of 6 values over the C chunks, in
  // chunk order, two lanes a group, and publishes them (wave 0: the first item's pair, wave 1: the last's) ----
  if (w < 2) {
    const int k = w == 0 ? 0 : ni - 1;
    const int Cc = ni > w ? __builtin_amdgcn_readfirstlane(sm.it[k].C) : 1;
    const int ci = ni > w ? __builtin_amdgcn_readfirstlane(sm.it[k].c) : 0;
    const int g0 = GRP * ci / Cc, ng = GRP * (ci + 1) / Cc - g0;
    if (Cc > 1 && ng > 0) {
      const int r0 = wgkey + __builtin_amdgcn_readfirstlane(sm.it[k].r0), k0 = __builtin_amdgcn_readfirstlane(sm.it[k].k0);
      const uint32_t o = uint32_t(2 + 2 * g0 + min(lane, 2 * ng - 1)) * 16u;
      float v[3] = {0.f, 0.f, 0.f};
      constexpr int N = 12;
      for (int c0 = 0; c0 < Cc; c0 += N) {
        u32x4 x[N];
        const int n = min(N, Cc - c0);
        C.template poll<N>(52, (1u << n) - 1u, [&](const u32x4& u) { return u.w == tg; }, [&](int) { return o; },
                           [&](int i) { return W::rec(r0 + c0 + i, c0 + i == 0 ? k0 : 0, 0); }, x);
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (i < n) {
            v[0] += __uint_as_float(x[i].x);
            v[1] += __uint_as_float(x[i].y);
            v[2] += __uint_as_float(x[i].z);
          }
      }
      float y[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) y[i] = dpp<0xb1>(0.f, v[i]);  // the pair's other lane
      if ((lane & 1) == 0 && lane < 2 * ng)
        C.st(W::vec_u(sm.it[k].g * 32 + g0 + (lane >> 1)) + W::vec_s(C_ATT, slot0 + sm.it[k].slot),
             u32x4{pack2(v[0], v[1]), pack2(v[2], y[0]), pack2(y[1], y[2]), tg});
    }
  }
  C.cbar();  // the attention buffers share storage with the staged rows
  tr(8);
}

template <class G, int PX>
__device__ __forceinline__ void consumer(const Params& p, const PlanC<G, PX>& P, SmemC<G, PX>& sm, uint32_t epoch,
                                         const void* region) {
  using S = CG<G, PX>;
  using W = CW<G>;
  CC<G, PX> C(p, P, sm, epoch, region);
  const int B = p.B;
  const int nuq = P.q1 - P.q0, nuo = P.o1 - P.o0, nua = P.a1 - P.a0;
  const int rg = C.lane >> 4, col = C.lane & 15;  // MFMA output row group and sequence column
  auto tr = [&](int l, int ev) { if (C.ct == 0) trace_at(p, l, ev, p.n_layers); };
  if (C.ct == 0) trace_tail(p, 0);
  // cos / sin of this lane's two RoPE pairs in its wave's QKV tile (the same in every layer)
  float rc[2] = {1.f, 1.f}, rs_[2] = {0.f, 0.f};
  const int uq = 4 * C.cw + rg;  // this lane's QKV unit within the workgroup's
  if (uq < nuq && col < C.ns && 4 * (P.q0 + uq) < (G::NH + G::KVH) * 64)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const size_t at = size_t(sm.sPos[sm.sid[col]]) * 64 + size_t((2 * (P.q0 + uq) + k) & 31);
      rc[k] = p.cs_fp32 ? reinterpret_cast<const float*>(p.cos_sin)[at] : bf2f(reinterpret_cast<const uint16_t*>(p.cos_sin)[at]);
      rs_[k] = p.cs_fp32 ? reinterpret_cast<const float*>(p.cos_sin)[at + 32]
                         : bf2f(reinterpret_cast<const uint16_t*>(p.cos_sin)[at + 32]);
    }
  const int seq = col < C.ns ? sm.sid[col] : 0;  // global sequence of this lane's column
  // layer 0's x: the embedding rows
  auto first_x = [&](const NormW<G, PX>& nw) {
    if (C.cw < C.ns) {
      const uint2* row = reinterpret_cast<const uint2*>(p.embed + size_t(sm.sId[sm.sid[C.cw]]) * G::H);
      uint2 v[S::LU];
#pragma unroll
      for (int j = 0; j < S::LU; ++j) v[j] = C.lane + 64 * j < S::HU ? row[C.lane + 64 * j] : make_uint2(0u, 0u);
      keep_rows(C, v);
      norm_row(C, v, C.cw, nw);
    }
    C.cbar();
  };
  for (int l = 0; l < p.n_layers && C.ns > 0; ++l) {
    // ---------------- RMSNorm(x) + QKV + RoPE ----------------
    C.refresh();
    C.begin_layer(l);
    tr(l, 0);
    const NormW<G, PX> nw1(C);
    const Weights<S::KSH, S::TQ, G, PX> wq(C, (4 * nuq + 7) / 8);
    if (l == 0) first_x(nw1);
    else stage_x(C, C_X, l - 1, nw1);
    tr(l, 1);
    {
      floatx4 acc[S::TQ];
      wq.apply(C, S::XH, acc, C.ns);
      to_red<4, S::TQ>(C, acc);
      skew_delay(p.skew, P.wg, l, C_QKV);
      if (uq < nuq && col < C.ns && C.cw < S::TQ) {
        const floatx4 d = red_sum<4>(C, C.cw, C.lane);
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = rnd(d[j]);
        u32x4 u = C.vec_unit(0u, 0u, l);
        if (4 * (P.q0 + uq) < (G::NH + G::KVH) * 64) {
          // bf16(bf16(x cos) + bf16(rotate_half(x) sin)) (modeling_llama.py:138-160)
          float e[4];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const float x0 = o[2 * k], x1 = o[2 * k + 1];
            e[k] = rnd(x0 * rc[k]) + rnd((-x1) * rs_[k]);
            e[2 + k] = rnd(x1 * rc[k]) + rnd(x0 * rs_[k]);
          }
          u.x = pack2(e[0], e[1]);
          u.y = pack2(e[2], e[3]);
        } else {
          u.x = pack2(o[0], o[1]);
          u.y = pack2(o[2], o[3]);
        }
        C.st(W::vec_u(P.q0 + uq) + W::vec_s(C_QKV, C.slot0() + col), u);
      }
    }
    tr(l, 3);
    // ---------------- attention ----------------
    C.refresh();
    if constexpr (S::E2E) attention_many<G, PX>(C, l);
    else attention_one<G, PX>(C, l);
    // ---------------- O + residual ----------------
    C.refresh();
    auto rows_out = [&](int kind, int site, bool outputs) {
      skew_delay(p.skew, P.wg, l, site);
#pragma unroll
      for (int t = 0; t < S::TO; ++t) {
        const int u = 4 * t + rg;
        if (t % NCW != C.cw || u >= nuo || col >= C.ns) continue;
        const floatx4 d = red_sum<4>(C, t, C.lane);
        const uint2 r = sm.res[col][u];
        const uint32_t y0 = pack2(bf_lo(r.x) + rnd(d[0]), bf_hi(r.x) + rnd(d[1]));
        const uint32_t y1 = pack2(bf_lo(r.y) + rnd(d[2]), bf_hi(r.y) + rnd(d[3]));
        C.st(W::vec_u(P.o0 + u) + W::vec_s(kind, C.slot0() + col), C.vec_unit(y0, y1, l));
        if (outputs && p.layer_outputs)
          *reinterpret_cast<uint2*>(p.layer_outputs + (size_t(l) * B + seq) * G::H + 4 * (P.o0 + u)) = make_uint2(y0, y1);
      }
    };
    const Weights<S::KSH, S::TO, G, PX> wo(C, (4 * nuo + 7) / 8);
    stage_att(C);
    tr(l, 9);
    {
      floatx4 acc[S::TO];
      wo.apply(C, S::XH, acc, C.ns);
      to_red<4, S::TO>(C, acc);
      rows_out(C_H1, C_H1, false);
    }
    tr(l, 11);
    // ---------------- RMSNorm(h1) + gate/up + SwiGLU ----------------
    C.refresh();
    const NormW<G, PX> nw2(C);
    const Weights<S::KSH, S::TA, G, PX> wa(C, nua);
    stage_x(C, C_H1, l, nw2);
    tr(l, 12);
    {
      floatx4 acc[S::TA];
      wa.apply(C, S::XH, acc, C.ns);
      to_red<4, S::TA>(C, acc);
      skew_delay(p.skew, P.wg, l, C_ACT);
#pragma unroll
      for (int t = 0; t < S::TA; ++t) {
        const int u = 2 * t + (rg >> 1);  // row groups of a tile: gate, up of unit 2t, gate, up of unit 2t + 1
        if (t % NCW != C.cw || (rg & 1) || u >= nua || col >= C.ns) continue;
        const floatx4 g = red_sum<4>(C, t, C.lane), x = red_sum<4>(C, t, C.lane + 16);
        float av[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float gv = rnd(g[j]);
          av[j] = rnd(gv / (1.0f + expf(-gv))) * rnd(x[j]);
        }
        C.st(W::vec_u(P.a0 + u) + W::vec_s(C_ACT, C.slot0() + col), C.vec_unit(pack2(av[0], av[1]), pack2(av[2], av[3]), l));
      }
    }
    tr(l, 14);
    // ---------------- down + residual ----------------
    C.refresh();
    const Weights<S::KSI, S::TO, G, PX> wd(C, (4 * nuo + 7) / 8);
    stage_act<G, PX>(C, l);
    tr(l, 15);
    {
      floatx4 acc[S::TO];
      wd.apply(C, S::XI, acc, C.ns);
      to_red<4, S::TO>(C, acc);
      rows_out(C_X, C_X, true);
    }
    tr(l, 17);
  }
  // ---------------- final RMSNorm of every sequence, LM head, argmax ----------------
  {
    // (a wave's sequences one after the other: all are there by the time the first is)
    const NormW<G, PX> nw(C);
    const uint32_t o = W::vec_u(C.lane), oe = W::vec_u(min(C.lane, S::HU - 1 - 64 * (S::LU - 1)));
#pragma unroll 1
    for (int b = C.cw; b < B; b += NCW) {
      u32x4 x[S::LU];
      uint2 v[S::LU];
      const uint32_t so = W::vec_s(C_X, __builtin_amdgcn_readfirstlane(sm.cs[b]));
      C.template poll<S::LU>(53, (1u << S::LU) - 1u, [&](const u32x4& u) { return C.vec_ok(u, p.n_layers - 1); },
                             [&](int j) { return j == S::LU - 1 ? oe : o; },
                             [&](int j) { return so + uint32_t(j) * W::STRIDE64; }, x);
#pragma unroll
      for (int j = 0; j < S::LU; ++j) v[j] = make_uint2(x[j].x, x[j].y);
      norm_row(C, v, b, nw);
    }
    C.cbar();
    if (P.wg == 0 && C.ct < S::HU)
      for (int i = 0; i < B; ++i)
        *reinterpret_cast<uint2*>(p.out_hidden + size_t(i) * G::H + 4 * C.ct) =
            *reinterpret_cast<const uint2*>(sm.xs + i * S::XH + 4 * C.ct);
  }
  float best = -INFINITY;
  int bidx = 0x7fffffff;
  if (P.v1 > P.v0) {
    floatx4 acc[S::TL / NCW];  // each wave whole tiles
    project<S::KSH, S::TL, 1, 2, 2 * S::TL>(C, 2 * S::TL, S::XH, acc, B);
    if (col < B)
#pragma unroll
      for (int t = 0; t < S::TL / NCW; ++t) {
        const floatx4 d = acc[t];
        const int r = P.v0 + 16 * (C.cw + t * NCW) + 4 * rg;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = rnd(d[j]);
          if (x > best || (x == best && r + j < bidx)) { best = x; bidx = r + j; }
        }
        if (p.out_logits)
          *reinterpret_cast<uint2*>(p.out_logits + size_t(col) * G::V + r) = make_uint2(pack2(d[0], d[1]), pack2(d[2], d[3]));
      }
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {  // lanes l, l+16, l+32, l+48 hold the same sequence
      const float ov = __shfl_xor(best, o);
      const int oi = __shfl_xor(bidx, o);
      if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
    }
  }
  if (C.lane < BMAX) { sm.lm_val[C.cw][C.lane] = best; sm.lm_idx[C.cw][C.lane] = bidx; }
  C.cbar();
  if (C.ct == 0) trace_tail(p, 1);
  // end records: one unit {best value, its index, gave up, epoch} per workgroup and sequence
  if (C.ct < B) {
    float bv = sm.lm_val[0][C.ct];
    int bi = sm.lm_idx[0][C.ct];
    for (int v = 1; v < NCW; ++v)
      if (sm.lm_val[v][C.ct] > bv || (sm.lm_val[v][C.ct] == bv && sm.lm_idx[v][C.ct] < bi)) {
        bv = sm.lm_val[v][C.ct];
        bi = sm.lm_idx[v][C.ct];
      }
    skew_delay(p.skew, P.wg, p.n_layers, 13);
    C.st(W::end(C.ct, P.wg), u32x4{__float_as_uint(bv), uint32_t(bi), C.dead ? 1u : 0u, epoch});
  }
  if (P.wg != 0) {
    if (p.out_logits && (C.dead || aborted(p.ws, epoch)))  // this workgroup's logits rows are not valid
      for (int b = 0; b < B; ++b)
        for (int i = P.v0 + C.ct; i < P.v1; i += NCT) p.out_logits[size_t(b) * G::V + i] = 0x7fc0;
    return;
  }
  C.cbar();  // lm_val is reused below
  uint32_t bad = 0;
  // workgroup 0: per sequence, argmax over the NWG candidates (first index on ties, as torch.argmax)
  for (int b = 0; b < B; ++b) {
    u32x4 x[1];
    C.template poll<1>(54, 1u, [&](const u32x4& u) { return u.w == epoch; }, [&](int) { return W::end(b, C.ct); },
                       [&](int) { return 0u; }, x);
    float bv = __uint_as_float(x[0].x);
    int bi = int(x[0].y);
    bad |= x[0].z != 0u || x[0].w != epoch ? 1u : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o);
      const int oi = __shfl_xor(bi, o);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (C.lane == 0) { sm.lm_val[C.cw][b] = bv; sm.lm_idx[C.cw][b] = bi; }
  }
  const bool any_bad = __builtin_amdgcn_ballot_w64(bad != 0u) != 0ull;
  if (C.lane == 0) sm.sums[C.cw][0] = any_bad ? 1.f : 0.f;
  C.cbar();
  bool fail = C.dead || aborted(p.ws, epoch);
  for (int w = 0; w < NCW; ++w) fail = fail || sm.sums[w][0] != 0.f;
  if (C.ct < B) {
    float bv = sm.lm_val[0][C.ct];
    int bi = sm.lm_idx[0][C.ct];
    for (int v = 1; v < NCW; ++v)
      if (sm.lm_val[v][C.ct] > bv || (sm.lm_val[v][C.ct] == bv && sm.lm_idx[v][C.ct] < bi)) {
        bv = sm.lm_val[v][C.ct];
        bi = sm.lm_idx[v][C.ct];
      }
    if (p.out_ids) p.out_ids[C.ct] = fail ? -1 : bi;
  }
  if (fail)
    for (int b = 0; b < B; ++b) {
      step_failed(p, epoch, C.ct, b);
      if (p.out_logits)  // every logits row of the sequence (best effort: see step_failed)
        for (int i = C.ct; i < G::V; i += NCT) p.out_logits[size_t(b) * G::V + i] = 0x7fc0;
    }
}

template <class G, int PX>
__global__ void __launch_bounds__(WG_THREADS, 1) decode_cell(Params p, const void* region) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
  using SM = SmemC<G, PX>;
  SM& sm = *reinterpret_cast<SM*>(smem_raw);
  if (threadIdx.x == 0) {
    for (int w = 0; w < NPW; ++w) sm.front[w] = 0;
    for (int w = 0; w < NCW; ++w) sm.consumed[w] = 0;
    sm.cbar = 0;
  }
  for (int i = threadIdx.x; i < p.n_layers; i += WG_THREADS) {
    const void* const* t = p.layers + size_t(i) * 6;
    LayerW w{};
    w.norm1 = t[0]; w.qkv = t[1]; w.o = t[2]; w.norm2 = t[3]; w.gate_up = t[4]; w.down = t[5];
    sm.lw[i] = w;
    sm.kvp[i] = p.kv[i];
  }
  if (threadIdx.x < p.B) {
    const int t = threadIdx.x;
    sm.sS[t] = min(max(p.seq_lens[t], 1), p.max_seq);
    sm.sPos[t] = int(max(p.positions[t], (int64_t)0));
    sm.sSlot[t] = p.slot_mapping[t];
    const long long id = p.ids_i64 ? reinterpret_cast<const int64_t*>(p.input_ids)[t]
                                   : reinterpret_cast<const int32_t*>(p.input_ids)[t];
    sm.sId[t] = int(min(max(id, 0LL), (long long)G::V - 1));
  }
  trace_begin(p);
  __syncthreads();
  const PlanC<G, PX> P(p, blockIdx.x);
  if (threadIdx.x < 64) setup<G, PX>(p, P, sm);
  __syncthreads();
  // block id of every tile of the workgroup's range (tiles are the cache's 16-token blocks)
  for (int i = threadIdx.x; i < sm.ntile; i += WG_THREADS) {
    int k = 0;
    while (i >= sm.it[k].tile0 + sm.it[k].ntile) ++k;
    sm.blk[i] = p.block_table[size_t(sm.it[k].b) * p.bt_stride + sm.it[k].t0 / 16 + (i - sm.it[k].tile0)];
  }
  wait_vmcnt<0>();
  __syncthreads();
  const uint32_t epoch = step_epoch(p.ws);
  if (threadIdx.x < 64 * NPW) {
    producer<G, PX>(p, P, sm, epoch);
  } else {
    __builtin_amdgcn_s_setprio(1);  // the consumer waves are the step's critical path
    consumer<G, PX>(p, P, sm, epoch, region);
  }
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x == 0) st_dev(p.ws + HDR_EPOCH, epoch);
  trace_end(p);
}

template <class G, int PX>
static int launch(const Params& p, const void* region, hipStream_t stream, int cooperative) {
  static_assert((sizeof(SmemC<G, PX>) + 15) / 16 * 16 + TRACE_LDS_BYTES <= LDS_CU, "LDS budget of one gfx950 workgroup");
  static_assert(SmemC<G, PX>::RING_BYTES >= 64 * PKT, "four k-steps, or five quads of tokens, of the ring");
  static int ready[64] = {};
  static int status[64] = {};
  const void* fn = reinterpret_cast<const void*>(decode_cell<G, PX>);
  size_t lds = sizeof(SmemC<G, PX>);
  const size_t trace_off = (lds + 15) / 16 * 16;
  const size_t lds_traced = trace_off + TRACE_LDS_BYTES;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return PK_ERR_RESIDENCY;
  if (!ready[dev]) {
    hipDeviceProp_t prop;
    int st = 0, max_lds = 0;
    if ((e = hipGetDeviceProperties(&prop, dev)) != hipSuccess) st = e;
    else if ((e = hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) != hipSuccess) st = e;
    else if (__builtin_strncmp(prop.gcnArchName, "gfx950", 6) != 0) st = PK_ERR_ARCH;
    else if (prop.multiProcessorCount < NWG || size_t(max_lds) < lds_traced) st = PK_ERR_RESIDENCY;
    else if ((e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds_traced))) != hipSuccess) st = e;
    status[dev] = st;
    ready[dev] = 1;
  }
  if (status[dev]) return status[dev];
  Params q = p;
  if (q.trace) {
    if (q.n_layers > TR_LAYERS) return PK_ERR_MODEL;
    q.trace_lds = uint32_t(trace_off);
    lds = lds_traced;
  }
  void* args[] = {&q, &region};
  if (cooperative) e = hipLaunchCooperativeKernel(fn, dim3(NWG), dim3(WG_THREADS), args, lds, stream);
  else e = hipLaunchKernel(fn, dim3(NWG), dim3(WG_THREADS), args, lds, stream);
  if (e != hipSuccess) return e;
  return hipGetLastError();
}

}  // namespace cell

// Cells of two XCDs: fewer XCDs a cell read the weights more often, more XCDs make every exchange wider.  us per
// step at 1 / 2 / 4 XCDs (and the kernel of one cell of eight, decode_kernel_b): batch 4: 684 / 596 / 624 (1,055);
// batch 16: 807 / 737 / 829 (1,342).
//
// Pairs in whole workgroups while the block tables' capacity is moderate, end to end above.  One chunk a workgroup takes
// two barriers and no staging of q and k, and P.V runs on the matrix cores; but rounded up to whole workgroups
// the longest chunk is longer than an even share (20 % at 16 sequences), which counts once the stream of
// K and V bounds the step.  us per step end to end / whole: batch 7, 100..2000: 620 / 588; batch 16, 100..2000: 653 /
// 635, 3000..9000: 973 / 1,059.  (The second and later items of a workgroup in the one-chunk form: slower than
// either.)
constexpr long long kWholeTokens = 61440;
constexpr int kPX = 2;
int cell_launch(const Params& p, const void* region, hipStream_t stream, int cooperative) {
  if ((long long)p.B * p.max_seq <= kWholeTokens) return cell::launch<G135, kPX>(p, region, stream, cooperative);
  return cell::launch<cell::EndToEnd<G135>, kPX>(p, region, stream, cooperative);
}
size_t cell_region_bytes() { return size_t(cell::CW<G135>::TOTAL) * 16; }

}  // namespace pk
