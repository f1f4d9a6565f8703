// plh_wavefront.hip -- the persistent layer-wavefront kernel (H <= 128) of the stacked LSTM +
// Linear inference forward on CDNA4 (gfx950).  Every workgroup of a launch is co-resident (the host
// sizes the grid to the device's occupancy) and loops over the time steps itself.
//
// One workgroup per (layer, batch tile of 8 or 16 rows):
//   * each wave owns 16 hidden units and keeps the i, f, g, o rows of [W_ih | W_hh] for them in
//     VGPRs for the whole sequence as fp16 MFMA A fragments (256 KB per layer at H = 128);
//   * per step a wave computes gates^T[64 gate cols, 16 cols] = W[64, K] * [in_t | h_{t-1}]^T with
//     v_mfma_f32_16x16x32_f16 (fp32 accumulate, bias as the initial accumulator); with 8-row tiles
//     the B columns 8..15 repeat rows 0..7 and each lane evaluates two of its four (unit, row)
//     pairs; the next step's input part is issued between this step's gate computations;
//   * the gate nonlinearities and the c/h update run on the accumulator registers; c never leaves
//     VGPRs; h goes to LDS (double-buffered by step) for the next step's recurrent MFMAs;
//   * activations live in "fragment order": a [R rows x 32 k] block is stored as [k/8][row][8],
//     i.e. exactly the B operand of one MFMA (lane l reads 16 B at l * 16), so LDS traffic is
//     conflict-free;
//   * a layer hands h to the next one step by step: each lane sends its units of h_t as one tagged word
//     through a ring of kHandoffSlots steps per (layer, tile), and the same lane of the next layer's
//     workgroup loads it four steps ahead, checks its tag two steps ahead and puts it into LDS.  No
//     counter, barrier or fence sits between the two layers, so layer l+1 runs about six steps behind
//     layer l (measured: the kernel of H 128, L = 4, B = 1, T = 64 87 -> 62 us against chunks of 8 steps, which lagged 18
//     steps per layer; C2 853 -> 787 us, where a chunk's copies also cost ~10% of the steps).  The sends,
//     loads and checks sit under the latency of the step's LDS reads of h.  Where the ring wraps,
//     counters read once per 8 steps keep a layer from running a whole ring ahead;
//   * layer 0 loads x a block of 8 steps at a time into a double-buffered LDS ring, so no step waits on
//     global memory;
//   * a tile's layers run on one XCD where the grid can be arranged so, and then hand h over through
//     its L2;
//   * the Linear head runs in the last layer's epilogue on the final h held in LDS;
//   * every wait between workgroups is bounded in wall-clock time; a failed wait sets a status bit,
//     fails every other wait and poisons the outputs, so the grid always drains.
//
// Reference behaviour restated (mantuoluozk/persistent_lstm_hip): gate order i, f, g, o and the
// c/h recurrence of persistent_lstm_reference.cpp:21-35; fp16 h storage per step and fp32 c of
// persistent_lstm_hip.cu:520-525; the fp32-accumulated head of persistent_lstm_hip.cu:1662-1682.
#include <type_traits>

#include "plh_device.h"

namespace plh {
namespace {

// Workgroup -> (layer, tile).  With xcd_map, workgroups are dispatched round-robin over the 8
// XCDs (block b lands on XCD b % 8), and the mapping puts all layers of a tile on one XCD; the grid
// covers ntile_grid tiles then, a multiple of 8.
__device__ __forceinline__ void block_coords(int b, int ntile, int ntile_grid, int xcd_map, int& layer, int& tile) {
  if (xcd_map) {
    const int per = ntile_grid >> 3;
    const int r = b >> 3;
    tile = r % per * 8 + (b & 7);
    layer = r / per;
  } else {
    layer = b / ntile;
    tile = b % ntile;
  }
}

template <int HP, int ROWS>
struct Tile {
  static_assert(ROWS == 8 || ROWS == 16, "tiles hold 8 or 16 batch rows");
  static constexpr int kWaves = HP / 16;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kKci = HP / 32;          // input-part K chunks (layers >= 1)
  static constexpr int kKcr = HP / 32;          // recurrent K chunks
  static constexpr int kKc = kKci + kKcr;
  static constexpr int kFragVec = 4 * ROWS;     // f16x8 per [ROWS x 32] fragment block
  static constexpr int kUpl = ROWS / 4;         // (unit, row) pairs per lane in the epilogue
  static constexpr int kNw = kUpl / 2;          // 32-bit hand-off words per lane and step
  static constexpr int kSlot = kThreads * kNw * 4;  // bytes of one step in the hand-off ring
};

// Steps per block of the unrolled step loop: layer 0 moves x a block at a time, and a workgroup looks
// at its consumer's progress (and reports its own) once per block.
constexpr int kBlock = 8;
static_assert(kHandoffSlots % kBlock == 0 && kHandoffSlots >= 3 * kBlock,
              "the ring covers the layers' lag and a stale report");

// LDS of one workgroup.  Layers >= 1 keep the inputs of two steps (step t in slot t & 1), layer 0 those
// of two blocks.
template <int HP, int ROWS>
struct WavefrontLds {
  using C = Tile<HP, ROWS>;
  f16x8 xin[2 * kBlock * C::kKci * C::kFragVec];
  f16x8 hist[2][C::kKcr * C::kFragVec];  // h after step t in slot t & 1
  int fail;
  int tlen;
};

// Hand-off words.  A lane's units of one step travel as one 32-bit (8-row tiles) or 64-bit word, tagged
// in one bit: bit 14 (the exponent's top bit) of its last fp16, clear in every h a step computes
// (|h| <= 1).  The tag alternates with the laps of the ring, starting at 1 (the ring is cleared to 0
// before the launch), and a slot is overwritten only once its consumer has read it, so a slot holds
// the wanted step or the one a lap before it, which the tag tells apart.  Sending is one bit-field
// insert of the tag; `word ^ tag` is the value itself, and one compare finds both a stale word (bit 14
// set) and NaN, which lost the bit when it was sent and so arrives as a magnitude above 1 (0x3C01 ..
// 0x3FFF).  The frozen h0 of rows of length 0 may arrive changed the same way: their values feed only
// their own frozen rows.  (A 2-bit lap tag in both halves, with the NaN encoding of the xw_* words, took
// ~11 more VALU instructions per wave and step: C2 0.92 ms.)
constexpr uint32_t kHandoffTag = 0x40000000u;
__device__ __forceinline__ uint32_t handoff_tag(int s) { return ((uint32_t)s / kHandoffSlots) & 1u ? 0u : kHandoffTag; }
// True unless the last fp16 of `w` (its upper half) is at most 1 in magnitude: |w| as a float against
// 0x3C00FFFF, ordered as integers are; "not less or equal" also holds for NaN patterns.
__device__ __forceinline__ bool handoff_special(uint32_t w) {
  return !(__builtin_fabsf(__builtin_bit_cast(float, w)) <= __builtin_bit_cast(float, 0x3C00FFFFu));
}

// Where a layer's step input comes from: the layer below (tagged words), x with one K chunk (I <= 32, so
// the input MFMAs on the other, all-zero chunks are skipped) or with all of them, or, for an input wider
// than the padded hidden size, its projection x_t W_ih^T from the projection GEMM (padded H 128).
enum class Src { kUp, kX1, kXn, kGates };

// The persistent layer-wavefront recurrence of one (layer, tile).  Template: padded hidden size HP,
// batch rows per workgroup ROWS (16, or 8 with the MFMA's B columns 8..15 duplicating rows 0..7 so
// each lane evaluates two (unit, row) pairs instead of four), RAGGED: rows may end before the
// tile's last step (lengths given; without it every row is live at every step and the
// state-freezing selects are compiled out), WIDE: the model's
// input is wider than HP, the step input's source, and DOWN: a layer above takes h.
template <int HP, int ROWS, bool RAGGED, bool WIDE, Src SRC, bool DOWN>
__device__ __forceinline__ void wavefront_body(const ForwardArgs& a, WavefrontLds<HP, ROWS>& lds, int layer, int tile) {
  using C = Tile<HP, ROWS>;
  constexpr int KCI = C::kKci, KCR = C::kKcr, KC = C::kKc, NT = C::kThreads, FV = C::kFragVec;
  constexpr bool UP = SRC == Src::kUp;
  constexpr bool GATES = SRC == Src::kGates;
  constexpr int KIN = SRC == Src::kX1 ? 1 : GATES ? 0 : KCI;  // input-part K chunks with MFMA work
  constexpr int UPL = C::kUpl, NW = C::kNw;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15;            // B-operand / D column
  const int kg = lane >> 4;           // K group of the A/B fragments, row group of D
  const int r = n & (ROWS - 1);       // batch row in the tile
  const int fl = kg * ROWS + r;       // this lane's B fragment within a block

  const int grow = a.row0 + tile * ROWS + r;
  const bool row_ok = grow < a.row_end;
  int len = 0, Tt = a.T;
  if (threadIdx.x == 0) lds.fail = 0;
  if constexpr (RAGGED) {
    if (row_ok) {
      len = a.lengths ? a.lengths[grow] : a.T;
      len = len < 0 ? 0 : (len > a.T ? a.T : len);
    }
    if (threadIdx.x == 0) lds.tlen = 0;
    __syncthreads();
    if (wave == 0 && kg == 0) atomicMax(&lds.tlen, len);
    __syncthreads();
    Tt = __builtin_amdgcn_readfirstlane(lds.tlen);  // steps this tile runs: the longest row in it
  }

  // A batch of equal rows (seen by the prologue's blocks): only the first tile runs, and its head writes
  // row 0's outputs for every row.
  bool uniform = false;
  if (!RAGGED && a.uniform) {
    uint32_t differs = 0;
    for (int i = threadIdx.x; i < a.n_uniform; i += NT) differs |= a.uniform[i];
    uniform = __syncthreads_or(differs != 0u) == 0;
    if (uniform && tile != 0) return;
  }

  // Resident weights: A fragments of [W_ih | W_hh] rows for this wave's 16 units, 4 gates.
  f16x8 w[KC][4];
  if constexpr (!WIDE) {
    const f16x8* wp = reinterpret_cast<const f16x8*>(a.wpack) + ((size_t)(layer * C::kWaves + wave) * KC * 4) * 64 + lane;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
      for (int q = 0; q < 4; ++q) w[kc][q] = (kc < KIN || kc >= KCI) ? wp[(kc * 4 + q) * 64] : f16x8{};
  } else {
    // Models with an input wider than the padded H are packed for the layer-sequential path only: gather
    // the same fragments (row: unit u of gate q, k: 8 kg .. + 7 of the chunk) from its W_hh fragments
    // (pack_rec_kernel: slice u / 64, wave u / 8 % 8, tile u / 4 % 2, row 4 (u % 4) + q) and from its W_ih
    // rows in lane order (rec_lane_column).
    const int u = wave * 16 + n;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        w[kc][q] = f16x8{};
        if (kc >= KCI)
          w[kc][q] = reinterpret_cast<const f16x8*>(a.wpack)[
              ((((size_t)layer * 16 + (u >> 3)) * KCR + kc - KCI) * 2 + ((u >> 2) & 1)) * 64 + kg * 16 + (u & 3) * 4 + q];
        else if (UP)
          w[kc][q] = *reinterpret_cast<const f16x8*>(
              a.wih_up + ((size_t)(layer - 1) * 4 * HP + ((u >> 3) * 4 + (u & 3)) * 8 + 2 * q + ((u >> 2) & 1)) * HP +
              kc * 32 + kg * 8);
      }
  }
  // D rows of this lane: units u0 .. u0+3 of row n; it evaluates UPL of them, starting at uo.
  const int u0 = wave * 16 + kg * 4;
  const int ibase = (ROWS == 8 && n >= 8) ? 2 : 0;
  const int uo = u0 + ibase;
  f32x4 bias[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) bias[q] = *reinterpret_cast<const f32x4*>(a.bias + ((size_t)layer * 4 + q) * HP + u0);

  // Initial state (nn.LSTM hx) or zeros; h_{-1} goes to slot 1.
  typedef _Float16 hvec __attribute__((ext_vector_type(UPL)));
  typedef uint32_t wvec __attribute__((ext_vector_type(NW)));
  float c[UPL];
  hvec hcur;
#pragma unroll
  for (int j = 0; j < UPL; ++j) {
    const int u = uo + j;
    const bool v = row_ok && u < a.H;
    const size_t si = ((size_t)layer * a.B + grow) * a.H + u;
    c[j] = (v && a.c0) ? (float)a.c0[si] : 0.0f;
    hcur[j] = (v && a.h0) ? a.h0[si] : (_Float16)0.0f;
  }
  const int hoff = frag_index<ROWS>(r, uo);  // where this lane's UPL h values go (contiguous)
  auto frag_at = [&](f16x8* block) -> _Float16* { return reinterpret_cast<_Float16*>(block) + hoff; };
  *reinterpret_cast<hvec*>(frag_at(lds.hist[1])) = hcur;

  // ---- hand-off from the layer below and to the layer above ----
  // Thread i takes the words that thread i of the workgroup below wrote (the same units and row), loaded
  // four steps ahead and checked two ahead, so that a step waits neither for the load nor, once the
  // layers have settled about six steps apart, for the words.
  const int slots = a.T < kHandoffSlots ? a.T : kHandoffSlots;
  const size_t ring_bytes = (size_t)slots * C::kSlot;
  char* const rings = reinterpret_cast<char*>(a.hseq);
  const __amdgpu_buffer_rsrc_t in_rs = __builtin_amdgcn_make_buffer_rsrc(
      UP ? rings + ((size_t)(layer - 1) * a.ntile + tile) * ring_bytes : nullptr, 0, UP ? (int)ring_bytes : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t out_rs = __builtin_amdgcn_make_buffer_rsrc(
      DOWN ? rings + ((size_t)layer * a.ntile + tile) * ring_bytes : nullptr, 0, DOWN ? (int)ring_bytes : 0, 0x00020000);
  const uint32_t woff = threadIdx.x * (4u * NW);
  uint32_t woff_out = woff;
  auto clamp_step = [&](int s) { return s < Tt ? s : Tt - 1; };
  auto slot_of = [&](int s) { return (s & (kHandoffSlots - 1)) * C::kSlot; };
  wvec words[2] = {};  // the words in flight, of an even and an odd step
  auto load_word = [&](int slot, wvec& rw) __attribute__((always_inline)) {
    if constexpr (NW == 1)
      rw[0] = __builtin_amdgcn_raw_buffer_load_b32(in_rs, woff, slot, 16);
    else
      rw = __builtin_bit_cast(wvec, __builtin_amdgcn_raw_buffer_load_b64(in_rs, woff, slot, 16));
  };
  // Bounded waits.  `dead`: a wait of this wave failed; it then waits for nothing any more and sends
  // nothing (its offset falls outside the ring), so nothing downstream takes a word it wrote later.
  bool dead = false;
  uint64_t t0 = 0;
  auto wait_failed = [&](int spin) -> bool {
    if (spin == 0) {
      t0 = __builtin_amdgcn_s_memrealtime();
      return false;
    }
    if ((spin & 3) == 0 &&
        __builtin_amdgcn_readfirstlane(__hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) {
      dead = true;
    } else if (__builtin_amdgcn_s_memrealtime() - t0 > a.wait_ticks) {
      __hip_atomic_fetch_or(a.status, PLH_STATUS_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      dead = true;
    }
    if (dead) woff_out = 0x80000000u;
    return dead;
  };
  // The loaded word rw (of a step with this tag and slot) as h.
  auto check_word = [&](uint32_t tag, int slot, wvec rw) __attribute__((always_inline)) -> wvec {
    rw[NW - 1] ^= tag;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(handoff_special(rw[NW - 1])) != 0ull, 0)) {
      for (int spin = 0; __builtin_amdgcn_ballot_w64((rw[NW - 1] & kHandoffTag) != 0u) != 0ull; ++spin) {
        if (dead || wait_failed(spin)) break;
        asm volatile("" ::: "memory");  // the re-polls are not loop-invariant loads
        load_word(slot, rw);
        rw[NW - 1] ^= tag;
      }
      if (handoff_special(rw[NW - 1])) rw[NW - 1] |= 0x7E000000u;  // NaN again
    }
    return rw;
  };
  auto put_word = [&](wvec v, f16x8* dst) __attribute__((always_inline)) { *reinterpret_cast<wvec*>(frag_at(dst)) = v; };
  // h (in hcur) with a tag into a slot of the ring.  Stored with sc1 (written through; visible to other CUs
  // and XCDs without an L2 write-back), or, with 8-row tiles and a consumer on this XCD, without: the word
  // then stays in the XCD's L2, where the consumer's sc1 loads read it, and is acknowledged sooner (loads
  // and stores retire in order, so the wait for a word also waits for the stores issued before its load).
  // C2's kernel 787-792 -> 778 us, H 60 L3 B200 T365 142 -> 140 us; with ragged rows it was 1% and with 16-row
  // tiles 3.5% slower (a second copy of the block in kernels short of registers), which keep sc1.
  constexpr bool kLocal = DOWN && ROWS == 8 && !RAGGED;
  bool local = false;
  auto send = [&](uint32_t tag, int slot, auto loc) __attribute__((always_inline)) {
    constexpr int POLICY = decltype(loc)::value ? 0 : 16;
    wvec v = __builtin_bit_cast(wvec, hcur);
    v[NW - 1] = (v[NW - 1] & ~kHandoffTag) | tag;
    if constexpr (NW == 1)
      __builtin_amdgcn_raw_buffer_store_b32(v[0], out_rs, woff_out, slot, POLICY);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned int, v),
                                            out_rs, woff_out, slot, POLICY);
  };
  // Pacing, where the ring wraps (T > kHandoffSlots): a (layer, tile) counter holds how many input steps of
  // that workgroup have left the ring (the workgroup below may overwrite their slots) and, in the top
  // four bits, its XCD's id + 1.  Once per block a workgroup reports its own and loads its consumer's; a
  // step later it waits until the slots of the sends up to the next look are free.  Each counter has a
  // 128-byte line of its own (behind the rings), and a report stays in the XCD's L2 where the workgroup
  // below shares it: its acknowledgement, too, sits in front of the words loaded after it.  (With
  // adjacent counters and written-through reports H 60, L = 3, B = 200, T = 365 took 185 us, now 147.)
  constexpr int kXcdShift = 28;
  const bool paced = a.T > kHandoffSlots;
  const uint32_t xcd = (xcc_id() + 1u) << kXcdShift;
  uint32_t* const counters = reinterpret_cast<uint32_t*>(rings + (size_t)(a.L - 1) * a.ntile * ring_bytes);
  auto counter = [&](int l) { return counters + ((size_t)l * a.ntile + tile) * kCounterStride; };
  uint32_t* const my_ctr = counter(layer);
  const uint32_t* const down_ctr = counter(DOWN ? layer + 1 : layer);
  auto shares_xcd = [&](int l) -> bool {
    return (__builtin_amdgcn_readfirstlane(__hip_atomic_load(counter(l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >>
            kXcdShift << kXcdShift) == xcd;
  };
  bool up_local = false;
  uint32_t down_seen = 0;
  auto report = [&](int n) __attribute__((always_inline)) {
    if (threadIdx.x != 0) return;
    if (up_local)
      __hip_atomic_store(my_ctr, (uint32_t)n | xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
      __hip_atomic_store(my_ctr, (uint32_t)n | xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto progress_poll = [&](int t) __attribute__((always_inline)) {
    if (!paced) return;
    if (UP) report(t + 2);
    if (DOWN) down_seen = __hip_atomic_load(down_ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto progress_wait = [&](int t) __attribute__((always_inline)) {
    if (!DOWN || !paced) return;
    const int need = t + kBlock - kHandoffSlots;  // sends of steps t - 1 .. t + kBlock - 1
    uint32_t seen = __builtin_amdgcn_readfirstlane(down_seen);
    for (int spin = 0; __builtin_expect((int)(seen & ((1u << kXcdShift) - 1u)) < need, 0); ++spin) {
      if (dead || wait_failed(spin)) break;
      // The consumer still has about two blocks of words: ~1 us between looks keeps the counters' lines quiet.
      __builtin_amdgcn_s_sleep(32);
      seen = __builtin_amdgcn_readfirstlane(__hip_atomic_load(down_ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
  };
  if ((UP || DOWN) && paced) report(0);  // this workgroup's XCD, for both neighbours (read after its first input)

  // ---- layer 0: x, a block of steps at a time ----
  // Loaded into registers at step 2 of the block before, written to the block's LDS buffer at step 6.
  // A step's source holds the first `per` f16x8 of its fragment blocks (the g_in0 8-wide K groups of x);
  // the rest are written as zeros.
  constexpr int XS = KIN * FV;  // f16x8 per step in LDS
  constexpr int RN = GATES ? 1 : (kBlock * XS + NT - 1) / NT;
  const int per = a.g_in0 * ROWS;
  const f16x8* const xsrc = a.xp + (size_t)tile * a.T * per;
  f16x8 R[RN];
  auto load_block = [&](int k) {
#pragma unroll
    for (int i = 0; i < RN; ++i) {
      const int p = (int)threadIdx.x + i * NT;
      const int st = p / (XS ? XS : 1), e = p % (XS ? XS : 1);
      const size_t s = (size_t)clamp_step(k * kBlock + (st < kBlock ? st : kBlock - 1));
      R[i] = xsrc[s * per + (e < per ? e : per - 1)];
    }
  };
  auto store_block = [&](int k) {
    f16x8* rb = lds.xin + (k & 1) * kBlock * XS;
#pragma unroll
    for (int i = 0; i < RN; ++i) {
      const int p = (int)threadIdx.x + i * NT;
      if (p < kBlock * XS) rb[p] = p % (XS ? XS : 1) < per ? R[i] : f16x8{};
    }
  };

  // ---- layer 0 with a wide input: the projections, loaded two steps before they are added ----
  // Step t's row of this lane is row t rows_pad + tile ROWS + r of the blocked [.. x 4 HP] projections; the 16
  // bytes of column group (u / 8, u % 4) hold the four gates of units u and u + 4, alternating.
  const f16x8* const gsrc = reinterpret_cast<const f16x8*>(a.gates);
  f16x8 gates[2][UPL];
  auto load_gates = [&](int t, f16x8 (&g)[UPL]) __attribute__((always_inline)) {
    const size_t row = (size_t)clamp_step(t) * a.rows_pad + tile * ROWS + r;
    const f16x8* src = gsrc + ((row >> 4) * (4 * HP / 32) + (uo >> 3)) * 64 + (uo & 3) * 16 + (row & 15);
#pragma unroll
    for (int j = 0; j < UPL; ++j) g[j] = src[j * 16];
  };
  // acc = bias + the projections (8-row tiles: both candidates of a lane's pair, as it evaluates one)
  const bool upper = ((uo >> 2) & 1) != 0;
  auto add_gates = [&](const f16x8 (&g)[UPL], f32x4 (&acc)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f16x8 v = g[j % UPL];
        acc[q][j] = bias[q][j] + (float)(upper ? v[2 * q + 1] : v[2 * q]);
      }
  };
  // LDS slot of step t's input.
  auto xin_at = [&](int t) -> f16x8* { return UP ? lds.xin + (t & 1) * XS : lds.xin + (t & (2 * kBlock - 1)) * XS; };

  // ---- outputs ----
  // The last layer's output sequence: this lane's units of its row, a step after they were computed
  // (stores before the step's input load, which is waited for a step later), in pairs where every
  // row of [.. x H] is 4-byte aligned.
  const bool seq = !DOWN && a.out_seq;
  const bool seq_pairs = (a.H & 1) == 0;
  _Float16* seq_dst = seq ? a.out_seq + (size_t)grow * a.T * a.H + uo : nullptr;
  auto store_seq = [&](int t) {
    if (!seq || t < 0) return;
    _Float16* const dst = seq_dst;
    seq_dst += a.H;
    if (!row_ok) return;
    const bool live = !RAGGED || t < len;
    const hvec v = live ? hcur : hvec{};
    if (seq_pairs) {
      const wvec p = __builtin_bit_cast(wvec, v);
#pragma unroll
      for (int i = 0; i < NW; ++i)
        if (uo + 2 * i < a.H) reinterpret_cast<uint32_t*>(dst)[i] = p[i];
    } else {
#pragma unroll
      for (int j = 0; j < UPL; ++j)
        if (uo + j < a.H) dst[j] = v[j];
    }
  };

  int probe_i = 0;
  // Probe steps are wave-uniform and kept in SGPRs (readfirstlane right after the load): a VGPR
  // loaded in the loop would make the compiler wait for every outstanding global access (vmcnt(0),
  // in order on gfx950) at each step.
  int probe_next = a.n_probe > 0 ? __builtin_amdgcn_readfirstlane(a.probe_steps[0]) : -1;
  auto write_probe = [&](int p) {
    if (!row_ok) return;
#pragma unroll
    for (int j = 0; j < UPL; ++j) {
      const int u = uo + j;
      if (u < a.H) {
        const size_t o = (((size_t)p * a.L + layer) * a.B + grow) * a.H + u;
        a.probe_h[o] = (float)hcur[j];
        a.probe_c[o] = c[j];
      }
    }
  };

  // ---- prologue: the first inputs into LDS, the next word in flight, step 0's input part ----
  f32x4 acc_next[4];
  if (Tt > 0) {
    if constexpr (UP) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int sc = clamp_step(s);
        load_word(slot_of(sc), words[s]);
        wait_vmem_all();
        put_word(check_word(handoff_tag(sc), slot_of(sc), words[s]), xin_at(s));
      }
    } else if constexpr (!GATES) {
      load_block(0);
      wait_vmem_all();
      store_block(0);
    }
    // The neighbours' first reports are out by now (a missing one costs speed only).
    if (paced) {
      if constexpr (UP) up_local = shares_xcd(layer - 1);
      if constexpr (kLocal) local = shares_xcd(layer + 1);
    }
    // The words of steps 2 and 3, each with a send (of no tag) behind it as in the steps, so that the wait
    // for a loaded word leaves the accesses behind it in flight from the first step on.
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if constexpr (UP) load_word(slot_of(clamp_step(2 + s)), words[s]);
      if constexpr (DOWN) send(0u, (slots - 1) * C::kSlot, std::false_type());
    }
  }
  __syncthreads();
  if (GATES && Tt > 0) {
    load_gates(0, gates[0]);
    wait_vmem_all();
    add_gates(gates[0], acc_next);
    load_gates(1, gates[1]);
    load_gates(2, gates[0]);
  } else if (Tt > 0) {
    const f16x8* xr = xin_at(0) + fl;
    f16x8 xv[KIN ? KIN : 1];
#pragma unroll
    for (int kc = 0; kc < KIN; ++kc) xv[kc] = xr[kc * FV];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc_next[q] = bias[q];
#pragma unroll
    for (int kc = 0; kc < KIN; ++kc)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc_next[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[kc][q], xv[kc], acc_next[q], 0, 0, 0);
  }
  lds_barrier();  // step 0 overwrites slot 0 (with x_2) once every wave has read x_0

  // ---- steps ----
  // Step t = 8 k + s: the LDS reads of h_{t-1}; under their latency the word of x_{t+2} into LDS, the load
  // of x_{t+4}'s and the send of h_{t-1}; the recurrent MFMAs; the gate math with the input MFMAs of
  // step t + 1; h_t into LDS; one barrier.  In a FULL block every step up to t + 4 exists, no probe
  // is due and s is a constant, so slots and tags come from the block's, without clamps.
  const bool hi = ibase != 0;
  auto step = [&](const int k, const int s, auto par, auto full, auto loc) __attribute__((always_inline)) {
    constexpr int P = decltype(par)::value;  // s & 1
    constexpr bool FULL = decltype(full)::value;
    const int t = k * kBlock + s;
    // slot and tag of step t + d, d constant
    const int s2 = FULL ? t + 2 : clamp_step(t + 2), s4 = FULL ? t + 4 : clamp_step(t + 4);
    auto block_slot = [&](int d) { return slot_of((k + (s + d >= kBlock ? 1 : s + d < 0 ? -1 : 0)) * kBlock) +
                                          ((s + d) & (kBlock - 1)) * C::kSlot; };
    auto block_tag = [&](int d) { return handoff_tag((k + (s + d >= kBlock ? 1 : s + d < 0 ? -1 : 0)) * kBlock); };
    f32x4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = acc_next[q];
    const f16x8* hr = lds.hist[P ^ 1] + fl;
    f16x8 hv[KCR];
#pragma unroll
    for (int kr = 0; kr < KCR; ++kr) hv[kr] = hr[kr * FV];
    __builtin_amdgcn_sched_barrier(0);
    wvec x2 = {};
    if constexpr (UP) x2 = check_word(FULL ? block_tag(2) : handoff_tag(s2), FULL ? block_slot(2) : slot_of(s2), words[P]);
    if constexpr (!UP && !GATES) {
      if (s == 2) {
        // (also ends what is outstanding: without it the compiler keeps the block loads "possibly
        // outstanding", their consumers being lane-conditional)
        wait_vmem_all();
        load_block(k + 1);
      } else if (s == kBlock - 2) {
        wait_vmem_all();
        store_block(k + 1);
      }
    }
    if (s == 0) progress_poll(t);
    if (s == 1) progress_wait(t);
    store_seq(t - 1);
    if constexpr (UP) load_word(FULL ? block_slot(4) : slot_of(s4), words[P]);
    if constexpr (DOWN) {
      if (s > 0 || t > 0)
        send(FULL ? block_tag(-1) : handoff_tag(t - 1), FULL ? block_slot(-1) : slot_of(t - 1), loc);
      else
        send(0u, (slots - 1) * C::kSlot, loc);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kr = 0; kr < KCR; ++kr)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[KCI + kr][q], hv[kr], acc[q], 0, 0, 0);

    // Next step's input part (the last step computes a discarded one), interleaved with this
    // step's gate math so the matrix core runs while the VALU evaluates the gates (in-order issue
    // would otherwise queue all VALU work behind a burst of MFMAs).
    const f16x8* xr = (UP ? lds.xin + (P ^ 1) * XS
                          : lds.xin + ((s + 1 < kBlock ? (k & 1) * kBlock + s + 1 : ((k + 1) & 1) * kBlock)) * XS) + fl;
    f16x8 xv[KIN ? KIN : 1];
#pragma unroll
    for (int kc = 0; kc < KIN; ++kc) xv[kc] = xr[kc * FV];
    if constexpr (UP) put_word(x2, lds.xin + P * XS);  // (after the reads, which then move up among the MFMAs)
    if constexpr (GATES) {
      add_gates(gates[P ^ 1], acc_next);  // step t + 1's
      load_gates(t + 3, gates[P ^ 1]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) acc_next[q] = bias[q];
    }
    const bool live = t < len;
    auto input_mfma = [&](int m) __attribute__((always_inline)) {
      const int kc = m / 4, q = m % 4;
      acc_next[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[kc][q], xv[kc], acc_next[q], 0, 0, 0);
    };
    // this lane's pair j: D element ibase + j of every gate tile (one v_cndmask each)
    auto cell_pair = [&](int j) __attribute__((always_inline)) {
      float z[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) z[q] = pick(hi, acc[q][j], acc[q][2 + j % 2]);
      float cn = c[j], hn;
      lstm_cell(z[0], z[1], z[2], z[3], cn, hn);
      if constexpr (RAGGED) {
        // selects, not a branch: rows past their length keep their state
        c[j] = live ? cn : c[j];
        hcur[j] = live ? (_Float16)hn : hcur[j];
      } else {
        c[j] = cn;
        hcur[j] = (_Float16)hn;
      }
    };
    if constexpr (ROWS == 8 && RAGGED) {
      // With ragged rows (the selects on `live` add VALU work) the gate math goes first and the
      // next step's input MFMAs follow it: 1.7-2.3% faster than the interleave below, which is
      // the faster one without them.
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < UPL; ++j) cell_pair(j);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < KIN * 4; ++m) input_mfma(m);
      __builtin_amdgcn_sched_barrier(0);
    } else if constexpr (ROWS == 8) {
      // Two pairs per lane (~80 VALU instructions per wave): one MFMA, then three VALU
      // instructions, and so on, so both waves of a SIMD keep the matrix core fed and neither
      // queues its gate math behind a burst of MFMAs.
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < KIN * 4; ++m) input_mfma(m);
#pragma unroll
      for (int j = 0; j < UPL; ++j) cell_pair(j);
#pragma unroll
      for (int m = 0; m < KIN * 4; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // three VALU
      }
      __builtin_amdgcn_sched_barrier(0);
    } else {
      // Four pairs per lane: each pair is preceded by its share of the MFMAs and fenced.
      constexpr int kMfmaPerPiece = (KIN * 4 + UPL - 1) / UPL;
#pragma unroll
      for (int j = 0; j < UPL; ++j) {
#pragma unroll
        for (int m = j * kMfmaPerPiece; m < (j + 1) * kMfmaPerPiece && m < KIN * 4; ++m) input_mfma(m);
        cell_pair(j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // One conversion feeds every use of h (the compiler would otherwise round it once per use, fused
    // with the product for some).
    wvec hw = __builtin_bit_cast(wvec, hcur);
#pragma unroll
    for (int i = 0; i < NW; ++i) asm volatile("" : "+v"(hw[i]));
    hcur = __builtin_bit_cast(hvec, hw);
    *reinterpret_cast<hvec*>(frag_at(lds.hist[P])) = hcur;
    if (!FULL && t + 1 == probe_next) {
      write_probe(probe_i);
      ++probe_i;
      probe_next = probe_i < a.n_probe ? __builtin_amdgcn_readfirstlane(a.probe_steps[probe_i]) : -1;
    }
    lds_barrier();
  };
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  auto full_block = [&](int k, auto loc) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < kBlock; s += 2) {
      step(k, s, Even(), std::true_type(), loc);
      step(k, s + 1, Odd(), std::true_type(), loc);
    }
  };
  for (int k = 0; k * kBlock < Tt; ++k) {
    const int left = Tt - k * kBlock;
    if (left >= kBlock + 4 && (probe_next < 0 || probe_next > (k + 1) * kBlock)) {
      if constexpr (kLocal) {
        if (local)
          full_block(k, std::true_type());
        else
          full_block(k, std::false_type());
      } else {
        full_block(k, std::false_type());
      }
    } else {
#pragma unroll 1
      for (int s = 0; s < kBlock && s < left; s += 2) {
        step(k, s, Even(), std::false_type(), std::false_type());
        if (s + 1 < left) step(k, s + 1, Odd(), std::false_type(), std::false_type());
      }
    }
  }
  if (Tt > 0) {
    store_seq(Tt - 1);
    if constexpr (DOWN) send(handoff_tag(Tt - 1), slot_of(Tt - 1), std::false_type());
  }
  if (dead) lds.fail = 1;
  __syncthreads();
  const bool ok = __builtin_amdgcn_readfirstlane(lds.fail) == 0;

  if (!ok) {
    // A hand-off wait failed (the status word records it and fails every other wait): poison every
    // output of this workgroup (states, probes, output sequence, head) and leave.
    if (row_ok) poison_lane_outputs(a, layer, grow, uo, UPL, !DOWN);
    if (!DOWN && a.out) {
      for (int idx = threadIdx.x; idx < (uniform ? a.B : ROWS) * a.O; idx += NT) {
        const int g = a.row0 + tile * ROWS + idx / a.O;
        if (g < a.row_end) a.out[(size_t)g * a.O + idx % a.O] = (_Float16)__builtin_nanf("");
      }
    }
    return;
  }
  // Steps past the tile's longest row were never visited: their output sequence is zero.
  if (!DOWN && a.out_seq && row_ok) {
    for (int t = Tt; t < a.T; ++t) {
      _Float16* dst = a.out_seq + ((size_t)grow * a.T + t) * a.H + uo;
#pragma unroll
      for (int j = 0; j < UPL; ++j)
        if (uo + j < a.H) dst[j] = (_Float16)0.0f;
    }
  }

  // States after the tile's last step (rows that ended earlier were frozen at their last step).
  while (probe_i < a.n_probe) {
    write_probe(probe_i);
    ++probe_i;
  }
  if (row_ok) {
#pragma unroll
    for (int j = 0; j < UPL; ++j) {
      const int u = uo + j;
      if (u < a.H) {
        const size_t si = ((size_t)layer * a.B + grow) * a.H + u;
        if (a.h_n) a.h_n[si] = hcur[j];
        if (a.c_n) a.c_n[si] = (_Float16)c[j];
      }
    }
  }

  // Linear head on the final h of the last layer (slot of the tile's last step).
  if (!DOWN && a.out) {
    const _Float16* hf = reinterpret_cast<const _Float16*>(lds.hist[(Tt + 1) & 1]);
    _Float16* const row0_out = reinterpret_cast<_Float16*>(lds.xin);  // (no step reads the inputs any more)
    static_assert(sizeof(lds.xin) >= 4096 * sizeof(_Float16), "one row of the widest head");
    for (int idx = threadIdx.x; idx < ROWS * a.O; idx += NT) {
      const int rr = idx / a.O, o = idx % a.O;
      const int g = a.row0 + tile * ROWS + rr;
      if (g >= a.row_end) continue;
      const float* wr = a.wlin + (size_t)o * HP;
      float s0 = 0.f, s1 = 0.f;
      for (int k8 = 0; k8 < HP; k8 += 8) {
        const f16x8 hv = *reinterpret_cast<const f16x8*>(hf + frag_index<ROWS>(rr, k8));
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          s0 = fmaf((float)hv[j], wr[k8 + j], s0);
          s1 = fmaf((float)hv[j + 1], wr[k8 + j + 1], s1);
        }
      }
      const _Float16 y = (_Float16)(a.blin[o] + (s0 + s1));
      a.out[(size_t)g * a.O + o] = y;
      if (rr == 0) row0_out[o] = y;
    }
    if (uniform) {
      __syncthreads();
      for (int idx = ROWS * a.O + threadIdx.x; idx < a.B * a.O; idx += NT) a.out[idx] = row0_out[idx % a.O];
    }
  }
}


// One workgroup per (layer, tile).  The body (its input's source, a layer above or not) is chosen once
// here, so no step branches on it.
// At least two waves per SIMD in the bounds keep a wave within 256 registers, where MFMAs take and leave
// their accumulators in VGPRs; with one (what 128- and 256-thread workgroups default to) they went to
// AGPRs, and every step copied its 16 gate sums back.
template <int HP, int ROWS, bool RAGGED, bool WIDE>
__global__ void __launch_bounds__(HP / 16 * 64, 2)
lstm_wavefront_kernel(ForwardArgs a) {
  __shared__ WavefrontLds<HP, ROWS> lds;
  int layer, tile;
  block_coords(blockIdx.x, a.ntile, a.ntile_grid, a.xcd_map, layer, tile);
  if (tile >= a.ntile) return;  // a tile that only rounds the grid up to a multiple of 8
  auto body = [&](auto src) __attribute__((always_inline)) {
    constexpr Src SRC = decltype(src)::value;
    if (layer + 1 < a.L)
      wavefront_body<HP, ROWS, RAGGED, WIDE, SRC, true>(a, lds, layer, tile);
    else
      wavefront_body<HP, ROWS, RAGGED, WIDE, SRC, false>(a, lds, layer, tile);
  };
  if (layer > 0) {
    body(std::integral_constant<Src, Src::kUp>());
  } else if constexpr (WIDE) {
    body(std::integral_constant<Src, Src::kGates>());
  } else if (a.g_in0 <= 4) {
    body(std::integral_constant<Src, Src::kX1>());
  } else {
    body(std::integral_constant<Src, Src::kXn>());
  }
}

}  // namespace

template <int ROWS, bool RAGGED>
static const void* wavefront_kernel_rows(int HP, bool wide) {
  if (wide) return HP == 128 ? reinterpret_cast<const void*>(&lstm_wavefront_kernel<128, ROWS, RAGGED, true>) : nullptr;
  switch (HP) {
    case 32: return reinterpret_cast<const void*>(&lstm_wavefront_kernel<32, ROWS, RAGGED, false>);
    case 64: return reinterpret_cast<const void*>(&lstm_wavefront_kernel<64, ROWS, RAGGED, false>);
    case 128: return reinterpret_cast<const void*>(&lstm_wavefront_kernel<128, ROWS, RAGGED, false>);
    default: return nullptr;
  }
}

const void* wavefront_kernel(int HP, int tile_rows, bool ragged, bool wide) {
  if (tile_rows == 8)
    return ragged ? wavefront_kernel_rows<8, true>(HP, wide) : wavefront_kernel_rows<8, false>(HP, wide);
  if (tile_rows == 16)
    return ragged ? wavefront_kernel_rows<16, true>(HP, wide) : wavefront_kernel_rows<16, false>(HP, wide);
  return nullptr;
}

}  // namespace plh
