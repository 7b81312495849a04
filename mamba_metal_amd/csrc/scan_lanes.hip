// Selective scan with time across the lanes of a wave: mm_selective_scan_fwd[_strided] for scans
// of few channels (see plan), where scan.hip's chains -- one lane per channel, walking time --
// are too few to fill the chip.  Semantics as in scan.hip.
//
// A wave takes one channel and walks its sequence in chunks of 512 steps, 8 consecutive steps
// per lane.  Per state: the lane's decays a = exp2(delta2 A) and inputs b = delta' u B are
// computed once and kept in registers; the lane's end state from zero (one fma per step); an
// inclusive scan of the lanes' (decay, end state) pairs through DPP (a lane's decay is
// exp2 of A times its sum of delta2, so it is not multiplied up); then the recurrence once more
// from the lane's true start state, and y += C h.  Per (channel, state, step) that is seven VALU slots
// (the sequential walk has six), and per state and chunk ~30 for the lane scan and three more
// exponentials, which is five more per update over a lane's eight steps; y needs no sum over waves.  B and C are staged in LDS as fp32, eight states at a time
// (the next group's loads in flight during this one's arithmetic), shared by the workgroup's
// channels.  SW > 1 shares a channel's states among SW waves, for launches that would leave
// SIMDs idle; with few channels and a long sequence time is split as well: a first launch
// (SUM) leaves every segment's end state from zero and its sum of delta2, and the second folds
// its predecessors' with one more lane scan.
//
// What bounds it: VALU issue (at B=4 D=1536 L=4096 along time, counted: fp16 12.1 instructions and 14.0
// issue slots per update, 91% of the VALU's cycles busy, fp32 27.3, 27.9 and 95%; by rows fp16 12.6, 14.5
// and 86%), against 9.6-12 slots for scan.hip where that one's
// chains fill the chip, and its 14-40 where they do not.  The registers allow four waves per SIMD,
// in fp32 at the price of 8 to 20 of them in scratch (along time on one and two waves per
// channel, by rows on one).  With a workgroup per CU or less, a chunk's dependent steps and the
// fetches of code that runs once.  Tried and not kept: 16 steps per
// lane (11 slots, but two waves per SIMD instead of four: B=4 D=1536 L=4096 149 -> 180 us), two
// states interleaved per wave where the chip is full (149 -> 186), the next state's LDS reads ahead
// (149 -> 151), by rows both state groups of B and C loaded together (1x2048x1536 40.8 -> 42.8).
#include <algorithm>
#include <type_traits>

#include "scan_common.h"

namespace mm {
namespace lscan {

constexpr int kTL = 8;                 // steps per lane and chunk
constexpr int kChunk = 64 * kTL;       // steps per chunk
constexpr int kNG = 8;                 // states of B and C staged at a time
constexpr int kItems = kNG * kChunk / 8;  // 8-element items of a staged tensor
constexpr int kXcds = 8, kCus = 256;
constexpr int kMaxSeg = 64;  // a wave folds its segment's predecessors, one per lane

// kTime: u, delta, z, y and B, C contiguous along time.  kRows: u, delta, z, y contiguous along
// channels (a multiple of 8), B, C along states (a multiple of 8).
enum Layout { kTime = 0, kRows = 1 };

struct Params {
  const void* u;
  const void* delta;
  const void* z;
  void* y;
  const float* A;
  const float* D;
  const void* B;
  const void* C;
  float* state_out;
  float* sum;    // [batch][dim][dstate + 1][nseg] segment summaries: end states, then sum of delta2
  int* ctl;
  int64_t us0, us1, us2, ds0, ds1, ds2, zs0, zs1, zs2, ys0, ys1, ys2;
  int64_t Bs0, Bs1, Bs2, Cs0, Cs1, Cs2, As0, As1, Ds;
  int32_t dim, dstate, seqlen, nseg, seg_chunks;
  float softplus_cut;
};

// N elements at any element-aligned address (the hardware takes unaligned global accesses), so
// odd lengths and strides need no path of their own.
template <int DT, int N>
struct Run {
  typedef typename Ty<DT>::T V __attribute__((ext_vector_type(N)));
  typedef typename Ty<DT>::T U __attribute__((ext_vector_type(N), aligned(sizeof(typename Ty<DT>::T))));
};

// Value of x in another lane through DPP; lanes without a source get `old`.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dpp_or(float old, float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), CTRL, ROWS, 0xF, false));
}
// ... get 0.
template <int CTRL>
__device__ __forceinline__ float dpp_or0(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
constexpr int kRowShr = 0x110;   // + n: lane i of a 16-lane row takes lane i - n
constexpr int kWaveShr1 = 0x138; // lane i takes lane i - 1
constexpr int kBcast15 = 0x142;  // rows 1 and 3 take the last lane of the row before
constexpr int kBcast31 = 0x143;  // rows 2 and 3 take lane 31

__device__ __forceinline__ bool is_inf(float v) { return __builtin_amdgcn_classf(v, 0x204); }

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// LDS rows of one state's B or C: the four steps 4q .. 4q + 3 of every lane lie together, so a
// lane reads its steps as float4s next to its neighbours'.  Each q's block is rotated, so
// that 64 consecutive steps lie on distinct banks when they are written one by one.
__device__ __forceinline__ int lds_lane(int lane, int q) { return q * 256 + ((lane * 4 + q * 32) & 255); }
__device__ __forceinline__ int lds_pos(int t) { return lds_lane(t / kTL, (t % kTL) >> 2) + (t & 3); }

// Inclusive prefix sums over the lanes: within each 16-lane row, within each half, whole.
__device__ __forceinline__ void prefix(float s, float& row, float& half, float& all) {
  s += dpp_or0<kRowShr + 1>(s);
  s += dpp_or0<kRowShr + 2>(s);
  s += dpp_or0<kRowShr + 4>(s);
  s += dpp_or0<kRowShr + 8>(s);
  row = s;
  half = s + dpp_or<kBcast15, 0xA>(0.0f, s);
  all = half + dpp_or<kBcast31, 0xC>(0.0f, half);
}

// Inclusive scan over the lanes of the recurrence's (decay, state) pairs: on entry P and h are
// a lane's decay over its own steps and its end state from a zero start; on return h is the
// end state from the start of the wave.  pr and ph: the lane's decay since the start of its
// 16-lane row and of its half-wave.  Lanes without a source in a row step read decay and state
// 0 (they are complete by then).  Each s_nop covers the two wait states between a VALU write
// of a register and its read through DPP.
__device__ __forceinline__ void lane_scan(float& P, float& h, float pr, float ph) {
  asm volatile(
      "s_nop 1\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "s_nop 0\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "s_nop 0\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "s_nop 0\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "s_nop 1\n\t"
      "v_fmac_f32_dpp %1, %1, %2 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_fmac_f32_dpp %1, %1, %3 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 1"
      : "+&v"(P), "+&v"(h)
      : "v"(pr), "v"(ph));
}

// lane_scan of two states: the second's instructions stand where the first's results would be waited
// for, so fewer s_nops are left.
__device__ __forceinline__ void lane_scan2(float& P0, float& h0, float pr0, float ph0, float& P1, float& h1,
                                           float pr1, float ph1) {
  asm volatile(
      "s_nop 1\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %3, %3, %2 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %2, %2, %2 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %3, %3, %2 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %2, %2, %2 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %3, %3, %2 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_mul_f32_dpp %2, %2, %2 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %1, %1, %0 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "v_fmac_f32_dpp %3, %3, %2 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
      "s_nop 0\n\t"
      "v_fmac_f32_dpp %1, %1, %4 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %3, %6 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 0\n\t"
      "v_fmac_f32_dpp %1, %1, %5 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %3, %7 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 1"
      : "+&v"(P0), "+&v"(h0), "+&v"(P1), "+&v"(h1)
      : "v"(pr0), "v"(ph0), "v"(pr1), "v"(ph1));
}

// B and C of NG states of a chunk on their way to LDS rows of fp32, zero past the sequence's
// end and past the last state: one vector of 8 steps of a state (kTime) or of 8 states of a
// step (kRows) per thread and tensor.
template <int DT, int LAYOUT, int NT>
struct Stage {
  using T = typename Ty<DT>::T;
  using V = typename Run<DT, 8>::V;
  using U = typename Run<DT, 8>::U;
  static constexpr int kPer = kChunk / 8;         // kTime: 8-step items of a state
  static_assert(NT == kItems, "one item of B and of C per thread");
  V v[2];           // of B and C
  const T* ptr[2];  // this thread's item of state group 0 and step 0

  // (As a call: with tid written out the compiler schedules the fp32 kernels otherwise, 1x1536x2048
  // 44 -> 47 us.)
  __device__ __forceinline__ int item(int tid) const { return tid; }

  __device__ __forceinline__ void init(const Params& p, int64_t bat, int tid) {
    const T* const pb = static_cast<const T*>(p.B) + bat * p.Bs0;
    const T* const pc = static_cast<const T*>(p.C) + bat * p.Cs0;
    const int i = item(tid);
    ptr[0] = pb + (LAYOUT == kTime ? (i / kPer) * p.Bs1 + 8 * (i % kPer) : i * p.Bs2);
    ptr[1] = pc + (LAYOUT == kTime ? (i / kPer) * p.Cs1 + 8 * (i % kPer) : i * p.Cs2);
  }

  __device__ __forceinline__ void load(const Params& p, bool with_c, int g0, int t0, int tid) {
    const bool full = t0 + kChunk <= p.seqlen && g0 + kNG <= p.dstate;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      if (x == 1 && !with_c) break;
      const int64_t s1 = x ? p.Cs1 : p.Bs1, s2 = x ? p.Cs2 : p.Bs2;
      int64_t o;
      if constexpr (LAYOUT == kTime) {
        o = g0 * s1 + t0;
        if (!full) {
          // states past the last read the last one, the sequence's last vector lies 8 steps
          // before its end
          const int n = item(tid) / kPer, t = 8 * (item(tid) % kPer);
          o += static_cast<int64_t>(std::min(n, p.dstate - 1 - g0) - n) * s1 + (std::min(t, p.seqlen - 8 - t0) - t);
        }
      } else {
        int dt = t0;
        if (!full) dt = t0 + item(tid) < p.seqlen ? dt : -item(tid);  // steps past the end read step 0
        o = dt * s2 + g0;
      }
      v[x] = *reinterpret_cast<const U*>(ptr[x] + o);
    }
  }

  __device__ __forceinline__ void store(const Params& p, bool with_c, int g0, int t0, int tid,
                                        float (*sb)[kChunk], float (*sc)[kChunk]) const {
    const bool full = t0 + kChunk <= p.seqlen && g0 + kNG <= p.dstate;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      float(*const dst)[kChunk] = x ? sc : sb;
      if (!with_c && dst == sc) break;
      if constexpr (LAYOUT == kTime) {
        const int n = item(tid) / kPer, t = 8 * (item(tid) % kPer);
        if (full) {
#pragma unroll
          for (int q = 0; q < 8; q += 4)
            *reinterpret_cast<float4*>(&dst[n][lds_pos(t + q)]) = make_float4(
                Ty<DT>::f(v[x][q]), Ty<DT>::f(v[x][q + 1]), Ty<DT>::f(v[x][q + 2]), Ty<DT>::f(v[x][q + 3]));
        } else {
          // Vectors past the end and past the last state as zeros.  The one that holds the end was read
          // 8 steps before it: its elements are moved down to their own steps through LDS, by eight
          // lanes of its wave (which has this state alone, and whose LDS accesses stay in order), not
          // in registers: code that runs once a call costs its fetches, 1x8x64 fp16 11 -> 7 us.
          const bool in = g0 + n < p.dstate && t0 + t < p.seqlen;
#pragma unroll
          for (int q = 0; q < 8; q += 4)
            *reinterpret_cast<float4*>(&dst[n][lds_pos(t + q)]) =
                make_float4(in ? Ty<DT>::f(v[x][q]) : 0.0f, in ? Ty<DT>::f(v[x][q + 1]) : 0.0f,
                            in ? Ty<DT>::f(v[x][q + 2]) : 0.0f, in ? Ty<DT>::f(v[x][q + 3]) : 0.0f);
          const int over = p.seqlen & 7, end = p.seqlen - over - t0;  // its steps inside, its first one
          if (end < kChunk && over > 0) {
            int l = item(tid) % kPer;
            asm volatile("" : "+v"(l));  // not worth registers in every chunk
            if (l < 8) {
              asm volatile("" ::: "memory");  // the read is of another lane's store
              const float f = dst[n][lds_pos(end + ((l - over) & 7))];
              asm volatile("" ::: "memory");
              dst[n][lds_pos(end + l)] = l < over ? f : 0.0f;
            }
          }
        }
      } else {
        const int t = item(tid), pos = lds_pos(t);
        const bool in = full || t0 + t < p.seqlen;
#pragma unroll
        for (int k = 0; k < 8; ++k) dst[k][pos] = in ? Ty<DT>::f(v[x][k]) : 0.0f;
      }
    }
  }
};

// CH channels per workgroup, each on SW waves that share its states.  kDirect: a lane loads and
// stores its own steps; otherwise every thread owns 8 / SW elements of the chunk (steps of a
// channel, or channels of a step) and they pass through an LDS tile.  PAIR: two states side by side, for
// launches of at most one workgroup per CU (two waves per SIMD), where a state's dependent steps are
// waited for; with more waves the second state's registers cost more than that (4x2048x1536 fp16 by
// rows 88 -> 108 us).
template <int DT, int LAYOUT, bool SUM, int CH, int SW, bool PAIR>
__global__ __launch_bounds__(64 * CH * SW, PAIR ? 2 : 4) void lane_scan_kernel(const Params p) {
  using T = typename Ty<DT>::T;
  static_assert(!(SUM && PAIR), "pairs for the pass that writes y");
  constexpr int NT = 64 * CH * SW;
  constexpr bool kDirect = LAYOUT == kTime && SW == 1;
  static_assert(LAYOUT == kTime || NT % kChunk == 0, "threads in whole chunks");
  constexpr int E = 8 / SW;          // elements of a thread per chunk and tensor
  constexpr int kStates = kNG / SW;  // states of a wave in a staged group
  using V = typename Run<DT, E>::V;
  using U = typename Run<DT, E>::U;

  __shared__ __attribute__((aligned(16))) float s_b[kNG][kChunk];
  __shared__ __attribute__((aligned(16))) float s_c[SUM ? 1 : kNG][kChunk];
  // the tile: delta2 and delta' * u, then the partial y's of the waves of a channel
  constexpr int kAreas = kDirect ? 0 : SUM || SW <= 2 ? 2 : SW;
  __shared__ __attribute__((aligned(16))) float s_x[kAreas > 0 ? kAreas : 1][kDirect ? 1 : CH][kDirect ? 4 : kChunk];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wch = wave % CH, part = wave / CH;
  // Workgroups go to the XCDs (each with an L2 of its own) in turn.  Neighbouring channel groups
  // share the 128-byte lines of channel-contiguous tensors, so each XCD takes a run of them.
  int unit;
  {
    const int n = gridDim.x, x = blockIdx.x % kXcds, k = blockIdx.x / kXcds;
    unit = x * (n / kXcds) + std::min(x, n % kXcds) + k;
  }
  const int ncg = (p.dim + CH - 1) / CH;
  const int ch0 = unit % ncg * CH;
  const int seg = unit / ncg % p.nseg;
  const int64_t b = unit / ncg / p.nseg;
  const int ch = ch0 + wch;
  const bool chok = ch < p.dim;
  const int c = chok ? ch : p.dim - 1;  // waves past dim repeat the last channel, unstored
  const bool has_z = p.z != nullptr;
  if (!SUM && unit == 0 && tid == 0) p.ctl[1] = 0;  // the call's status

  // lane n holds the channel's A[n] and the carried state n
  float Al = lane < p.dstate ? p.A[c * p.As0 + lane * p.As1] : 0.0f;
  // A = -inf keeps no state from step to step; over steps past the sequence's end and between
  // neighbouring segments (delta2 0) it would be NaN
  Al = Al == -__builtin_inff() ? -__FLT_MAX__ : Al;
  const bool mine = SW == 1 || lane % kNG / kStates == part;  // whether this wave has state n = lane
  const bool Apos = __any(Al > 0.0f);
  const bool may_grow = Apos || p.softplus_cut != p.softplus_cut;
  float carry = 0.0f;
  float dsum = 0.0f;  // SUM: delta2 over the segment

  if (!SUM && seg > 0) {
    // carry into the segment: predecessors' end states decayed over what lies between.  Lane i
    // takes segment seg - 1 - i; its distance is the sum of delta2 of the segments after.
    const float* const sm = p.sum + (b * p.dim + c) * (p.dstate + 1) * static_cast<int64_t>(p.nseg);
    const int j = lane < seg ? seg - 1 - lane : 0;
    const float ds = lane < seg ? sm[static_cast<int64_t>(p.dstate) * p.nseg + j] : 0.0f;
    float r, hf, all;
    prefix(ds, r, hf, all);
    const float w = dpp_or<kWaveShr1>(0.0f, all);
    const bool grows = Apos || __any(ds < 0.0f);  // see `serial` below
    for (int g0 = 0; g0 < p.dstate; g0 += kNG) {
      float v[kStates];
#pragma unroll
      for (int k = 0; k < kStates; ++k) {
        const int n = g0 + part * kStates + k;
        v[k] = (lane < seg && n < p.dstate) ? sm[static_cast<int64_t>(n) * p.nseg + j] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < kStates; ++k) {
        const int n = g0 + part * kStates + k;
        const float An = lane_value(Al, n & 63);
        float hin;
        if (grows || __any(is_inf(v[k]))) {
          hin = 0.0f;
          for (int i = seg - 1; i >= 0; --i) {
            // a segment's factor may overflow where its product with a small state does not: in
            // sixteen steps (and not at all on a zero or infinite state)
            const float f = exp2_decay<DT>(An * lane_value(ds, i) * 0.0625f);
            float g = hin;
            for (int r = 0; r < 16; ++r) g *= f;
            hin = (hin == 0.0f || is_inf(hin) ? hin : g) + lane_value(v[k], i);
          }
        } else {
          float vr, vh, va;
          prefix(v[k] * exp2_decay<DT>(w * An), vr, vh, va);
          hin = lane_value(va, 63);
        }
        carry = lane == n ? hin : carry;
      }
    }
  }

  const int nch = (p.seqlen + kChunk - 1) / kChunk;
  const int c_begin = seg * p.seg_chunks;
  const int c_end = c_begin + p.seg_chunks < nch ? c_begin + p.seg_chunks : nch;

  const T* const up = static_cast<const T*>(p.u) + b * p.us0;
  const T* const dp = static_cast<const T*>(p.delta) + b * p.ds0;
  const T* const zp = has_z ? static_cast<const T*>(p.z) + b * p.zs0 : up;
  const int64_t zs1 = has_z ? p.zs1 : p.us1, zs2 = has_z ? p.zs2 : p.us2;
  T* const yp = static_cast<T*>(p.y) + b * p.ys0;
  // this thread's elements: from step et of the chunk (and, by rows, from channel ch0 + ec)
  const int et = LAYOUT == kTime ? (kDirect ? lane * kTL : part * 64 * E + lane * E) : tid & (kChunk - 1);
  const int ec = LAYOUT == kTime ? wch : tid / kChunk * E;
  float Dv[LAYOUT == kTime ? 1 : E];
#pragma unroll
  for (int k = 0; k < (LAYOUT == kTime ? 1 : E); ++k)
    Dv[k] = (!SUM && p.D) ? p.D[(ch0 + ec + k < p.dim ? ch0 + ec + k : p.dim - 1) * p.Ds] : 0.0f;

  auto load = [&](const T* base, int64_t s1, int64_t s2, int t0, V& v) __attribute__((always_inline)) {
    if constexpr (LAYOUT == kTime) {
      const T* const r = base + c * s1 + t0 + et;
      if (t0 + kChunk <= p.seqlen) {
        v = *reinterpret_cast<const U*>(r);
      } else {
        // The lane that holds the sequence's end reads its last E steps and moves them down to its
        // own; lanes past it read step 0 (masked, see `inside`).
        int left = p.seqlen - t0 - et;
        asm volatile("" : "+v"(left));  // not worth registers in every chunk
        const int off = left >= E ? et + t0 : left > 0 ? p.seqlen - E : 0;
        v = *reinterpret_cast<const U*>(base + c * s1 + off);
        if (left > 0 && left < E) {
#pragma unroll
          for (int m = 1; m < E; m *= 2) {
            const bool by = (E - left) & m;
#pragma unroll
            for (int k = 0; k + m < E; ++k) v[k] = by ? v[k + m] : v[k];
          }
        }
      }
    } else {
      v = *reinterpret_cast<const U*>(base + (t0 + et < p.seqlen ? t0 + et : 0) * s2 + ch0 + ec);
    }
  };
  // whether element k of this thread lies inside the sequence (tt: its first step)
  auto inside = [&](int tt, int k) { return (LAYOUT == kTime ? tt + k : tt) < p.seqlen; };

  V ru, rd, rz, ku;  // the chunk's u, delta, z, and u kept for the skip term
  Stage<DT, LAYOUT, NT> st;
  load(up, p.us1, p.us2, c_begin * kChunk, ru);
  load(dp, p.ds1, p.ds2, c_begin * kChunk, rd);
  st.init(p, b, tid);
  st.load(p, !SUM, 0, c_begin * kChunk, tid);

  for (int chunk = c_begin; chunk < c_end; ++chunk) {
    const int t0 = chunk * kChunk;
    float d2[kTL], du[kTL], y[kTL];
    float S, Srow, Shalf;
    bool serial = false;

    for (int g0 = 0; g0 < p.dstate; g0 += kNG) {
      const bool last = g0 + kNG >= p.dstate;
      __syncthreads();  // the staged states and the tile are read
      st.store(p, !SUM, g0, t0, tid, s_b, s_c);
      if (g0 == 0) {
        // this thread's elements: delta2 and delta' * u
        float ed[E], eu[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
          ed[k] = scan::delta_log2<DT>(Ty<DT>::f(rd[k]), p.softplus_cut);
          eu[k] = ed[k] * kLn2 * Ty<DT>::f(ru[k]);
        }
        if (t0 + kChunk > p.seqlen) {
          int tt = t0 + et;
          asm volatile("" : "+v"(tt));  // keeps this a branch
#pragma unroll
          for (int k = 0; k < E; ++k) {
            ed[k] = inside(tt, k) ? ed[k] : 0.0f;  // identity step past the end
            eu[k] = inside(tt, k) ? eu[k] : 0.0f;
          }
        }
        ku = ru;
        if constexpr (kDirect) {
#pragma unroll
          for (int j = 0; j < kTL; ++j) d2[j] = ed[j], du[j] = eu[j];
        } else if constexpr (LAYOUT == kTime) {
          typedef float FV __attribute__((ext_vector_type(E)));
          FV dv, uv;
#pragma unroll
          for (int k = 0; k < E; ++k) dv[k] = ed[k], uv[k] = eu[k];
          *reinterpret_cast<FV*>(&s_x[0][ec][lds_pos(et)]) = dv;
          *reinterpret_cast<FV*>(&s_x[1][ec][lds_pos(et)]) = uv;
        } else {
          const int pos = lds_pos(et);
#pragma unroll
          for (int k = 0; k < E; ++k) {
            s_x[0][ec + k][pos] = ed[k];
            s_x[1][ec + k][pos] = eu[k];
          }
        }
      }
      if (!last) st.load(p, !SUM, g0 + kNG, t0, tid);
      else if (chunk + 1 < c_end) st.load(p, !SUM, 0, t0 + kChunk, tid);
      __syncthreads();

      if (g0 == 0) {
        if constexpr (!kDirect) {
#pragma unroll
          for (int q = 0; q < kTL / 4; ++q) {
            const float4 dv = *reinterpret_cast<const float4*>(&s_x[0][wch][lds_lane(lane, q)]);
            const float4 uv = *reinterpret_cast<const float4*>(&s_x[1][wch][lds_lane(lane, q)]);
            d2[4 * q] = dv.x, d2[4 * q + 1] = dv.y, d2[4 * q + 2] = dv.z, d2[4 * q + 3] = dv.w;
            du[4 * q] = uv.x, du[4 * q + 1] = uv.y, du[4 * q + 2] = uv.z, du[4 * q + 3] = uv.w;
          }
        }
        S = d2[0];
#pragma unroll
        for (int j = 1; j < kTL; ++j) S += d2[j];
        float Sall;
        prefix(S, Srow, Shalf, Sall);
        if constexpr (SUM) dsum += lane_value(Sall, 63);
#pragma unroll
        for (int j = 0; j < kTL; ++j) y[j] = 0.0f;
        // Growing states (A > 0, or delta < 0 without the softplus): products of decays may
        // overflow where the recurrence itself does not, so then the lanes go one by one -- unless
        // the steps that grow a state multiply it by less than 2^60 in all, which bounds every
        // product (without this 1x1536x2048 fp16 by rows 41 -> 202 us for a rate of 0.01 or a few small
        // negative steps).
        serial = false;
        if (may_grow) {
          float pos = 0.0f, r, hf, all;
#pragma unroll
          for (int j = 0; j < kTL; ++j) pos += fmaxf(d2[j], 0.0f);
          prefix(pos, r, hf, all);  // of the steps above zero; those below it: Sall - all
          serial = __any(!(lane_value(all, 63) * Al < 60.0f && lane_value(Sall - all, 63) * Al < 60.0f));
        }
      }
      if (last) {  // in flight during these states
        if (!SUM) load(zp, zs1, zs2, t0, rz);
        if (chunk + 1 < c_end) {
          load(up, p.us1, p.us2, t0 + kChunk, ru);
          load(dp, p.ds1, p.ds2, t0 + kChunk, rd);
        }
      }

      const int n_end = std::min((part + 1) * kStates, p.dstate - g0);
      int n = part * kStates;
      if constexpr (PAIR) {
        if (!serial) {
          float y_in[kTL];
          const float carry_in = carry;
          const int n_in = n;
          float most = 0.0f;
#pragma unroll
          for (int j = 0; j < kTL; ++j) y_in[j] = y[j];
#pragma unroll 1
          for (; n + 2 <= n_end; n += 2) {
            float cin[2], a[2][kTL], bb[2][kTL], h[2], P[2], Pr[2], Ph[2], hx[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const float A = lane_value(Al, g0 + n + i);
              cin[i] = lane_value(carry, g0 + n + i);
#pragma unroll
              for (int q = 0; q < kTL / 4; ++q) {
                const float4 v = *reinterpret_cast<const float4*>(&s_b[n + i][lds_lane(lane, q)]);
                bb[i][4 * q] = du[4 * q] * v.x;
                bb[i][4 * q + 1] = du[4 * q + 1] * v.y;
                bb[i][4 * q + 2] = du[4 * q + 2] * v.z;
                bb[i][4 * q + 3] = du[4 * q + 3] * v.w;
              }
#pragma unroll
              for (int j = 0; j < kTL; ++j) a[i][j] = exp2_decay<DT>(d2[j] * A);
              h[i] = lane == 0 ? cin[i] : 0.0f;
              P[i] = exp2_decay<DT>(S * A);
              Pr[i] = exp2_decay<DT>(Srow * A);
              Ph[i] = exp2_decay<DT>(Shalf * A);
            }
#pragma unroll
            for (int j = 0; j < kTL; ++j)
#pragma unroll
              for (int i = 0; i < 2; ++i) h[i] = __builtin_fmaf(a[i][j], h[i], bb[i][j]);
            most = fmaxf(fmaxf(most, fabsf(h[0])), fabsf(h[1]));
            lane_scan2(P[0], h[0], Pr[0], Ph[0], P[1], h[1], Pr[1], Ph[1]);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              hx[i] = dpp_or<kWaveShr1>(cin[i], h[i]);
              carry = lane == g0 + n + i ? lane_value(h[i], 63) : carry;
            }
#pragma unroll
            for (int q = 0; q < kTL / 4; ++q) {
              const float4 v0 = *reinterpret_cast<const float4*>(&s_c[n][lds_lane(lane, q)]);
              const float4 v1 = *reinterpret_cast<const float4*>(&s_c[n + 1][lds_lane(lane, q)]);
              const float cc[2][4] = {{v0.x, v0.y, v0.z, v0.w}, {v1.x, v1.y, v1.z, v1.w}};
#pragma unroll
              for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                  hx[i] = __builtin_fmaf(a[i][4 * q + j], hx[i], bb[i][4 * q + j]);
                  y[4 * q + j] = __builtin_fmaf(hx[i], cc[i][j], y[4 * q + j]);
                }
            }
          }
          if (__any(is_inf(most))) {  // the states once more below, see there
            n = n_in;
            carry = carry_in;
#pragma unroll
            for (int j = 0; j < kTL; ++j) y[j] = y_in[j];
          }
        }
      }
#pragma unroll 1
      for (; n < n_end; ++n) {
        const float A = lane_value(Al, g0 + n), cin = lane_value(carry, g0 + n);
        float a[kTL], bb[kTL];
#pragma unroll
        for (int q = 0; q < kTL / 4; ++q) {
          const float4 v = *reinterpret_cast<const float4*>(&s_b[n][lds_lane(lane, q)]);
          bb[4 * q] = du[4 * q] * v.x;
          bb[4 * q + 1] = du[4 * q + 1] * v.y;
          bb[4 * q + 2] = du[4 * q + 2] * v.z;
          bb[4 * q + 3] = du[4 * q + 3] * v.w;
        }
#pragma unroll
        for (int j = 0; j < kTL; ++j) a[j] = exp2_decay<DT>(d2[j] * A);
        float hx, hend;  // the state before this lane's steps, and at the chunk's end
        bool one_by_one = serial;
        if (!serial) {
          float h = lane == 0 ? cin : 0.0f;
#pragma unroll
          for (int j = 0; j < kTL; ++j) h = __builtin_fmaf(a[j], h, bb[j]);
          // An infinite state stays infinite while each step's decay is above zero, but its product
          // with the decay over many steps, which may underflow, is NaN: then, too, the lanes go
          // one by one.  The test costs 0 to 4% of a call (1x1024x2048 fp16 21.7 -> 22.6 us, fp32 4x1024x4096
          // 174 -> 175), one per chunk of its inputs or end states 1 to 12%; the pairs above test once
          // a group of states and keep y as it was, for which the registers do not suffice here.
          one_by_one = __any(is_inf(h));
          float P = exp2_decay<DT>(S * A);
          lane_scan(P, h, exp2_decay<DT>(Srow * A), exp2_decay<DT>(Shalf * A));
          hx = dpp_or<kWaveShr1>(cin, h);
          hend = lane_value(h, 63);
        }
        if (one_by_one) {
          hx = hend = cin;
          for (int l = 0; l < 64; ++l) {
            hx = lane == l ? hend : hx;
            float v = hend;
#pragma unroll
            for (int j = 0; j < kTL; ++j) v = __builtin_fmaf(a[j], v, bb[j]);
            hend = lane_value(v, l);
          }
        }
        carry = lane == g0 + n ? hend : carry;
        if constexpr (!SUM) {
#pragma unroll
          for (int q = 0; q < kTL / 4; ++q) {
            const float4 v = *reinterpret_cast<const float4*>(&s_c[n][lds_lane(lane, q)]);
            const float cc[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              hx = __builtin_fmaf(a[4 * q + j], hx, bb[4 * q + j]);
              y[4 * q + j] = __builtin_fmaf(hx, cc[j], y[4 * q + j]);
            }
          }
        }
      }
    }

    if constexpr (SUM) continue;
    // ---- skip term, gate and store ----
    float ey[E];
    if constexpr (kDirect) {
#pragma unroll
      for (int k = 0; k < E; ++k) ey[k] = y[k];
    } else {
      __syncthreads();  // the tile's delta2 and delta' * u are read
#pragma unroll
      for (int q = 0; q < kTL / 4; ++q)
        *reinterpret_cast<float4*>(&s_x[part][wch][lds_lane(lane, q)]) =
            make_float4(y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]);
      __syncthreads();
      const int pos = lds_pos(et);
#pragma unroll
      for (int k = 0; k < E; ++k) {
        ey[k] = LAYOUT == kTime ? s_x[0][ec][pos + k] : s_x[0][ec + k][pos];
#pragma unroll
        for (int w = 1; w < SW; ++w) ey[k] += LAYOUT == kTime ? s_x[w][ec][pos + k] : s_x[w][ec + k][pos];
      }
    }
    V o;
#pragma unroll
    for (int k = 0; k < E; ++k) ey[k] = __builtin_fmaf(Dv[LAYOUT == kTime ? 0 : k], Ty<DT>::f(ku[k]), ey[k]);
    if (has_z) {
#pragma unroll
      for (int k = 0; k < E; ++k) o[k] = Ty<DT>::from(ey[k] * silu_f(Ty<DT>::f(rz[k])));
    } else {
#pragma unroll
      for (int k = 0; k < E; ++k) o[k] = Ty<DT>::from(ey[k]);
    }
    if constexpr (LAYOUT == kTime) {
      T* const r = yp + c * p.ys1 + t0 + et;
      if (!chok) continue;
      if (t0 + et + E <= p.seqlen) {
        *reinterpret_cast<U*>(r) = o;
      } else {
#pragma unroll
        for (int k = 0; k < E; ++k)
          if (t0 + et + k < p.seqlen) r[k] = o[k];
      }
    } else if (t0 + et < p.seqlen) {
      *reinterpret_cast<U*>(yp + (t0 + et) * p.ys2 + ch0 + ec) = o;
    }
  }

  if (!chok || !mine) return;
  if constexpr (SUM) {
    float* const sm = p.sum + (b * p.dim + c) * (p.dstate + 1) * static_cast<int64_t>(p.nseg) + seg;
    if (lane < p.dstate) sm[static_cast<int64_t>(lane) * p.nseg] = carry;
    if (lane == 0) sm[static_cast<int64_t>(p.dstate) * p.nseg] = dsum;
  } else if (p.state_out != nullptr && seg + 1 == p.nseg) {
    if (lane < p.dstate) p.state_out[(b * p.dim + c) * p.dstate + lane] = carry;
  }
}

// How a call runs here, if it does (sw == 0: it does not, scan.hip has it).
struct Plan {
  int layout, sw, nseg;
};
// Channels of a workgroup: eight waves in all.
inline int channels_of(int layout, int sw) { return layout == kTime && sw == 4 ? 2 : sw == 2 ? 4 : 8; }

// Which calls: unit strides along one axis, B and C in x's type (anything else keeps scan.hip's
// packed B/C), and few enough channels.  The lines below are where scan.hip's time and this one's
// cross, measured over 8 to 16384 channels, 8 to 65536 steps, 1 to 64 states, fp16 and fp32,
// along time and by rows; of 15549 calls that come here (drawn and large ones, in all types) 7 are
// slower than scan.hip by 3% or more (14% at most), and they take 0.36 of its time on average.  us, scan.hip's
// first, fp16 and 16 states unless said, batch x channels x steps:
//   - A chunk costs the same for 1 or 512 steps, and a launch as many rounds of a workgroup per CU as
//     it has begun: `waste` is the work done over the work asked for.  One chunk nearly always
//     pays (1x1536x512 20 -> 12, 1x1024x64 13 -> 9.4), more of them while the waste is small:
//     1x2560x896 (1.4) 30 -> 28, 1x2560x768 (1.6) 25 -> 28; 1x2048x1152 (1.3) 31 -> 27, 1x2560x1152 (1.6)
//     32 -> 39; 1x3072x2304 (1.1) 69 -> 60, 1x2560x2304 (1.3) 51 -> 60; by rows 1x2560x896 (1.8) 0.83 of the
//     time, 1x2560x768 (2.1) 1.12.  Rows of a length that scan.hip cannot load as vectors cost it
//     a third (1x2560x3001 92 -> 73), and few states cost this kernel less, and scan.hip no less.
//   - Up to 8 thousand channels (16-bit rows 10): 4x2048x2048 116 -> 96, 4x1536x8192 335 -> 289.  Above,
//     scan.hip's chains fill the chip.
//   - Few channels and long: time is split, in two launches (1x16x32768 90 -> 14, 1x64x8192 36 ->
//     17, 1x256x2048 22 -> 17; 1x256x4608 29 -> 33, 1x512x1280 21 -> 23).  Between these and 2048 (fp32
//     1024) channels, long sequences keep scan.hip's split, which takes fewer slots (1x1024x32768 247
//     against 292).
//   - dstate > 16, where scan.hip has 64-channel blocks of 32 or 64 states that walk all of time: any length,
//     without a split (1x16x65536 at 32 states in 0.07 of the time), until those blocks fill the chip with
//     states that are no padding: 1x16384x1024 at 32 and 64 states 0.9 to 1.1 of the time, at 24 and 48 0.5 to 0.8.
inline Plan plan(const mm_scan_params* a, size_t sum_bytes) {
  Plan pl = {kTime, 0, 1};
  const int64_t ch = a->batch * a->dim, L = a->seqlen;
  if (L < 8 || L > (1 << 30) || ch > (1 << 20) || a->bc_dtype != a->x_dtype) return pl;
  bool time_c = a->B_stride[2] == 1 && a->C_stride[2] == 1;
  bool chan_c = a->B_stride[1] == 1 && a->C_stride[1] == 1 && a->dim % 8 == 0 && a->dstate % 8 == 0;
  const int64_t* st[4] = {a->u_stride, a->delta_stride, a->y_stride, a->z_stride};
  for (int i = 0; i < (a->z ? 4 : 3); ++i) {
    time_c = time_c && st[i][2] == 1;
    chan_c = chan_c && st[i][1] == 1;
  }
  if (!time_c && !chan_c) return pl;
  pl.layout = time_c ? kTime : kRows;
  const bool f32 = a->x_dtype == MM_F32;
  const int64_t nch = ceil_div(L, kChunk);

  int64_t most = time_c || f32 ? 8192 : 10240;
  if (a->dstate > 16)
    most = ceil_div(a->dstate, 8) % 4 != 0 ? 16384 : ch > 2048 && L <= 256 ? 12288 : ch > 6144 ? 14200 : 16384;
  if (ch * nch * kChunk > most * L) return pl;
  const bool low = a->dstate <= (f32 ? 4 : 8);
  bool split = false;
  if (a->dstate <= 16) {
    const int64_t w = low ? 2 : 1;
    const bool few = (ch <= 256 * w && nch <= 4) || (ch <= 192 * w && ch * nch <= 2048) || (ch <= 128 * w && ch * nch <= 4096);
    const bool some = a->dstate > 4 && a->dstate <= 8;  // one state per lane of scan.hip's, and not few of them
    if (time_c) {
      if (nch > 2 && ch < (f32 && nch <= (some ? 16 : 32) ? 1024 : f32 || nch <= 16 || low ? 2048 : 4096) && !(ch >= 768 && nch <= 4)) {
        if (!few) return pl;
        split = true;
      }
    } else if (f32 && some && nch > 16) {
      if (!few) return pl;
      split = true;
    } else if (nch > 1 && ch < 3072 && !(ch >= (f32 ? 1024 : 2048) && nch <= 8) && !(ch >= 1536 && nch <= 4) &&
               !(ch >= 768 && nch <= 2)) {
      if (!few || nch < 4) return pl;
      split = true;
    }
  }

  // Waves per channel.  Unsplit, until the channels alone give four waves per SIMD: 1x1536x2048
  // fp32 61 (SW = 1), 52 (2), 48 us (4), 2x1536x4096 fp16 104, 95, 114; by rows a second wave,
  // on four channels a workgroup instead of eight, pays up to 1024 channels (a workgroup per CU) and
  // in fp32 always (B x L x D, against eight channels on one wave each): fp16 1x1000x1024 20.7 -> 15.2, 2x700x512 19.9
  // -> 14.3, 1x2048x1536 40.8 and 41.2, 4x2048x1536 88 and 107; fp32 1x2048x1536 71 -> 55,
  // 1x2048x3072 108 -> 82, 4x2048x1536 165 -> 147 (two waves on eight channels: 20.7, 19.5, 42.6,
  // 121; 57, 109, 166).  Split, as long as the segments leave room.
  if (split) {
    const int64_t seg = std::min<int64_t>(nch, kMaxSeg), bytes = 4 * ch * (a->dstate + 1);
    // (without room for summaries one pass over all chunks is still the faster one)
    const int64_t nseg = std::min<int64_t>({seg, static_cast<int64_t>(sum_bytes) / bytes, std::max<int64_t>(1, 4096 / ch)});
    if (nseg > 1) {
      const int64_t per = ceil_div(nch, nseg);
      pl.nseg = static_cast<int>(ceil_div(nch, per));
    }
    const int64_t w = ch * pl.nseg;
    pl.sw = time_c ? (w <= 1024 ? 4 : w <= 2048 ? 2 : 1) : (w <= 2048 ? 2 : 1);
    return pl;
  }
  pl.sw = time_c ? (ch <= 1536 ? 4 : ch < 4096 ? 2 : 1) : (f32 || ch <= 1024 ? 2 : 1);
  if (a->dstate <= 16 && ch > 1024 && !(nch <= 2 && ch <= 2048 && (nch == 2 || !time_c))) {
    const int64_t wgs = a->batch * ceil_div(a->dim, channels_of(pl.layout, pl.sw));
    const double waste = static_cast<double>(nch * kChunk) / L * round_up(wgs, kCus) / wgs;
    double limit;
    if (nch == 1) limit = ch <= 3072 ? 5.0 : time_c && f32 && ch > 4096 ? 1.5 : 2.5;
    else if (low && ch >= 4096 && time_c) limit = 5.0;
    else if (time_c && nch == 2) limit = 1.45;
    else if (time_c && f32) limit = nch <= 4 ? 1.45 : ch >= 2048 ? 1.25 : 1.19;
    else if (time_c) limit = ch <= 1536 ? 1.1 : nch == 3 ? 1.4 : nch == 4 ? 1.33 : ch < 4096 ? 1.1 : 1.19;
    else if (f32) limit = nch == 2 ? 1.5 : nch == 3 ? 1.4 : nch == 4 && ch < 2048 ? 1.9 : 1.3;
    else limit = nch == 2 ? 1.95 : nch <= 4 ? 1.5 : 1.25;
    if (low && (nch <= 8 || (f32 && ch > 1536))) limit *= 1.1;
    if (time_c && L % 4 != 0) limit *= 1.3;
    if (waste > limit) pl.sw = 0;
  }
  return pl;
}

bool preferred(const mm_scan_params* a, size_t sum_bytes) { return plan(a, sum_bytes).sw > 0; }

int segments(const mm_scan_params* a, size_t sum_bytes, int* sw) {
  const Plan pl = plan(a, sum_bytes);
  *sw = pl.sw;
  return pl.nseg;
}

template <int DT, int LAYOUT, int CH, int SW, bool PAIR = false>
void launch_n(const Params& p, int64_t batch, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(ceil_div(p.dim, CH) * p.nseg * batch));
  const dim3 block(64 * CH * SW);
  if (p.nseg > 1)
    hipLaunchKernelGGL((lane_scan_kernel<DT, LAYOUT, true, CH, SW, false>), grid, block, 0, s, p);
  hipLaunchKernelGGL((lane_scan_kernel<DT, LAYOUT, false, CH, SW, PAIR>), grid, block, 0, s, p);
}

template <int DT>
void launch_dt(const Params& p, int64_t batch, const Plan& pl, hipStream_t s) {
  if (pl.layout == kTime) {
    if (pl.sw == 4) launch_n<DT, kTime, 2, 4>(p, batch, s);
    else if (pl.sw == 2) launch_n<DT, kTime, 4, 2>(p, batch, s);
    else launch_n<DT, kTime, 8, 1>(p, batch, s);
  } else {
    // 16-bit, unsplit, at most a workgroup per CU: states in pairs (fp32's longer decays keep a SIMD's
    // two waves busy: 1x1000x1024 19.7 and 19.6 us, 2x2048x3072 155 and 203)
    if constexpr (DT != MM_F32) {
      if (p.nseg == 1 && ceil_div(p.dim, channels_of(kRows, pl.sw)) * batch <= kCus) {
        if (pl.sw == 2) launch_n<DT, kRows, 4, 2, true>(p, batch, s);
        else launch_n<DT, kRows, 8, 1, true>(p, batch, s);
        return;
      }
    }
    if (pl.sw == 2) launch_n<DT, kRows, 4, 2>(p, batch, s);
    else launch_n<DT, kRows, 8, 1>(p, batch, s);
  }
}

int launch(const mm_scan_params* a, int* ctl, float* sum, size_t sum_bytes, void* stream) {
  const Plan pl = plan(a, sum_bytes);
  Params p = {};
  p.u = a->u;
  p.delta = a->delta;
  p.z = a->z;
  p.y = a->y;
  p.A = a->A;
  p.D = a->D;
  p.B = a->B;
  p.C = a->C;
  p.state_out = a->state_out;
  p.sum = sum;
  p.ctl = ctl;
  p.us0 = a->u_stride[0], p.us1 = a->u_stride[1], p.us2 = a->u_stride[2];
  p.ds0 = a->delta_stride[0], p.ds1 = a->delta_stride[1], p.ds2 = a->delta_stride[2];
  p.zs0 = a->z_stride[0], p.zs1 = a->z_stride[1], p.zs2 = a->z_stride[2];
  p.ys0 = a->y_stride[0], p.ys1 = a->y_stride[1], p.ys2 = a->y_stride[2];
  p.Bs0 = a->B_stride[0], p.Bs1 = a->B_stride[1], p.Bs2 = a->B_stride[2];
  p.Cs0 = a->C_stride[0], p.Cs1 = a->C_stride[1], p.Cs2 = a->C_stride[2];
  p.As0 = a->A_stride[0], p.As1 = a->A_stride[1];
  p.Ds = a->D_stride;
  p.dim = static_cast<int32_t>(a->dim);
  p.dstate = static_cast<int32_t>(a->dstate);
  p.seqlen = static_cast<int32_t>(a->seqlen);
  p.softplus_cut = a->delta_softplus ? 20.0f : __builtin_nanf("");
  p.nseg = pl.nseg;
  p.seg_chunks = static_cast<int32_t>(ceil_div(ceil_div(a->seqlen, kChunk), pl.nseg));
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (a->x_dtype) {
    case MM_F32: launch_dt<MM_F32>(p, a->batch, pl, s); break;
    case MM_F16: launch_dt<MM_F16>(p, a->batch, pl, s); break;
    default: launch_dt<MM_BF16>(p, a->batch, pl, s); break;
  }
  return check_launch("lane_scan");
}

}  // namespace lscan
}  // namespace mm
