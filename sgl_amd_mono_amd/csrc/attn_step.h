// Sparse-attention phase of one decode step on gfx950, as ONE persistent launch (one
// 512-thread workgroup per CU). The reference runs it as stages of its decoder-layer
// launch: FP4 index scores (deepseek_v4/gfx950/kernels/stages/indexer.py:460-602 and
// the native-FP4 scorer deepseek_v41/gfx950/indexer/score_fp4.py:254-296), the exact
// top-2048 (indexer.py:604-802, glm53/gfx950/kernel.py:3000-3636), the sparse MLA
// split (kernel.py:3638-3973) and the split merge (kernel.py:3975-4123).
//
// Tasks, dealt round-robin over the workgroups in this order. A workgroup waits only on
// tasks earlier in the list or on its own top-k team, whose members share one round
// of the deal (teams never straddle a round), so the launch cannot deadlock while all
// workgroups are resident; every wait is guarded (sync.h):
//   score  (row, 1024 keys): 8 waves x 128 keys. The row's FP4 query (64 heads x 128
//          dims, E2M1 + E8M0 per 32) is the A operand and 16 keys of SGLang's FP4 index
//          plane the B operand of v_mfma_scale_f32_16x16x128_f8f6f4 with FP4 formats:
//          the plane's E8M0 bytes are the MFMA's per-lane B scales as they lie (a
//          lane's dword holds its key's scale for the page's four 16-key tiles).
//          score = sum_h w_h relu(q_h . k) -> mailbox score, and the histogram of the
//          keys' leading 8-bit digits -> mailbox rowh. Only rows of more than TOPK keys
//          are scored (a shorter row selects every key). One chunk a workgroup where the
//          grid holds a workgroup for every chunk of max_ctx; else each workgroup takes a
//          contiguous run of the step's chunks (score_run)
//   topk   (row, member of a team of 16): the row's scores as order-preserving u32
//          keys, 2048 a member; an MSB-first 8-bit radix select of the 2048th largest
//          key: digit 1 from the chunk histograms, digit 2 from the sum of the members'
//          histograms (mailbox hist; a wave's most common digits go in as one atomic).
//          The keys sharing both digits with the threshold (mailbox cand) are ranked by
//          every member; a crowded bin (ties) takes digits 3 and 4 the same way as digit
//          2 and a stable compaction from the members' counts (mailbox cnt). Every key
//          above the threshold and the lowest positions equal to it, ascending -> cache
//          slots (page_table[p / 64] * 64 + p % 64) -> mailbox sel (glm53/check.py:100-117)
//   split  (row, 64 selected tokens): sub-tiles of 64 tokens gathered from the FP8
//          cache into LDS as they lie, two buffers: q.k operands, and p.v operands by
//          transposed LDS reads, both widened exactly to bf16 in registers; q in
//          registers; bf16 MFMA 16x16x32 for q.k (two waves a token tile, each half of
//          the 576 dims) and p.v, the per-token scale folded into the logit and the
//          probability, online softmax -> the split's partials (bf16, 32 KB in one
//          contiguous run) and (m, l), then its done word (mailbox sdone)
//   merge  (row, head): once every split of the row is done,
//          out = sum_j e^(m_j - M) acc_j / sum_j e^(m_j - M) l_j, bf16
#pragma once

#include "attn_ops.h"
#include "common.h"
#include "proj_ops.h"
#include "sync.h"

namespace mono {
namespace attn {

namespace {

#ifdef MONO_ATTN_LONG
constexpr bool kLongSplits = true;
constexpr int TMK = TEAM_LONG;  // members of a row's top-k team in this launch
#else
constexpr bool kLongSplits = false;
constexpr int TMK = TEAM;
#endif

constexpr int AT = 512;
constexpr int AW = AT / WAVE;
constexpr int KPM = MAX_CTX / TMK;           // keys a top-k team member owns
constexpr int KPT = KPM / AT;                // keys a thread of a member holds
// a member of many keys stages its selected slots in LDS and stores them as one run: each
// thread storing its own took 4.3 us for a member that holds its row alone (staged 1.9; 33
// rows of 1500-12000 keys 44.2 -> 43.1 us a launch, 48 rows of 32768 71.0 -> 70.1)
constexpr bool kStageSel = KPM > TOPK;
constexpr int SUB = 64;                      // tokens a split sub-tile
constexpr int QK_HALF = DQK / 2;             // dims of q.k a wave sums (two waves a token tile)
constexpr int QK_STEPS = QK_HALF / 32;       // its bf16 MFMA k steps
// dwords a cached FP8 row in LDS: 16-byte aligned, and 20 banks (mod 64) from the next
// row, so the 16 rows of a q.k operand read fall on distinct banks
constexpr int KF_W = DQK / 4 + 4;
constexpr int PF_STRIDE = SUB + 4;           // f32 a logit row in LDS
constexpr int PB_STRIDE = SUB + 8;           // bf16 a probability row in LDS
constexpr int ROPE_CH = (DQK - DV) / 16;     // 16-byte chunks of a row past the value dims
// 16-byte units a staged q row (one head): padded by one, so the 16 heads of a q
// operand read fall on distinct banks
constexpr int Q_UNITS = DQK / 8 + 1;
static_assert(DV / 16 * (SUB / 4) == AT && ROPE_CH * SUB <= AT && QK_HALF % 32 == 0, "gather tiling");
constexpr int KEYS_WAVE = CHUNK / AW;        // 128 keys a wave of a score task
constexpr int KTILES = KEYS_WAVE / 16;
constexpr float NEG_INF = -__builtin_huge_valf();
static_assert(KPM % AT == 0 && PAGE % KPT == 0 && TMK <= 16 && KPT % 4 == 0 && KEYS_WAVE % PAGE == 0 && SPLIT_MAX <= AT, "tiling");
static_assert(AT == NH * DV / 32, "tiling");

enum { W_SCORE = 0, W_SEL = 1, W_PART = 2, W_TEAM = 3 };



constexpr int RUN = 8;  // chunks of a score run held in LDS at a time (64 rows of 32 chunks: 8 a CU)
static_assert(RUN <= AW, "a wave looks a chunk up");

struct ScoreLds {
  uint32_t hist[256];  // the leading-digit histogram of the row's chunks scored here
  // a run's chunks: their page numbers, and the query (E2M1 rows, E8M0 scales, head
  // weights) of the row that starts at, or runs into, chunk j
  int32_t pg[RUN][CHUNK / PAGE];
  u32x4 q[RUN][IH * ID / 32];
  uint32_t qs[RUN][IH];
  u32x2 qw[RUN][IH / 4];
};

struct TopkLds {
  uint32_t hist[256];       // this member's digit histogram
  uint32_t tot[256];        // the team's
  uint32_t pre[256];        // the members' before this one
  uint32_t cu[CMAX];        // the team's threshold candidates, 0 past the last
  int32_t sl[kStageSel ? TOPK : 1];  // this member's selected slots, in position order
  int32_t xw[TMK];          // the members' keys above the first digit
  int32_t cnt[TMK][2];      // the team's keys above / at the threshold
  uint32_t digit, uT;
  int32_t above, pre_above;
};

// Typed views of 16- and 8-byte units: an access through a pointer cast from a narrower
// element type is split by the compiler into 4-byte pairs (the cast's alignment is
// not known to it); through an array of the unit type it is one b128 / b64 access.
struct SplitLds {
  // the cached rows of two sub-tiles as they lie (E4M3), sub-tile st in buffer st % 2:
  // the q.k operands (8 dims a unit) and, read transposed, the p.v operands
  union {
    u32x4 kf16[2][SUB][KF_W / 4];
    u32x2 kf8[2][SUB][KF_W / 2];
    struct {
      u32x4 first[SUB][KF_W / 4];  // kf16[0]
      u32x4 q16[NH][Q_UNITS];      // until the second sub-tile's rows: the row's q (bf16)
    };
    u32x2 ot[2][SUB][KF_W / 2];  // after the last sub-tile: the partials, in the buffer it does not use
  };
  union {  // logits [dim half][head][token]: sums over dims [0, 288) and [288, 576)
    f32x4 pf4[2][NH][PF_STRIDE / 4];
    float pf[2][NH][PF_STRIDE];
  };
  union {  // probabilities times the tokens' scales, bf16 [head][token]
    u32x4 pb16[NH][PB_STRIDE / 8];
    u32x2 pb8[NH][PB_STRIDE / 4];
  };
  union {
    int32_t slot[SPLIT_MAX];
    i32x4 slot4[SPLIT_MAX / 4];
  };
  union {
    float kvs[2][SUB];
    f32x4 kvs4[2][SUB / 4];
  };
  float alpha[NH];
};
static_assert(KF_W % 4 == 0 && PF_STRIDE % 4 == 0 && PB_STRIDE % 8 == 0, "16-byte units");
static_assert(sizeof(SplitLds::q16) <= sizeof(SplitLds::first), "q inside the second sub-tile's buffer");
static_assert(NH * 16 == AT && SUB == 16 * 4, "softmax: a 16-lane row a head, 4 tokens a lane");

struct MergeLds {
  float w[8][SPLITS];  // each split's weight e^(m_j - M) a head of the task, 0 for an empty split
  float den[8];        // sum_j w_j l_j a head
};

struct Lds {
  union {
    ScoreLds sc;
    TopkLds t;
    SplitLds sp;
    MergeLds mg;
  } u;
  int32_t scan[AW];
};

struct Args {
  const uint8_t* iq;
  const uint8_t* iqs;
  const uint16_t* iw;
  const uint8_t* ikv;
  const uint8_t* iks;
  const uint16_t* q;
  const uint8_t* kv;
  const float* kv_scale;
  int kv_mask;  // slot & kv_mask indexes kv_scale (0: one scale for every row)
  const int32_t* pt;
  const int32_t* seq_lens;
  int pt_stride;
  int n_pages;
  uint16_t* out;
  int rows;
  float* scores;
  int32_t* topk;
  int64_t* timeline;
  float scale;
  // the front of the layer ran earlier in this launch: its replicated done words
  // (proj::Mail::fdone: FD_B + s row s's index key and head weights, FD_E + 8 s + j its
  // index query, FD_D + h head h of q), awaited at wait sites fsite and fsite + 1; only a
  // build with MONO_ATTN_FRONT has the waits, so no other build can name done words
#ifdef MONO_ATTN_FRONT
  const uint64_t* fdone;
  int fsite;
#endif
  bool publish_out;  // a later stage of the launch reads `out`: each merge puts a done word
  // the row histograms: 1, two copies by launch parity (each launch clears its
  // successor's copy, the guard's flip words); 0, one copy that the launch's caller
  // clears once every reader is done (a layer of a multi-layer launch)
  int rowh_flip;
  Mail mail;
  GuardArgs guard;
};

MONO_DEV uint32_t radix_key(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// FP4 x FP4 16x16x128 with per-lane E8M0 scales; the B scale byte is picked by OPB.
template <int OPB>
MONO_DEV f32x4 mfma_fp4_opb(const u32x4& a, const u32x4& b, int sa, int sb) {
  const i32x8 A = {(int)a[0], (int)a[1], (int)a[2], (int)a[3], 0, 0, 0, 0};
  const i32x8 B = {(int)b[0], (int)b[1], (int)b[2], (int)b[3], 0, 0, 0, 0};
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, z, 4, 4, 0, sa, OPB, sb);
}

// E4M3 bytes 2 HW, 2 HW + 1 of a dword -> two bf16 as a dword, the first in the low half
// (exact: every E4M3 value is a bf16 value)
template <bool HW>
MONO_DEV uint32_t fp8x2_bf16(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, HW));
}

// A 16-lane group's transposed read of 8 rows x 16 bytes of LDS: lane l gives the address
// of bytes 8 (l % 2) .. of row l / 2 and gets byte l of each of the 8 rows.
MONO_DEV u32x2 lds_tr8(const u32x2* p) {
  typedef int32_t i32x2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)p));
}

// 8 E4M3 bytes (two dwords) -> 8 bf16: an MFMA operand of 8 consecutive k
MONO_DEV bf16x8 fp8x8_bf16x8(const u32x2& w) {
  const u32x4 o = {fp8x2_bf16<false>(w[0]), fp8x2_bf16<true>(w[0]), fp8x2_bf16<false>(w[1]), fp8x2_bf16<true>(w[1])};
  return __builtin_bit_cast(bf16x8, o);
}

class Step {
 public:
  MONO_DEV Step(const Args& a, Lds& l) : A(a), L(l) {
    tid = thread_index();
    lane = tid % WAVE;
    wave = tid / WAVE;
    g = lane / 16;
    r = lane % 16;
    G = gridDim.x;
    CH = a.mail.max_ctx / CHUNK;
  }

  MONO_DEV void run() {
    if (!begin()) return poison(true);
    if (!tasks()) poison(false);
  }

  // NaN over the launch's output (sync.h poison_bf16)
  MONO_DEV void poison(bool share) const { poison_bf16(A.out, (size_t)A.rows * NH * DV, share); }

  // The launch's tag and deadline (false: the guard refused the launch or its epoch
  // scrub failed). The row histograms are the guard's flip accumulators: the launch
  // start clears the copy the next launch adds into.
  MONO_DEV bool begin() { return guard_begin(A.guard, gd); }

  // Run under a guard the caller set up (a layer of a multi-layer launch).
  MONO_DEV void adopt(const Guard& g) { gd = g; }

  MONO_DEV const Guard& guard() const { return gd; }

  // tasks in the list: score tasks padded to a multiple of TMK so no top-k team
  // straddles a round, then top-k members, splits, merges
  MONO_DEV int n_score() const { return (A.rows * CH + TMK - 1) / TMK * TMK; }
  // (a row's merges_of(rows) merges of 32 / merges_of(rows) heads each cover its NH heads)
  MONO_DEV int n_tasks() const { return n_score() + A.rows * TMK + A.rows * (splits_of(A.rows) + merges_of(A.rows)); }
  MONO_DEV int n_topk() const { return A.rows * TMK; }
  // after the scores: the list index at which the tasks after them are dealt
  MONO_DEV int list_base() const { return base; }

  // This workgroup's tasks (false, workgroup-uniform: a wait failed).
  MONO_DEV bool tasks() {
    return tasks([] { return true; });
  }

  // The same with `between()` (workgroup-uniform; false: a wait failed) run after this
  // workgroup's top-k tasks and before its splits: the fused layer's deferred work.
  template <class Between>
  MONO_DEV bool tasks(Between&& between) {
    const int n_topk = A.rows * TMK;
    if (kLongSplits || A.rows * CH > G) row_n = lane < A.rows ? row_len(lane) : 0;
    if (!scores()) return false;
    // a workgroup's list is ordered by stage: one loop a stage keeps each loop body to
    // one task kind (and its registers). The list after the scores starts at `base` (a
    // multiple of TMK); a task's timeline row is its list index + tl0.
    const int tl0 = n_score() - base, at = base + n_topk;
    int T = first_at_or_after(base);
    for (; T < at; T += G) {
      const uint64_t t0 = now_ticks();
      const bool ok = topk_member((T - base) / TMK, (T - base) % TMK);
      stamp(T + tl0, t0, 1);
      if (!ok) return false;  // workgroup-uniform
    }
    if (!between()) return false;
    // one sub-tile a split up to LONG_ROWS rows (its loop over sub-tiles compiles away),
    // splits of the plan above, in k_attn_long alone (MONO_ATTN_LONG): every other launch
    // takes at most LONG_ROWS rows.
    const int n_split = kLongSplits ? first_split(A.rows) : A.rows * SPLITS;
    for (T = first_at_or_after(at); T < at + n_split; T += G) {
      const uint64_t t0 = now_ticks();
      const int i = T - at;
      bool ok;
      if (kLongSplits) {
        const int s = (int)__popcll(__ballot(sp_inc <= i)), j = i - first_split(s);
        const int nst = sub_tiles(__builtin_amdgcn_readlane(row_n, s)), nsp = first_split(s + 1) - first_split(s);
        const int rcp = recip(nsp), lo = j * nst * rcp >> 16, hi = (j + 1) * nst * rcp >> 16;
        ok = split_task<true>(s, j, lo * SUB, (hi - lo) * SUB);
        if (i < A.rows * splits_of(A.rows)) stamp(T + tl0, t0, 2);
      } else {
        ok = split_task<false>(i / SPLITS, i % SPLITS, i % SPLITS * SUB, SUB);
        stamp(T + tl0, t0, 2);
      }
      if (!ok) return false;
    }
    const int tlm = n_score() + n_topk + A.rows * splits_of(A.rows);
    const bool ok = !kLongSplits               ? merges<1>(at + n_split, tlm)
                    : merges_of(A.rows) == 8 ? merges<4>(at + n_split, tlm)
                                             : merges<8>(at + n_split, tlm);
    if (A.timeline) stamp_idle(n_split);
    return ok;
  }

 private:
  const Args& A;
  Lds& L;
  Guard gd;
  int tid, lane, wave, g, r, G, CH;
  int base = 0;
  int row_n = 0;   // lane s: row s's length (wide steps)
  int sp_inc = 0;  // lane s: the splits of rows 0 .. s (k_attn_long)
  bool q_ready = false;  // the front's q has been awaited (a fused launch)
  uint64_t waited = 0;

  // sub-tiles of selected tokens of a row of n keys
  MONO_DEV static int sub_tiles(int n) { return (min(n, TOPK) + SUB - 1) / SUB; }
  // The splits of a wide step: as few sub-tiles a split (sp) as let the step's splits fit
  // one round of the grid; row s has ceil(its sub-tiles / sp) splits of even length. A
  // fixed count a row (8 to 32 rows, 5 to 48, 4 above) gave 33 rows splits of 7 sub-tiles
  // where 5 fit, 17 rows 4 where 3 fit, and a short row's first splits as much as they held
  // (33 rows of 1500-12000 keys: 47.9 -> 42.6 us a launch). Taken while the first keys are
  // on their way. It takes in every row's length: a row's cuts, and with them its last bits,
  // depend on the step's other rows (its error does not: 0.0026 of the exact values either way).
  MONO_DEV void plan_splits() {
    const int nst = sub_tiles(row_n);
    const int total = wave_incl_scan(nst);
    int sp = 1;  // at least the even share
    for (int left = __builtin_amdgcn_readlane(total, WAVE - 1) - G; left > 0 && sp < SPLIT_MAX / SUB; left -= G) ++sp;
#pragma unroll 1
    for (;; ++sp) {
      sp_inc = wave_incl_scan((nst + sp - 1) * recip(sp) >> 16);
      if (sp == SPLIT_MAX / SUB || __builtin_amdgcn_readlane(sp_inc, WAVE - 1) <= G) break;
    }
  }
  // x * recip(d) >> 16 == x / d for 1 <= d <= 32 and 0 <= x <= 1024 (a reciprocal rounded up)
  MONO_DEV static int recip(int d) { return (int)(65536.0f * hw_rcp((float)d)) + 1; }
  // the list index (from the first split) of row s's first split
  MONO_DEV int first_split(int s) const { return s > 0 ? __builtin_amdgcn_readlane(sp_inc, s - 1) : 0; }
  // a row's chunks that are scored
  MONO_DEV int live_chunks(int n) const { return n > TOPK || A.scores ? (n + CHUNK - 1) / CHUNK : 0; }
  MONO_DEV int row_len(int s) const { return min(max(A.seq_lens[s], 0), A.mail.max_ctx); }
  // row s's leading-digit histogram of the launch with this tag: launches alternate
  // between two copies, and each launch clears the copy its successor uses
  MONO_DEV uint32_t* row_hist(uint32_t tag, int s) const {
    return A.mail.rowh + ((size_t)(A.rowh_flip ? tag & 1u : 0u) * A.mail.max_rows + s) * ROWH;
  }
  MONO_DEV int page_of(int s, int p) const {
    const int pg = A.pt[(size_t)s * A.pt_stride + p / PAGE];
    return min(max(pg, 0), A.n_pages - 1);
  }
  MONO_DEV int slot_of(int s, int p) const { return page_of(s, p) * PAGE + p % PAGE; }

  // this workgroup's first task at or after list index `at` (tasks are dealt round-robin)
  MONO_DEV int first_at_or_after(int at) const {
    const int b = block_index();
    return at <= b ? b : b + ((at - b + G - 1) / G) * G;
  }

  // timeline row of task T: start, inputs-ready and end ticks, workgroup << 8 | kind
  // (kind 0 score .. 3 merge); `waited` is 0 for a task that waits on nothing
  MONO_DEV void stamp(int T, uint64_t t0, int kind) const {
    if (A.timeline && tid == 0) {
      int64_t* tl = A.timeline + (size_t)T * 4;
      tl[0] = (int64_t)t0;
      tl[1] = (int64_t)waited;
      tl[2] = (int64_t)now_ticks();
      tl[3] = ((int64_t)block_index() << 8) | kind;
    }
  }
  MONO_DEV void mark_waited() { waited = now_ticks(); }
  // The timeline rows that no task of this step has, as tasks that end where they start:
  // chunks that are not scored (with the padding to whole teams) and splits past the plan.
  MONO_DEV void stamp_idle(int n_split) {
    waited = 0;
    for (int T = block_index(); T < n_score(); T += G) {
      const int s = T / CH;
      if (s >= A.rows || T % CH >= live_chunks(row_len(s))) stamp(T, now_ticks(), 0);
    }
    if (kLongSplits)
      for (int i = first_at_or_after(n_split); i < A.rows * splits_of(A.rows); i += G)
        stamp(n_score() + n_topk() + i, now_ticks(), 2);
  }

  // ---------------------------------------------------------------- score
  // The row's FP4 query in a wave's MFMA operands (64 heads x 128 dims: head tile ht =
  // heads 16 ht ..) with its scales and head weights.
  struct Query {
    u32x4 qa[IH / 16];
    int qsc[IH / 16];
    uint32_t w2[IH / 16][2];
  };
  // A wave's 128 keys of a chunk = 2 pages = 8 tiles of 16 keys (lane (g, r) holds chunk
  // g of key 16 t + r) with their pages' E8M0 dwords.
  struct Keys {
    u32x4 kb[KTILES];
    uint32_t ks[KEYS_WAVE / PAGE];
  };
  // The wave's two pages of a chunk as buffer resources: the page is the base, so a
  // lane's offset is the same for every tile and chunk; with no records (past a run's
  // last chunk) the loads return zeros without touching memory, and every turn issues
  // the same loads.
  struct Pages {
    __amdgpu_buffer_rsrc_t kv[KEYS_WAVE / PAGE], sc[KEYS_WAVE / PAGE];
  };
  static constexpr int NT_LOAD = 2;  // buffer cache policy: nontemporal

  // The lane's and the wave's indices afresh (from an opaque copy of the thread index), so
  // a loop's addresses are derived inside it, not hoisted out of it and held across it.
  struct Lane {
    int lane, g, r, wave;
  };
  MONO_DEV Lane lane_now() const {
    const unsigned t = (unsigned)opaque_v(tid);
    __builtin_assume(t < AT);
    return {(int)(t % WAVE), (int)(t % WAVE / 16), (int)(t % 16), __builtin_amdgcn_readfirstlane((int)(t / WAVE))};
  }

  MONO_DEV Pages pages(const int (&pg)[KEYS_WAVE / PAGE], bool any) const {
    Pages p;
#pragma unroll
    for (int i = 0; i < KEYS_WAVE / PAGE; ++i) {
      const size_t u = (size_t)__builtin_amdgcn_readfirstlane(pg[i]);
      p.kv[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(A.ikv) + u * (PAGE * ID / 2), 0,
                                                  any ? PAGE * ID / 2 : 0, BUF_DWORD3);
      p.sc[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(A.iks) + u * (PAGE * ID / 32), 0,
                                                  any ? PAGE * ID / 32 : 0, BUF_DWORD3);
    }
    return p;
  }
  MONO_DEV static void key_tile(const Lane& z, Keys& k, const Pages& p, int kt) {
    k.kb[kt] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(p.kv[kt / 4], z.g * (PAGE * 16) + z.r * 16,
                                                                               (kt % 4) * 256, NT_LOAD));
  }
  MONO_DEV static void key_scales(const Lane& z, Keys& k, const Pages& p, int i) {
    k.ks[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(p.sc[i], z.g * PAGE + z.r * 4, 0, 0));
  }
  MONO_DEV static void key_load(const Lane& z, Keys& k, const Pages& p) {
#pragma unroll
    for (int kt = 0; kt < KTILES; ++kt) {  // issued in the order in which a run's turns issue and use them
      key_tile(z, k, p, kt);
      if (kt % 4 == 3) key_scales(z, k, p, kt / 4);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  MONO_DEV void query_load(int s, Query& o) const {
#pragma unroll
    for (int ht = 0; ht < IH / 16; ++ht) {
      const size_t row = (size_t)s * IH + 16 * ht + r;
      o.qa[ht] = ld_u32x4(A.iq + row * (ID / 2) + g * 16);
      o.qsc[ht] = A.iqs[row * (ID / 32) + g];
      const u32x2 w4 = *reinterpret_cast<const u32x2*>(A.iw + (size_t)s * IH + 16 * ht + 4 * g);
      o.w2[ht][0] = w4[0];
      o.w2[ht][1] = w4[1];
    }
  }

  // key tile kt's logits against the four head tiles of the query
  MONO_DEV static void score_mfmas(const Query& q, const Keys& k, int kt, f32x4 (&d)[IH / 16]) {
#pragma unroll
    for (int ht = 0; ht < IH / 16; ++ht) {
      switch (kt % 4) {
        case 0: d[ht] = mfma_fp4_opb<0>(q.qa[ht], k.kb[kt], q.qsc[ht], (int)k.ks[kt / 4]); break;
        case 1: d[ht] = mfma_fp4_opb<1>(q.qa[ht], k.kb[kt], q.qsc[ht], (int)k.ks[kt / 4]); break;
        case 2: d[ht] = mfma_fp4_opb<2>(q.qa[ht], k.kb[kt], q.qsc[ht], (int)k.ks[kt / 4]); break;
        default: d[ht] = mfma_fp4_opb<3>(q.qa[ht], k.kb[kt], q.qsc[ht], (int)k.ks[kt / 4]); break;
      }
    }
  }

  // The wave's 128 scores of a chunk: lane (g, r) ends with those of its keys 16 g + r and
  // 64 + 16 g + r. NEXT: the keys of pages `np` are loaded into k, tile by tile, as this
  // chunk's are consumed (they are used two chunks later: a run holds two chunks' keys).
  template <bool NEXT>
  MONO_DEV static void chunk_scores(const Lane& z, const Query& q, Keys& k, const Pages& np, float (&sc)[2]) {
    float wv[IH / 16][4];
#pragma unroll
    for (int ht = 0; ht < IH / 16; ++ht) {
      wv[ht][0] = bf16_lo(q.w2[ht][0]);
      wv[ht][1] = bf16_hi(q.w2[ht][0]);
      wv[ht][2] = bf16_lo(q.w2[ht][1]);
      wv[ht][3] = bf16_hi(q.w2[ht][1]);
    }
    // a key tile's four head-tile MFMAs are issued together and the next tile's before
    // this tile's results are consumed, so no MFMA's latency sits in front of its use
    // (32 MFMAs a wave, each consumed at once, cost ~1 us of exposed latency)
    f32x4 d[2][IH / 16];
    float part[KTILES];
    score_mfmas(q, k, 0, d[0]);
#pragma unroll
    for (int kt = 0; kt < KTILES; ++kt) {
      if (kt + 1 < KTILES) score_mfmas(q, k, kt + 1, d[(kt + 1) % 2]);
      if (NEXT) {
        __builtin_amdgcn_sched_barrier(0);  // the tile's registers are free from here on
        key_tile(z, k, np, kt);
        if (kt % 4 == 3) key_scales(z, k, np, kt / 4);
      }
      part[kt] = 0.f;
#pragma unroll
      for (int ht = 0; ht < IH / 16; ++ht)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[kt] += wv[ht][i] * (d[kt % 2][ht][i] > 0.f ? d[kt % 2][ht][i] : 0.f);
      asm volatile("" : "+v"(part[kt]));  // summed here: eight tiles' logits would not fit the registers
    }
    // each key's sum over the four lane groups, (0 + 1) + (2 + 3): two tiles meet in a
    // swap of 16-lane rows, two such pairs in a swap of halves, and tile 4 h + j's sums
    // end in lane group j
#pragma unroll
    for (int h = 0; h < 2; ++h)
      sc[h] = swap_sum<32>(swap_sum<16>(part[4 * h], part[4 * h + 1]), swap_sum<16>(part[4 * h + 2], part[4 * h + 3]));
  }
  // 16: rows (a0 + a1, b0 + b1, a2 + a3, b2 + b3); 32: halves (a lo + a hi, b lo + b hi)
  template <int LANES>
  MONO_DEV static float swap_sum(float a, float b) {
    const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
    const auto v = LANES == 16 ? __builtin_amdgcn_permlane16_swap(x, y, false, false)
                               : __builtin_amdgcn_permlane32_swap(x, y, false, false);
    return __uint_as_float(v[0]) + __uint_as_float(v[1]);
  }

  // The wave's scores of chunk c of row s (n keys) -> mailbox score (each store covers 64
  // consecutive positions; the buffer drops those past the row) and the workgroup's
  // leading-digit histogram.
  MONO_DEV void chunk_store(const Lane& z, int s, int c, int n, const float (&sc)[2]) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(A.mail.score + (size_t)s * A.mail.max_ctx, 0, n * 4, BUF_DWORD3);
    const int p0 = c * CHUNK + z.wave * KEYS_WAVE + z.lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sc[i]), rs, (p0 + 64 * i) * 4, 0, SC1);
    if (A.scores)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (p0 + 64 * i < n) A.scores[(size_t)s * A.mail.max_ctx + p0 + 64 * i] = sc[i];
#pragma unroll
    for (int i = 0; i < 2; ++i) hist_add(L.u.sc.hist, p0 + 64 * i < n, radix_key(sc[i]) >> 24);
  }

  // Chunks c .. c + k - 1 of row s are scored here: their histogram is added into the row's
  // (the top-k's first radix pass) and, once every score and count is performed, they are
  // marked done (mailbox cdone). Frees the histogram for the next row.
  MONO_DEV void row_flush(int s, int c, int k) {
    uint32_t* hist = L.u.sc.hist;
    __syncthreads();
    uint32_t* rh = row_hist(gd.tag, s);
    if (tid < 256 && hist[tid] != 0u)
      __hip_atomic_fetch_add(&rh[tid], hist[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < 256) hist[tid] = 0u;
    __builtin_amdgcn_s_waitcnt(0);  // every score is stored and every add performed
    __syncthreads();
    if (tid < k) mb_put(&A.mail.cdone[(size_t)s * CH + c + tid], 0u, gd.tag);
  }

  // In a launch that runs the front too, it writes each row's index query, head weights
  // and new key: keys may be read before the wait for it (await_front), except a wave's
  // whose pages may hold a key written in this launch (the row's last `rows` positions: its
  // own new key and, for the rows of a verify chain, those of the chain's earlier rows;
  // a wave past the row reads the row's last page).
  MONO_DEV bool fresh(int k0, int n) const { return front_here() && k0 + KEYS_WAVE > n - A.rows; }  // wave-uniform
  MONO_DEV bool front_here() const { return front_done() != nullptr; }
  // the done words of the front of this launch (null, at compile time: it runs no front)
  // and the wait site of its first outputs
#ifdef MONO_ATTN_FRONT
  MONO_DEV const uint64_t* front_done() const { return A.fdone; }
  MONO_DEV int front_site() const { return A.fsite; }
#else
  MONO_DEV const uint64_t* front_done() const { return nullptr; }
  MONO_DEV int front_site() const { return 0; }
#endif
  MONO_DEV bool await_front() {
    const uint64_t* fd = done_copy(front_done());
    const int nr = A.rows;
    return hint_wait(nr * (1 + IH / 8), [fd, nr](int i) { return fd + (i < nr ? proj::FD_B + i : proj::FD_E + i - nr); },
                     front_site(), gd);
  }

  // This workgroup's share of the scores, and `base` for the tasks after them.
  MONO_DEV bool scores() {
    if (A.rows * CH > G) {
      if (!score_run()) return false;
    } else {
      // a workgroup for every chunk of max_ctx: chunk b, with no look at the other rows'
      // lengths in front of its loads (a round trip, ~1 us at 8 rows)
      base = n_score();
      if (kLongSplits) plan_splits();
      const int b = block_index();
      if (b < A.rows * CH) {
        const int s = b / CH, c = b % CH, n = row_len(s);
        if (c < live_chunks(n) && !score_one(s, c, n)) return false;  // workgroup-uniform
      }
    }
    __syncthreads();  // the top-k tasks reuse the LDS
    return true;
  }

  MONO_DEV bool score_one(int s, int c, int n) {
    const uint64_t t0 = now_ticks();
    const Lane z = lane_now();
    if (tid < 256) L.u.sc.hist[tid] = 0u;
    const int k0 = c * CHUNK + z.wave * KEYS_WAVE;
    int pg[KEYS_WAVE / PAGE];
#pragma unroll
    for (int i = 0; i < KEYS_WAVE / PAGE; ++i) pg[i] = page_of(s, min(k0 + i * PAGE, n - 1));
    Query q;
    Keys k;
    if (!front_here()) query_load(s, q);
    const Pages p = pages(pg, true);
    const bool fr = fresh(k0, n);
    if (!fr) key_load(z, k, p);
    if (front_here()) {
      if (!await_front()) return false;
      if (fr) key_load(z, k, p);
      query_load(s, q);
    } else {
      __syncthreads();  // the histogram is cleared
    }
    float sc[2];
    chunk_scores<false>(z, q, k, p, sc);
    chunk_store(z, s, c, n, sc);
    row_flush(s, c, 1);
    stamp(s * CH + c, t0, 0);
    return true;
  }

  // The step's scored chunks, row by row, in contiguous runs of equal length (a chunk a
  // workgroup while they last): every CU streams the same share whatever the rows'
  // lengths, and a run pays the histogram's flush, its acknowledgement and the query once
  // a row. Each chunk's keys are loaded two chunks ahead, so 64 to 128 KB a CU stay in
  // flight and no wait drains them but a row's flush. Chunks dealt round-robin over
  // max_ctx left three quarters of the grid idle at 33 rows of 1500-12000 keys (scores
  // done after 22.4 us, now 6.0; the launch 63.6 -> 51.6), and each chunk's own flush
  // drained its successor's loads (48 rows of 32768: 31.2 us, 3.4 TB/s, now 23.9, 4.5;
  // the launch 76.0 -> 70.5).
  MONO_DEV bool score_run() {
    ScoreLds& P = L.u.sc;
    const int nl = row_n;
    const int inc = wave_incl_scan(live_chunks(nl));
    const int total = __builtin_amdgcn_readlane(inc, WAVE - 1), b = block_index();
    base = (min(total, G) + TMK - 1) / TMK * TMK;
    int i0 = total > G ? (int)((int64_t)b * total / G) : min(b, total);
    const int i1 = total > G ? (int)((int64_t)(b + 1) * total / G) : min(b + 1, total);
    if (i0 >= i1) {  // workgroup-uniform
      if (kLongSplits) plan_splits();
      return true;
    }
    if (tid < 256) P.hist[tid] = 0u;
    // row s of scored chunk i, and the row's first one
    const auto row_at = [inc](int i) { return (int)__popcll(__ballot(inc <= i)); };
    const auto first_of = [inc](int s) { return s > 0 ? __builtin_amdgcn_readlane(inc, s - 1) : 0; };
    bool awaited = !front_here(), planned = !kLongSplits;
#pragma unroll 1
    for (; i0 < i1; i0 += RUN) {
      const Lane z = lane_now();
      const int m = min(i1 - i0, RUN);  // chunks of this piece
      __syncthreads();  // the piece before is done with the LDS; the histogram is cleared
      bool lead = false;
      int s = 0;
      if (z.wave < m) {  // wave w looks up chunk w
        s = row_at(i0 + z.wave);
        const int f = first_of(s), n = __builtin_amdgcn_readlane(nl, s);
        const int p0 = (i0 + z.wave - f) * CHUNK + (z.lane % (CHUNK / PAGE)) * PAGE;
        const int pg = page_of(s, min(p0, n - 1));
        lead = z.wave == 0 || f == i0 + z.wave;  // wave-uniform: the row's first chunk of the piece
        if (awaited && lead) run_query(z, s);
        if (z.lane < CHUNK / PAGE) P.pg[z.wave][z.lane] = pg;
      }
      __syncthreads();
      const auto pages_of = [&](const Lane& z, int j) {
        int pg[KEYS_WAVE / PAGE];
#pragma unroll
        for (int i = 0; i < KEYS_WAVE / PAGE; ++i) pg[i] = P.pg[min(j, m - 1)][z.wave * (KEYS_WAVE / PAGE) + i];
        return pages(pg, j < m);
      };
      Keys ka, kb;
      if (awaited) {
        key_load(z, ka, pages_of(z, 0));
        key_load(z, kb, pages_of(z, 1));
      } else {
        const auto fresh_at = [&](int j) {
          const int sj = row_at(i0 + min(j, m - 1));
          return fresh((i0 + j - first_of(sj)) * CHUNK + z.wave * KEYS_WAVE, __builtin_amdgcn_readlane(nl, sj));
        };
        const bool fa = fresh_at(0), fb = fresh_at(1);
        if (!fa) key_load(z, ka, pages_of(z, 0));
        if (!fb) key_load(z, kb, pages_of(z, 1));
        if (!await_front()) return false;
        awaited = true;
        if (lead) run_query(z, s);
        if (fa) key_load(z, ka, pages_of(z, 0));
        if (fb) key_load(z, kb, pages_of(z, 1));
        __syncthreads();
      }
      if (!planned) plan_splits();
      planned = true;
      Query q;
      int n = 0, c = -1, c0 = 0;
      const auto turn = [&](Keys& k, int j) {  // chunk j of the piece
        const uint64_t t0 = now_ticks();
        const Lane z = lane_now();
        if (c < 0) {  // the row's first chunk of the piece
          s = row_at(i0 + j);
          n = __builtin_amdgcn_readlane(nl, s);
          c = c0 = i0 + j - first_of(s);
          query_from(z, j, q);
        }
        float sc[2];
        chunk_scores<true>(z, q, k, pages_of(z, j + 2), sc);
        chunk_store(z, s, c, n, sc);
        const bool last = j + 1 == m || (c + 1) * CHUNK >= n;
        if (last) row_flush(s, c0, c + 1 - c0);
        stamp(s * CH + c, t0, 0);
        c = last ? -1 : c + 1;
      };
#pragma unroll 1
      for (int j = 0; j < m; j += 2) {
        turn(ka, j);
        if (j + 1 == m) break;
        turn(kb, j + 1);
      }
    }
    return true;
  }
  // Row s's query into the wave's LDS slot, and from slot j into a wave's operands.
  MONO_DEV void run_query(const Lane& z, int s) {
    ScoreLds& P = L.u.sc;
    constexpr int N = IH * ID / 32 / WAVE;
    u32x4 v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = ld_u32x4(A.iq + (size_t)s * (IH * ID / 2) + (WAVE * i + z.lane) * 16);
    const uint32_t qs = *reinterpret_cast<const uint32_t*>(A.iqs + ((size_t)s * IH + z.lane) * (ID / 32));
    const u32x2 w = *reinterpret_cast<const u32x2*>(A.iw + (size_t)s * IH + z.lane % (IH / 4) * 4);
#pragma unroll
    for (int i = 0; i < N; ++i) P.q[z.wave][WAVE * i + z.lane] = v[i];
    P.qs[z.wave][z.lane] = qs;
    if (z.lane < IH / 4) P.qw[z.wave][z.lane] = w;
  }
  MONO_DEV void query_from(const Lane& z, int j, Query& o) const {
    const ScoreLds& P = L.u.sc;
#pragma unroll
    for (int ht = 0; ht < IH / 16; ++ht) {
      o.qa[ht] = P.q[j][(16 * ht + z.r) * (ID / 32) + z.g];
      o.qsc[ht] = (int)((P.qs[j][16 * ht + z.r] >> (8 * z.g)) & 0xffu);
      const u32x2 w4 = P.qw[j][4 * ht + z.g];
      o.w2[ht][0] = w4[0];
      o.w2[ht][1] = w4[1];
    }
  }

  // ---------------------------------------------------------------- top-k
  // exclusive prefix sum of v over the workgroup (a full barrier)
  MONO_DEV int block_excl_scan(int v) {
    int total;
    return block_excl_scan(v, total);
  }
  MONO_DEV int block_excl_scan(int v, int& total) {
    const int incl = wave_incl_scan(v);
    if (lane == WAVE - 1) L.scan[wave] = incl;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < AW; ++w) {
      before += w < wave ? L.scan[w] : 0;
      total += L.scan[w];
    }
    __syncthreads();
    return before + incl - v;
  }

  MONO_DEV void publish_sel(int s, int j, int slot) {
    mb_put(&A.mail.sel[(size_t)s * TOPK + j], (uint32_t)slot, gd.tag);
    if (A.topk) A.topk[(size_t)s * TOPK + j] = slot;
  }

  // Count a key digit into an LDS histogram: the lanes sharing the first live lane's
  // digit (scores share sign and exponent bits, so leading digits pile onto few bins)
  // as one atomic, every other live lane as a plain atomic (the LDS resolves spread
  // addresses quickly; a wave of same-address atomics would serialize).
  MONO_DEV void hist_add(uint32_t* hist, bool live, uint32_t d) {
    const uint64_t act = __ballot(live);
    if (act == 0) return;  // wave-uniform
    if (__popcll(act) <= 16) {  // few live lanes (wave-uniform): plain atomics, no scalar chain
      if (live) atomicAdd(&hist[d], 1u);
      return;
    }
    const int first = __builtin_ctzll(act);
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, first);
    const uint64_t same = __ballot(live && d == d0);
    if (live && d != d0) atomicAdd(&hist[d], 1u);
    if (lane == first) atomicAdd(&hist[d0], (uint32_t)__popcll(same));
  }

  // Pick the next digit from a 256-bin histogram (wave 0): the highest digit d with
  // (keys above d) < need <= (keys above d) + hist[d] -> K.digit, K.above; with `pre`,
  // also K.pre_above = the sum of pre over the bins above d.
  MONO_DEV void pick_digit(TopkLds& K, const uint32_t* hist, int need, const uint32_t* pre) {
    if (wave != 0) return;
    int c[4], tot = 0;  // lane l holds bins 255 - 4l .. 252 - 4l, highest first
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      c[j] = (int)hist[255 - 4 * lane - j];
      tot += c[j];
    }
    const int incl = wave_incl_scan(tot);
    const int excl = incl - tot;
    const bool mine = excl < need && need <= incl;
    int dg = 0, ab = 0, run = excl;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (mine && dg == 0 && run + c[j] >= need) {
        dg = 256 + 255 - 4 * lane - j;  // + 256: found
        ab = run;
      }
      run += c[j];
    }
    const uint64_t who = __ballot(mine);
    const int src = who ? __ffsll((long long)who) - 1 : 0;
    dg = __builtin_amdgcn_readlane(dg, src) & 0xff;
    ab = __builtin_amdgcn_readlane(ab, src);
    if (pre) {
      int x = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) x += 255 - 4 * lane - j > dg ? (int)pre[255 - 4 * lane - j] : 0;
      x = wave_sum_i(x);
      if (lane == 0) K.pre_above = x;
    }
    if (lane == 0) {
      K.digit = (uint32_t)dg;
      K.above = ab;
    }
  }

  // This member's keys under `prefix` counted by the digit at `shift` into an LDS histogram:
  // plain atomics unless a quarter of the wave's first keys share the first lane's digit
  // (ties: their atomics would serialize; hist_add takes those together, by a scalar chain
  // a key: 8 rows of 32768 keys 31.9 -> 31.7 us a launch without it, 48 rows 71.1 -> 69.5)
  MONO_DEV void hist_keys(uint32_t* hist, const uint32_t (&key)[KPT], int cnt, uint32_t prefix, uint32_t mask, int shift) {
    cnt = opaque_v(cnt);  // (each pass over a thread's keys compares anew, see topk_member)
    const uint32_t first = (key[0] >> shift) & 0xffu;
    if (__popcll(__ballot(first == (uint32_t)__builtin_amdgcn_readfirstlane((int)first))) >= WAVE / 4) {  // wave-uniform
#pragma unroll
      for (int q = 0; q < KPT; ++q) hist_add(hist, q < cnt && (key[q] & mask) == prefix, (key[q] >> shift) & 0xffu);
    } else {
#pragma unroll
      for (int q = 0; q < KPT; ++q)
        if (q < cnt && (key[q] & mask) == prefix) atomicAdd(&hist[(key[q] >> shift) & 0xffu], 1u);
    }
  }

  // One exchanged radix pass: member m's histogram of the digit at `shift` over its keys
  // matching prefix under mask -> mailbox hist as 128 words of two 16-bit bins (a member
  // holds at most KPM keys), plus `count` as word 128 when count >= 0; the team's sum
  // -> K.tot, the sum over the members before m -> K.pre, the members' counts -> K.xw.
  // `lone`: the member holds the whole row. Workgroup-uniform result.
  MONO_DEV bool exchange_hist(int s, int m, bool lone, int pass, const uint32_t (&key)[KPT], int cnt, uint32_t prefix,
                              uint32_t mask, int shift, int count) {
    static_assert(KPM < 65536, "16-bit bins");
    TopkLds& K = L.u.t;
    if (tid < 256) K.hist[tid] = 0u;
    __syncthreads();
    hist_keys(K.hist, key, cnt, prefix, mask, shift);
    __syncthreads();
    if (lone) {  // team-uniform: nobody to exchange with
      if (tid < 256) {
        K.tot[tid] = K.hist[tid];
        K.pre[tid] = 0u;
      }
      __syncthreads();
      return true;
    }
    uint64_t* hb = &A.mail.hist[((size_t)s * PASSES + pass) * TMK * HW];
    bool ok = true;
    if (tid < 128) {
      mb_put(&hb[m * HW + tid], K.hist[2 * tid] | (K.hist[2 * tid + 1] << 16), gd.tag);
      uint32_t v[TMK];
      const uint64_t* col = hb + tid;
      const auto at = [col](int j) { return col + j * HW; };
      ok = poll_words<TMK, decltype(at), false>(at, v, (1u << TMK) - 1u, W_TEAM, gd);
      uint32_t t = 0, p = 0;  // two 16-bit sums side by side (at most TMK KPM keys)
#pragma unroll
      for (int j = 0; j < TMK; ++j) {
        t += v[j];
        p += j < m ? v[j] : 0u;
      }
      K.tot[2 * tid] = t & 0xffffu;
      K.tot[2 * tid + 1] = t >> 16;
      K.pre[2 * tid] = p & 0xffffu;
      K.pre[2 * tid + 1] = p >> 16;
    } else if (count >= 0 && tid < 128 + TMK) {
      const int j = tid - 128;
      if (j == m) mb_put(&hb[m * HW + 128], (uint32_t)count, gd.tag);
      uint32_t v = 0;
      ok = poll_word(&hb[j * HW + 128], v, W_TEAM, gd);
      K.xw[j] = (int)v;
    }
    return block_all(ok);
  }

  // a threshold candidate's rank word: larger first = score desc, position asc (the
  // candidates share their keys' upper 16 bits)
  MONO_DEV static uint32_t cand_word(uint32_t key, int pos) { return (key << 16) | (uint32_t)(0x7fff - pos); }

  // Member m of row s's top-k team. The team selects the exact top-TOPK of the row
  // (score desc, position asc) -> cache slots, ascending. Member m owns positions
  // [m KPM, (m + 1) KPM), KPT of them in each thread's registers. An MSB-first 8-bit
  // radix select of the threshold key: digit 1 from the score tasks' chunk histograms,
  // digit 2 from the members' exchanged histograms. The keys left sharing both digits
  // with the threshold (the candidates, few unless scores tie) are exchanged as (low
  // key bits, position) and every member ranks them all; a crowded threshold bin
  // instead takes digits 3 and 4 the same way as digit 2 and then the members' counts
  // above / at the threshold (mailbox cnt). Each member writes its selected slots at
  // its offset in position order. A row that its first member holds alone exchanges
  // nothing (33 rows of 1500-12000 keys: 4.3 us of 16.5 a lone member's selection took).
  MONO_DEV bool topk_member(int s, int m) {
    TopkLds& K = L.u.t;
    const int n = row_len(s);
    if (n <= TOPK) {  // every key is selected, in place (split_task); only a caller's copy is written here
      if (A.topk && m == 0)
        for (int j = tid; j < TOPK; j += AT) A.topk[(size_t)s * TOPK + j] = j < n ? slot_of(s, j) : -1;
      return true;
    }
    const bool lone = kStageSel && n <= KPM;
    if (lone && m > 0) return true;
    const int p0 = m * KPM + tid * KPT;
    const int cnt = min(max(n - p0, 0), KPT);
    const int page = cnt > 0 ? page_of(s, p0) : 0;  // a thread's keys share one page
    bool ok = true;
    // thread c < (scored chunks) waits for chunk c's scores and counts (done word)
    if (tid < (n + CHUNK - 1) / CHUNK) {
      uint32_t v;
      ok = poll_word(&A.mail.cdone[(size_t)s * CH + tid], v, W_SCORE, gd);
    }
    if (!block_all(ok)) return false;
    // then a thread's KPT consecutive scores: 16-byte device-coherent loads (the buffer
    // reads zeros past the row), and the row histogram
    uint32_t key[KPT];
    {
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc(A.mail.score + (size_t)s * A.mail.max_ctx, 0, n * 4, BUF_DWORD3);
      u32x4 k4[KPT / 4];
#pragma unroll
      for (int i = 0; i < KPT / 4; ++i)
        k4[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (p0 + 4 * i) * 4, 0, SC1));
#pragma unroll
      for (int q = 0; q < KPT; ++q) key[q] = radix_key(__uint_as_float(k4[q / 4][q % 4]));
    }
    if (tid < 256) K.tot[tid] = ld_agent_u32(&row_hist(gd.tag, s)[tid]);
    __syncthreads();
    mark_waited();
    pick_digit(K, K.tot, TOPK, nullptr);
    __syncthreads();
    int need = TOPK - K.above;
    const uint32_t d1 = K.digit;
    uint32_t prefix = d1 << 24, mask = 0xff000000u;
    // Each pass over a thread's keys compares its positions and keys anew (opaque copies):
    // shared between the passes, KPT lane masks a comparison would be held in scalar
    // registers and spilled
    int above1 = 0;  // this member's keys above digit 1
    {
      const int cn = opaque_v(cnt);
#pragma unroll
      for (int q = 0; q < KPT; ++q) above1 += (q < cn && (key[q] >> 24) > d1) ? 1 : 0;
    }
    above1 = wave_sum_i(above1);
    if (lane == 0) L.scan[wave] = above1;
    __syncthreads();
    above1 = 0;
#pragma unroll
    for (int w = 0; w < AW; ++w) above1 += L.scan[w];
    if (!exchange_hist(s, m, lone, 1, key, cnt, prefix, mask, 16, above1)) return false;
    pick_digit(K, K.tot, need, K.pre);
    __syncthreads();
    need -= K.above;
    int above_before = K.pre_above;  // the earlier members' keys above the threshold's upper 16 bits
    // a fixed trip count: the LDS reads issue together (a loop to m waits on each one;
    // 0.4-0.5 us of the top-k at 1 and 8 rows)
#pragma unroll
    for (int j = 0; j < TMK; ++j) above_before += j < m ? K.xw[j] : 0;
    prefix |= K.digit << 16;
    mask |= 0x00ff0000u;
    const int n_cand = (int)K.tot[K.digit], cand_before = (int)K.pre[K.digit];
    int sel_before;
    uint32_t uT = 0;  // candidates: the lowest selected rank word
    bool cand = n_cand <= CMAX;  // team-uniform
    if (cand) {
      const uint32_t P16 = prefix >> 16;
      int c_my = 0;
      {
        const int cn = opaque_v(cnt);
#pragma unroll
        for (int q = 0; q < KPT; ++q) c_my += (q < cn && (key[q] >> 16) == P16) ? 1 : 0;
      }
      static_assert(CMAX == AT, "a thread a candidate");
      if (lone) K.cu[tid] = 0u;
      int idx = cand_before + block_excl_scan(c_my);
      uint64_t* cb = &A.mail.cand[(size_t)s * CMAX];
      uint32_t u = 0;
      ok = true;
      const int cn = opaque_v(cnt);
      const uint32_t P16b = (uint32_t)opaque_v((int)P16);
      if (lone) {
#pragma unroll
        for (int q = 0; q < KPT; ++q)
          if (q < cn && (key[q] >> 16) == P16b) K.cu[idx++] = cand_word(key[q], p0 + q);
        __syncthreads();
        u = K.cu[tid];
      } else {
#pragma unroll
        for (int q = 0; q < KPT; ++q)
          if (q < cn && (key[q] >> 16) == P16b) mb_put(&cb[idx++], cand_word(key[q], p0 + q), gd.tag);
        if (tid < n_cand) ok = poll_word(&cb[tid], u, W_TEAM, gd);
        K.cu[tid] = u;
        if (!block_all(ok)) return false;
      }
      if (wave * WAVE < n_cand) {  // wave-uniform
        // candidates ranked before this thread's, 32 a step with the step's LDS reads issued
        // together (K.cu holds zeros past the last candidate, and a step starting below
        // n_cand <= CMAX ends inside K.cu)
        static_assert(CMAX % 32 == 0, "whole steps");
        int rank = 0;
        for (int j = 0; j < n_cand; j += 32) {
          u32x4 x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = *reinterpret_cast<const u32x4*>(&K.cu[j + 4 * i]);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            rank += (x[i][0] > u ? 1 : 0) + (x[i][1] > u ? 1 : 0) + (x[i][2] > u ? 1 : 0) + (x[i][3] > u ? 1 : 0);
        }
        if (tid < n_cand && rank == need - 1) K.uT = u;
      }
      __syncthreads();
      uT = K.uT;
      sel_before = above_before + __syncthreads_count(tid < cand_before && u >= uT);
    } else {
#pragma unroll 1
      for (int pass = 2; pass < PASSES; ++pass) {
        const int shift = 24 - 8 * pass;
        __syncthreads();  // K.digit and K.tot are read
        if (!exchange_hist(s, m, lone, pass, key, cnt, prefix, mask, shift, -1)) return false;
        pick_digit(K, K.tot, need, nullptr);
        __syncthreads();
        need -= K.above;
        prefix |= K.digit << shift;
        mask |= 0xffu << shift;
      }
      // the team's counts above / at T, then this member's offset
      int c_gt = 0, c_eq = 0;
#pragma unroll
      for (int q = 0; q < KPT; ++q) {
        c_gt += (q < cnt && key[q] > prefix) ? 1 : 0;
        c_eq += (q < cnt && key[q] == prefix) ? 1 : 0;
      }
      const int gt_in = block_excl_scan(c_gt), eq_in = block_excl_scan(c_eq);
      if (tid == AT - 1) {  // the last thread's inclusive sums are the member's totals
        mb_put(&A.mail.cnt[((size_t)s * TMK + m) * 2], (uint32_t)(gt_in + c_gt), gd.tag);
        mb_put(&A.mail.cnt[((size_t)s * TMK + m) * 2 + 1], (uint32_t)(eq_in + c_eq), gd.tag);
      }
      ok = true;
      if (tid < 2 * (lone ? 1 : TMK)) {
        uint32_t v = 0;
        ok = poll_word(&A.mail.cnt[(size_t)s * TMK * 2 + tid], v, W_TEAM, gd);
        K.cnt[tid / 2][tid % 2] = (int)v;
      }
      if (!block_all(ok)) return false;
      int eq_before = 0;  // over the members before m, in position order
      sel_before = 0;
      for (int j = 0; j < m; ++j) {
        const int take_j = min(max(need - eq_before, 0), K.cnt[j][1]);
        sel_before += K.cnt[j][0] + take_j;
        eq_before += K.cnt[j][1];
      }
      // this thread's share of the keys equal to T: the lowest positions first
      uT = (uint32_t)min(max(need - (eq_before + eq_in), 0), c_eq);
    }
    // the selected keys in position order: above the threshold prefix, and the
    // threshold's share (candidates ranked at or above uT / the first uT equal to T)
    uint32_t take = 0;  // bit q: key q is selected
    {
      const int cn = opaque_v(cnt);
      if (cand) {
#pragma unroll
        for (int q = 0; q < KPT; ++q) {
          const uint32_t hi = key[q] >> 16, P16 = prefix >> 16;
          const bool t = q < cn && (hi > P16 || (hi == P16 && cand_word(key[q], p0 + q) >= uT));
          take |= t ? 1u << q : 0u;
        }
      } else {
        int te = 0;
#pragma unroll
        for (int q = 0; q < KPT; ++q) {
          const bool eq = q < cn && key[q] == prefix;
          const bool t = (q < cn && key[q] > prefix) || (eq && te < (int)uT);
          te += eq ? 1 : 0;
          take |= t ? 1u << q : 0u;
        }
      }
    }
    const int c_take = __popc(take);
    if (kStageSel) {
      int n_sel;
      int idx = block_excl_scan(c_take, n_sel);
#pragma unroll
      for (int q = 0; q < KPT; ++q)
        if ((take >> q & 1u) && idx < TOPK) K.sl[idx++] = page * PAGE + (p0 + q) % PAGE;
      __syncthreads();
      for (int j = tid; j < n_sel && sel_before + j < TOPK; j += AT) publish_sel(s, sel_before + j, K.sl[j]);
      __syncthreads();  // the next task may rewrite the LDS
    } else {
      int idx = sel_before + block_excl_scan(c_take);
      // (a key not taken stores past the row's words: the buffer drops it, no branch a key;
      // 8 rows of 32768 keys: 31.4 -> 31.3 us a launch)
      const __amdgpu_buffer_rsrc_t rs = coherent_rsrc(A.mail.sel + (size_t)s * TOPK, TOPK * 8);
#pragma unroll
      for (int q = 0; q < KPT; ++q) {
        const bool t = take >> q & 1u;
        const u32x2 w = {(uint32_t)(page * PAGE + (p0 + q) % PAGE), gd.tag};
        __builtin_amdgcn_raw_buffer_store_b64(w, rs, t ? idx * 8 : TOPK * 8, 0, SC1);
        if (A.topk && t && idx < TOPK) A.topk[(size_t)s * TOPK + idx] = (int)w[0];
        idx += t ? 1 : 0;
      }
    }
    return true;
  }

  // ---------------------------------------------------------------- split
  // A thread's share of a sub-tile's rows: value chunk c = tid % 32 (dims 16 c .. 16 c +
  // 15) of the 4 tokens 4 m .. 4 m + 3, m = tid / 32 (a wave's load covers 512
  // contiguous bytes of each of 2 rows), and (the first SUB x ROPE_CH threads) one
  // 16-byte chunk past the value dims; the scale of token tid % SUB.
  struct Gather {
    u32x4 v[4];
    u32x4 rope;
    float sc;
  };

  // Issue sub-tile st's cache-row loads. Every load is unconditional (an empty slot reads
  // row 0, zeroed at the store): a load under a condition is waited for at the join,
  // which would serialize the gather's round trips.
  MONO_DEV void gather_load(const SplitLds& P, int st, Gather& gt) {
#pragma unroll
    for (int part = 0; part < 3; ++part) gather_load_part(P, st, gt, part);
  }
  // part 0: value chunks of tokens 4 m, 4 m + 1; part 1: of 4 m + 2, 4 m + 3; part 2: the
  // chunk past the value dims and the scale (a long split issues the next sub-tile's
  // parts between its phases, so no wave stalls in one burst)
  MONO_DEV void gather_load_part(const SplitLds& P, int st, Gather& gt, int part) {
    const int c = tid % (DV / 16), m = tid / (DV / 16);
    const int32_t* sl = P.slot + st * SUB;
    if (part < 2) {
#pragma unroll
      for (int k = 2 * part; k < 2 * part + 2; ++k)
        gt.v[k] = ld_nt_u32x4(A.kv + (size_t)max(sl[4 * m + k], 0) * DQK + 16 * c);
    } else {
      const int f = min(tid, ROPE_CH * SUB - 1);
      gt.rope = ld_nt_u32x4(A.kv + (size_t)max(sl[f / ROPE_CH], 0) * DQK + DV + 16 * (f % ROPE_CH));
      gt.sc = A.kv_scale[max(sl[tid % SUB], 0) & A.kv_mask];
    }
  }

  // Every slot of sub-tile st is a cached row (wave-uniform): no row to clear, no token to
  // leave out (all but a row's last sub-tile; 30 of a thread's ~400 VALU a sub-tile).
  MONO_DEV bool sub_full(const SplitLds& P, int st) const { return __ballot(P.slot[st * SUB + lane] < 0) == 0; }

  // Store sub-tile st's rows into its buffer as they lie, the rows of empty slots as
  // zeros, and its scales. One copy serves q.k and p.v: a second, widened and transposed
  // one (64 KB of LDS stores, 64 VALU a thread and two more barriers a sub-tile) put 0.7
  // us on the chain of a one-sub-tile split (one row of 700 keys: 13.2 -> 12.5 us a launch).
  MONO_DEV void gather_store(SplitLds& P, int st, const Gather& gt) {
    if (sub_full(P, st))
      gather_store_rows<true>(P, st, gt);
    else
      gather_store_rows<false>(P, st, gt);
  }
  template <bool FULL>
  MONO_DEV void gather_store_rows(SplitLds& P, int st, const Gather& gt) {
    const int c = tid % (DV / 16), m = tid / (DV / 16);
    const int32_t* sl = P.slot + st * SUB;
    u32x4(*kf)[KF_W / 4] = P.kf16[st % 2];
#pragma unroll
    for (int k = 0; k < 4; ++k) kf[4 * m + k][c] = FULL || sl[4 * m + k] >= 0 ? gt.v[k] : u32x4{0u, 0u, 0u, 0u};
    if (tid < ROPE_CH * SUB) {
      const int t = tid / ROPE_CH;
      kf[t][DV / 16 + tid % ROPE_CH] = FULL || sl[t] >= 0 ? gt.rope : u32x4{0u, 0u, 0u, 0u};
    }
    if (tid < SUB) P.kvs[st % 2][tid] = FULL || sl[tid] >= 0 ? gt.sc : 0.f;
  }

  // Split j of row s: its selected tokens lo .. lo + len - 1 (whole sub-tiles of SUB). LONG:
  // a split may hold several sub-tiles.
  template <bool LONG>
  MONO_DEV bool split_task(int s, int j, int lo, int len) {
    SplitLds& P = L.u.sp;
    const int n = row_len(s);
    const int cnt = min(max(min(n, TOPK) - lo, 0), len);
    const size_t mlb = ((size_t)s * SPLITS + j) * NH;
    if (cnt == 0) {  // an empty split contributes nothing to the merge
      if (tid < NH) {
        st_agent_f32(&A.mail.ml[(mlb + tid) * 2], NEG_INF);
        st_agent_f32(&A.mail.ml[(mlb + tid) * 2 + 1], 0.f);
      }
      split_done(s, j);
      return true;
    }
    if (front_here() && !q_ready) {
      // every head of q from the front of this launch, and every row's cache row (a row that
      // selects all its keys waits for no scores, which would follow them)
      const uint64_t* fd = done_copy(front_done());
      if (!hint_wait(NH + A.rows, [fd](int i) { return fd + (i < NH ? proj::FD_D + i : proj::FD_B + i - NH); },
                     front_site() + 1, gd))
        return false;
      q_ready = true;
    }
    {
      constexpr int QN = NH * DQK / 8, QL = (QN + AT - 1) / AT;
      u32x4 qv[QL];
#pragma unroll
      for (int i = 0; i < QL; ++i) qv[i] = ld_u32x4(A.q + (size_t)s * NH * DQK + (size_t)min(tid + i * AT, QN - 1) * 8);
#pragma unroll
      for (int i = 0; i < QL; ++i) {
        const int f = tid + i * AT;  // unconditional loads (see gather_load), guarded stores
        if (f < QN) P.q16[f / (DQK / 8)][f % (DQK / 8)] = qv[i];
      }
    }
    bool ok = true;
    if (tid < len) {
      int slot = -1;
      if (tid < cnt && n <= TOPK) {
        // every key of the row is selected: no selection to wait for (one row of 700 keys:
        // 12.3 -> 11.9 us a launch)
        slot = slot_of(s, lo + tid);
      } else if (tid < cnt) {
        uint32_t v = 0;
        ok = poll_word(&A.mail.sel[(size_t)s * TOPK + lo + tid], v, W_SEL, gd);
        slot = (int)v;
        if (slot < 0 || slot >= A.n_pages * PAGE) slot = -1;
      }
      P.slot[tid] = slot;
    }
    if (!block_all(ok)) return false;
    mark_waited();

    // p.v of wave w: dims 64 w + 16 b + [0, 16) (b = 0..3) x heads 16 a + [0, 16) (a = 0, 1);
    // lane (g, r) holds dims 64 w + 16 b + 4 g + i of head 16 a + r. Softmax: each
    // 16-lane row of the workgroup one head (tid / 16), a lane 4 tokens; the head's
    // running maximum and sum (every lane of the row holds them).
    f32x4 acc[4][2];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) acc[b][a] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = NEG_INF, l_run = 0.f;
    const int nsub = (cnt + SUB - 1) / SUB;
    Gather gt;
    gather_load(P, 0, gt);
    // q.k of wave (kh, tt): dims QK_HALF kh .. of tokens 16 tt .. 16 tt + 15 against every
    // head; its q operands (heads 16 a + r, 8 dims a k step) held in registers
    bf16x8 qa[2][QK_STEPS];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int ks = 0; ks < QK_STEPS; ++ks)
        qa[a][ks] = __builtin_bit_cast(bf16x8, P.q16[16 * a + r][QK_HALF / 8 * (wave / 4) + 4 * ks + g]);
    gather_store(P, 0, gt);
    __syncthreads();
    if (LONG && nsub > 1) gather_load(P, 1, gt);

#pragma unroll 1
    for (int st = 0; st < nsub; ++st) {
      // a long split: the lane's indices afresh each sub-tile (opaque copies), so the q.k,
      // softmax and p.v LDS addresses are derived inside the loop, not hoisted out of it
      // and held across it
      const int lane = LONG ? opaque_v(tid) % WAVE : this->lane, g = lane / 16, r = lane % 16;
      const int wv = LONG ? opaque_v(tid) / WAVE : wave;
      const int buf = LONG ? st % 2 : 0;
      const bool next = LONG && st + 1 < nsub, next2 = LONG && st + 2 < nsub;
      // logits, transposed: A = 16 cached rows (FP8, widened in registers), B = 16 heads
      // of q; lane (g, r) ends with tokens 16 tt + 4 g + i of head 16 a + r
      {
        const u32x2* krow = &P.kf8[buf][16 * (wv % 4) + r][QK_HALF / 8 * (wv / 4) + g];
        u32x2 kw[QK_STEPS];
#pragma unroll
        for (int ks = 0; ks < QK_STEPS; ++ks) kw[ks] = krow[4 * ks];
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int ks = 0; ks < QK_STEPS; ++ks) {
          const bf16x8 ka = fp8x8_bf16x8(kw[ks]);
          s0 = mfma_bf16(ka, qa[0][ks], s0);
          s1 = mfma_bf16(ka, qa[1][ks], s1);
        }
        P.pf4[wv / 4][r][4 * (wv % 4) + g] = s0;
        P.pf4[wv / 4][16 + r][4 * (wv % 4) + g] = s1;
      }
      __syncthreads();
      // online softmax: head tid / 16, tokens 4 (tid % 16) .. + 3; the head's reductions
      // inside the lane's 16-lane row (DPP)
      {
        const int ti = LONG ? opaque_v(tid) : tid, h = ti / 16, tq = ti % 16;
        const f32x4 x0 = P.pf4[0][h][tq], x1 = P.pf4[1][h][tq], ks = P.kvs4[buf][tq];
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = (x0[i] + x1[i]) * (ks[i] * A.scale);
        if (!sub_full(P, st)) {
          const i32x4 sl = P.slot4[st * (SUB / 4) + tq];
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = sl[i] >= 0 ? x[i] : NEG_INF;
        }
        float mx = row_reduce<16>(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), OpMax());
        if (LONG) mx = fmaxf(m_run, mx);
        float pr[4], ps = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pr[i] = (mx == NEG_INF || x[i] == NEG_INF) ? 0.f : hw_exp(x[i] - mx);
          ps += pr[i];
        }
        ps = row_reduce<16>(ps, OpAdd());
        const float al = m_run == NEG_INF ? (mx == NEG_INF ? 1.f : 0.f) : hw_exp(m_run - mx);
        l_run = LONG ? l_run * al + ps : ps;
        m_run = mx;
        P.pb8[h][tq] = u32x2{pack_bf16x2(pr[0] * ks[0], pr[1] * ks[1]), pack_bf16x2(pr[2] * ks[2], pr[3] * ks[3])};
        if (LONG && tq == 0) P.alpha[h] = al;
      }
      // the next sub-tile's rows into the other buffer (its last readers, the p.v of the
      // sub-tile before, are behind this phase's first barrier) and the rows after them
      // on their way, in three parts, so no wave stalls in one issue burst
      if (next) gather_store(P, st + 1, gt);
      if (next2) gather_load_part(P, st + 2, gt, 0);
      __syncthreads();
      if (next2) gather_load_part(P, st + 2, gt, 1);
      // o^T[dims x heads] = alpha o^T + v^T p^T: A = 16 dims of the values, read transposed
      // (a 16-lane group reads 8 tokens x 16 dims, two lanes a token, and each lane gets
      // one dim of the 8 tokens) and widened, B = 16 heads' probabilities, k = 32 tokens
      // a step
      {
        if (LONG) {
          float alh[2];
#pragma unroll
          for (int a = 0; a < 2; ++a) alh[a] = P.alpha[16 * a + r];
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
              for (int i = 0; i < 4; ++i) acc[b][a][i] *= alh[a];
        }
#pragma unroll
        for (int kt = 0; kt < SUB / 32; ++kt) {
          bf16x8 pv[2], va[4];  // every operand of the k step read before its MFMAs
#pragma unroll
          for (int a = 0; a < 2; ++a) pv[a] = __builtin_bit_cast(bf16x8, P.pb16[16 * a + r][4 * kt + g]);
#pragma unroll
          for (int b = 0; b < 4; ++b)
            va[b] = fp8x8_bf16x8(lds_tr8(&P.kf8[buf][32 * kt + 8 * g + r / 2][8 * wv + 2 * b + r % 2]));
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a) acc[b][a] = mfma_bf16(va[b], pv[a], acc[b][a]);
        }
      }
      if (next2) gather_load_part(P, st + 2, gt, 2);
      // (no barrier: the next q.k reads the other buffer and writes the logits, read
      // before this phase's barrier)
    }
    // the partials (bf16, the reference's split partials, kernel.py:4040-4066) staged as
    // [head][dim] in LDS (a lane's 4 consecutive dims of a head as 8 bytes), then stored
    // as the split's contiguous 32 KB by 16-byte device-coherent stores (whole lines);
    // then (m, l); then the split's done word
    // (a head's row padded by 16 bytes: the 16 heads of a lane group's store fall on
    // distinct banks)
    constexpr int OT_ROW = DV / 8 + 1;  // 16-byte units a staged head row
    // the buffer that the last sub-tile does not use (its readers are two barriers back)
    u32x2* ot = &P.ot[LONG ? nsub % 2 : 1][0][0];
    static_assert(sizeof(P.ot[0]) >= NH * OT_ROW * 16, "partial staging");
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const u32x2 o = {pack_bf16x2(acc[b][a][0], acc[b][a][1]), pack_bf16x2(acc[b][a][2], acc[b][a][3])};
        ot[(16 * a + r) * 2 * OT_ROW + (64 * wave + 16 * b + 4 * g) / 4] = o;
      }
    __syncthreads();
    {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          A.mail.part + ((size_t)s * SPLITS + j) * NH * DV, 0, NH * DV * 2, BUF_DWORD3);
      const u32x4* ot16 = &P.kf16[LONG ? nsub % 2 : 1][0][0];
      constexpr int CH16 = NH * DV * 2 / 16;  // 16-byte chunks of the split's partials
#pragma unroll
      for (int q = 0; q < CH16 / AT; ++q) {
        const int c = tid + AT * q;
        __builtin_amdgcn_raw_buffer_store_b128(ot16[(c / (DV / 8)) * OT_ROW + c % (DV / 8)], rs, 16 * c, 0, SC1);
      }
    }
    if (tid % 16 == 0) {
      st_agent_f32(&A.mail.ml[(mlb + tid / 16) * 2], m_run);
      st_agent_f32(&A.mail.ml[(mlb + tid / 16) * 2 + 1], l_run);
    }
    split_done(s, j);  // its barrier also frees the LDS for the next task
    return true;
  }

  // every store of the split performed (each thread waits for its own), then its done word
  MONO_DEV void split_done(int s, int j) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) mb_put(&A.mail.sdone[(size_t)s * SPLITS + j], 0u, gd.tag);
  }

  // ---------------------------------------------------------------- merge
  // This workgroup's merges: list index `at` + k (timeline row tl + k) is merge k (row
  // k / (32 / HM), heads (k % (32 / HM)) HM ..), HM heads a task.
  template <int HM>
  MONO_DEV bool merges(int at, int tl) {
    constexpr int MPR = NH / HM;  // merges a row
    const int n = A.rows * MPR;
    for (int T = first_at_or_after(at); T < at + n; T += G) {
      const uint64_t t0 = now_ticks();
      const int k = T - at, s = k / MPR;
      const bool ok = merge_task<HM>(s, k % MPR, kLongSplits ? first_split(s + 1) - first_split(s) : SPLITS);
      stamp(tl + k, t0, 3);
      if (!ok) return false;
    }
    return true;
  }

  // N dwords at uniform offset `u` plus lane offset `v` of a device-coherent resource
  template <int N>
  MONO_DEV static void load_words(__amdgpu_buffer_rsrc_t rs, int v, int u, uint32_t (&w)[N]) {
    if constexpr (N == 4) {
      const u32x4 x = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, v, u, SC1));
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = x[i];
    } else if constexpr (N == 2) {
      const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, v, u, SC1));
      w[0] = x[0];
      w[1] = x[1];
    } else {
      static_assert(N == 1, "4, 8 or 16 bytes");
      w[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(rs, v, u, SC1));
    }
  }

  // Merge (row s, heads hg HM .. hg HM + HM - 1) over the row's nsp splits: each thread
  // combines CPT consecutive channels of a head, BATCH splits at a time (a task takes in
  // nsp x HM KB of partials, by loads of up to 16 bytes).
  template <int HM>
  MONO_DEV bool merge_task(int s, int hg, int nsp) {
    constexpr int CPT = HM > 2 ? HM : 2;  // channels a thread
    constexpr int BATCH = kLongSplits ? 8 : SPLITS;
    static_assert(SPLITS <= WAVE && HM <= AW && HM <= 8 && HM * DV / CPT <= AT && NH % HM == 0,
                  "a lane a split; a wave a head's weights");
    MergeLds& Q = L.u.mg;
    const int h0 = hg * HM;
    const size_t rb = (size_t)s * SPLITS;
    // every split of the row done: lane j of wave 0 polls split j's word
    bool ok = true;
    if (wave == 0 && lane < nsp) {
      uint32_t v;
      ok = poll_word(&A.mail.sdone[rb + lane], v, W_PART, gd);
    }
    if (!block_all(ok)) return false;
    mark_waited();
    // the split weights: wave w takes head h0 + w, lane j split j (0 past the last)
    if (wave < HM) {
      const int h = h0 + wave;
      const int jl = max(min(lane, nsp - 1), 0);
      const float m = ld_agent_f32(&A.mail.ml[((rb + jl) * NH + h) * 2]);
      const float l = lane < nsp ? ld_agent_f32(&A.mail.ml[((rb + jl) * NH + h) * 2 + 1]) : 0.f;
      const bool live = l > 0.f;
      const float M = wave_max(live ? m : NEG_INF);
      const float w = live ? hw_exp(m - M) : 0.f;
      const float den = wave_sum(w * l);
      if (lane < SPLITS) Q.w[wave][lane] = w;
      if (lane == 0) Q.den[wave] = den;
    }
    // the channels of the batch's splits (unconditional loads; an empty split's words are
    // read and ignored)
    const int c0 = tid * CPT, hh = c0 / DV;  // channel of the task's HM heads, its head
    const bool mine = c0 < HM * DV;          // wave-uniform
    const __amdgpu_buffer_rsrc_t rs = coherent_rsrc(A.mail.part + rb * NH * DV, SPLITS * NH * DV * 2);
    float o[CPT];
#pragma unroll
    for (int i = 0; i < CPT; ++i) o[i] = 0.f;
    uint32_t av[BATCH][CPT / 2];
    const auto load = [&](int j0) {
#pragma unroll
      for (int j = 0; j < BATCH; ++j) {
        const int jl = kLongSplits ? max(min(j0 + j, nsp - 1), 0) : j;
        load_words(rs, c0 * 2, (jl * NH + h0) * DV * 2, av[j]);
      }
    };
    const auto add = [&](int j0) {
#pragma unroll
      for (int j = 0; j < BATCH; ++j) {
        const float w = Q.w[hh][j0 + j];
        if (w > 0.f)
#pragma unroll
          for (int i = 0; i < CPT / 2; ++i) {
            o[2 * i] += w * bf16_lo(av[j][i]);
            o[2 * i + 1] += w * bf16_hi(av[j][i]);
          }
      }
    };
    if (mine) load(0);
    __syncthreads();
    if (mine) {
      add(0);
      if (kLongSplits)
#pragma unroll 1
        for (int j0 = BATCH; j0 < nsp; j0 += BATCH) {
          load(j0);
          add(j0);
        }
      const float den = Q.den[hh];
      const float inv = den > 0.f ? 1.0f / den : 0.f;
      uint32_t* po = reinterpret_cast<uint32_t*>(A.out + ((size_t)s * NH + h0) * DV + c0);
#pragma unroll
      for (int i = 0; i < CPT / 2; ++i) {
        const uint32_t ov = pack_bf16x2(o[2 * i] * inv, o[2 * i + 1] * inv);
        if (A.publish_out) {  // read in this launch: a device-coherent store, complete before the done word
          __hip_atomic_store(po + i, ov, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          po[i] = ov;
        }
      }
      if (A.publish_out) __builtin_amdgcn_s_waitcnt(0);
    }
    __syncthreads();  // (and the next task may rewrite the LDS weights)
    if (A.publish_out && tid < HM) mb_put(&A.mail.mdone[(size_t)s * NH + h0 + tid], 0u, gd.tag);
    return true;
  }
};

// The kernel arguments of a launch (shared by k_attn and the fused attention + back).
void fill_args(Args& a, const AttnArgs& g, const Mail& mail, const GuardArgs& guard) {
  a.iq = static_cast<const uint8_t*>(g.iq);
  a.iqs = static_cast<const uint8_t*>(g.iqs);
  a.iw = static_cast<const uint16_t*>(g.iw);
  a.ikv = static_cast<const uint8_t*>(g.ikv);
  a.iks = static_cast<const uint8_t*>(g.iks);
  a.q = static_cast<const uint16_t*>(g.q);
  a.kv = static_cast<const uint8_t*>(g.kv);
  a.kv_scale = g.kv_scale;
  a.kv_mask = g.kv_mask;
  a.pt = g.page_table;
  a.seq_lens = g.seq_lens;
  a.pt_stride = g.pt_stride;
  a.n_pages = g.n_pages;
  a.out = static_cast<uint16_t*>(g.out);
  a.rows = g.rows;
  a.scores = g.scores;
  a.topk = g.topk;
  a.timeline = g.timeline;
  a.scale = g.softmax_scale;
  a.publish_out = false;
  a.rowh_flip = 1;
#ifdef MONO_ATTN_FRONT
  a.fdone = nullptr;
  a.fsite = 0;
#endif
  a.mail = mail;
  a.guard = guard;
}

}  // namespace
}  // namespace attn
}  // namespace mono
