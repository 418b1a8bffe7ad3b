// Chunked gated delta rule for few sequences: the state-independent work of
// every chunk in one parallel launch, then a recurrence with little left in
// its serial chain.
//
// The one-launch kernel (chunk_chain.hip) gives each (sequence, v-head,
// 64-column slice) a workgroup that forms the chunk's tiles itself: 2.3-2.4 us
// a chunk, whatever else runs, and one sequence of 32 heads occupies 64 of 256
// CUs.  With few sequences that serial time is all there is.  Here
//   * chunk_records_kernel forms, for every (chunk, v-head) at once, the parts
//     that do not depend on the state: the gate table, the solve's operands
//     A11, A22, -L21 and the masked tiles M, stored as MFMA fragments in the
//     order the recurrence reads them (1 KB per fragment, 16 bytes a lane);
//   * chunk_scan_kernel runs the recurrence.  A workgroup takes 16 state
//     columns of one (sequence, v-head) in six waves: the chain (P = K h, R,
//     the two-half solve, the state update), the output one chunk behind it
//     (o = scale (2^G q h + M v') from the chain's f16 state and v' operands,
//     handed over in LDS) and four that stage K, Q, V and the records, loaded
//     two chunks ahead.  One barrier per chunk.
// The operands, the order of every sum and the roundings are those of
// chunk_chain_kernel, so both give the same bits.
//
// Bound: the chain wave's dependent steps, 0.88 us a chunk with nothing else
// in the workgroup, and 1.22 us with the other waves' loads and LDS traffic
// beside it (LDS active 35 % of the cycles, no conflicts; deeper prefetch, a
// warmed L2 and tiles laid out contiguously for the staging waves changed
// nothing or cost their own writes).  With frame tables and a token log (EXT)
// 1.9 us a chunk: a checkpoint inside it, the v' rows' stores, and some 100 SGPR
// spills at d_k 128 (14 without EXT).  One sequence of 8192 tokens, 16 / 32 heads
// of 128: 165 us for both launches against 290 us in one; the prefill 312 -> 228
// us (with v written out by the front end), replayed from a graph.  16 columns a
// workgroup: 32 took 10 % longer for one sequence and gained only where the
// one-launch form is the better one anyway.
#include <type_traits>

#include "chunk_tile.hpp"

namespace gdn {
namespace {

// Record of one (chunk, v-head): A fragments, M fragments (6 x 1 KB each: lane
// l's 16 bytes at 16 l), the gate table's G, 2^G, 2^(G_last - G), beta (64
// floats each), then with a token log the byte offsets of the tokens' v' rows
// (64 int64 per 64-column slice).
constexpr int kFrag = 1024;
constexpr int kRecG = 12 * kFrag, kRecLog = 13 * kFrag;

struct ScanParams {
  ChunkParams c;
  char* rec;
  int64_t rec_stride;
  int64_t chunks;  // upper bound of the chunk count (the records grid)
};

int64_t record_bytes(int64_t dv, bool logging) { return kRecLog + (logging ? (dv + 63) / 64 * 512 : 0); }

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Sequence and chunk of global chunk index gc (chunks of all sequences in
// order), by a scan over the sequences' chunk counts, 64 at a time; false
// past the last chunk.
__device__ __forceinline__ bool find_chunk(const ChunkParams& p, int64_t gc, int lane, int64_t& n, int64_t& c) {
  int64_t base = 0;
  for (int64_t n0 = 0; n0 < p.N; n0 += 64) {
    const int64_t i = n0 + lane;
    int count = 0;
    if (i < p.N)
      count = static_cast<int>((load_index(p.cu, i + 1, p.cu_is64) - load_index(p.cu, i, p.cu_is64) + kC - 1) / kC);
    int sum = count;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(sum, o);
      sum += lane >= o ? up : 0;
    }
    const int64_t total = uniform(__builtin_amdgcn_readlane(sum, 63));
    if (gc < base + total) {
      const int l = uniform(__builtin_ctzll(__ballot(base + sum > gc)));
      n = n0 + l;
      c = gc - base - (__builtin_amdgcn_readlane(sum, l) - __builtin_amdgcn_readlane(count, l));
      return true;
    }
    base += total;
  }
  return false;
}

// K / Q rows into a tile: thread st moves rows 4 (st / DB).. and 8 columns.
template <int DK, int LDK, class QKT>
__device__ __forceinline__ void stage_rows(_Float16* tile, int st, const uint4 (&raw)[4]) {
  constexpr int DB = DK / 8;
  const int tb = st / DB, db = st % DB;
  const int a = tb & 3;
  const int o0 = 4 * ((2 * db) ^ a), o1 = 4 * ((2 * db + 1) ^ a);
  _Float16* d = tile + 4 * tb * LDK;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const uint4 v = to_f16x8<QKT>(raw[u]);
    *reinterpret_cast<uint2*>(d + u * LDK + o0) = make_uint2(v.x, v.y);
    *reinterpret_cast<uint2*>(d + u * LDK + o1) = make_uint2(v.z, v.w);
  }
}

// grid: XCD-aware (chunk, key head) groups x the key head's v-heads; 4 waves:
// 0-1 the inverses, 2-3 seven tiles each (and the gate tables before them).
constexpr int kRecThreads = 256;
template <int DK, class IOT, bool LOG>
__global__ __launch_bounds__(kRecThreads, 4) void chunk_records_kernel(ScanParams sp) {
  const ChunkParams& p = sp.c;
  constexpr int KS = DK / 32, LDK = DK + 16, DB = DK / 8, KBLK = 16 * DB;
  __shared__ __align__(16) _Float16 sK[kC * LDK];
  __shared__ __align__(16) _Float16 sQ[kC * LDK];
  __shared__ __align__(16) float gt[GTS];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int64_t slot = blockIdx.x / 8;
  const int heads = static_cast<int>(p.HV / p.H);
  const int64_t group = (slot / heads) * 8 + blockIdx.x % 8;
  const int64_t gc = group / p.H, kh = group % p.H;
  if (gc >= sp.chunks) return;
  const int64_t h = kh * heads + slot % heads;
  int64_t n, c;
  if (!find_chunk(p, gc, lane, n, c)) return;
  const int64_t bos = uniform_index(p.cu, n, p.cu_is64);
  const int64_t len = uniform_index(p.cu, n + 1, p.cu_is64) - bos;
  const int64_t left = len - c * kC;
  const int nk = static_cast<int>(left < kC ? left : kC);
  const int64_t t0 = bos + c * kC;

  // rows past the sequence end read as zeros (the buffer's range)
  uint4 pk[4], pq[4];
  const uint32_t row_bytes = static_cast<uint32_t>(p.H * DK * 2);
  const int64_t first = (t0 * p.H + kh) * DK;
  const bool kq = tid < KBLK;
  {
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(static_cast<const uint16_t*>(p.k) + first), 0, nk * row_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t qr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(static_cast<const uint16_t*>(p.q) + first), 0, nk * row_bytes, 0x00020000);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t o = static_cast<uint32_t>(4 * (tid / DB) + u) * row_bytes + 16 * (tid % DB);
      pk[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kr, o, 0, 0));
      pq[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qr, o, 0, 0));
    }
  }
  if (wave >= 2) {
    const bool ok = lane < nk;
    const int64_t gi = (t0 + (ok ? lane : 0)) * p.HV + h;
    const float g = p.g[gi], b = p.beta[gi];
    if (wave == 2) gate_table(gt, lane, nk, ok ? g : 0.f, ok ? b : 0.f);
    else factor_table(gt, lane, ok ? g : 0.f);
  }
  if (kq) {
    stage_rows<DK, LDK, IOT>(sK, tid, pk);
    stage_rows<DK, LDK, IOT>(sQ, tid, pq);
  }
  __syncthreads();

  char* rec = sp.rec + (gc * p.HV + h) * sp.rec_stride;
  reinterpret_cast<float*>(rec + kRecG)[tid] = gt[tid];
  if (LOG && wave == 0) {
    // byte offset in the frame storage of each token's value row, per 64-column slice (as the chunk kernel's log rows)
    const int64_t t = t0 + (lane < nk ? lane : 0);
    const int slot_ = static_cast<int>(load_index(p.log_slots, t, p.log_is64));
    const int pos = static_cast<int>(load_index(p.log_pos, t, p.log_pos_is64));
    const bool valid = lane < nk && slot_ >= 0 && slot_ < p.log_rows && pos >= 0 && pos < p.log_page;
    const uint32_t ps = valid ? static_cast<uint32_t>(pos) : 0u;
    const uint32_t g = static_cast<uint32_t>(p.gran), sh = static_cast<uint32_t>(__builtin_ctz(g));
    const uint32_t key_size = g * static_cast<uint32_t>(p.log_key_heads) * DK;
    const uint32_t layer_size = key_size + g * static_cast<uint32_t>(p.HV) * static_cast<uint32_t>(p.DV);
    const uint32_t elem = ((ps >> sh) * static_cast<uint32_t>(p.log_layers) + static_cast<uint32_t>(p.layer)) * layer_size +
                          key_size + (static_cast<uint32_t>(h) * g + (ps & (g - 1))) * static_cast<uint32_t>(p.DV);
    for (uint32_t col = 0; col < static_cast<uint32_t>(p.DV); col += 64) {
      const uint32_t byte = 2u * (elem + col);
      const int64_t fr = load_index(p.log_table, valid ? static_cast<int64_t>(slot_) * p.fps + p.fdiv.div(byte) : 0,
                                    p.log_table_is64);
      reinterpret_cast<int64_t*>(rec + kRecLog)[col + lane] =
          valid && fr >= 0 && fr < p.num_frames ? fr * p.frame_bytes + p.fdiv.mod(byte) : -1;
    }
  }
  // Fragment f from the two C-layout tiles of its 16 rows (columns 4 g.. and
  // 16 + 4 g.. of its 32): lane (g, c) holds row c, as the tiles do.
  auto put = [&](int f, f4_t lo, f4_t hi) __attribute__((always_inline)) {
    *reinterpret_cast<h8_t*>(rec + f * kFrag + lane * 16) = cat(hfrag(lo), hfrag(hi));
  };
  if (wave < 2) {
    HalfInverse inv;
    inv.first<KS, LDK>(sK, gt, 32 * wave, lr, lg);
    f4_t a00, a10, a11;
    inv.second(a00, a10, a11);
    put(4 * wave, a00, zero4());  // A11: fragments 0, 1; A22: 4, 5
    put(4 * wave + 1, a10, a11);
  } else {
    auto frags = [&](const _Float16* X, int r, h8_t (&f)[KS]) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < KS; ++m) f[m] = kqfrag(X, LDK, 16 * r + lr, 32 * m, lg);
    };
    auto dot = [&](const h8_t (&a)[KS], const h8_t (&b)[KS]) __attribute__((always_inline)) {
      f4_t acc = zero4();
#pragma unroll
      for (int m = 0; m < KS; ++m) acc = mma(a[m], b[m], acc);
      return acc;
    };
    auto l = [&](int ti, int tj, f4_t x) __attribute__((always_inline)) {
      return -masked_off(gt, x, 16 * ti + lr, 16 * tj + 4 * lg, true);
    };
    auto m = [&](int ti, int tj, f4_t x) __attribute__((always_inline)) {
      const int t = 16 * ti + lr, s0 = 16 * tj + 4 * lg;
      return ti > tj ? masked_off(gt, x, t, s0, false) : masked(gt, x, t, s0, false, false);
    };
    h8_t k0[KS], k1[KS], k2[KS], k3[KS], qa[KS], qb[KS];
    frags(sK, 0, k0);
    frags(sK, 1, k1);
    frags(sK, 2, k2);
    frags(sK, 3, k3);
    if (wave == 2) {  // -L21, M rows 0-31
      frags(sQ, 0, qa);
      frags(sQ, 1, qb);
      const f4_t l20 = dot(k0, k2), l21 = dot(k1, k2), l30 = dot(k0, k3), l31 = dot(k1, k3);
      const f4_t m00 = dot(k0, qa), m10 = dot(k0, qb), m11 = dot(k1, qb);
      put(2, l(2, 0, l20), l(2, 1, l21));
      put(3, l(3, 0, l30), l(3, 1, l31));
      put(6, m(0, 0, m00), zero4());
      put(7, m(1, 0, m10), m(1, 1, m11));
    } else {  // M rows 32-63
      frags(sQ, 2, qa);
      frags(sQ, 3, qb);
      const f4_t m20 = dot(k0, qa), m21 = dot(k1, qa), m22 = dot(k2, qa);
      const f4_t m30 = dot(k0, qb), m31 = dot(k1, qb), m32 = dot(k2, qb), m33 = dot(k3, qb);
      put(8, m(2, 0, m20), m(2, 1, m21));
      put(9, m(3, 0, m30), m(3, 1, m31));
      put(10, m(2, 2, m22), zero4());
      put(11, m(3, 2, m32), m(3, 3, m33));
    }
  }
}

// ---------------------------------------------------------------- recurrence
constexpr int kStagers = 256;
constexpr int kScanThreads = 128 + kStagers;
constexpr int kDepth = 2;  // register sets of the staging waves: loads go out this many chunks before they are staged

// Keeps the LDS reads issued above it above what follows.
__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }

// The barrier of chunk c, B(c), comes after the chain's solve of chunk c.
// Between B(c - 1) and B(c):
//   chain    h update of chunk c - 1 (K^T and v' in registers), then P, R and
//            the solve of chunk c; reads K(c), A(c), V(c), gates(c)
//   output   o of chunk c - 1: reads Q, M, gates and the chain's operands of c - 1
//   staging  writes K, A, V, gates of chunk c + 1, Q and M of chunk c, and
//            issues the loads of chunk c + 1 + kDepth
// so everything has 2 buffers (the chain's last reads of K(c - 1), its K^T
// fragments, come before B(c - 1)) but the gates: the output wave reads those of
// chunk c - 1 while the chain reads chunk c's and chunk c + 1's are written (a
// ring of 4).
// EXT: checkpoints every 16 or 32 tokens, frame-table states and the token
// log's v' rows (as chunk_chain_kernel's).
template <int DK, class IOT, class ST, bool EXT>
__global__ __launch_bounds__(kScanThreads) void chunk_scan_kernel(ScanParams sp) {
  const ChunkParams& p = sp.c;
  constexpr int HT = DK / 16, KS = DK / 32, LDK = DK + 16, DB = DK / 8, KBLK = 16 * DB;
  constexpr int TILE = kC * LDK * 2;     // bytes of a K or Q tile
  constexpr int COLS = 16;
  constexpr int BUF = TILE + 6 * kFrag;  // a K tile and the A fragments, or a Q tile and the M fragments
  __shared__ __align__(16) char sKA[2 * BUF];
  __shared__ __align__(16) char sQM[2 * BUF];
  __shared__ __align__(16) _Float16 sV[2 * kC * COLS];  // (a transpose read's four 32-byte rows: distinct banks)
  __shared__ __align__(16) float sG[4 * 256];  // a chunk's G, 2^G, 2^(G_last - G), beta
  __shared__ int sSlot[4];                     // its last checkpoint slot
  // EXT: byte offset in the frame storage of each token's logged v' row, at the slice's 64-column group (-1: none)
  __shared__ __align__(16) int64_t sLog[EXT ? 2 * kC : 1];
  __shared__ __align__(16) char sH[2 * KS * kFrag];  // the chain's f16 state operands, per chunk parity
  __shared__ __align__(16) char sX[2 * 2 * kFrag];   // its v' operands

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int64_t bslot = blockIdx.x / 8;
  const int members = p.members;
  const int64_t group = (bslot / members) * 8 + blockIdx.x % 8;
  if (group >= p.N * p.H) return;
  const int member = static_cast<int>(bslot % members);
  const int slices = static_cast<int>(p.DV / COLS);
  const int64_t n = group / p.H, kh = group % p.H;
  const int64_t h = kh * (p.HV / p.H) + member / slices;
  const int64_t col_base = static_cast<int64_t>(member % slices) * COLS;

  const int64_t bos = uniform_index(p.cu, n, p.cu_is64);
  const int64_t len = uniform_index(p.cu, n + 1, p.cu_is64) - bos;
  const int nchunks = static_cast<int>((len + kC - 1) / kC);
  const int last_rows = static_cast<int>(len - (nchunks - 1) * static_cast<int64_t>(kC));  // of the last chunk
  // chunks of the sequences before this one, and their checkpoint intervals
  const int gran = EXT ? p.gran : kC;
  int64_t chunk_base = 0, sub_base = 0;
  for (int64_t m = 0; m < n; ++m) {
    const int64_t lm = uniform_index(p.cu, m + 1, p.cu_is64) - uniform_index(p.cu, m, p.cu_is64);
    chunk_base += (lm + kC - 1) / kC;
    sub_base += (lm + gran - 1) / gran;
  }
  // every wave runs the same number of barriers: the chunks, rounded up to the staging waves' unrolled sets
  const int iters = (nchunks + kDepth - 1) / kDepth * kDepth;

  if (wave == 0) {
    // ==================================================================== chain wave
    const StateSlots<ST, EXT> slots{p, h, col_base};
    f4_t hT[HT];
    auto lane_off = [&]() {
      uint32_t o = static_cast<uint32_t>((4 * lg * p.DV + lr) * sizeof(ST));
      asm volatile("" : "+v"(o));
      return o;
    };
    auto store_state = [&](int64_t s) __attribute__((always_inline)) {
      slots.template store<HT>(s, lane_off(), [&](int ti) __attribute__((always_inline)) { return hT[ti]; });
    };
    slots.load(uniform_index(p.read_slots, n, p.read_is64), lane_off(), hT);
#pragma unroll
    for (int ti = 0; ti < HT; ++ti) asm volatile("" ::"v"(hT[ti]));
    const int64_t fw = p.fw_slots ? uniform_index(p.fw_slots, n, p.fw_is64) : -1;
    if (nchunks == 0) {  // empty sequence: the final state is the initial state
      if (fw >= 0) store_state(fw);
      return;
    }
    uint16_t* vng = p.v_new ? static_cast<uint16_t*>(p.v_new) + (bos * p.HV + h) * p.DV + col_base : nullptr;
    const int64_t tok_stride = p.HV * p.DV;
    uint32_t ktr = lane_tr_offset(LDK, lr, lg);
    asm volatile("" : "+v"(ktr));
    h8_t kT[2 * HT];  // K^T of the chunk being updated
    h8_t db0, db1;    // its 2^(G_last - G) v'
    float gl;         // 2^G_last
    int cw;           // its checkpoint slot
    auto update = [&]() __attribute__((always_inline)) {  // h <- 2^G_last h + K^T (2^(G_last - G) v')
#pragma unroll
      for (int ti = 0; ti < HT; ++ti) hT[ti] = mma(kT[2 * ti + 1], db1, mma(kT[2 * ti], db0, hT[ti] * gl));
      if (cw >= 0) store_state(cw);
    };
    __builtin_amdgcn_s_setprio(3);
    lds_barrier();  // chunk 0 staged
    for (int c = 0; c < nchunks; ++c) {
      const _Float16* K = reinterpret_cast<const _Float16*>(sKA + (c & 1) * BUF);
      const _Float16* Vt = sV + (c & 1) * kC * COLS;
      const float* gt = sG + (c & 3) * 256;
      char* hx = sH + (c & 1) * KS * kFrag + lane * 16;
      char* vx = sX + (c & 1) * 2 * kFrag + lane * 16;
      const char* A = sKA + (c & 1) * BUF + TILE + lane * 16;
      // the first half of K goes out before the update, the rest after it (with K^T the whole would not fit)
      constexpr int KH = KS > 1 ? KS / 2 : KS;
      h8_t kf[KS][4];
      auto read_k = [&](int m) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) kf[m][i] = kqfrag(K, LDK, 16 * i + lr, 32 * m, lg);
      };
#pragma unroll
      for (int m = 0; m < KH; ++m) read_k(m);
      sched_fence();
      if (c) update();
#pragma unroll
      for (int m = KH; m < KS; ++m) read_k(m);
      sched_fence();
      // P = K h; the state operands also go to the output wave
      f4_t P[4], R[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) P[i] = zero4();
      auto p_step = [&](int m) __attribute__((always_inline)) {
        const h8_t hb = bfrag(hT[2 * m], hT[2 * m + 1]);
        *reinterpret_cast<h8_t*>(hx + m * kFrag) = hb;
#pragma unroll
        for (int i = 0; i < 4; ++i) P[i] = mma(kf[m][i], hb, P[i]);
      };
#pragma unroll
      for (int m = 0; m < KH; ++m) p_step(m);
      sched_fence();
      // the other operands of this chunk: their latency passes under P (not
      // more than the 15 LDS operations a wait can tell apart before K is in)
      h8_t a[6];
      f4_t e4[4], b4[4];
      h4_t vr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        e4[i] = *reinterpret_cast<const f4_t*>(gt + G_EXP + 16 * i + 4 * lg);
        b4[i] = *reinterpret_cast<const f4_t*>(gt + G_BETA + 16 * i + 4 * lg);
        vr[i] = tr_read(Vt + (16 * i + 4 * lg + (lr >> 2)) * COLS + 4 * (lr & 3));
      }
      sched_fence();
#pragma unroll
      for (int m = KH; m < KS; ++m) p_step(m);
#pragma unroll
      for (int f = 0; f < 6; ++f) a[f] = *reinterpret_cast<const h8_t*>(A + f * kFrag);
      sched_fence();
      // this chunk's K^T, decays and slot, read for its update
      const int nv = c == nchunks - 1 ? last_rows : kC;
      f4_t d[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = *reinterpret_cast<const f4_t*>(gt + G_DEC + 16 * i + 4 * lg);
      gl = gt[G_EXP + nv - 1];
      const int cwv = sSlot[c & 3];
      {
        const char* kl = reinterpret_cast<const char*>(K) + ktr;
#pragma unroll
        for (int ti = 0; ti < HT; ++ti) {
          kT[2 * ti] = kq_tfrag<LDK>(kl, 0, 16 * ti);
          kT[2 * ti + 1] = kq_tfrag<LDK>(kl, 32, 16 * ti);
        }
      }
      sched_fence();
      // R = beta (v - 2^G P)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v4[4];
        v_rows<IOT>(vr[i], v4);
#pragma unroll
        for (int e = 0; e < 4; ++e) R[i][e] = b4[i][e] * (v4[e] - e4[i][e] * P[i][e]);
      }
      // v'_top = A11 R_top; R_bot -= L21 v'_top; v'_bot = A22 R_bot
      f4_t V[4];
      const h8_t rb0 = bfrag(R[0], R[1]);
      V[0] = mma(a[0], rb0, zero4());
      V[1] = mma(a[1], rb0, zero4());
      const h8_t vb0 = bfrag(V[0], V[1]);
      R[2] = mma(a[2], vb0, R[2]);
      R[3] = mma(a[3], vb0, R[3]);
      const h8_t rb1 = bfrag(R[2], R[3]);
      V[2] = mma(a[4], rb1, zero4());
      V[3] = mma(a[5], rb1, zero4());
      const h8_t vb1 = bfrag(V[2], V[3]);
      *reinterpret_cast<h8_t*>(vx) = vb0;
      *reinterpret_cast<h8_t*>(vx + kFrag) = vb1;
      db0 = bfrag(V[0] * d[0], V[1] * d[1]);
      db1 = bfrag(V[2] * d[2], V[3] * d[3]);
      cw = uniform(cwv);
      if (vng || (EXT && p.logging)) {  // v'^T = R^T A^T: a lane writes 4 consecutive columns of one token
        const f4_t vt[4] = {mma(rb0, a[0], zero4()), mma(rb0, a[1], zero4()), mma(rb1, a[4], zero4()),
                            mma(rb1, a[5], zero4())};
        char* vb = reinterpret_cast<char*>(vng + static_cast<int64_t>(c) * kC * tok_stride);
        uint32_t ov = static_cast<uint32_t>((lr * tok_stride + 4 * lg) * 2);
        asm volatile("" : "+v"(ov));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          char* dst = vb + 16 * i * tok_stride * 2 + ov;
          bool on = 16 * i + lr < nv;
          if (EXT && p.logging) {
            const int64_t off = sLog[(c & 1) * kC + 16 * i + lr];
            dst = static_cast<char*>(p.state) + off + (col_base % 64 + 4 * lg) * 2;
            on = off >= 0;
          }
          if (on) {
            uint2 w;
            w.x = out_pack2<IOT>(vt[i][0], vt[i][1]);
            w.y = out_pack2<IOT>(vt[i][2], vt[i][3]);
            *reinterpret_cast<uint2*>(dst) = w;
          }
        }
      }
      // checkpoints inside the chunk: the state after token te = (s + 1) gran - 1
      // is 2^G_te h + K^T (2^(G_te - G) v'), the decay taken over tokens t <= te
      for (int sc = 0; EXT && sc + 1 < (nv + gran - 1) / gran; ++sc) {
        const int64_t ws = uniform_index(p.cw_slots, sub_base + static_cast<int64_t>(c) * (kC / gran) + sc, p.cw_is64);
        if (ws < 0) continue;
        const int te = (sc + 1) * gran - 1;
        const float Ge = gt[te], ge = gt[G_EXP + te];
        f4_t dm[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f4_t g4 = *reinterpret_cast<const f4_t*>(gt + 16 * i + 4 * lg);
#pragma unroll
          for (int e = 0; e < 4; ++e) dm[i][e] = 16 * i + 4 * lg + e <= te ? V[i][e] * fast_exp2(Ge - g4[e]) : 0.f;
        }
        const h8_t m0 = bfrag(dm[0], dm[1]), m1 = bfrag(dm[2], dm[3]);
        slots.template store<HT>(ws, lane_off(), [&](int ti) __attribute__((always_inline)) {
          f4_t r = mma(kT[2 * ti], m0, hT[ti] * ge);
          if (te >= 32) r = mma(kT[2 * ti + 1], m1, r);
          return r;
        });
      }
      lds_barrier();  // B(c)
    }
    update();
    if (fw >= 0) store_state(fw);
    for (int c = nchunks; c < iters; ++c) lds_barrier();
  } else if (wave == 1) {
    // ==================================================================== output wave
    if (nchunks == 0) return;
    const int64_t tok_stride = p.HV * p.DV;
    const uint32_t tok_bytes = static_cast<uint32_t>(tok_stride * 2);
    uint16_t* og = static_cast<uint16_t*>(p.out) + (bos * p.HV + h) * p.DV + col_base;
    uint32_t ooff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ooff[i] = static_cast<uint32_t>(16 * i + lr) * tok_bytes + 8 * lg;
    lds_barrier();  // chunk 0 staged
    for (int c = 0; c < nchunks; ++c) {
      lds_barrier();  // B(c)
      const _Float16* Q = reinterpret_cast<const _Float16*>(sQM + (c & 1) * BUF);
      const char* hx = sH + (c & 1) * KS * kFrag + lane * 16;
      const char* vx = sX + (c & 1) * 2 * kFrag + lane * 16;
      const char* M = sQM + (c & 1) * BUF + TILE + lane * 16;
      const float* gt = sG + (c & 3) * 256;
      h8_t qf[KS][4], hb[KS], mf[6];
      float e[4];
#pragma unroll
      for (int m = 0; m < KS; ++m) {
        hb[m] = *reinterpret_cast<const h8_t*>(hx + m * kFrag);
#pragma unroll
        for (int i = 0; i < 4; ++i) qf[m][i] = kqfrag(Q, LDK, 16 * i + lr, 32 * m, lg);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = gt[G_EXP + 16 * i + lr];
      const h8_t vb0 = *reinterpret_cast<const h8_t*>(vx), vb1 = *reinterpret_cast<const h8_t*>(vx + kFrag);
#pragma unroll
      for (int f = 0; f < 6; ++f) mf[f] = *reinterpret_cast<const h8_t*>(M + f * kFrag);
      sched_fence();
      f4_t Ot[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) Ot[i] = zero4();
#pragma unroll
      for (int m = 0; m < KS; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) Ot[i] = mma(hb[m], qf[m][i], Ot[i]);
#pragma unroll
      for (int i = 0; i < 4; ++i) Ot[i] *= e[i];
#pragma unroll
      for (int i = 0; i < 4; ++i) Ot[i] = mma(vb0, mf[i], Ot[i]);
      Ot[2] = mma(vb1, mf[4], Ot[2]);
      Ot[3] = mma(vb1, mf[5], Ot[3]);
      // rows past the sequence end fall outside the buffer's range and are dropped
      const int nv = c == nchunks - 1 ? last_rows : kC;
      const __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc(
          og + static_cast<int64_t>(c) * kC * tok_stride, 0, nv * tok_bytes, 0x00020000);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
        const u2_t w = {out_pack2<IOT>(p.scale * Ot[i][0], p.scale * Ot[i][1]),
                        out_pack2<IOT>(p.scale * Ot[i][2], p.scale * Ot[i][3])};
        __builtin_amdgcn_raw_buffer_store_b64(w, orsrc, ooff[i], 0, 0);
      }
    }
    for (int c = nchunks; c < iters; ++c) lds_barrier();
  } else {
    // ==================================================================== staging waves
    if (nchunks == 0) return;
    const int st = tid - 128;
    const uint32_t vrow = static_cast<uint32_t>(p.HV * p.DV * 2);
    const bool vt = st < 2 * kC;  // two 16-byte pieces of a V row
    const uint32_t voff = vt ? static_cast<uint32_t>(st / 2) * vrow + static_cast<uint32_t>(16 * (st % 2)) : 0u;
    // Sources of the next chunk to load.  Rows past the sequence end read as
    // zeros (the buffers' ranges); past the last chunk the record pointers
    // stay on it.
    const char* vp = static_cast<const char*>(p.v) + ((bos * p.HV + h) * p.DV + col_base) * 2;
    const int64_t vstep = static_cast<int64_t>(kC) * vrow;
    const char* ra = sp.rec + (chunk_base * p.HV + h) * sp.rec_stride;
    const char* rm = ra;
    const int64_t rstep = p.HV * sp.rec_stride;
    const bool kq = st < KBLK;
    const uint32_t krow = static_cast<uint32_t>(p.H * DK * 2);
    uint32_t koff[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      koff[u] = static_cast<uint32_t>(4 * (st / DB) + u) * krow + static_cast<uint32_t>(16 * (st % DB));
    const char* kp = static_cast<const char*>(p.k) + (bos * p.H + kh) * DK * 2;
    const char* qp = static_cast<const char*>(p.q) + (bos * p.H + kh) * DK * 2;
    const int64_t kstep = static_cast<int64_t>(kC) * krow;
    int qrows = 0;  // rows of chunk next - 1
    int next = 0;  // chunk to load
    struct Set {
      uint4 k[4], q[4], r[3], v, g, log;
      int cw;
    } set[kDepth];
    const int64_t logged = EXT && p.logging ? kRecLog + col_base / 64 * 512 : kRecG;  // (any 512 bytes without a log)
    // K, V, A, gates and slot of chunk `next`, Q and M of the chunk before it (itself for chunk 0)
    auto issue = [&](Set& s, bool first) __attribute__((always_inline)) {
      const int rows = next < nchunks - 1 ? kC : (next == nchunks - 1 ? last_rows : 0);
      const __amdgpu_buffer_rsrc_t vr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vp), 0, rows * vrow, 0x00020000);
      const __amdgpu_buffer_rsrc_t kr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kp), 0, rows * krow, 0x00020000);
      const __amdgpu_buffer_rsrc_t qr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(qp), 0, (first ? rows : qrows) * krow, 0x00020000);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s.k[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kr, koff[u], 0, 0));
        s.q[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qr, koff[u], 0, 0));
      }
      // 384 16-byte pieces of A, then 384 of M: three per thread
      s.r[0] = *reinterpret_cast<const uint4*>(ra + 16 * st);
      s.r[1] = *reinterpret_cast<const uint4*>((st < 128 ? ra : rm) + 16 * (256 + st));
      s.r[2] = *reinterpret_cast<const uint4*>(rm + 16 * (512 + st));
      s.v = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vr, voff, 0, 0));
      s.g = *reinterpret_cast<const uint4*>(ra + kRecG + 16 * (st & 63));
      if constexpr (EXT) s.log = *reinterpret_cast<const uint4*>(ra + logged + 16 * (st & 31));
      // the slot of the chunk's last interval
      const int64_t end = static_cast<int64_t>(next < nchunks ? next : nchunks - 1) * kC + (next < nchunks - 1 ? kC : last_rows);
      s.cw = static_cast<int>(load_index(p.cw_slots, sub_base + (end + gran - 1) / gran - 1, p.cw_is64));
      if (!first) {
        qp += kstep;
        rm = ra;
      }
      kp += kstep;
      vp += vstep;
      qrows = rows;
      ++next;
      if (next < nchunks) ra += rstep;
    };
    auto stage = [&](const Set& s, int c) __attribute__((always_inline)) {
      const int cq = c > 0 ? c - 1 : 0;
      char* ka = sKA + (c & 1) * BUF;
      char* qm = sQM + (cq & 1) * BUF;
      if (kq) {
        stage_rows<DK, LDK, IOT>(reinterpret_cast<_Float16*>(ka), st, s.k);
        stage_rows<DK, LDK, IOT>(reinterpret_cast<_Float16*>(qm), st, s.q);
      }
      ka += TILE;
      qm += TILE;
      *reinterpret_cast<uint4*>(ka + 16 * st) = s.r[0];
      *reinterpret_cast<uint4*>(st < 128 ? ka + 16 * (256 + st) : qm + 16 * (st - 128)) = s.r[1];
      *reinterpret_cast<uint4*>(qm + 16 * (128 + st)) = s.r[2];
      if (vt) *reinterpret_cast<uint4*>(reinterpret_cast<char*>(sV + (c & 1) * kC * COLS) + 16 * st) = s.v;
      if (st < 64) *reinterpret_cast<uint4*>(sG + (c & 3) * 256 + 4 * st) = s.g;
      if (st == 64) sSlot[c & 3] = s.cw;
      if (EXT && st >= 128 && st < 160) *reinterpret_cast<uint4*>(sLog + (c & 1) * kC + 2 * (st & 31)) = s.log;
    };
    issue(set[0], true);
    stage(set[0], 0);
#pragma unroll
    for (int u = 0; u < kDepth; ++u) issue(set[u], false);
    lds_barrier();  // chunk 0 staged
    for (int c = 0; c < iters; c += kDepth) {
#pragma unroll
      for (int u = 0; u < kDepth; ++u) {
        stage(set[u], c + u + 1);
        issue(set[u], false);
        lds_barrier();  // B(c + u)
      }
    }
  }
}

template <int DK, class IOT, class ST>
int launch_typed(const ScanParams& s, hipStream_t stream) {
  const ChunkParams& p = s.c;
  const int64_t rec_blocks = (s.chunks * p.H + 7) / 8 * 8 * (p.HV / p.H);
  const int64_t scan_blocks = (p.N * p.H + 7) / 8 * 8 * p.members;
  if (rec_blocks > 0x7fffffff || scan_blocks > 0x7fffffff) {
    set_error("gdn chunk scan: grid too large");
    return GDN_ERR_INVALID;
  }
  const dim3 rgrid(static_cast<unsigned>(rec_blocks)), grid(static_cast<unsigned>(scan_blocks));
  if (p.logging)
    hipLaunchKernelGGL((chunk_records_kernel<DK, IOT, true>), rgrid, dim3(kRecThreads), 0, stream, s);
  else
    hipLaunchKernelGGL((chunk_records_kernel<DK, IOT, false>), rgrid, dim3(kRecThreads), 0, stream, s);
  if (p.gran < kC || p.frames)
    hipLaunchKernelGGL((chunk_scan_kernel<DK, IOT, ST, true>), grid, dim3(kScanThreads), 0, stream, s);
  else
    hipLaunchKernelGGL((chunk_scan_kernel<DK, IOT, ST, false>), grid, dim3(kScanThreads), 0, stream, s);
  return GDN_LAUNCH_CHECK("gdn chunk scan launch");
}

}  // namespace

int64_t chunk_scan_workspace(int64_t num_seqs, int64_t total_tokens, int64_t HV, int64_t dv, bool logging) {
  return (total_tokens / kC + num_seqs) * HV * record_bytes(dv, logging);
}

// The scan's workgroups (16 columns each) must fit the 256 CUs at one apiece,
// which is where the one-launch form leaves three CUs of four idle; beyond
// that its parallel launches, whose time grows with all tokens, cost more than
// the shorter chain saves.  Whole prefill, replayed from a graph, us, one launch
// / two, heads of 128: 1 x 8192 x 32 heads 312 / 228, 2 x 8000 x 16 305 / 228, but
// 2 x 4096 x 32 184 / 233, 4 x 4096 x 16 184 / 236.  From about 12 tokens a sequence
// and one-launch workgroup on two launches win by 10 % and more (1 x 768 x 32
// 44.8 / 40.5, 1 x 1000 x 32 54.0 / 46.3, 2 x 800 x 16 48.5 / 42.6; heads of 64: 16
// x 800 x 4 58.0 / 53.1, 16 x 2500 x 4 131 / 105).  Below, the two are within 7 % of
// each other (1 x 128 x 32 19.8 / 20.3, 1 x 300 x 32 26.5 / 26.2, 1 x 500 x 32 33.6 /
// 33.4, 1 x 700 x 32 42.4 / 39.9, 1 x 300 x 16 26.0 / 24.2, 16 x 200 x 4 of 64 26.6 /
// 26.5), and one launch needs no workspace.
bool chunk_scan_preferred(int64_t num_seqs, int64_t total_tokens, int64_t HV, int64_t dv) {
  const int64_t groups = num_seqs * HV * ((dv + 63) / 64);  // workgroups of the one-launch form
  const int64_t least = 12 * groups > 128 ? 12 * groups : 128;
  return groups <= 64 && total_tokens >= least * num_seqs;
}

int launch_chunk_scan(const ChunkParams& p, int64_t dk, int io_dtype, int state_dtype, void* workspace,
                      hipStream_t stream) {
  ScanParams s{};
  s.c = p;
  s.rec = static_cast<char*>(workspace);
  s.rec_stride = record_bytes(p.DV, p.logging);
  s.chunks = p.T / kC + p.N;
  s.c.members = static_cast<int>((p.HV / p.H) * (p.DV / 16));
  auto by_dk = [&](auto dkc) {
    constexpr int DK = decltype(dkc)::value;
    if (io_dtype == GDN_BF16 && state_dtype == GDN_F32) return launch_typed<DK, bf16, float>(s, stream);
    if (io_dtype == GDN_BF16 && state_dtype == GDN_BF16) return launch_typed<DK, bf16, bf16>(s, stream);
    if (io_dtype == GDN_F16 && state_dtype == GDN_F32) return launch_typed<DK, f16, float>(s, stream);
    if (io_dtype == GDN_F16 && state_dtype == GDN_F16) return launch_typed<DK, f16, f16>(s, stream);
    return static_cast<int>(GDN_ERR_UNSUPPORTED);
  };
  if (dk == 128) return by_dk(std::integral_constant<int, 128>{});
  if (dk == 64) return by_dk(std::integral_constant<int, 64>{});
  if (dk == 32) return by_dk(std::integral_constant<int, 32>{});
  return GDN_ERR_UNSUPPORTED;
}

}  // namespace gdn
