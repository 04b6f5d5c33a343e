// Kernel instantiations and launch sequences for ONE element type, selected with -DGN_INST_DTYPE=0..3
// (f32, f64, f16, bf16).  Built four times so the four types compile in parallel.
#include "gn_host.h"
#include <algorithm>

#include "gn_fused.h"
#include "gn_kernels.h"

#ifndef GN_INST_DTYPE
#error "compile with -DGN_INST_DTYPE=<0|1|2|3>"
#endif
// One data type's kernels are spread over four translation units so that they compile in parallel: the single-launch
// kernels of the forward (part 0), the backward (part 1) and the forward with fused additions (part 2); the streaming
// kernels of both directions and the choice between the families (part 3).
#ifndef GN_INST_PART
#error "compile with -DGN_INST_PART=<0|1|2|3>"
#endif
#define GN_PART_FWD (GN_INST_PART == 0)
#define GN_PART_BWD (GN_INST_PART == 1)
#define GN_PART_ADD (GN_INST_PART == 2)
#define GN_PART_STREAM (GN_INST_PART == 3)

namespace gn {

// wide_param_t: the other type weight / bias may have (f32 parameters with 16-bit data)
#if GN_INST_DTYPE == 0
typedef float elem_t;
typedef float wide_param_t;
#define GN_SUFFIX f32
#elif GN_INST_DTYPE == 1
typedef double elem_t;
typedef double wide_param_t;
#define GN_SUFFIX f64
#elif GN_INST_DTYPE == 2
typedef f16_t elem_t;
typedef float wide_param_t;
#define GN_SUFFIX f16
#else
typedef bf16_t elem_t;
typedef float wide_param_t;
#define GN_SUFFIX bf16
#endif
#define GN_CAT2(a, b) a##b
#define GN_CAT(a, b) GN_CAT2(a, b)

// The single-launch families (parts 0 to 2): true if the call was launched, false if it does not fit one.
bool GN_CAT(try_resident_fwd_, GN_SUFFIX)(const FwdArgs &a);
bool GN_CAT(try_resident_fwd_added_, GN_SUFFIX)(const FwdArgs &a);
bool GN_CAT(try_resident_bwd_, GN_SUFFIX)(const BwdArgs &a);

namespace {

typedef acc_t<elem_t> A;
constexpr int kVec = vec_of<elem_t>::value;

dim3 tile_grid(const Plan &p, int extra_x) {
  return dim3((unsigned)(p.tiles + extra_x), (unsigned)p.nchunk, (unsigned)(p.N < 65535 ? p.N : 65535));
}

// dy stored in a 16-bit type while the data are float (only the float instantiation has such kernels)
[[maybe_unused]] constexpr bool kHasDy16 = GN_INST_DTYPE == 0;

#if GN_PART_STREAM
size_t input_bytes(const FwdArgs &a) { return (size_t)a.plan.N * a.plan.R * a.plan.C * sizeof(elem_t); }
bool input_stays_cached(const FwdArgs &a) { return input_bytes(a) <= kCacheBytes; }
template <typename PT, int VEC, int ACT> void launch_apply(const FwdArgs &a, const A *part, const PartialGeo &q, const Plan &p) {
  auto kernel = apply_kernel<elem_t, PT, VEC, ACT, false>;
  // (an input too large for the memory-side cache is read here for the last time anyone could find it there: non-temporal
  // loads, which pass that cache by, 6 % faster on a 537 MB copy; a smaller one may yet be wanted by the backward)
  if constexpr (VEC == kVec) {
    if (!input_stays_cached(a)) kernel = apply_kernel<elem_t, PT, VEC, ACT, true>;
  }
  launch(kKindFwdApply, kernel, tile_grid(p, 0), dim3(kBlock), a.stream, (const elem_t *)a.x, (elem_t *)a.y, part, q, a.w, a.b,
         a.mean, a.rstd, a.sdtype, a.ydtype, (A)a.eps, p);
}
template <typename PT, int VEC> void launch_apply_act(const FwdArgs &a, const A *part, const PartialGeo &q, const Plan &p) {
  switch (a.act) {
    case GN_ACT_IDENTITY: launch_apply<PT, VEC, GN_ACT_IDENTITY>(a, part, q, p); break;
    case GN_ACT_RELU: launch_apply<PT, VEC, GN_ACT_RELU>(a, part, q, p); break;
    case GN_ACT_SILU: launch_apply<PT, VEC, GN_ACT_SILU>(a, part, q, p); break;
    case GN_ACT_GELU: launch_apply<PT, VEC, GN_ACT_GELU>(a, part, q, p); break;
    default: launch_apply<PT, VEC, GN_ACT_GELU_TANH>(a, part, q, p); break;
  }
}
#else  // single-launch families

// ---- resident (single-launch) path ----------------------------------------------------------------
// Workgroups that can be resident at once for a kernel: occupancy reported by the runtime times the CUs.
template <typename K> int resident_slots(K kernel) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  const int slots = per_cu * cus;
  return slots < kMaxResidentBlocks ? slots : kMaxResidentBlocks;
}

// Row tiling of a resident launch with a register capacity of nv rows per lane: tiles of exactly nv rows per
// lane (all loads useful; only the last tile of a sample may be short), every workgroup resident.
// Returns false if it does not fit.  `rolling`: only the workgroups that exchange records (a set) have to be resident
// together, and they may take half of the device at most.  A set that fills the device waits for whatever else holds a
// single slot of it, and while an expired set recovers (milliseconds) the set behind it could not become resident either,
// so that its waits would expire as well, and so on through the launch.  With two sets' room the next one completes beside
// it, a tenant may hold the other half, and two rolling launches (replayed graphs) do not starve each other.
// What the other half gave: float16 (1, R, 256, 32), R = 320 / 384 / 448 / 512 Ki rows, 87 / 97 / 120 / 129 us against the
// streaming pair's 91 / 114 / 118 / 134 us; at half, R = 256 Ki, 56 against 73.
bool resident_tiling(const Plan &base, int64_t samples, int nv, int slots, Plan &out, bool rolling = false) {
  const int64_t columns = samples * base.nchunk;
  if (slots <= 0 || samples > 65535) return false;
  const int64_t together = rolling ? exchange_chunks(base) : columns;
  if (rolling) slots /= 2;
  if (together > slots) return false;
  if (base.G > 8192 || base.C >= (1 << 23)) return false;  // the kernels index their records with 24-bit multiplies
  if ((base.lpr & (base.lpr - 1)) != 0) return false;  // ... and find a lane's row and column by shifts
  const int64_t rows = (int64_t)nv * base.rpi;
  const int64_t tiles = (base.R + rows - 1) / rows;
  if (together * tiles > slots) return false;
  out = base;
  out.N = samples;
  out.tile_rows = (int)rows;
  out.tiles = (int)tiles;
  out.nblocks = columns * tiles;
  set_divisors(out);
  return true;
}


struct ResidentWorkspace {
  SyncArea sync;
};
// Captured launches take their per-replay epoch from the library's generation word and a sequence number.
void arm_generation(ResidentWorkspace &r, const CapturedEpoch &c) {
  r.sync.generation = c.generation;
  if (c.generation) r.sync.epoch = c.next_sequence();
}
ResidentWorkspace resident_fwd_ws(void *ws, const Plan &p, const FwdRecords &records) {
  ResidentWorkspace r;
  char *base = (char *)ws + kWorkspaceHeader;
  r.sync.area = base;
  r.sync.area_bytes = (unsigned)(records.rec + records.frec);
  r.sync.rec_first = 0;
  r.sync.frec_first = (unsigned)(records.rec / 16);
  r.sync.crec_first = 0;  // (no channel records in the forward)
  r.sync.two_level = two_level_exchange(p) ? 1 : 0;
  r.sync.status = resident_status();
  r.sync.generation = nullptr;
  r.sync.max_spins = resident_spin_limit();
  r.sync.epoch = next_epoch();
  r.sync.trace = trace_buffer();
  r.sync.trace_wait = trace_waits() ? 1 : 0;
  return r;
}
ResidentWorkspace resident_bwd_ws(void *ws, const Plan &p, const BwdRecords &records) {
  ResidentWorkspace r;
  char *base = (char *)ws + kWorkspaceHeader;
  r.sync.area = base;
  r.sync.area_bytes = (unsigned)(records.crec + records.rec + records.frec);
  r.sync.crec_first = 0;  // channel records of the whole tensor, [N][tiles][C]
  r.sync.rec_first = (unsigned)(records.crec / 16);
  r.sync.frec_first = (unsigned)((records.crec + records.rec) / 16);
  r.sync.two_level = two_level_exchange(p) ? 1 : 0;
  r.sync.status = resident_status();
  r.sync.generation = nullptr;
  r.sync.max_spins = resident_spin_limit();
  r.sync.epoch = next_epoch();
  r.sync.trace = trace_buffer();
  r.sync.trace_wait = trace_waits() ? 1 : 0;
  return r;
}

// How many consecutive single-launch kernels over groups of samples still beat the streaming kernels in the backward.  Each
// launch pays a fixed latency of roughly 9 microseconds but moves 3 S bytes instead of 5 S (about 5.4 bytes per nanosecond
// either way, and about 14 us fixed for the streaming kernels).  Measured on (N, 320, 128, 128) bf16, cold tensors: one
// launch 27.0 against 44.4 us at N = 4 and 35.9 against 67.4 at N = 6, two 52.5 against 87.6 at N = 8 and 71.0 against 121.0
// at N = 12, three 103.4 against 162.2 at N = 16.
int worthwhile_batches(const Plan &p) {
  const double s_mb = (double)p.N * p.R * p.C * sizeof(elem_t) / 1e6;
  const double k = (14.0 + 0.405 * s_mb) / 9.0;
  const int kk = k < 1.0 ? 1 : (int)k;
  return kk < kMaxBatches ? kk : kMaxBatches;
}
size_t stat_size(int sdtype) { return sdtype == GN_F32 ? 4 : sdtype == GN_F64 ? 8 : 2; }

#if GN_PART_FWD || GN_PART_ADD
// One NV variant: the tensor resident as a whole, or (rolling) set by set.  A rolling launch reads x once where the streaming
// pair reads it twice, and its sets overlap each other's loads, exchanges and stores; on cold tensors, rolling against the
// streaming pair: bf16 (8 / 12 / 16, 320, 128, 128) 39.1 / 58.3 / 76.7 against 48.1 / 70.7 / 99.0 us, float32
// (2, 256, 256, 256) 58.8 against 70.3, float16 (1, 256, 512, 512) 55.7 against 73.4; with a residual and the sum written,
// bf16 (16, 320, 128, 128) 145 against 193.  One set has to fit half of the device (resident_tiling): with groups inside a
// chunk, samples of 262144 rows of 128 bytes.
template <typename PT, int ACT, int NV, int ADD>
bool try_resident_fwd_nv(const FwdArgs &a, const FwdRecords &records, bool rolling) {
  if (NV < resident_min_rows()) return false;
  auto kernel_all = fused_fwd_kernel<elem_t, PT, kVec, ACT, NV, ADD, false>;  // every workgroup polls every tile
  auto kernel_two = fused_fwd_kernel<elem_t, PT, kVec, ACT, NV, ADD, true>;   // two-level exchange (many tiles)
  static const int slots = std::min(resident_slots(kernel_all), resident_slots(kernel_two));
  Plan p;
  if (rolling && cooperative_launches()) return false;  // the runtime refuses a cooperative grid larger than the device
  if (!resident_tiling(a.plan, a.plan.N, NV, slots, p, rolling)) return false;
  // A rolling launch works with 16 rows per lane while a set is at most an eighth of what is resident -- several sets are
  // then in every phase at any time -- and with 32 beyond that, where a set's exchange weighs more.  Where every workgroup polls
  // every tile, the exchange weighs more already: there a sample of 18 tiles or more keeps 16 rows only while the whole launch is at
  // most 4/3 of what is resident.  16 / 32 rows, us: with 1.2 - 1.3 of it bf16 (8, 320, 128, 128) 32.0 / 34.3, (6, 320, 100, 215)
  // 33.2 / 37.3, float32 (2, 256, 200, 210) 33.3 / 33.2; with 1.35 - 1.5 (2, 256, 200, 220) 37.2 / 34.5, (2, 256, 200, 250) 51.1 / 41.7,
  // bf16 (2, 512, 200, 230) 41.8 / 39.6; with 2.2 and more float32 (4, 256, 200, 250) 106 / 86, bf16 (16, 320, 128, 128) 75.1 / 71.0,
  // (20, 320, 96, 96) 54.0 / 48.1.  Shorter samples: bf16 (24, 320, 92, 92), 17 tiles, 55.9 / 62.4, (30, 640, 80, 80), 13, 99 / 102.  In
  // two levels float32 (4, 128, 256, 256) 52.4 / 60.9.  (With a residual, three workgroups of 16 rows to a CU, the first line alone, and
  // for 16-bit gelu, which the vector ALUs bound and which wants the wavefronts: (16, 320, 128, 128) 83.6 / 93.8; float32, half as many
  // elements to a row, (2, 256, 200, 250) 53.7 / 46.9, and 16-bit gelu_tanh (16, 320, 128, 128) 78.0 / 75.7.)
  const int64_t set = exchange_chunks(p) * p.tiles;
  constexpr int kTallSample = 18, kManyRecords = 900;
  constexpr bool alu_bound = sizeof(elem_t) == 2 && ACT == GN_ACT_GELU;
  const bool polled_by_all = ADD != kAddResidual && !alu_bound && !two_level_exchange(p) && p.tiles >= kTallSample;
  if (rolling && NV < 32 && (set > slots / 8 || (polled_by_all && p.nblocks * 3 > (int64_t)slots * 4))) return false;
  // A launch that is resident as a whole: the fourth workgroup per CU is not worth it where all of them poll nearly as many records
  // as are merged in two levels.  16 / 32 rows, us: float32 (1, 256, 200, 250), 980 records, 21.6 / 19.3, with a channel addend
  // 31.0 / 27.0; bf16 (1, 512, 200, 250) 23.4 / 22.7; but float32 (1, 256, 250, 256) in groups of 16, 750 records, 24.5 / 23.9 and
  // (1, 256, 256, 256) in groups of 32, 512, 23.1 / 23.5; bf16 (1, 512, 240, 250), two levels, 23.8 / 25.1.
  if (!rolling && NV == 16 && polled_by_all && exchange_records(p) > kManyRecords && p.nblocks > 3 * (kMaxResidentBlocks / 4)) return false;
  if (!resident_status()) return false;
  CapturedEpoch cap;
  if (!captured_epoch(a.stream, cap)) return false;
  ResidentOrder order(a.stream, cap.generation != nullptr);
  mark_resident_launch();
  ResidentWorkspace r = resident_fwd_ws(a.ws, p, records);
  arm_generation(r, cap);
  FusedFwdParams k = {};
  k.x = a.x;
  k.y = a.y;
  k.sync = r.sync;
  k.w = a.w;
  k.b = a.b;
  k.mean_out = a.mean;
  k.rstd_out = a.rstd;
  k.sdtype = a.sdtype;
  k.ydtype = a.ydtype;
  k.eps = (float)a.eps;
  k.add = a.add;
  k.p = p;
  launch(ADD != kAddNone ? kKindFusedFwdAdd : kKindFusedFwd, r.sync.two_level ? kernel_two : kernel_all, tile_grid(p, 0),
         dim3(kBlock), a.stream, k);
  note_resident_launch(ADD != kAddNone ? kKindFusedFwdAdd : kKindFusedFwd, NV, 0, 0, r.sync.two_level, 1, p.nblocks);
  return true;
}
template <typename PT, int ACT, int ADD> bool try_resident_fwd_add(const FwdArgs &a) {
  const FwdRecords records = resident_fwd_records(a.plan);
  if (try_resident_fwd_nv<PT, ACT, 4, ADD>(a, records, false) || try_resident_fwd_nv<PT, ACT, 8, ADD>(a, records, false) ||
      try_resident_fwd_nv<PT, ACT, 16, ADD>(a, records, false) || try_resident_fwd_nv<PT, ACT, 32, ADD>(a, records, false))
    return true;
  return records.rolling &&
         (try_resident_fwd_nv<PT, ACT, 16, ADD>(a, records, true) || try_resident_fwd_nv<PT, ACT, 32, ADD>(a, records, true));
}
template <typename PT, int ACT> bool try_resident_fwd_act(const FwdArgs &a) {
#if GN_PART_ADD
  // a sum of x and a channel addend alone, or a copy of x (sum_out only), needs no second tile
  return a.add.residual ? try_resident_fwd_add<PT, ACT, kAddResidual>(a) : try_resident_fwd_add<PT, ACT, kAddChannel>(a);
#else
  return try_resident_fwd_add<PT, ACT, kAddNone>(a);
#endif
}
template <typename PT> bool try_resident_fwd_pt(const FwdArgs &a) {
  switch (a.act) {
    case GN_ACT_IDENTITY: return try_resident_fwd_act<PT, GN_ACT_IDENTITY>(a);
    case GN_ACT_RELU: return try_resident_fwd_act<PT, GN_ACT_RELU>(a);
    case GN_ACT_SILU: return try_resident_fwd_act<PT, GN_ACT_SILU>(a);
    case GN_ACT_GELU: return try_resident_fwd_act<PT, GN_ACT_GELU>(a);
    default: return try_resident_fwd_act<PT, GN_ACT_GELU_TANH>(a);
  }
}
bool try_resident_fwd(const FwdArgs &a) {
  if (!resident_enabled() || a.plan.vec != kVec) return false;
  return a.pdtype == GN_INST_DTYPE ? try_resident_fwd_pt<elem_t>(a) : try_resident_fwd_pt<wide_param_t>(a);
}

#endif  // GN_PART_FWD || GN_PART_ADD

#if GN_PART_BWD
// A backward that no one launch can hold runs as a few launches over groups of samples where these fill the device well
// (80 % of the workgroups that can be resident), else as one launch set by set, as the forward does (try_resident_fwd_nv), in the form
// that holds the most rows per workgroup.  Full launches load, exchange and store in step and reach 5.6 TB/s; set by set, no
// launch is left half empty and no gap lies between two.  Launches against set by set: bf16 (16, 320, 128, 128), 83 % full,
// 89.5 / 96 us; (12, 320, 128, 128), 94 %, 80.5 / 89; float32 (2, 256, 256, 256), full, 73 / 76; at 78 % float32 (5, 320, 128, 128)
// 58.0 / 58.6 and bf16 (3, 640, 200, 200) 97 / 88; at 70 % bf16 (3, 640, 150, 160) 51.0 / 49.7, (9, 320, 128, 128) 61.6 / 48.8; at
// 68 % (5, 320, 140, 200) 60.7 / 49.3, (7, 320, 125, 160) 60.6 / 48.6.  Where only the streaming kernels were left: float32
// (1, 128, 512, 512) 107.9 / 73.7; for 16-bit data see try_resident_bwd_act.
// (set by set with 16 or 22 rows of both tensors in registers: bf16 (16, 320, 128, 128) 128 and 101 us.)
constexpr int kRolling = 0;  // in the place of a number of launches: one launch, set by set
template <typename PT, int ACT, int NV, int XW, int XL, bool EXACT, bool DY16>
bool try_resident_bwd_one(const BwdArgs &a, const BwdRecords &records, int batches, bool *underfilled);
template <typename PT, int ACT, int NV, int XW = 0, int XL = 0, bool EXACT = false>
bool try_resident_bwd_nv(const BwdArgs &a, const BwdRecords &records, int batches, bool *underfilled) {
  if (a.dydtype != GN_INST_DTYPE) {
    if constexpr (kHasDy16) return try_resident_bwd_one<PT, ACT, NV, XW, XL, EXACT, true>(a, records, batches, underfilled);
    else return false;
  }
  return try_resident_bwd_one<PT, ACT, NV, XW, XL, EXACT, false>(a, records, batches, underfilled);
}
template <typename PT, int ACT, int NV, int XW, int XL, bool EXACT, bool DY16>
bool try_resident_bwd_one(const BwdArgs &a, const BwdRecords &records, int batches, bool *underfilled) {
  if (NV < resident_min_rows()) return false;
  // (kernels that park rows of x in LDS have statistics slots for chunks of at most kBlock channels)
  if (XL > 0 && a.plan.lpr * a.plan.vec > kBlock) return false;
  auto kernel_all = fused_bwd_kernel<elem_t, PT, kVec, ACT, NV, false, XW, XL, DY16, EXACT>;
  auto kernel_two = fused_bwd_kernel<elem_t, PT, kVec, ACT, NV, true, XW, XL, DY16, EXACT>;
  static const int slots = std::min(resident_slots(kernel_all), resident_slots(kernel_two));
  const int64_t per = batches == kRolling ? a.plan.N : (a.plan.N + batches - 1) / batches;
  Plan p;
  const bool rolling = batches == kRolling;
  if (rolling && cooperative_launches()) return false;  // the runtime refuses a cooperative grid larger than the device
  if (!resident_tiling(a.plan, per, NV, slots, p, rolling)) return false;
  if (rolling && tail_blocks_per_chunk(p, a.plan.N) > p.tiles) return false;  // (tail_blocks relies on it)
  const int64_t count = rolling ? 1 : (a.plan.N + per - 1) / per;  // launches
  // (the windowed form addresses the rows of a tile by 32-bit byte offsets from the tile's first row)
  if (XW > 0 && (int64_t)p.tile_rows * p.C * (int64_t)sizeof(elem_t) >= ((int64_t)1 << 31)) return false;
  // the channel records of every sample stay in the workspace until the last launch has summed them
  const size_t crec_need = (size_t)a.plan.N * p.tiles * a.plan.C * 16;
  if (crec_need > (rolling ? records.crec : resident_crec_bytes((int64_t)p.lpr * p.vec))) return false;
  if (underfilled && a.plan.N * p.nchunk * p.tiles * 10 < count * slots * 8) {
    *underfilled = true;
    return false;
  }
  if (!resident_status()) return false;
  CapturedEpoch cap;
  if (!captured_epoch(a.stream, cap)) return false;
  ResidentOrder order(a.stream, cap.generation != nullptr);
  mark_resident_launch();
  const int64_t sample = a.plan.R * a.plan.C;
  const size_t ssz = stat_size(a.sdtype);
  for (int64_t n0 = 0; n0 < a.plan.N; n0 += per) {
    Plan pb = p;
    if (a.plan.N - n0 < per) resident_tiling(a.plan, a.plan.N - n0, NV, slots, pb);  // the last, shorter group
    pb.tiles = p.tiles;  // same row tiling in every group (it depends on R and NV only)
    ResidentWorkspace r = resident_bwd_ws(a.ws, pb, records);
    arm_generation(r, cap);
    const bool last = n0 + per >= a.plan.N;
    FusedBwdParams k = {};
    k.x = (const elem_t *)a.x + n0 * sample;
    k.dy = (const char *)a.dy + n0 * sample * stat_size(a.dydtype);
    k.dydtype = a.dydtype;
    k.dx = (elem_t *)a.dx + n0 * sample;
    k.mean = (const char *)a.mean + n0 * a.plan.G * ssz;
    k.rstd = (const char *)a.rstd + n0 * a.plan.G * ssz;
    k.w = a.w;
    k.b = a.b;
    k.sync = r.sync;
    k.dw = last ? a.dw : nullptr;
    k.db = last ? a.db : nullptr;
    k.mean_all = a.mean;
    k.rstd_all = a.rstd;
    k.n0 = n0;
    k.n_all = a.plan.N;
    k.sdtype = a.sdtype;
    k.tail_last = rolling ? 1 : 0;
    k.p = pb;
    launch(kKindFusedBwd, r.sync.two_level ? kernel_two : kernel_all, tile_grid(pb, 0), dim3(kBlock), a.stream, k);
    note_resident_launch(kKindFusedBwd, NV, XW, XL, r.sync.two_level, rolling ? 1 : batches, pb.nblocks);
  }
  return true;
}
template <typename PT, int ACT> bool try_resident_bwd_act(const BwdArgs &a) {
  // the form that keeps g' and reads most of x twice
  // (window: what the registers leave beside 32 rows of g', 16 rows for 16-bit data; parked: the rows of x that two
  // workgroups per CU can keep in LDS beside their reduction arrays, 14 x 4 KB for 16-bit data, 16 x 4 KB for float)
  constexpr int window = sizeof(elem_t) == 2 ? 16 : 12;
  constexpr int parked = sizeof(elem_t) == 2 ? 14 : 16;
  const BwdRecords records = resident_bwd_records(a.plan);
  const int most = a.plan.N < worthwhile_batches(a.plan) ? (int)a.plan.N : worthwhile_batches(a.plan);
  const auto launches = [&](int b, bool *underfilled) {
    if (try_resident_bwd_nv<PT, ACT, 4>(a, records, b, underfilled) || try_resident_bwd_nv<PT, ACT, 8>(a, records, b, underfilled) ||
        try_resident_bwd_nv<PT, ACT, 16>(a, records, b, underfilled) || try_resident_bwd_nv<PT, ACT, 22>(a, records, b, underfilled) ||
        try_resident_bwd_nv<PT, ACT, 32>(a, records, b, underfilled))
      return true;
    // too large for two tiles in registers: that form, before the tensor is cut into more launches (measured on bf16
    // (N, 320, 128, 128): 32.6 against 39.3 us at N = 5, 37.2 against 43.4 at N = 6)
    return try_resident_bwd_nv<PT, ACT, 32, window, parked>(a, records, b, underfilled) ||
           try_resident_bwd_nv<PT, ACT, 36, 8, parked>(a, records, b, underfilled);
  };
  bool underfilled = false;
  for (int b = 1; b <= most && !underfilled; ++b) {  // as few launches as it takes, each well filled ...
    if (launches(b, b > 1 ? &underfilled : nullptr)) return true;
  }
  // Set by set.  Where launches that keep g' could serve the call, so may the set-by-set form that does.  Where only the streaming
  // kernels could, which use g' in float, it is not rounded here either (EXACT; the identity's and relu's g', dy or 0, never is):
  // relative error of dx (2-norm), bf16 silu, 1.66e-3 as in the streaming kernels, 2.35e-3 with g' rounded.  The second
  // evaluation of the derivative, and a window that leaves it registers, cost bf16 (32, 320, 128, 128) 190 -> 218 us (streaming
  // 321), (1, 640, 256, 256) 50.9 -> 57.4 (77).  (A window of 16 rows spills 46 registers, 226 and 59.5 us.)
  constexpr bool rounds = sizeof(elem_t) == 2 && ACT != GN_ACT_IDENTITY && ACT != GN_ACT_RELU;
  constexpr int exact_window = 12;
  if (records.rolling && (underfilled || !rounds)) {
    if (try_resident_bwd_nv<PT, ACT, kRollingBwdRows, window, parked>(a, records, kRolling, nullptr)) return true;
  }
  if constexpr (rounds) {
    if (records.rolling && !underfilled && try_resident_bwd_nv<PT, ACT, kRollingBwdRows, exact_window, parked, true>(a, records, kRolling, nullptr))
      return true;
  }
  for (int b = 2; b <= most && underfilled; ++b) {  // ... or filled as they may be
    if (launches(b, nullptr)) return true;
  }
  return false;
}
template <typename PT> bool try_resident_bwd_pt(const BwdArgs &a) {
  switch (a.act) {
    case GN_ACT_IDENTITY: return try_resident_bwd_act<PT, GN_ACT_IDENTITY>(a);
    case GN_ACT_RELU: return try_resident_bwd_act<PT, GN_ACT_RELU>(a);
    case GN_ACT_SILU: return try_resident_bwd_act<PT, GN_ACT_SILU>(a);
    case GN_ACT_GELU: return try_resident_bwd_act<PT, GN_ACT_GELU>(a);
    default: return try_resident_bwd_act<PT, GN_ACT_GELU_TANH>(a);
  }
}
bool try_resident_bwd(const BwdArgs &a) {
  if (!resident_enabled() || a.plan.vec != kVec) return false;
  return a.pdtype == GN_INST_DTYPE ? try_resident_bwd_pt<elem_t>(a) : try_resident_bwd_pt<wide_param_t>(a);
}

#endif  // GN_PART_BWD
#endif  // GN_PART_STREAM

#if GN_PART_STREAM
// The single-launch kernel if the call fits one (64-bit data has none).
bool try_resident(const BwdArgs &a) {
  if constexpr (sizeof(A) != 4) return false;
  else return GN_CAT(try_resident_bwd_, GN_SUFFIX)(a);
}
bool try_resident(const FwdArgs &a) {
  if constexpr (sizeof(A) != 4) return false;
  else return a.has_add() ? GN_CAT(try_resident_fwd_added_, GN_SUFFIX)(a) : GN_CAT(try_resident_fwd_, GN_SUFFIX)(a);
}
template <int VEC> hipError_t fwd_impl(const FwdArgs &a) {
  if (VEC == kVec && !a.streaming_only && try_resident(a)) return hipGetLastError();
  note_streaming_call();
  if (a.has_add()) {
    // multi-launch form: materialise the sum (in sum_out, or in y when the caller does not want it), then
    // normalise it from there (in place when it sits in y)
    const Plan &p = a.plan;
    elem_t *dst = (elem_t *)(a.add.sum_out ? a.add.sum_out : a.y);
    if (a.add.residual && !a.add.channel_bias) {
      const int64_t nvec = p.N * p.R * p.C / VEC;
      const int64_t want = (nvec + 4 * kBlock - 1) / (4 * kBlock);
      const unsigned grid = (unsigned)(want < 8 * kNumCU ? (want > 0 ? want : 1) : 8 * kNumCU);
      launch(kKindAdd, (add_flat_kernel<elem_t, VEC>), dim3(grid), dim3(kBlock), a.stream, (const elem_t *)a.x,
             (const elem_t *)a.add.residual, dst, nvec);
    } else {
      launch(kKindAdd, (add_kernel<elem_t, VEC>), tile_grid(p, 0), dim3(kBlock), a.stream, (const elem_t *)a.x, a.add, dst,
             (const void *)a.ws, p);
    }
    FwdArgs plain = a;
    plain.x = dst;
    plain.add = AddArgs{nullptr, nullptr, a.add.channel_bias_dtype, nullptr};
    return fwd_impl<VEC>(plain);
  }
  const Plan &p = a.plan;
  const FwdWorkspace ws = fwd_workspace(p);
  A *base = (A *)((char *)a.ws + kWorkspaceHeader);
  A *part = base + ws.part, *compact = base + ws.compact;
  PartialGeo q = producer_geo(p);
  {
    launch(kKindFwdStats, (stats_kernel<elem_t, VEC>), tile_grid(p, 0), dim3(kBlock), a.stream, (const elem_t *)a.x, part, p,
           make_sweep(p, (double)kCacheBytes / (double)input_bytes(a)));
  }
  const A *src = part;
  const Plan c = consumer_plan(p, VEC * (int)sizeof(elem_t));
  if (needs_compaction(p, c)) {
    const int64_t items = p.N * p.G;
    const unsigned grid = (unsigned)((items + kBlock / 64 - 1) / (kBlock / 64));
    launch(kKindFwdStatsCompact, (stats_compact_kernel<A>), dim3(grid), dim3(kBlock), a.stream, (const A *)part, compact, q, p);
    q = compacted_geo(p);
    src = compact;
  }
  {
    if (a.pdtype == GN_INST_DTYPE) launch_apply_act<elem_t, VEC>(a, src, q, c);
    else launch_apply_act<wide_param_t, VEC>(a, src, q, c);
  }
  return hipGetLastError();
}

// Channels a workgroup of the dgamma / dbeta sums takes (a power of two; kBlock / columns lanes share a channel's
// `entries` tile sums): 32, a 256-byte line per entry, while that leaves a lane at most two rounds of four loads, fewer
// for more entries down to 8, a 64-byte sector.
int dwdb_columns(int64_t entries) {
  int cols = 32;
  while (cols > 8 && entries > 8 * (kBlock / cols)) cols >>= 1;
  return cols;
}
template <typename PT, int VEC, int ACT, bool DY16> void launch_bwd_act(const BwdArgs &a) {
  const Plan &p = a.plan;
  const BwdWorkspace ws = bwd_workspace(p);
  A *base = (A *)((char *)a.ws + kWorkspaceHeader);
  A *partC = base + ws.partC, *partG = base + ws.partG, *compactC = base + ws.compactC, *compactG = base + ws.compactG;
  PartialGeo q = producer_geo(p);
  {
    launch(kKindBwdReduce, (bwd_reduce_kernel<elem_t, PT, VEC, ACT, DY16>), tile_grid(p, 0), dim3(kBlock), a.stream,
                       (const elem_t *)a.x, (const elem_t *)a.dy, a.mean, a.rstd, a.sdtype, a.w, a.b, partC, partG, p, a.dydtype);
  }
  const A *srcC = partC, *srcG = partG;
  const Plan c = consumer_plan(p, VEC * (int)sizeof(elem_t));
  if (needs_compaction(p, c)) {
    const int nG = (int)((p.N * p.G + kBlock / 64 - 1) / (kBlock / 64));
    int cpb = 32;  // channels per workgroup: fewer when N C is small, so that about a CU's worth of workgroups exist
    while (cpb > 2 && p.N * p.C / cpb < kNumCU) cpb >>= 1;
    const int64_t nC = (p.N * p.C + cpb - 1) / cpb;
    launch(kKindBwdCompact, (bwd_compact_kernel<A>), dim3((unsigned)(nG + nC)), dim3(kBlock), a.stream, (const A *)partC,
           (const A *)partG, compactC, compactG, q, nG, cpb, p);
    q = compacted_geo(p);
    srcC = compactC;
    srcG = compactG;
  }
  {
    const int dcols = dwdb_columns(p.N * q.tiles);
    const int pieces = (c.lpr * c.vec + dcols - 1) / dcols;  // per chunk, handed out over the samples of the grid
    const int samples = (int)(p.N < 65535 ? p.N : 65535);
    const int extra = a.dw || a.db ? (pieces + samples - 1) / samples : 0;
    launch(kKindBwdDx, (bwd_dx_kernel<elem_t, PT, VEC, ACT, DY16>), tile_grid(c, extra), dim3(kBlock), a.stream,
                       (const elem_t *)a.x, (const elem_t *)a.dy, (elem_t *)a.dx, a.mean, a.rstd, a.sdtype, a.w, a.b, srcC,
                       srcG, q, a.dw, a.db, c, a.dydtype, dcols);
  }
}
template <typename PT, int VEC, bool DY16> void bwd_act_dy(const BwdArgs &a) {
  switch (a.act) {
    case GN_ACT_IDENTITY: launch_bwd_act<PT, VEC, GN_ACT_IDENTITY, DY16>(a); break;
    case GN_ACT_RELU: launch_bwd_act<PT, VEC, GN_ACT_RELU, DY16>(a); break;
    case GN_ACT_SILU: launch_bwd_act<PT, VEC, GN_ACT_SILU, DY16>(a); break;
    case GN_ACT_GELU: launch_bwd_act<PT, VEC, GN_ACT_GELU, DY16>(a); break;
    default: launch_bwd_act<PT, VEC, GN_ACT_GELU_TANH, DY16>(a); break;
  }
}
template <typename PT, int VEC> void bwd_act(const BwdArgs &a) {
  if constexpr (kHasDy16) {
    if (a.dydtype != GN_INST_DTYPE) return bwd_act_dy<PT, VEC, true>(a);
  }
  bwd_act_dy<PT, VEC, false>(a);
}
template <int VEC> hipError_t bwd_impl(const BwdArgs &a) {
  if (VEC == kVec && try_resident(a)) return hipGetLastError();
  note_streaming_call();
  if (a.pdtype == GN_INST_DTYPE) bwd_act<elem_t, VEC>(a);
  else bwd_act<wide_param_t, VEC>(a);
  return hipGetLastError();
}

#endif  // GN_PART_STREAM

}  // namespace

#if GN_PART_STREAM
// The widths below the full 16 bytes serve channel counts and addresses that only a half, a quarter or one element divides.
hipError_t GN_CAT(launch_fwd_, GN_SUFFIX)(const FwdArgs &a) {
  if (a.plan.vec == kVec) return fwd_impl<kVec>(a);
  if constexpr (kVec >= 8) if (a.plan.vec == 4) return fwd_impl<4>(a);
  if constexpr (kVec >= 4) if (a.plan.vec == 2) return fwd_impl<2>(a);
  return fwd_impl<1>(a);
}
hipError_t GN_CAT(launch_bwd_, GN_SUFFIX)(const BwdArgs &a) {
  if (a.plan.vec == kVec) return bwd_impl<kVec>(a);
  if constexpr (kVec >= 8) if (a.plan.vec == 4) return bwd_impl<4>(a);
  if constexpr (kVec >= 4) if (a.plan.vec == 2) return bwd_impl<2>(a);
  return bwd_impl<1>(a);
}
#elif GN_PART_FWD
bool GN_CAT(try_resident_fwd_, GN_SUFFIX)(const FwdArgs &a) { return try_resident_fwd(a); }
#elif GN_PART_BWD
bool GN_CAT(try_resident_bwd_, GN_SUFFIX)(const BwdArgs &a) { return try_resident_bwd(a); }
#else
bool GN_CAT(try_resident_fwd_added_, GN_SUFFIX)(const FwdArgs &a) { return try_resident_fwd(a); }
#endif

}  // namespace gn
