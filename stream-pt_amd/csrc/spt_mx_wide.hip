// spt_mx_wide.hip -- grouped MXFP4 x Q8_0 product for up to 64 list entries
// per pass over an expert's weights, on the gfx950 block-scaled MFMA
// (v_mfma_scale_f32_32x32x64_f8f6f4, A = E2M1, B = E2M3).
//
// One MFMA is one 32-element block of 32 weight rows x 32 entries:
//   A (32 rows x 64 K): lane l holds row l % 32; both half-waves hold the
//     same 16 nibble bytes of the MXFP4 block, as stored, and its E8M0 byte
//     as the scale.  Nothing is decoded.
//   B (64 K x 32 entries): lane l holds entry l % 32.  A Q8_0 code is split
//     exactly into two digits q = 16 h + l (h in [-8, 7], l in [0, 15]),
//     each an E2M3 value (digit / 8, exact for magnitudes up to 15): lanes
//     0-31 hold the h digits of the block's 32 codes with scale 2^(3+4),
//     lanes 32-63 the l digits with scale 2^3, both in nibble order
//     (position p <-> element (p >> 1) + 16 (p & 1)).
//   D = 2^(e-127) * sum(E2M1 * q) = isum * 2^(e-128) exactly (products and
//     partial sums are integers below 2^24 times one power of two), for e in
//     [4, 240]; D lane l, register r is row 8 (r/4) + 4 (l/32) + r%4, entry
//     l % 32 (lane layouts measured on the hardware).
//   acc = fma(D, d_x, acc) per block, the value of the integer form.
// A 32-row step holding an E8M0 outside [4, 240] in some row recomputes that
// row with the integer decode (keeps the reference's Inf/NaN semantics).
//
// What bounds it: an expert's weights are read once per 64 entries, so below
// about 64 entries the weight stream (HBM) is the floor, and beyond it the
// one FMA per output and block (16 per MFMA and lane, twice the MFMA's own
// cycles).  Measured at GPT-OSS-120B shape, gate/up + down: 2,000 tokens
// (8,000 selections, 62 per expert) 588 + 265 us, 0.47 PFLOP/s, 1.9 TB/s of
// weights; the bf16 MFMA form it replaces (16-row fragments, the weights in
// 96-byte row windows) took 1,016 + 462 us in the two slices it ran as; 512
// tokens, Zipf(1.1): the layer 452 -> 412 us.  Of a step's 10,000 cycles per
// compute unit the products take half, the waves' sums and the epilogue a
// quarter, waiting for loads the rest.

#include <type_traits>

#include "spt_device.h"
#include "spt_kernels.h"

namespace spt {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2s __attribute__((ext_vector_type(2)));
typedef unsigned u32x4s __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kStages = 3;
// Blocks of a row per stage, as the LDS allows: half a row, a whole row, a whole
// row of each of two row tiles.
constexpr int kMaxHalf = 45, kMaxRow = 48, kMaxRow2 = 24;
constexpr int kLoadWaves = 4;        // waves that issue the loads (one per SIMD)
constexpr int kPartsLds = kWaves * kWideRows * kGemmTokens * 4;  // the waves' partial sums of a step
constexpr int kStaticLds1 = 11 * 1024, kStaticLds2 = 19 * 1024;  // static LDS of a workgroup, rows in one part and in two
constexpr int kDownStores = 1, kActStores = 4;  // vector stores of an epilogue that stores (down; up step)
constexpr int kBiasWave = kLoadWaves - 1;  // loads the biases
constexpr int kEMin = 4, kEMax = 240;
constexpr int kXcds = 8;
constexpr uint32_t kOOR = 0x80000000u;  // buffer offset past every range: reads zero
constexpr int kVmcnt0 = 0x0F70;          // s_waitcnt vmcnt(0)
// 16-byte slots of a row's window in a stage: its blocks and up to 15 bytes
// before them; an odd number, so that 16 rows begin at 16 different groups of
// banks (2,560 inputs, 40 blocks a part: down of 105 experts 251 us with 44
// slots a row, every fourth row in the same banks).
__host__ __device__ constexpr int row_slots(int blocks) { return ((blocks * kMxBlock + 15 + 15) / 16) | 1; }
// 1 KB DMA loads of a stage of RT row tiles, and of each loading wave (the last
// of those waves has one fewer: the bias in its place).
template <int RT>
__host__ __device__ constexpr int stage_loads(int blocks) { return (RT * kWideRows * row_slots(blocks) + 63) / 64; }
template <int RT>
__host__ __device__ constexpr int wave_loads(int blocks) { return (stage_loads<RT>(blocks) + 1 + kLoadWaves - 1) / kLoadWaves; }
// Row slot p of a stage holds row slot_row(p), row r of a tile lies in its slot
// row_slot(r): rows 16-31 of a tile are rotated by one, so that the two rows
// whose slots are 16 apart (the same LDS banks) begin at different bytes of
// their first 16 (with 2,880 inputs a row is 10 bytes past a multiple of 16) and
// the 32 lanes' reads meet no bank twice.
__device__ inline int slot_row(int p) { return (p & 16) == 0 ? p : (p & ~15) + ((p + 1) & 15); }
__device__ inline int row_slot(int r) { return r < 16 ? r : 16 + ((r - 1) & 15); }
static_assert(2 * kMaxHalf >= kMxMaxInput / 32, "a row is at most two parts");
// dynamic LDS of a workgroup: the stages and the waves' partial sums
template <int RT>
constexpr int dynamic_lds(int blocks) { return kStages * 1024 * stage_loads<RT>(blocks) + kPartsLds; }
static_assert(dynamic_lds<1>(kMaxHalf) + kStaticLds2 <= 160 * 1024, "LDS, rows in two parts");
static_assert(dynamic_lds<1>(kMaxRow) + kStaticLds1 <= 160 * 1024, "LDS, rows in one part");
static_assert(dynamic_lds<2>(kMaxRow2) + kStaticLds1 <= 160 * 1024, "LDS, two row tiles");
static_assert(kGemmTokens == 64, "two 32-entry tiles per pass");

// Waits for a stage (the waves that load; the barrier after it does for the
// others): at most N operations may be outstanding, the loads of the stage
// issued after it and the stores of one epilogue.  The counter retires
// in order, so every wave must issue exactly these since (anything more only
// makes the wait longer): loads and stores are never skipped by a branch but
// given an offset past the range.
template <int N>
__device__ __attribute__((always_inline)) inline void wait_stage(int wave) {
    if (wave < kLoadWaves)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
    else
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

__device__ __attribute__((always_inline)) inline void raw_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The kernel's arguments where they lie in memory (`p`, the kernel's own
// argument segment: only a kernel may ask for it), read where they are used
// by scalar loads rather than held in scalar registers across the loop.
typedef __attribute__((address_space(4))) const MxWideArgs WideArgs;
__device__ __attribute__((always_inline)) inline WideArgs &wide_args(WideArgs *p) {
    asm volatile("" : "+s"(p));
    return *p;
}
#define SPT_INLINE __attribute__((always_inline))

// The value of the lane 16 (32) away, and the larger of it and this lane's.
__device__ __attribute__((always_inline)) inline float max_permlane16(float v) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __attribute__((always_inline)) inline float max_permlane32(float v) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
// (after the swap of two copies the first holds the low half's values in
// both halves, the second the high half's)
__device__ __attribute__((always_inline)) inline uint32_t other_half(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32) ? (uint32_t)r[0] : (uint32_t)r[1];
}

// 16-byte slot of a wave's partial sums: row quad rq (0..7) of entry t of a
// tile.  The entries of quad rq are permuted, so that the epilogue's lanes (4
// or 8 entries times all quads) spread over the banks as well as the writes
// (all 32 entries of a quad) do.
__device__ __attribute__((always_inline)) inline int part_slot(int tile, int rq, int t) { return tile * 256 + rq * 32 + (t ^ (4 * rq)); }

// Where a workgroup stands in its range of units: (slot, pass, unit) with
// the slot's expert, list begin and entry count.
struct Walk {
    int slot, p, u, e, begin, count;
};

// A value that is the same in every lane, in a scalar register.
__device__ __attribute__((always_inline)) inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __attribute__((always_inline)) inline void walk_slot(const WideArgs &a, Walk &w) {
    w.e = uniform(a.active[w.slot]);
    w.begin = uniform(a.offsets[w.e]);
    w.count = uniform(a.offsets[w.e + 1]) - w.begin;
}

// Next unit (the caller has one left); true when the pass changed.
__device__ __attribute__((always_inline)) inline bool walk_next(const WideArgs &a, Walk &w, int units) {
    if (++w.u < units) return false;
    w.u = 0;
    if (++w.p * kGemmTokens >= w.count) {
        w.p = 0;
        ++w.slot;
        walk_slot(a, w);
    }
    return true;
}

// Integer-decode dot of one weight row with one entry's Q8_0 row (rows with
// special E8M0 scales).
__device__ float lut_dot(const ByteView &v, uint32_t row_pos, int nb, const int8_t *codes, const uint8_t *tab) {
    float acc = 0.0f;
    const uint32_t *cw = reinterpret_cast<const uint32_t *>(codes);
    for (int b = 0; b < nb; b++) {
        uint32_t d[5], o;
        load_block5(v, row_pos + (uint32_t)b * kMxBlock, d, &o);
        MxDecoded dec;
        mx_decode(d, o, dec);
        uint32_t q[8];
#pragma unroll
        for (int k = 0; k < 8; k++) q[k] = cw[b * 8 + k];
        const int32_t s = mx_isum(dec, q);
        const float dx = *reinterpret_cast<const float *>(tab + (size_t)b * kDigitBytes + digit_scale(0));
        acc = __builtin_fmaf((float)s, mx_block_scale(dx, dec.e), acc);
    }
    return acc;
}

}  // namespace

// Persistent workgroups of eight waves, one per CU.  A unit is RT tiles of 32
// outputs: gate/up takes it in two steps (its gate rows, then its up rows),
// down in one.  The packing deals each workgroup a contiguous range of
// (expert, pass of 64 entries, unit) whose cost is its share of the whole
// (k_pack), so a workgroup changes pass once or twice in a launch.
//
// The eight waves split K, not the entries: within each part of a row wave w
// multiplies blocks w, w + 8, ..., so its B digits for all 64 entries stay in
// registers for the whole pass (P * NJ blocks x 2 tiles x 6 VGPRs) and every
// weight byte is read from LDS once.  Short rows leave a wave a block or two of
// that: with RT = 2 four waves split K on the first 32 rows of a step, four on
// the next (the last step's second tile may lie past the rows: its results go
// nowhere).  Weights come by LDS DMA in stages of one part (half a row beyond
// 48 blocks) of a step's rows -- a ring of three stages, two in flight while one
// is multiplied; a row's part is contiguous in memory, so a stage is 32 or 64
// runs of up to 765 bytes.
//
// The waves' partial sums of a step meet in LDS, and each output's partials
// (eight, or four with RT = 2) are added in wave order, so it does not depend
// on its entry's place in the list.  A wave takes eight entries of a two-tile
// pass (four of a one-tile pass), all 32 rows of a tile, so a 32-element Q8_0
// block of act stays within it.  This epilogue of a step runs at the start of
// the next one.
template <int MODE, int P, int NJ, int RT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_mx_wide(MxWideArgs) {
    constexpr int kSub = MODE == kGateUp ? 2 : 1;  // steps per unit
    constexpr int KS = kWaves / RT, kStepRows = RT * kWideRows;  // parts of K; rows of a step
    constexpr int kBlocks = P == 2 ? kMaxHalf : RT == 1 ? kMaxRow : kMaxRow2;
    constexpr int kLoads = wave_loads<RT>(NJ * KS < kBlocks ? NJ * KS : kBlocks);
    static_assert(RT == 1 || P == 1, "rows in parts: one row tile");
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ uint32_t s_bias[8][64];      // raw bias dwords of a step's rows
    __shared__ int s_ent[2][kGemmTokens];   // per pass parity: list entries (-1 past the end)
    __shared__ uint32_t s_apos[kLoads][64 * kLoadWaves];  // each loading thread's offsets of a stage
    __shared__ v4f s_gate[MODE == kGateUp && P == 2 ? kThreads : 1];  // gate sums of a unit, for its up step
    __shared__ uint32_t s_spare[256];       // where the loads past a stage's go
    __shared__ uint32_t s_special[2][RT];   // per step parity and row tile: rows with special scales

    WideArgs *const args = (WideArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    WideArgs &a = wide_args(args);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The lane's roles, from the lane index made opaque where they are used:
    // the addresses derived from it are recomputed (a few VALU operations)
    // rather than held across the loop, whose registers are full.
    auto lane_now = [&]() SPT_INLINE {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    const int kp = RT == 1 ? wave : wave % KS, rt = RT == 1 ? 0 : wave / KS;  // the wave's part of K and row tile
    const int nb = a.nb, units = (a.rows + kStepRows - 1) / kStepRows;
    const uint32_t row_bytes = (uint32_t)nb * kMxBlock;
    const int G = gridDim.x;
    // the ranges are dealt XCD-major (workgroup b runs on XCD b % 8), so
    // passes over one expert share an L2
    const int vb = (G % kXcds == 0) ? ((int)blockIdx.x % kXcds) * (G / kXcds) + (int)blockIdx.x / kXcds : (int)blockIdx.x;
    const int32_t *st = a.start + (size_t)vb * kGvStartWords;
    const int n_units = uniform(st[0]);
    if (n_units <= 0) return;
    Walk cur;
    cur.slot = uniform(st[1]);
    cur.p = uniform(st[2]);
    cur.u = uniform(st[3]);
    cur.e = uniform(st[4]);
    cur.begin = uniform(st[5]);
    cur.count = uniform(st[6]);

    // parts of a row, and this lane's share of a stage's loads: load i =
    // wave + kLoadWaves * k fills 16-byte slots 64i .. 64i+63 (slot q: row q / slots,
    // piece q % slots)
    const int nb0 = P == 1 ? nb : (nb + 1) / 2;
    const int slots = row_slots(nb0);
    const int nloads = stage_loads<RT>(nb0);
    const uint32_t stage_bytes = 1024u * (uint32_t)nloads;
#pragma unroll
    for (int k = 0; k < kLoads; k++) {
        if (wave >= kLoadWaves) break;
        const int q = 64 * (wave + kLoadWaves * k) + lane, r = q / slots, pc = q - r * slots;
        s_apos[k][tid] = r < kStepRows ? (uint32_t)slot_row(r) * row_bytes + 16u * (uint32_t)pc : kOOR;
    }
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    typedef __attribute__((address_space(3))) const uint32_t lds_cu32;
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_u8 *)lds);
    const uint32_t bias0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_u8 *)&s_bias[0][0]);
    const uint32_t spare0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_u8 *)&s_spare[0]);
    uint8_t *parts = lds + kStages * stage_bytes;
    if (tid < 2 * RT) (&s_special[0][0])[tid] = 0u;

    // ---- the issue side: walks ahead of the multiply -----------------------
    Walk iw = cur;
    int i_left = n_units, i_sub = 0, i_part = 0, i_stage = 0, i_step = 0;
    const uint32_t expert_bytes = (uint32_t)a.expert_bytes;  // (mx_wide_fits)
    // the expert's matrices (gate/up: both) of the issue side and, of the
    // multiply, their offsets in the first 16 bytes
    uint64_t i_mb[kSub];
    uint32_t c_le[kSub];
    auto matrices = [&](const Walk &w, uint64_t (&mb)[kSub]) SPT_INLINE {
        WideArgs &a = wide_args(args);
#pragma unroll
        for (int m = 0; m < kSub; m++) mb[m] = reinterpret_cast<uintptr_t>(a.w[m]) + (uint64_t)w.e * expert_bytes;
    };
    matrices(iw, i_mb);
#pragma unroll
    for (int m = 0; m < kSub; m++) c_le[m] = (uint32_t)i_mb[m] & 15u;
    // Load k of this wave of the next stage; past the range it reads nothing
    // (and fills its slots, or the spare ones past a stage's loads, with
    // zeros), so that every wave and stage counts the same loads.
    auto issue_load = [&](const u32x4v &rs, int k, uint32_t adv, int ln) SPT_INLINE {
        const uint32_t ap = s_apos[k][64 * wave + ln];  // (written by the same thread)
        const int i = wave + kLoadWaves * k;
        dma16_nt_other_stage(rs, i < nloads ? lds0 + (uint32_t)i_stage * stage_bytes + 1024u * (uint32_t)i : spare0,
                             (ap + adv) & ~15u, 0u);
    };
    // the raw dwords holding a step's 32 bias elements (zeros without a bias)
    auto issue_bias = [&](int ln) SPT_INLINE {
        WideArgs &a = wide_args(args);
        const int m = MODE == kGateUp ? i_sub : 0;
        const uintptr_t bb = reinterpret_cast<uintptr_t>(a.bias[m]);
        const uint32_t lead = (uint32_t)(bb & 3u);
        const u32x4v rb = rsrc_words(reinterpret_cast<const void *>(bb - lead), a.bias[m] ? (uint32_t)((a.bias_bytes[m] + lead + 3u) & ~3ull) : 0u);
        const uint32_t idx = (uint32_t)iw.e * (uint32_t)a.rows + (uint32_t)(iw.u * kStepRows + (ln & (kStepRows - 1)));
        const uint32_t off = (lead + idx * (a.bias_type[m] == 0 ? 4u : 2u)) & ~3u;
        dma4(rb, bias0 + 256u * (uint32_t)(i_step & 7), i_left > 0 && ln < kStepRows ? off : kOOR, 0u);
    };
    // after them: on to the next stage
    auto issue_end = [&]() SPT_INLINE {
        i_stage = i_stage == kStages - 1 ? 0 : i_stage + 1;
        if (P == 2 && i_part == 0) {
            i_part = 1;
            return;
        }
        i_part = 0;
        i_step++;
        if (kSub == 2 && i_sub == 0) {
            i_sub = 1;
            return;
        }
        i_sub = 0;
        if (--i_left > 0) {
            const int slot = iw.slot;
            walk_next(wide_args(args), iw, units);
            if (iw.slot != slot) matrices(iw, i_mb);
        }
    };
    auto issue = [&]() SPT_INLINE {
        if (wave >= kLoadWaves) {
            issue_end();
            return;
        }
        // (offsets past 2^31 are past every matrix: mx_wide_fits)
        const uint64_t mb = kSub == 2 && i_sub ? i_mb[kSub - 1] : i_mb[0];
        const uint32_t le = (uint32_t)mb & 15u;
        // from the 16-byte boundary at or below the matrix to the one at or
        // above its end
        const u32x4v rs = rsrc_words(reinterpret_cast<const void *>(mb - le), (expert_bytes + le + 15u) & ~15u);
        const uint32_t adv = i_left > 0 ? le + (uint32_t)(iw.u * kStepRows) * row_bytes + (P == 2 && i_part ? (uint32_t)nb0 * kMxBlock : 0u) : kOOR;
        const int ln = lane_now();
#pragma unroll
        for (int k = 0; k < kLoads - 1; k++) issue_load(rs, k, adv, ln);
        // the last loading wave has one load fewer (kBiasWave): the bias in its place
        if (wave == kBiasWave && i_part == 0)
            issue_bias(ln);
        else
            issue_load(rs, kLoads - 1, adv, ln);
        issue_end();
    };
    issue();
    issue();

    // ---- the pass: entries to LDS, B digits and d_x to registers -------------
    v8i B[P][NJ][2];
    f16x2 dx[P][NJ];
    int ntile = 0, parity = 1;
    auto load_pass = [&]() SPT_INLINE {
        WideArgs &a = wide_args(args);
        parity ^= 1;
        const int ln = lane_now(), l32 = ln & 31, half = ln >> 5;
        const int base = cur.begin + cur.p * kGemmTokens, nt = min(kGemmTokens, cur.count - cur.p * kGemmTokens);
        ntile = (nt + 31) >> 5;
        if (tid < kGemmTokens) s_ent[parity][tid] = tid < nt ? a.list[base + tid] : -1;
        const rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.tab), (short)0, (int)a.tab_bytes, kRsrcWord3);
        // entries past the end repeat the first (their results go nowhere)
        uint32_t tpos[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int ent = a.list[base + (32 * t + l32 < nt ? 32 * t + l32 : 0)];
            tpos[t] = (uint32_t)(MODE == kGateUp ? ent / a.topk : ent) * (uint32_t)nb * (uint32_t)kDigitBytes;
        }
        // A block's two 16-byte pieces lie in one 64-byte line: they are asked
        // for together (every block's first piece before any second one fetched
        // the lines twice: down at 2,000 tokens 264.7 -> 267.1 us).
        uint32_t d[P][NJ][2];
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int so = KS * kDigitBytes * j;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    // (past the part: some block's digits, or zeros, with d_x = 0)
                    const uint32_t o = tpos[t] + (uint32_t)((p * nb0 + kp) * kDigitBytes);
                    const u32x4 lo = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rt, o + 16u * (uint32_t)half + so, 0, 0));
                    const u32x4 hi = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rt, o + 16u * (uint32_t)half + 32u + so, 0, 0));
                    B[p][j][t] = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, 0, 0};
                    d[p][j][t] = hi.z;
                }
                asm volatile("" ::: "memory");
            }
        // All of it arrives here: waited for where the products use it, the
        // compiler's waits of every later step would drain the loads of the next
        // stages too (512 tokens, Zipf(1.1): gate/up 179.9 -> 178.1 us).
        __builtin_amdgcn_s_waitcnt(kVmcnt0);
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const bool ok = kp + KS * j < (p ? nb - nb0 : nb0);
                asm volatile("" : "+v"(d[p][j][0]), "+v"(d[p][j][1])::"memory");
                // exact: d_x is an fp16 value
                dx[p][j] = f16x2{(_Float16)(ok ? __uint_as_float(d[p][j][0]) : 0.0f), (_Float16)(ok ? __uint_as_float(d[p][j][1]) : 0.0f)};
                asm volatile("" : "+v"(dx[p][j]));
            }
    };

    v16f acc[2];
    uint32_t emin, emax;
    // this wave's blocks of part p in buffer `buf`
    auto multiply = [&](auto nt_c, auto p_c, int stage, uint32_t lead) SPT_INLINE {
        constexpr int NT = decltype(nt_c)::value, p = decltype(p_c)::value;
        const int ln = lane_now(), l32 = ln & 31;
        const int sb = ln < 32 ? 134 : 130;  // B scale: digit / 8, times 16 for h
        const uint32_t pos = lds0 + (uint32_t)stage * stage_bytes + (uint32_t)((kWideRows * rt + row_slot(l32)) * slots) * 16u + lead +
                             (uint32_t)(kp * kMxBlock);
        lds_cu32 *pa = reinterpret_cast<lds_cu32 *>((uintptr_t)(pos & ~3u));
        const uint32_t sel = 0x04030201u + (pos & 3u) * 0x01010101u, esh = (pos & 3u) * 8u;
        const int cnt = p ? nb - nb0 : nb0;
        uint32_t d[5];
#pragma unroll
        for (int i = 0; i < 5; i++) d[i] = pa[i];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const bool ok = kp + KS * j < cnt;
            const uint32_t e = __builtin_amdgcn_ubfe(d[0], esh, 8u);
            emin = min(emin, ok ? e : 127u);
            emax = max(emax, ok ? e : 127u);
            const int sa = ok ? (int)e : 127;  // past the part: d_x = 0 times a finite value
            const v8i A = {(int)__builtin_amdgcn_perm(d[1], d[0], sel), (int)__builtin_amdgcn_perm(d[2], d[1], sel),
                           (int)__builtin_amdgcn_perm(d[3], d[2], sel), (int)__builtin_amdgcn_perm(d[4], d[3], sel), 0, 0, 0, 0};
            // the next block's reads fly during this one's products; blocks KS
            // (4 or 8) apart are 17 or 34 dwords apart: one alignment
            if (j + 1 < NJ) {
#pragma unroll
                for (int i = 0; i < 5; i++) d[i] = pa[KS * kMxBlock / 4 * (j + 1) + i];
            }
            const v16f z = {};
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const v16f D = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B[p][j][t], z, 4, 2, 0, sa, 0, sb);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[t][r] = __builtin_fmaf(D[r], (float)dx[p][j][t], acc[t][r]);
                if (P == 2) __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- the epilogue of the previous step ---------------------------------------
    v4f gate_sums[RT];  // s_gate where registers are left (rows in one part; the LDS goes to longer stages)
    int q_u = 0, q_e = 0, q_sub = 0, q_par = 0, q_ntile = 0, q_step = 0;
    // NT tiles, row tile S: lane l of wave v takes TW = 4 NT entries' rows, R =
    // 2 NT rows each: entry TW * v + l % TW, rows R * (l / TW) .. + R - 1.
    auto epilogue_of = [&](auto nt_c, auto s_c) SPT_INLINE {
        constexpr int NT = decltype(nt_c)::value, S = decltype(s_c)::value, TW = 4 * NT, R = 2 * NT;
        typedef float vRf __attribute__((ext_vector_type(R)));
        typedef uint32_t vRu __attribute__((ext_vector_type(R)));
        WideArgs &a = wide_args(args);
        const int ln = lane_now(), t = TW * wave + (ln & (TW - 1)), r0 = R * (ln / TW);
        const int tile = q_u * RT + S;  // of 32 rows
        const vRf *pp = reinterpret_cast<const vRf *>(parts + S * KS * (kPartsLds / kWaves) + part_slot(t >> 5, r0 >> 2, t & 31) * 16 + 4 * (r0 & 3));
        vRf y[KS];
#pragma unroll
        for (int w = 0; w < KS; w++) y[w] = pp[w * (kPartsLds / kWaves / (4 * R))];
        const int m = MODE == kGateUp ? q_sub : 0;
        const vRu braw = *reinterpret_cast<const vRu *>(&s_bias[q_step & 7][kWideRows * S + r0]);
        vRf s = y[0];
#pragma unroll
        for (int w = 1; w < KS; w++)
#pragma unroll
            for (int i = 0; i < R; i++) s[i] += y[w][i];
        // (a last step's tile past the rows goes nowhere)
        const int ent = RT == 1 || tile * kWideRows < a.rows ? s_ent[q_par][t] : -1;
        const uint32_t spec = s_special[q_step & 1][S];
        if (spec && ent >= 0) {
            const ByteView cv = make_view((MODE == kGateUp && q_sub ? a.w[1] : a.w[0]) + (uint64_t)q_e * a.expert_bytes,
                                          a.expert_bytes);
            const size_t ar = MODE == kGateUp ? ent / a.topk : ent;
            for (int i = 0; i < R; i++) {
                if (!((spec >> (r0 + i)) & 1u)) continue;
                const float v = lut_dot(cv, (uint32_t)(tile * kWideRows + r0 + i) * row_bytes, nb, a.codes + ar * nb * 32,
                                        a.tab + ar * nb * kDigitBytes);
#pragma unroll
                for (int k = 0; k < R; k++) s[k] = k == i ? v : s[k];
            }
        }
        const int bt = a.bias_type[m];
        if (bt == 0) {
#pragma unroll
            for (int i = 0; i < R; i++) s[i] += __uint_as_float(braw[i]);
        } else {
            // (rows per expert are even, so the element's parity is the row's)
            const uint32_t blead = (uint32_t)(reinterpret_cast<uintptr_t>(a.bias[m]) & 3u);
#pragma unroll
            for (int i = 0; i < R; i++) {
                const uint32_t h = (((uint32_t)i * 2u + blead) & 2u) ? braw[i] >> 16 : braw[i] & 0xFFFFu;
                const float f16 = f16_bits_to_f32(h);
                s[i] += bt == 1 ? f16 : __uint_as_float(h << 16);
            }
        }
        if constexpr (MODE == kDown) {
            const rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(a.out, (short)0, (int)kOOR, kRsrcWord3);
            const uint32_t o = ent < 0 ? kOOR : ((uint32_t)ent * (uint32_t)a.rows + (uint32_t)(tile * kWideRows + r0)) * 4u;
            if constexpr (R == 4)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4s, s), ro, o, 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2s, s), ro, o, 0, 0);
            return;
        }
        // (a gate sum is read back by the thread that wrote it, in the same pass)
        v4f *const sg = &s_gate[P == 2 ? 64 * wave + ln : 0];
        if (q_sub == 0) {
#pragma unroll
            for (int i = 0; i < R; i++)
                if (P == 1) gate_sums[S][i] = s[i];
            if (P == 2) *reinterpret_cast<vRf *>(sg) = s;
            return;
        }
        vRf gv;
#pragma unroll
        for (int i = 0; i < R; i++) gv[i] = gate_sums[S][i];
        if (P == 2) gv = *reinterpret_cast<const vRf *>(sg);
        vRf act;
        {
            float g[R], u[R], v[R];
#pragma unroll
            for (int i = 0; i < R; i++) g[i] = gv[i], u[i] = s[i];
            swiglu_n<R>(g, u, v);
#pragma unroll
            for (int i = 0; i < R; i++) act[i] = v[i];
        }
        float amax = 0.0f;
        bool nan = false;
#pragma unroll
        for (int i = 0; i < R; i++) {
            nan |= act[i] != act[i];
            amax = fmaxf(amax, __builtin_fabsf(act[i]));  // (a NaN operand loses)
        }
        // over the entry's lanes (l % TW alike)
        amax = fmaxf(amax, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, amax), 0x128, 0xF, 0xF, false)));
        if (TW == 4) amax = fmaxf(amax, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, amax), 0x124, 0xF, 0xF, false)));
        amax = max_permlane16(amax);
        amax = max_permlane32(amax);
        const bool nan_any = ((__ballot(nan) >> (ln & (TW - 1))) & (TW == 8 ? 0x0101010101010101ull : 0x1111111111111111ull)) != 0;
        const float d = nan_any ? __builtin_nanf("") : amax / 127.0f;
        const float rd = 1.0f / d, id = d != 0.0f ? rd : 0.0f;
        const uint16_t dh = __builtin_bit_cast(uint16_t, static_cast<_Float16>(d));  // (a NaN d is the quiet one: 0x7e00)
        uint32_t qw = 0;  // the R codes
#pragma unroll
        for (int i = 0; i < R; i++) qw |= (uint32_t)(q8_code(act[i] * id) & 0xff) << (8 * i);
        const uint32_t qo = other_half(qw);  // elements 16 away
        // digits of elements r0 % 16 .. + R - 1 and 16 away: positions 2 (r0 %
        // 16) .. + 2 R - 1; the lanes of the low elements store the h digits,
        // the others the l digits
        const int g = ln >> 5;
        const uint32_t qlo = g ? qo : qw, qhi = g ? qw : qo;
        const uint32_t gm = g ? 0xFFFFFFFFu : 0u;  // (selects without a branch)
        const uint32_t dl = (gm & qlo & 0x0F0F0F0Fu) | (~gm & e2m3_high4(qlo)), dh4 = (gm & qhi & 0x0F0F0F0Fu) | (~gm & e2m3_high4(qhi));
        // bytes (low, high, low, high) of elements 2k, 2k + 1 -> 24 bits
        const uint32_t w0 = pack6x4(__builtin_amdgcn_perm(dh4, dl, 0x05010400u));
        const uint32_t w1 = R == 4 ? pack6x4(__builtin_amdgcn_perm(dh4, dl, 0x07030602u)) : 0u;
        const uint64_t w = (uint64_t)w0 | (uint64_t)w1 << 24;
        // Four stores, always: codes, the two pieces of the digits (which begin
        // at 3 R/2 bytes times an odd or even number: the 16-bit or 8-bit piece
        // first where odd) and the scale.
        const uint32_t blk = (uint32_t)ent * (uint32_t)(a.rows / kWideRows) + (uint32_t)tile;
        const rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(a.act_codes, (short)0, (int)kOOR, kRsrcWord3);
        const rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(a.act_tab, (short)0, (int)kOOR, kRsrcWord3);
        const uint32_t oc = ent < 0 ? kOOR : blk * 32u + (uint32_t)r0, ot = ent < 0 ? kOOR : blk * (uint32_t)kDigitBytes;
        const int o6 = 3 * ((r0 & 15) >> 1), odd = ((r0 & 15) / R) & 1;
        const uint32_t big = ot + (uint32_t)digit_byte(g, o6 + (odd ? R / 2 : 0)), small = ot + (uint32_t)digit_byte(g, odd ? o6 : o6 + R);
        if constexpr (R == 4) {
            __builtin_amdgcn_raw_buffer_store_b32(qw, rc, oc, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)(odd ? w >> 16 : w), rt, big, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(odd ? w : w >> 32), rt, small, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b16((uint16_t)qw, rc, oc, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(odd ? w0 >> 8 : w0), rt, big, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(odd ? w0 : w0 >> 16), rt, small, 0, 0);
        }
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(f16_bits_to_f32(dh)), rt, (r0 & 15) == 0 ? ot + digit_scale(g) : kOOR, 0, 0);
        if (ent >= 0 && (a.tap[0] || a.tap[1] || a.out || a.act_blocks34)) {
            const size_t o = (size_t)ent * a.rows + tile * kWideRows + r0;
            if (a.tap[0]) *reinterpret_cast<vRf *>(a.tap[0] + o) = gv;
            if (a.tap[1]) *reinterpret_cast<vRf *>(a.tap[1] + o) = s;
            if (a.out) *reinterpret_cast<vRf *>(a.out + o) = act;
            if (a.act_blocks34) {
                uint8_t *b34 = a.act_blocks34 + (size_t)blk * kQ80Block;
                if (r0 == 0) {
                    b34[0] = (uint8_t)(dh & 0xff);
                    b34[1] = (uint8_t)(dh >> 8);
                }
#pragma unroll
                for (int i = 0; i < R; i++) b34[2 + r0 + i] = (uint8_t)(qw >> (8 * i));
            }
        }
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    auto epilogue = [&]() SPT_INLINE {
        if (q_ntile == 2) {
            epilogue_of(C2{}, C0{});
            if constexpr (RT == 2) epilogue_of(C2{}, C1{});
        } else {
            epilogue_of(C1{}, C0{});
            if constexpr (RT == 2) epilogue_of(C1{}, C1{});
        }
    };

    // ---- the steps -----------------------------------------------------------------
    int stage = 0;
    bool fresh = true;
    int sub = 0, left = n_units;
    for (int step = 0;; step++) {
        // since this stage's loads: the next stage's, and the epilogue of step - 2
        // (which stored if it was an up step, as this one then is)
        if (MODE == kDown && step > 1)
            wait_stage<kLoads + RT * kDownStores>(wave);
        else if (MODE == kGateUp && step > 1 && sub == 1)
            wait_stage<kLoads + RT * kActStores>(wave);
        else
            wait_stage<kLoads>(wave);
        raw_barrier();  // this stage has landed; the previous step's partial sums are in place
        issue();
        if (step > 0) epilogue();
        if (fresh) {
            load_pass();
            fresh = false;
        }
        const uint32_t rpos = (kSub == 2 && sub ? c_le[kSub - 1] : c_le[0]) + (uint32_t)(cur.u * kStepRows + kWideRows * rt + (lane_now() & 31)) * row_bytes;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
        emin = 127u;
        emax = 127u;
        if (ntile == 2)
            multiply(C2{}, C0{}, stage, rpos & 15u);
        else
            multiply(C1{}, C0{}, stage, rpos & 15u);
        stage = stage == kStages - 1 ? 0 : stage + 1;
        if constexpr (P == 2) {
            // since: the next stage's loads and the epilogue of step - 1
            if (MODE == kDown && step > 0)
                wait_stage<kLoads + RT * kDownStores>(wave);
            else if (MODE == kGateUp && step > 0 && sub == 0)
                wait_stage<kLoads + RT * kActStores>(wave);
            else
                wait_stage<kLoads>(wave);
            raw_barrier();  // this stage; every wave is past the epilogue
            issue();
            if (step > 0 && tid < RT) s_special[q_step & 1][tid] = 0u;
            const uint32_t lead = (rpos + (uint32_t)nb0 * kMxBlock) & 15u;
            if (ntile == 2)
                multiply(C2{}, C1{}, stage, lead);
            else
                multiply(C1{}, C1{}, stage, lead);
            stage = stage == kStages - 1 ? 0 : stage + 1;
        } else {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            raw_barrier();  // every wave is past the epilogue
            if (step > 0 && tid < RT) s_special[q_step & 1][tid] = 0u;
        }
        const int ln = lane_now();
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (t < ntile) {
#pragma unroll
                for (int m = 0; m < 4; m++)
                    reinterpret_cast<v4f *>(parts)[wave * (kPartsLds / kWaves / 16) + part_slot(t, 2 * m + (ln >> 5), ln & 31)] =
                        v4f{acc[t][4 * m], acc[t][4 * m + 1], acc[t][4 * m + 2], acc[t][4 * m + 3]};
            }
        }
        const uint64_t sm = __ballot(emin < (uint32_t)kEMin || emax > (uint32_t)kEMax);
        if (sm && ln == 0) atomicOr(&s_special[step & 1][rt], (uint32_t)sm | (uint32_t)(sm >> 32));
        q_u = cur.u;
        q_e = cur.e;
        q_sub = sub;
        q_par = parity;
        q_ntile = ntile;
        q_step = step;
        if (kSub == 2 && sub == 0) {
            sub = 1;
            continue;
        }
        sub = 0;
        if (--left == 0) break;
        const int slot = cur.slot;
        fresh = walk_next(wide_args(args), cur, units);
        if (cur.slot != slot) {
            uint64_t mb[kSub];
            matrices(cur, mb);
#pragma unroll
            for (int m = 0; m < kSub; m++) c_le[m] = (uint32_t)mb[m] & 15u;
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    raw_barrier();
    epilogue();
}

int mx_wide_grid() { return device_cus(); }

template <int MODE, int P, int NJ, int RT>
static hipError_t launch_wide_form(hipStream_t s, const MxWideArgs &a, int nb0) {
    // one-time opt-in to more than 64 KB of dynamic LDS
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mx_wide<MODE, P, NJ, RT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       dynamic_lds<RT>(P == 2 ? kMaxHalf : RT == 1 ? kMaxRow : kMaxRow2));
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((k_mx_wide<MODE, P, NJ, RT>), dim3(mx_wide_grid()), dim3(kThreads), dynamic_lds<RT>(nb0), s, a);
    return hipGetLastError();
}

// Rows of a step of a launch over rows of nb blocks: two row tiles as long as
// their stages fit the LDS and there are five steps or more for a workgroup.  A
// step's exchange of partial sums, its barriers and the start of its loads cost
// about 4,000 cycles however short the rows are (at 90 blocks the whole step is
// 10,000); with few steps the last one, twice as long, costs as much.  Us, one
// tile / two: gate/up of 256 experts of 512 x 512, two entries each (8 steps a
// workgroup) 74.9 / 58.1, 768 x 768 (12) 110 / 86.6; 128 experts, eight each, (4)
// 40.6 / 32.8, (6) 58.6 / 47.6; 32 experts, 64 each, (1) 19.9 / 19.9, (1.5) 27.6 /
// 31.1; layers of 768 x 768 with three to four steps 2 to 5 us the longer.
// `passes` is a lower bound: the experts in use are not known here.
int mx_wide_unit_rows(int nb, int rows, int passes) {
    const int64_t steps = (int64_t)passes * ((rows + 2 * kWideRows - 1) / (2 * kWideRows));
    return nb <= kMaxRow2 && steps >= 5 * mx_wide_grid() ? 2 * kWideRows : kWideRows;
}

// The form with exactly the blocks per wave and part of this row, rounded up:
// a block past the part costs its products, a load past the stage's its issue
// (1,536 inputs, 128 experts, gate/up and down: 162 + 77 us in two parts with four
// blocks a wave and 28 loads a stage, 139 + 64 with three and 15, 136 + 60 in one
// part of six).
template <int MODE>
static hipError_t launch_wide_mode(hipStream_t s, const MxWideArgs &a) {
    if (a.unit_rows == 2 * kWideRows) {
        switch ((a.nb + 3) / 4) {
        case 1:
        case 2: return launch_wide_form<MODE, 1, 2, 2>(s, a, a.nb);
        case 3: return launch_wide_form<MODE, 1, 3, 2>(s, a, a.nb);
        case 4: return launch_wide_form<MODE, 1, 4, 2>(s, a, a.nb);
        case 5: return launch_wide_form<MODE, 1, 5, 2>(s, a, a.nb);
        default: return launch_wide_form<MODE, 1, 6, 2>(s, a, a.nb);
        }
    }
    if (a.nb <= kMaxRow) {
        switch ((a.nb + kWaves - 1) / kWaves) {
        case 1:
        case 2: return launch_wide_form<MODE, 1, 2, 1>(s, a, a.nb);
        case 3: return launch_wide_form<MODE, 1, 3, 1>(s, a, a.nb);
        case 4: return launch_wide_form<MODE, 1, 4, 1>(s, a, a.nb);
        case 5: return launch_wide_form<MODE, 1, 5, 1>(s, a, a.nb);
        default: return launch_wide_form<MODE, 1, 6, 1>(s, a, a.nb);
        }
    }
    const int nb0 = (a.nb + 1) / 2;
    switch ((nb0 + kWaves - 1) / kWaves) {
    case 4: return launch_wide_form<MODE, 2, 4, 1>(s, a, nb0);
    case 5: return launch_wide_form<MODE, 2, 5, 1>(s, a, nb0);
    default: return launch_wide_form<MODE, 2, 6, 1>(s, a, nb0);
    }
}
static_assert((kMaxRow + 2) / 2 > 3 * kWaves, "a half row is four blocks a wave or more");

hipError_t launch_mx_wide(hipStream_t s, GemvMode mode, const MxWideArgs &a) {
    if (a.rows <= 0) return hipSuccess;
    if (a.nb <= 0 || a.nb > 2 * kMaxHalf || a.rows % kWideRows != 0 || !a.start || !mx_wide_fits(a.expert_bytes) ||
        (a.unit_rows != kWideRows && (a.unit_rows != 2 * kWideRows || a.nb > kMaxRow2)))
        return hipErrorInvalidConfiguration;
    if (mode == kGateUp) return launch_wide_mode<kGateUp>(s, a);
    if (mode == kDown) return launch_wide_mode<kDown>(s, a);
    return hipErrorInvalidValue;
}

#undef SPT_INLINE

}  // namespace spt
