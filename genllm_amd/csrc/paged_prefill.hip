// paged_prefill.hip -- causal paged FlashAttention on bf16 MFMA (gfx950).
//
// Same result as the attention loop of PagedAttentionImpl<CPU>::execute
// (src/backend/cpu/attention.cpp:148-215) for a chunk of S queries: query s sits
// at q_abs = n_cached - S + s and attends keys 0..q_abs (causal, :164-181),
// kv head = q head / groups (:158).
//
// Rows: the queries of a q head or, in short chunks and split launches, the S x
// groups (query, q head) pairs of a kv head, q heads fastest, in row tiles of 64
// (fewer where CUs would stay idle), so a short chunk fills its tiles.  Grid: row
// tiles x (batch entry, head) pairs, workgroups of 8 waves: the long half of the
// row tiles from the last down, then the short half from the first up; or, where
// that would leave the chip idle, row tiles x key splits, merged by a second
// kernel (prefill_splits).
// All batch entries go in one launch: two prompts of 1000 tokens (16 q / 8 kv
// heads of 128) 16.9 us in one launch of 512 workgroups, 29.5 us in two.
// Wave w = qb + 4 kh owns row block qb (16 rows) of the tile and key
// part kh (32 keys) of every key tile of 64 tokens (4 pages; 128 tokens and
// four parts in the 16-wave form, below), so the two key
// halves of a row block share a SIMD (waves w and w + 4; measured 30.9
// against 31.5 us at config 4 and 47.4 against 48.1 us at head_dim 256 with
// the halves of two row blocks paired instead); the two halves of a row
// block are merged through LDS at the end.  At
// head_dim 128 a workgroup holds 66 KB of LDS and at most 128 VGPRs per lane,
// so two workgroups share a CU (4 waves per SIMD: one workgroup's barrier
// waits and dependent chains are filled by the other's work); the grid's
// order puts a long and a short row tile on each CU.  At head_dim 256 (130
// KB) one workgroup runs per CU.
// Key tiles are staged in two LDS buffers (one tile in flight while the other
// is computed), K and V each as [token][dim] rows whose 16-byte chunks are
// swizzled per 256-byte half: chunk c of row r sits at position
// 16 (c / 16) + ((c % 16) ^ swz(r % 16)), with swz(r) = 2 ((r % 8) ^ 4 (r / 8))
// + r / 8.
// Wave w < 4 (8 in the 16-wave form) moves the K rows, then the V rows of page w of every tile
// straight from HBM into LDS with 16-byte buffer loads in LDS mode (lane i's
// 16 bytes land at base + 16 i), so a tile costs no registers, no VALU and no
// LDS store instructions; one buffer resource per
// page (base = the page of this kv head, size = the bytes its rows below the
// key limit span) bounds every load.  The other waves issue no loads.
// Per tile and wave:
//   S^T = K Q^T  (v_mfma_f32_16x16x32_bf16 x 2 D/32; A = K from LDS: lane l ->
//        key l%16, dims 32ks+8(l/16)..; B = Q^T held in registers).
//        D[key][q] lands in lane q%16 + 16*(key/4), register key%4: every
//        lane holds 4 keys of ONE query row per 16-key block, so the online
//        softmax state (m, l) of a row is per lane.
//   O^T += V^T P^T  (v_mfma_f32_16x16x32_bf16 x D/16, full rate: 32 keys; B =
//        P^T is the lane's own 8 exponentials; A = V^T from two
//        ds_read_b64_tr_b16 per 16 dims).  O^T[dim][q] belongs to the lane's
//        own query column, so the rescale by 2^(m_old-m_new) stays lane-local.
// Causal masking is applied only to the key parts that reach past the first
// query of the wave (the diagonal) or past the cache end.
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace genllm {

namespace {

constexpr int KH = 32;          // keys of a tile per wave (the K dimension of the P.V MFMA)
constexpr int QW = 16;          // rows per wave (one 16-column block of O^T)
constexpr int QT = 4 * QW;      // rows per row tile: 4 row blocks
constexpr int IDS_BLOCK = 64;   // tiles whose page ids one vector load brings
constexpr int kMaxPrefillSplits = 32;

// Unsigned division by a divisor known at launch (Granlund and Montgomery,
// "Division by invariant integers using multiplication", 1994, figure 4.1):
// exact for every 32-bit dividend, four instructions where the compiler's
// division takes about thirty (17 queries of 17 keys, 16 q / 8 kv heads: 5.8 ->
// 5.4 us; 300 of 2000: 21.2 -> 20.3 us).
struct FastDiv {
    uint32_t m = 1;
    uint16_t s1 = 0, s2 = 0;
    FastDiv() = default;
    explicit FastDiv(uint32_t d) {
        uint32_t l = 0;
        while (l < 32 && (uint64_t(1) << l) < d) ++l;
        m = uint32_t(((uint64_t(1) << 32) * ((uint64_t(1) << l) - d)) / d + 1);
        s1 = uint16_t(l ? 1 : 0);
        s2 = uint16_t(l ? l - 1 : 0);
    }
    __device__ __forceinline__ int operator()(int x) const {
        const uint32_t t = __umulhi(m, uint32_t(x));
        return int((t + ((uint32_t(x) - t) >> uint32_t(s1))) >> uint32_t(s2));
    }
};

// What a launch adds to the attention parameters: batch entries (element
// strides between them) and the key splits.  The kernels take it ahead of
// AttnParams, in this order, so that what the prologue reads of both lies in
// the first four 64-byte lines of the argument block: every line is fetched
// anew in each launch, and with the fields spread over six of them, or held in
// scalar registers through the tile loop, a launch took 0.3-0.5 us longer
// (late_args; both: 16 q / 8 kv heads, 1700 tokens 24.0 against 24.7 us, 2048
// tokens 29.0 against 29.4; 8 / 2 heads of 256, 2048 tokens 42.7 against 43.5;
// medians of three traces each, taken in turn).
struct PrefillGrid {
    int64_t q_batch = 0, o_batch = 0, kv_batch = 0;
    int32_t batch = 1, n_splits = 1;
    int32_t tile_rows = QT;    // rows per row tile: 16, 32 or 64
    int32_t pack = 1;          // q heads whose rows share row tiles: the groups of a kv head, or 1
    int32_t units = 1;         // batch entries x (q heads / pack)
    // pack, units, q heads / pack, groups / pack, kv heads, n_splits
    int32_t n_rt = 0;          // row tiles of a unit
    FastDiv by_units, by_heads, by_groups, by_pack, by_splits, by_hkv;
    float* partial = nullptr;  // n_splits > 1: o [split][unit][row][D], then {m, l} [split][unit][row]
};

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) float lds_float;

struct NoAppend {};
template <bool kNew>
using AppendArg = std::conditional_t<kNew, PrefillAppend, NoAppend>;

// chunk-position swizzle of a 256-byte LDS row, bijective on r % 16.  The
// K reads (16 rows, one chunk each) hit 16 distinct positions.  A transposing
// V read takes 32 bytes (one chunk pair) of each of 16 rows, and the LDS
// serves it in two halves, lanes 0-15 with 32-47 (rows 0-3 and 8-11 of the
// 16) and lanes 16-31 with 48-63 (rows 4-7 and 12-15): the XOR with 4 (r / 8)
// puts the chunk pairs of rows r and r + 8 in different halves of the row,
// so each half of the read covers all 64 banks once (PMC: 2 conflict cycles
// per transposing read without it, none with it; config 4 34.3 -> 33.3 us)
__device__ __forceinline__ constexpr int swz(int r) { return (((r & 7) ^ ((r >> 1) & 4)) << 1) | ((r >> 3) & 1); }

__device__ __forceinline__ s16x4_t ds_read_tr(const lds_char* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        reinterpret_cast<__attribute__((address_space(3))) s16x4_t*>(const_cast<lds_char*>(p)));
}

// Workgroup barrier for the tile pipeline.  A release fence here would wait
// for every LDS-mode load still in flight (they write LDS); the tiles are
// instead waited for explicitly, by count, before it.  The LDS reads before
// it have all been consumed (their results feed the MFMAs), and the empty
// asm statements keep the compiler from moving memory accesses across it.
__device__ __forceinline__ void tile_barrier() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

// The key part kh (keys KT t + KH kh .. + KH - 1 of every key tile t) below
// wave_end, for query q0 + n16 (lane n16 + 16 g), formed the reference's way:
// per query over the keys it sees, in fp32, one key after another.  res: the
// O^T values of the lane's dims 16 db + 4 g + i, then m (log2 units) and l
// (the row's, in lane g = 0; 0 elsewhere, as the hand-over adds the four
// lanes).  Called only by waves whose tiled state came out NaN or infinite.
template <int D, bool F16, int KT, bool kNew>
__device__ __forceinline__ void prefill_exact_part(const AttnParams& p, const uint16_t* qrow, int64_t kv_off, int hkv, int s_row,
                                                   int kh, int wave_end, int t_begin, int t_end, float* res) {
    using E = Elem<F16>;
    constexpr int KS = D / 32, DB = D / 16;
    const int g = (threadIdx.x & 63) >> 4;
    const int n_cached = p.n_cached;
    const int lim = p.causal ? min(p.n_cached - p.S + s_row + 1, n_cached) : n_cached;
    const bool paged = p.k_ids != nullptr;
    const float c = fmaxf(p.scale_log2, __FLT_MIN__);
    float m = -INFINITY, l = 0.0f;
    f32x4_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = t_begin; t < t_end; ++t) {
        for (int j = 0; j < KH; ++j) {
            const int tok = t * KT + KH * kh + j;
            if (tok >= wave_end) break;  // wave-uniform
            const int64_t in_page = int64_t(tok % kPage) * p.kv_row;
            const uint16_t *krow, *vrow;
            if (kNew && tok >= p.new_from) {  // appended by this call: its pages may not be written yet
                const int64_t at = hkv * p.new_head_stride + int64_t(tok - p.new_from) * p.new_tok_stride;
                krow = p.k_new + at;
                vrow = p.v_new + at;
            } else {
                krow = p.k_pool + kv_off + (paged ? int64_t(p.k_ids[tok / kPage]) * p.page_elems + in_page : int64_t(tok) * p.kv_row);
                vrow = p.v_pool + kv_off + (paged ? int64_t(p.v_ids[tok / kPage]) * p.page_elems + in_page : int64_t(tok) * p.kv_row);
            }
            float sp = 0.0f;  // this lane's dims 32 ks + 8 g .. + 7, then the row's four lanes
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const uint4 qq = *reinterpret_cast<const uint4*>(qrow + 32 * ks + 8 * g);
                const uint4 kk = *reinterpret_cast<const uint4*>(krow + 32 * ks + 8 * g);
                const uint32_t qw[4] = {qq.x, qq.y, qq.z, qq.w}, kw[4] = {kk.x, kk.y, kk.z, kk.w};
#pragma unroll
                for (int w2 = 0; w2 < 4; ++w2) {
                    sp = __builtin_fmaf(E::lo(qw[w2]), E::lo(kw[w2]), sp);
                    sp = __builtin_fmaf(E::hi(qw[w2]), E::hi(kw[w2]), sp);
                }
            }
            sp += __shfl_xor(sp, 16);
            sp += __shfl_xor(sp, 32);
            const bool vis = tok < lim;
            const float x = sp * c;
            const float mn = vis ? __builtin_fmaxf(m, x) : m;
            const float alpha = m == -INFINITY ? 0.0f : exp2_fast(m - mn);
            const float pk = exp2_fast(x - mn);
            l = vis ? __builtin_fmaf(l, alpha, pk) : l;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const uint2 u = *reinterpret_cast<const uint2*>(vrow + 16 * db + 4 * g);
                const float v4[4] = {E::lo(u.x), E::hi(u.x), E::lo(u.y), E::hi(u.y)};
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[db][i] = vis ? __builtin_fmaf(pk, v4[i], acc[db][i] * alpha) : acc[db][i];
            }
            m = mn;
        }
    }
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) res[4 * db + i] = acc[db][i];
    res[4 * DB] = m;
    res[4 * DB + 1] = g == 0 ? l : 0.0f;
}

// The launch arguments as they lie in a kernel's argument block (pa where it
// appends).  late_args() reads them where they are used: after the tile loop,
// or in the one step that patches a page.  Taken from the kernel's parameters
// they are held in scalar registers through the loop (head_dim 128: 97 instead
// of 76, and 20-50 spilled in the forms that append: a 512-token chunk of 8192
// keys 101.0 -> 98.0 us).
struct KernelArgs {
    PrefillGrid gr;
    AttnParams p;
    PrefillAppend pa;
};
__device__ __forceinline__ const KernelArgs& late_args() {
    typedef const __attribute__((address_space(4))) KernelArgs args_t;
    args_t* a = (args_t*)__builtin_amdgcn_kernarg_segment_ptr();
    __asm__ volatile("" : "+s"(a));
    return *(const KernelArgs*)a;
}

// The op's append, inside the attention launch: the chunk's K and V rows
// ([Hkv][S][D]) copied to their page slots bit for bit, 16 bytes per thread and
// step, kCopy steps in flight; workgroup 0 also writes the ids of the pages
// opened by this call into the device table.  The attention reads the chunk's
// rows from k_new / v_new, so nothing waits for these stores; the waves that
// have handed their state over run it while the others write the output (at
// the start of the kernel it cost every workgroup 2.5 us).  tid of n_threads:
// the thread among those of the workgroup that take part.
constexpr int kCopy = 4;
template <int D>
__device__ __forceinline__ void append_chunk(int tid, int n_threads) {
    const KernelArgs& a = late_args();
    const AttnParams& p = a.p;
    const PrefillGrid& gr = a.gr;
    const PrefillAppend& pa = a.pa;
    constexpr int CH = D / 8;  // 16-byte chunks per row
    const int half = p.S * p.Hkv * CH;
    const int64_t step = int64_t(gridDim.x) * n_threads;
    if (blockIdx.x == 0)
        for (int i = tid; i < pa.upd.count; i += n_threads) {
            p.k_ids_w[pa.upd.first + i] = pa.upd.k[i];
            p.v_ids_w[pa.upd.first + i] = pa.upd.v[i];
        }
    for (int64_t i0 = int64_t(blockIdx.x) * n_threads + tid; i0 < 2 * int64_t(half); i0 += kCopy * step) {
        uint4 x[kCopy];
        uint16_t* dst[kCopy];
#pragma unroll
        for (int u = 0; u < kCopy; ++u) {
            const int64_t i = i0 + u * step;
            dst[u] = nullptr;
            if (i < 2 * int64_t(half)) {
                const bool v = i >= half;
                const int j = int(v ? i - half : i), row = j / CH, c = j % CH;
                const int t = gr.by_hkv(row), h = row - t * p.Hkv, pos = p.new_from + t;
                const int rel = pos / kPage - pa.upd.first;
                const int id = rel >= 0 && rel < pa.upd.count ? (v ? pa.upd.v : pa.upd.k)[rel] : (v ? p.v_ids : p.k_ids)[pos / kPage];
                x[u] = *reinterpret_cast<const uint4*>((v ? p.v_new : p.k_new) + h * p.new_head_stride + t * p.new_tok_stride + 8 * c);
                if (id >= 0 && id < pa.max_blocks)
                    dst[u] = (v ? p.v_pool_w : p.k_pool_w) + id * p.page_elems + (pos % kPage) * p.kv_row + h * D + 8 * c;
            }
        }
#pragma unroll
        for (int u = 0; u < kCopy; ++u)
            if (dst[u]) *reinterpret_cast<uint4*>(dst[u]) = x[u];
    }
}

template <int D, bool F16, bool kSplit, int KQ, bool kNew>
__device__ __forceinline__ void prefill_tiles(const AttnParams& p, const PrefillGrid& gr) {
    using E = Elem<F16>;
    constexpr int KS = D / 32, DB = D / 16;
    constexpr int ROWB = D * 2;       // bytes per token row (256 or 512)
    constexpr int KT = KQ * KH;       // keys per tile
    constexpr int KP = KT / kPage;    // pages per tile
    constexpr int TILEB = KT * ROWB;  // bytes of K (or V) per tile
    constexpr int XO = DB * 4 * 64;   // floats a wave hands over at the end: O^T, [value][lane]
    static_assert(KQ == 2 || KQ == 4, "key parts per tile");
    static_assert(KQ * XO * 4 <= 2 * TILEB, "a buffer holds the hand-overs of KQ waves");
    __shared__ __attribute__((aligned(16))) char lds_b0[2 * TILEB];
    __shared__ __attribute__((aligned(16))) char lds_b1[2 * TILEB];
    __shared__ float lds_ml[2 * KQ][2][64];  // m and l handed over
    lds_char* const buf0 = (lds_char*)lds_b0;
    lds_char* const buf1 = (lds_char*)lds_b1;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qblk = wv & 3, kh = wv >> 2;  // row block, key part (waves w, w + 4, ... share a SIMD)
    const int n16 = lane & 15, g = lane >> 4;
    const int pack = gr.pack, R = p.S * pack;  // rows of a unit: row r is q head r % pack of query r / pack
    const int tile_rows = gr.tile_rows;
    const int n_rt = gr.n_rt;
    // Workgroup i runs on XCD i % 8: with the (batch entry, head) pairs fastest
    // and 8 kv heads, XCD x holds kv head x (single q heads, in multiples of 8:
    // q heads [x heads / 8, (x + 1) heads / 8)) and its tiles are read through
    // one L2 (config 4: FETCH_SIZE 16.2 against 24.2 MiB per launch
    // with a kv head's rows spread over two XCDs)
    const int units = gr.units, heads = kSplit ? p.Hkv : pack == 1 ? p.Hq : p.Hkv;
    const int rank = gr.by_units(int(blockIdx.x));
    const int unit = int(blockIdx.x) - rank * units;
    const int bat = gr.by_heads(unit);
    int hg = unit - bat * heads;  // the unit's heads: hg * pack .. + pack - 1
    if (!kSplit && pack == 1 && (heads & 7) == 0) hg = (hg & 7) * (heads >> 3) + (hg >> 3);
    const int hkv = kSplit ? hg : gr.by_groups(hg);
    // Unsplit: the first half of the grid runs the row tiles with the most
    // keys, from the last tile down; the second half the others from the first
    // tile up, so that workgroups i and i + half the grid -- the two a CU holds
    // when every workgroup is resident (head_dim 128: 512 workgroups of two per
    // CU at 16 heads) -- carry the same sum of key tiles (A/B at config 4:
    // 34.5-34.7 against 36.0-36.2 us with the second half running down too).
    // Split: every workgroup has about the same number of key tiles.
    const int half = (n_rt + 1) / 2;
    const int rt = kSplit ? gr.by_splits(rank) : rank < half ? n_rt - 1 - rank : rank - half;
    const int sp = kSplit ? rank - rt * gr.n_splits : 0;
    const int qabs0 = p.n_cached - p.S;
    const int q0 = rt * tile_rows + qblk * QW;  // first row of the wave
    const int n_cached = p.n_cached;

    // Q^T operands: lane -> row q0 + n16, dims 32ks + 8g..+7 (a row past the
    // last one loads the last row: its column stays finite and is not written)
    const int row = min(q0 + n16, R - 1);
    const int s_row = gr.by_pack(row);  // the row's query
    const uint16_t* const qrow = p.q + bat * gr.q_batch + int64_t(hg * pack + (row - s_row * pack)) * p.q_head_stride +
                                 int64_t(s_row) * p.q_tok_stride;
    uint4 qb[KS];  // raw 16-bit elements
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qb[ks] = *reinterpret_cast<const uint4*>(qrow + 32 * ks + 8 * g);
    float m = -INFINITY, l = 0.0f;
    // nm = -m (0 while m = -inf); th = the raw score above which the scaled
    // score exceeds m + 8 (-inf while m = -inf)
    float nm = 0.0f, th = -INFINITY;
    f32x4_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int s_last = gr.by_pack(min(rt * tile_rows + tile_rows, R) - 1);  // last query of the workgroup
    const int kv_last = p.causal ? min(qabs0 + s_last + 1, n_cached) : n_cached;
    const int n_tiles = (kv_last + KT - 1) / KT;
    // key tiles [t_begin, t_end) of this workgroup; keys at or past kv_end are
    // another split's, or no row of the tile sees them
    const int t_begin = kSplit ? gr.by_splits(n_tiles * sp) : 0;  // n_tiles * 32 < 2^31
    const int t_end = kSplit ? gr.by_splits(n_tiles * (sp + 1)) : n_tiles;
    const int kv_end = kSplit ? min(kv_last, t_end * KT) : kv_last;
    const bool wave_has_rows = q0 < R && qblk * QW < tile_rows;
    // keys below wave_lim are visible to every row of the wave, keys at or
    // past wave_end to none of them (or not this split's)
    const int wave_lim = p.causal ? min(qabs0 + gr.by_pack(q0) + 1, n_cached) : n_cached;
    const int wave_end = !wave_has_rows ? 0
                         : p.causal     ? min(qabs0 + gr.by_pack(min(q0 + QW, R) - 1) + 1, kv_end)
                                        : kv_end;

    // ---- staging: wave w < KP moves page w of each tile, its K rows, then its
    // V rows; the other half of the waves issue no tile loads.  (8 waves:) waves
    // 4-7 share their SIMDs with waves 0-3 and reach their S^T MFMAs after them, so the step waits
    // for them: keeping the loads' issue off their path measured 31.3 against
    // 31.5 us at config 4 and 48.9 against 50.2 us at head_dim 256 (A/B on one
    // box; the mirror split, waves 4-7 loading, 32.2 and 50.7).  Every K row
    // of the tile is requested before any V row (needed first): 30.6 against
    // 30.9 us at config 4, 47.0 against 47.3 at head_dim 256, against one
    // kind per wave over two pages.
    const bool paged = p.k_ids != nullptr;
    const int pg = wv & (KP - 1);  // this wave's page of the tile (the first KP waves)
    const bool dma_wave = wv < KP;
    const int64_t head_off = bat * gr.kv_batch + int64_t(hkv) * (p.kv_head_stride ? p.kv_head_stride : D);
    const int64_t kv_row = p.kv_row, page_elems = p.page_elems;
    const int kv_row_bytes = int(kv_row) * 2;
    // lane i <- the K (kindx 0) or V (1) id of page pg of tile t0 + i
    auto load_ids = [&](int t0, int kindx) -> int {
        const int page = KP * (t0 + lane) + pg;
        const int end = kNew ? min(kv_end, p.new_from) : kv_end;  // pages that hold earlier tokens
        return page * kPage < end ? (kindx ? p.v_ids : p.k_ids)[page] : 0;
    };
    // instruction e fills rows RPI e .. RPI e + RPI-1 of the page (4 rows of
    // 256 B at D = 128, 2 of 512 B at D = 256): lane -> row RPI e + lane/LPR,
    // position p = lane % LPR <- chunk 16 (p/16) + ((p%16) ^ swz(row))
    constexpr int LPR = ROWB / 16, RPI = 64 / LPR, NI = kPage / RPI;  // lanes per row, rows per load, loads per page
    uint32_t dma_off[NI];
#pragma unroll
    for (int e = 0; e < NI; ++e) {
        const int row = RPI * e + lane / LPR, pos = lane % LPR;
        const int chunk = 16 * (pos >> 4) + ((pos & 15) ^ swz(row));
        dma_off[e] = uint32_t(row * kv_row_bytes + 16 * chunk);
    }

    // The buffer resource of a page spans exactly its rows below kv_end, so
    // rows past the causal limit, the cache end or the table read as zeros:
    // their keys are masked and their zero values meet zero probabilities.
    // kNew: pages that hold only tokens of this call's chunk are read from its
    // own rows, which follow each other (ROWB bytes apart); of the page where
    // the chunk starts only the earlier rows are loaded here (patch_page).
    const int new_from = kNew ? __builtin_amdgcn_readfirstlane(p.new_from) : INT_MAX;
    const uint16_t* const k_chunk = kNew ? p.k_new + hkv * p.new_head_stride - int64_t(new_from) * D : nullptr;
    const uint16_t* const v_chunk = kNew ? p.v_new + hkv * p.new_head_stride - int64_t(new_from) * D : nullptr;
    // kAny: the page may hold tokens of the chunk.
    auto issue_page = [&](auto any, int t, int ids, lds_char* buf, int kindx) {  // K (0) or V (1) rows of page pg of tile t
        constexpr bool kAny = decltype(any)::value;
        const int tok_page = t * KT + kPage * pg;
        if constexpr (!kAny) {
            const uint16_t* const src = (kindx ? p.v_pool : p.k_pool) + head_off;
            const int valid = min(max(kv_end - tok_page, 0), kPage);
            const uint32_t span = uint32_t(__builtin_amdgcn_readfirstlane(valid > 0 ? (valid - 1) * kv_row_bytes + ROWB : 0));
            const int64_t base = paged ? int64_t(__builtin_amdgcn_readlane(ids, t & (IDS_BLOCK - 1))) * page_elems
                                       : int64_t(tok_page) * kv_row;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(src + base), 0, span, kBufferFlags);
#pragma unroll
            for (int e = 0; e < NI; ++e)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    r, (__attribute__((address_space(3))) void*)(buf + (kindx * TILEB + pg * (kPage * ROWB) + e * 1024)), 16,
                    dma_off[e], 0, 0, 0);
        } else {
            const int ahead = tok_page - new_from;
            const bool fresh = ahead >= 0;
            const uint16_t* const src = fresh ? (kindx ? v_chunk : k_chunk) : (kindx ? p.v_pool : p.k_pool) + head_off;
            const int64_t base = fresh ? int64_t(tok_page) * D
                                       : int64_t(__builtin_amdgcn_readlane(ids, t & (IDS_BLOCK - 1))) * page_elems;
            const int row_bytes = fresh ? ROWB : kv_row_bytes, less = kv_row_bytes - row_bytes;
            const int rows = min(max(kv_end - tok_page, 0), kPage), valid = fresh ? rows : min(rows, -ahead);
            const uint32_t span = uint32_t(__builtin_amdgcn_readfirstlane(valid > 0 ? (valid - 1) * row_bytes + ROWB : 0));
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(src + base), 0, span, kBufferFlags);
            const uint32_t lane_less = uint32_t(lane / LPR) * uint32_t(less);
#pragma unroll
            for (int e = 0; e < NI; ++e)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    r, (__attribute__((address_space(3))) void*)(buf + (kindx * TILEB + pg * (kPage * ROWB) + e * 1024)), 16,
                    dma_off[e] - lane_less - uint32_t(RPI * e) * uint32_t(less), 0, 0, 0);
        }
    };
    // The chunk's rows of the page where it starts inside a page, into the
    // landed tile (the loads above left zeros there).
    auto patch_page = [&](lds_char* buf) {
        const AttnParams& p = late_args().p;
        const int tok_page = new_from & ~(kPage - 1), cut = new_from - tok_page;
        const int valid = min(max(kv_end - tok_page, 0), kPage);
#pragma clang loop unroll(disable)
        for (int kindx = 0; kindx < 2; ++kindx)
#pragma clang loop unroll(disable)
            for (int e = 0; e < NI; ++e) {
                const int prow = RPI * e + lane / LPR, pos = lane % LPR;
                const int chunk = 16 * (pos >> 4) + ((pos & 15) ^ swz(prow));
                if (prow < cut || prow >= valid) continue;
                const u32x4_t x = *reinterpret_cast<const u32x4_t*>((kindx ? p.v_new : p.k_new) + hkv * p.new_head_stride + int64_t(prow - cut) * D + 8 * chunk);
                *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(
                    buf + (kindx * TILEB + pg * (kPage * ROWB) + e * 1024 + 16 * lane)) = x;
            }
        __builtin_amdgcn_s_waitcnt(0);
    };
    auto issue_tile = [&](auto any, int t, int ids0, int ids1, lds_char* buf) {  // ids0, ids1: K and V ids of page pg
        if (dma_wave) {
            issue_page(any, t, ids0, buf, 0);
            issue_page(any, t, ids1, buf, 1);
        }
    };

    // ---- this wave's 32 keys of one tile against its 16 queries (buf: K at
    // 0, V at TILEB).  masked: the keys reach past the first query of the wave
    // or past the cache end.
    const float c = fmaxf(p.scale_log2, __FLT_MIN__);  // > 0: masked -inf scores give exactly 0
    const float inv_c = 1.0f / c;                       // may be inf (then no row grows after its first tile)
    auto compute_tile = [&](int t, const lds_char* buf, bool masked, auto&& after_s) {
        const int tok0 = t * KT + KH * kh;  // first key of the part
        const int r0 = KH * kh;             // its first LDS row (a multiple of 16)
        f32x4_t s[2] = {f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const int krow = r0 + 16 * kb + n16;
                const int pos = 16 * (ks >> 2) + ((4 * (ks & 3) + g) ^ swz(n16));
                const u32x4_t a = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(
                    buf + (krow * ROWB + pos * 16));
                s[kb] = E::mma32(__builtin_bit_cast(uint4, a), qb[ks], s[kb]);
            }
        after_s();
        if (masked) {
            __asm__ volatile("");  // keep a branch: full tiles carry no selects
            const int lim = p.causal ? min(qabs0 + s_row + 1, n_cached) : n_cached;
            const int rel = lim - tok0 - 4 * g;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[kb][i] = (16 * kb + i < rel) ? s[kb][i] : -INFINITY;
        }
        // raw row max, IEEE maximum (NaN-propagating: v_maximum3_f32, no quieting)
        float mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(s[0][0], s[0][1]),
                                                 __builtin_elementwise_maximum(s[0][2], s[0][3]));
        mx = __builtin_elementwise_maximum(mx, __builtin_elementwise_maximum(__builtin_elementwise_maximum(s[1][0], s[1][1]),
                                                                             __builtin_elementwise_maximum(s[1][2], s[1][3])));
        if (__any(mx > th)) {  // lazy rescale, as in the decode kernel
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const bool grow = mx > th;
            const float mn = grow ? mx * c : m;
            const float alpha = grow ? exp2_fast(m - mn) : 1.0f;
            l *= alpha;
            m = mn;
            nm = grow ? -mn : nm;
            th = grow ? (mn + 8.0f) * inv_c : th;
#pragma unroll
            for (int db = 0; db < DB; ++db) acc[db] *= alpha;
        }
        float e[2][4];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) e[kb][i] = exp2_fast(__builtin_fmaf(s[kb][i], c, nm));
        l += ((e[0][0] + e[0][1]) + (e[0][2] + e[0][3])) + ((e[1][0] + e[1][1]) + (e[1][2] + e[1][3]));
        const uint4 pb = make_uint4(E::pack_p(e[0][0], e[0][1]), E::pack_p(e[0][2], e[0][3]),
                                    E::pack_p(e[1][0], e[1][1]), E::pack_p(e[1][2], e[1][3]));
        // V^T from two transposing reads per 16 dims: rows r0 + 4g + n16/4 and
        // + 16, dims 16db + 4(n16%4)..+3 (chunk 2db + (n16%4)/2, half n16%2);
        // each read's LDS offset is one integer added to the buffer base, which
        // lets the compiler tell these reads from the loads streaming into the
        // other buffer
        const int row0 = r0 + 4 * g + (n16 >> 2), row1 = row0 + 16;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const int chunk = 2 * db + ((n16 & 3) >> 1), half = (n16 & 1) * 8;
            const int pos = 16 * (chunk >> 4) + ((chunk & 15) ^ swz(row0 & 15));
            const int off0 = TILEB + row0 * ROWB + pos * 16 + half;
            const int off1 = TILEB + row1 * ROWB + pos * 16 + half;  // row1 % 16 == row0 % 16
            const s16x4_t lo = ds_read_tr(buf + off0);
            const s16x4_t hi = ds_read_tr(buf + off1);
            const s16x4_t a8[2] = {lo, hi};
            acc[db] = E::mma32(__builtin_bit_cast(uint4, a8), pb, acc[db]);
        }
    };

    // ---- pipeline: one barrier per tile, two buffers.  Step t waits for its
    // own loads of tile t, meets the other waves (tile t complete in LDS;
    // everybody done with tile t-1), starts tile t+1 into the other buffer,
    // then computes its key part of tile t.  Every step issues the same 2 NI
    // loads in each loading wave; a tile past the last one has no rows below
    // kv_end and reads as zeros.  Page ids arrive IDS_BLOCK tiles per load; the rare reload
    // drains the loads in flight.
    const int t_ids = t_begin & ~(IDS_BLOCK - 1);
    int ids0 = paged && dma_wave ? load_ids(t_ids, 0) : 0;
    int ids1 = paged && dma_wave ? load_ids(t_ids, 1) : 0;
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // q and ids landed
    issue_tile(std::bool_constant<kNew>{}, t_begin, ids0, ids1, buf0);
    auto step = [&](auto any, int t, lds_char* cur, lds_char* nxt) {
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        if constexpr (decltype(any)::value) {
            const bool mixed = (new_from & (kPage - 1)) && new_from / KT == t && (new_from % KT) / kPage == pg;
            if (mixed && dma_wave) patch_page(cur);  // wave-uniform, once per workgroup at most
        }
        tile_barrier();
        if (((t + 1) & (IDS_BLOCK - 1)) == 0 && t + 1 < t_end) {
            if (paged && dma_wave) {
                ids0 = load_ids(t + 1, 0);
                ids1 = load_ids(t + 1, 1);
            }
            __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        }
        // At head_dim 256 the next tile's V rows are requested after this
        // tile's S^T MFMAs: the K reads right after the barrier then share the
        // LDS with half the incoming rows, and the longer step still hides the
        // V rows' latency (46.6-46.9 against 48.1-48.2 us at 2048 tokens; at
        // head_dim 128 the step is too short: 32.6 against 30.4 us; A/B on
        // one box).
        constexpr bool late_v = D == 256;
        if (late_v) {
            if (dma_wave) issue_page(any, t + 1, ids0, nxt, 0);
        } else {
            issue_tile(any, t + 1, ids0, ids1, nxt);
        }
        auto issue_v = [&]() {
            if (late_v && dma_wave) issue_page(any, t + 1, ids1, nxt, 1);
        };
        const int tok0 = t * KT + KH * kh;
        if (tok0 < wave_end)
            compute_tile(t, cur, tok0 + KH > wave_lim, issue_v);
        else
            issue_v();
    };
    int t = t_begin;
    if constexpr (kNew) {
        // the steps that neither hold nor request a row of the chunk, in a loop
        // without the selects between its rows and the pages (512 of
        // 4096, 16 waves: 58.7 -> 55.9 us)
        const int t_new = new_from / KT;
        for (; t + 2 < t_new && t < t_end; t += 2) {
            step(std::false_type{}, t, buf0, buf1);
            step(std::false_type{}, t + 1, buf1, buf0);
        }
    }
    for (; t < t_end; t += 2) {
        step(std::bool_constant<kNew>{}, t, buf0, buf1);
        step(std::bool_constant<kNew>{}, t + 1, buf1, buf0);
    }
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // the trailing (empty) loads have landed: LDS is free
    const AttnParams& pl = late_args().p;
    const PrefillGrid& gl = late_args().gr;

    // Keys of a masked half that a query may not see meet a zero probability
    // in the P.V MFMA, and 0 x NaN is NaN: a NaN or infinite V row there would
    // reach queries the reference never lets it reach.  A wave whose state
    // came out NaN or infinite (only ever with such inputs) forms its key part
    // again from the pools (the chunk's keys, in the forms that append, from
    // k_new / v_new), in fp32, visiting for each query only the keys it sees, as
    // the reference's loop does.  The check is one sum of the state
    // (a NaN or an infinity in it makes the sum non-finite); measured at
    // config 4, 30.85-30.93 against 30.65-30.80 us (A/B on one box, two passes;
    // checking each value instead cost 0.3-0.4 us).
    {
        float tsum = l;  // NaN or infinite when any of the state is
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) tsum += acc[db][i];
        if (__any(!(fabsf(tsum) <= __FLT_MAX__))) {
            float res[DB * 4 + 2];
            prefill_exact_part<D, F16, KT, kNew>(pl, qrow, head_off, hkv, s_row, kh, wave_end, t_begin, t_end, res);
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[db][i] = res[4 * db + i];
            m = res[4 * DB];
            l = res[4 * DB + 1];
        }
    }

    // ---- merge the key parts of each row block, pair by pair: one wave hands
    // (O^T, m, l) over through LDS, the other combines m = max(m0, m1), O = O0
    // 2^(m0-m) + O1 2^(m1-m), l likewise (a part that saw no key has m = -inf,
    // weight 0).  Four parts: 2 -> 0 and 3 -> 1, then 1 -> 0.
    __syncthreads();  // every wave is done with the tiles
    auto slot = [&](int i) { return (lds_float*)(i < KQ ? buf0 : buf1) + (i & (KQ - 1)) * XO + lane; };
    auto hand_over = [&](int i) {
        lds_float* const x = slot(i);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) x[(db * 4 + j) * 64] = acc[db][j];
        lds_ml[i][0][lane] = m;
        lds_ml[i][1][lane] = l;
    };
    if constexpr (KQ == 4) {
        if (kh >= 2) hand_over((kh - 2) * 4 + qblk);
        __syncthreads();
        if (kh < 2) {
            const int i = kh * 4 + qblk;
            const lds_float* const x = slot(i);
            const float m1 = lds_ml[i][0][lane], l1 = lds_ml[i][1][lane], mt = fmaxf(m, m1);
            const float a0 = mt == -INFINITY ? 0.0f : exp2_fast(m - mt), a1 = mt == -INFINITY ? 0.0f : exp2_fast(m1 - mt);
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[db][j] = acc[db][j] * a0 + x[(db * 4 + j) * 64] * a1;
            m = mt;
            l = l * a0 + l1 * a1;
        }
        __syncthreads();  // the slots are free
    }
    if (kh == 1) hand_over(qblk);
    __syncthreads();
    if constexpr (kNew)
        if (kh != 0) append_chunk<D>(tid - 256, (KQ - 1) * 256);
    if (kh != 0 || !wave_has_rows) return;
    const lds_float* const xch = slot(qblk);
    const float m1 = lds_ml[qblk][0][lane], l1 = lds_ml[qblk][1][lane];
    const float mt = fmaxf(m, m1);
    const float a0 = mt == -INFINITY ? 0.0f : exp2_fast(m - mt), a1 = mt == -INFINITY ? 0.0f : exp2_fast(m1 - mt);
    float lt = l * a0 + l1 * a1;
    lt += __shfl_xor(lt, 16);
    lt += __shfl_xor(lt, 32);
    const int r_out = q0 + n16;
    if (r_out >= R) return;
    if constexpr (kSplit) {
        // partials: o [split][unit][row][D], then {m, l} [split][unit][row]
        const int64_t at = (int64_t(sp) * gl.units + unit) * R + r_out;
        float* const po = gl.partial + at * D + 4 * g;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            f32x4_t o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = acc[db][i] * a0 + xch[(db * 4 + i) * 64] * a1;
            *reinterpret_cast<f32x4_t*>(po + 16 * db) = o;
        }
        if (g == 0)
            *reinterpret_cast<float2*>(gl.partial + int64_t(gl.n_splits) * gl.units * R * D + 2 * at) = make_float2(mt, lt);
        return;
    }
    const float inv = 1.0f / lt;
    const int s_out = gl.by_pack(r_out);
    uint16_t* orow = pl.out + bat * gl.o_batch + int64_t(hg * gl.pack + (r_out - s_out * gl.pack)) * pl.o_head_stride +
                     int64_t(s_out) * pl.o_tok_stride;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = (acc[db][i] * a0 + xch[(db * 4 + i) * 64] * a1) * inv;
        uint2 w;
        if constexpr (F16) {
            w.x = pack2(E::out(o[0]), E::out(o[1]));
            w.y = pack2(E::out(o[2]), E::out(o[3]));
        } else {
            w.x = bf16_pair_out(o[0], o[1]);
            w.y = bf16_pair_out(o[2], o[3]);
        }
        *reinterpret_cast<uint2*>(orow + 16 * db + 4 * g) = w;
    }
}

// D = 128: 66 KB of LDS and at most 128 VGPRs, so two workgroups share a CU
// (4 waves per SIMD: at config 4 36.2 us, against 41.9 us for the earlier
// form of one 128 KB, 196-VGPR workgroup per CU running two query tiles of
// 2 x 32 queries, A/B on one box); D = 256: 130 KB, one workgroup per CU.
template <bool F16, bool kSplit, bool kNew>
__global__ __launch_bounds__(512, kNew ? 4 : 2) void paged_prefill_d128_kernel(PrefillGrid gr, AttnParams p, AppendArg<kNew>) {
    prefill_tiles<128, F16, kSplit, 2, kNew>(p, gr);
}
// 16 waves on 128-key tiles, one workgroup per CU: the same waves per CU as
// two workgroups of the kernel above, for launches that have only one for
// each CU.  512 queries (32 q / 8 kv heads) at the end of 2048, 4096 keys:
// 33.6 against 36.3, 58.2 against 66.1 us.  Two
// independent workgroups stay faster where there are enough (0.63 against
// 0.87 us per 64 x 64 tile and CU: one barrier holds all 16 waves in step),
// and below kWideFrom keys the longer start and hand-over cost more than the
// tiles save (16 q / 8 kv heads, 1024 of 1024: 16.0 against 15.7 us, 100 of 1100
// 16.0 against 15.6, 600 of 1500 18.9 against 19.7; 40 of 40: 8.7 against 6.3).
constexpr int kWideFrom = 1280;
template <bool F16, bool kNew>
__global__ __launch_bounds__(1024) void paged_prefill_d128_wide_kernel(PrefillGrid gr, AttnParams p, AppendArg<kNew>) {
    prefill_tiles<128, F16, false, 4, kNew>(p, gr);
}
template <bool F16, bool kSplit, bool kNew>
__global__ __launch_bounds__(512) void paged_prefill_d256_kernel(PrefillGrid gr, AttnParams p, AppendArg<kNew>) {
    prefill_tiles<256, F16, kSplit, 2, kNew>(p, gr);
}

// Merge of the key splits: 4 dims per lane (D / 4 lanes per row), kMergeU
// splits in flight, with the log-sum-exp rule
//   M = max m_s, L = sum l_s 2^(m_s - M), O = sum o_s 2^(m_s - M), out = O / L.
// A split without a maximum (m_s = -inf) has weight 0, which its l and o are
// multiplied by all the same: they are zeros where the row sees no key of the
// split, but NaN where every score is NaN, and that NaN is the row's result.
constexpr int kMergeThreads = 256, kMergeU = 8;
template <int D, bool F16>
__global__ __launch_bounds__(kMergeThreads) void paged_prefill_merge_kernel(AttnParams p, PrefillGrid gr) {
    constexpr int LR = D / 4;
    const int G = p.G, R = p.S * G, units = gr.batch * p.Hkv;
    const int rows = units * R;  // at most 64 for each resident workgroup
    const int at = int(blockIdx.x) * (kMergeThreads / LR) + int(threadIdx.x) / LR;
    if (at >= rows) return;
    const int ns = gr.n_splits, d0 = 4 * (threadIdx.x % LR);
    const float2* const ml = reinterpret_cast<const float2*>(gr.partial + int64_t(ns) * rows * D) + at;
    const float* const po = gr.partial + int64_t(at) * D + d0;
    float M = -INFINITY, L = 0.0f;
    f32x4_t O = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < ns; s0 += kMergeU) {
        f32x4_t ov[kMergeU];
        float2 mv[kMergeU];
#pragma unroll
        for (int u = 0; u < kMergeU; ++u) {
            const bool in = s0 + u < ns;
            const int64_t off = int64_t(in ? s0 + u : s0) * rows;
            ov[u] = *reinterpret_cast<const f32x4_t*>(po + off * D);
            mv[u] = ml[off];
            if (!in) {  // the first of them again: weighs nothing
                ov[u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                mv[u] = make_float2(-INFINITY, 0.0f);
            }
        }
        float bm = M;
#pragma unroll
        for (int u = 0; u < kMergeU; ++u) bm = fmaxf(bm, mv[u].x);
        const float ref = bm == -INFINITY ? 0.0f : bm;
        const float a = exp2_fast(M - ref);  // 0 while M = -inf
        L *= a;
        O *= a;
#pragma unroll
        for (int u = 0; u < kMergeU; ++u) {
            const float w = exp2_fast(mv[u].x - ref);
            L += mv[u].y * w;
#pragma unroll
            for (int i = 0; i < 4; ++i) O[i] += ov[u][i] * w;
        }
        M = bm;
    }
    const float inv = 1.0f / L;
    const int unit = at / R, r = at - unit * R, s = gr.by_pack(r);
    const int bat = gr.by_hkv(unit), hkv = unit - bat * p.Hkv;
    uint16_t* const orow = p.out + bat * gr.o_batch + int64_t(hkv * G + (r - s * G)) * p.o_head_stride +
                           int64_t(s) * p.o_tok_stride + d0;
    *reinterpret_cast<uint2*>(orow) = make_uint2(pack2(Elem<F16>::out(O[0] * inv), Elem<F16>::out(O[1] * inv)),
                                                 pack2(Elem<F16>::out(O[2] * inv), Elem<F16>::out(O[3] * inv)));
}

bool wide_launch(const AttnParams& p, const PrefillGrid& gr, int head_dim) {
    return head_dim == 128 && gr.n_splits == 1 && p.n_cached >= kWideFrom &&
           int64_t(gr.n_rt) * gr.units <= device_cu_count();
}

template <int D, bool F16, bool kNew>
int launch_prefill_d(const AttnParams& p, const PrefillGrid& gr, const AppendArg<kNew>& pa, hipStream_t stream) {
    const int64_t rows = int64_t(p.S) * gr.pack, units = gr.units;
    const int64_t wgs = gr.n_rt * units * gr.n_splits;
    const bool split = gr.n_splits > 1;
    void (*k)(PrefillGrid, AttnParams, AppendArg<kNew>);
    int threads = 512;
    if constexpr (D == 128) {
        k = split ? paged_prefill_d128_kernel<F16, true, kNew> : paged_prefill_d128_kernel<F16, false, kNew>;
        if (wide_launch(p, gr, D)) {
            k = paged_prefill_d128_wide_kernel<F16, kNew>;
            threads = 1024;
        }
    } else {
        k = split ? paged_prefill_d256_kernel<F16, true, kNew> : paged_prefill_d256_kernel<F16, false, kNew>;
    }
    hipLaunchKernelGGL(k, dim3(unsigned(wgs)), dim3(threads), 0, stream, gr, p, pa);
    GENLLM_LAUNCH_CHECK("paged_prefill kernel");
    if (!split) return GENLLM_OK;
    constexpr int kMergeWgRows = kMergeThreads / (D / 4);
    hipLaunchKernelGGL((paged_prefill_merge_kernel<D, F16>), dim3(unsigned((rows * units + kMergeWgRows - 1) / kMergeWgRows)),
                       dim3(kMergeThreads), 0, stream, p, gr);
    GENLLM_LAUNCH_CHECK("paged_prefill_merge_kernel");
    return GENLLM_OK;
}

// The append runs inside the attention launch in the 16-wave form and where a
// workgroup walks few key tiles: it saves a launch of 3.3-7 us, and costs a
// step of the 8-wave forms about a tenth (the choice between the pages and the
// chunk's rows).  Both kernels against the one, us (q / kv heads, head_dim,
// queries of keys, key tiles of a workgroup): 32/8, 128, 512 of 4096 (16 waves)
// 61.2, 55.9; 16/8, 128, 200 of 200 (4) 11.8, 9.1; 32/8, 128, 256 of 4096 (16)
// 37.4, 36.1; 32/8, 128, 512 of 8192 (64) 93.1, 93.5; 32/8, 128, 1024 of 8192
// (128) 154.1, 168.6; 8/2, 256, 128 of 1128 (3) 22.2, 20.6; 8/2, 256, 2048 of
// 2048 (32) 54.6, 61.1.  Unsplit and with the keys still in the caches the line
// lies lower (32/8, 128, chunks of 269 of 536..1326: 82.5 us a session with
// kAppendTiles 8, 85.9 with 20).
constexpr int kAppendTiles = 8, kAppendSplitTiles = 20;
bool append_in_launch(const AttnParams& p, const PrefillGrid& gr, int head_dim) {
    if (int64_t(2) * p.S * p.Hkv * (head_dim / 8) > INT32_MAX) return false;  // the copy counts in 32 bits
    // an output that overlaps the chunk's rows must not be written before they are read
    const auto overlaps = [&](const uint16_t* x) {
        const uintptr_t o = reinterpret_cast<uintptr_t>(p.out), a = reinterpret_cast<uintptr_t>(x);
        return o < a + size_t(p.S) * p.Hkv * head_dim * 2 && a < o + size_t(gr.batch) * p.S * p.Hq * head_dim * 2;
    };
    if (overlaps(p.k_new) || overlaps(p.v_new)) return false;
    return wide_launch(p, gr, head_dim) ||
           p.n_cached <= int64_t(gr.n_splits > 1 ? kAppendSplitTiles : kAppendTiles) * 64 * gr.n_splits;
}

int append_before(const AttnParams& p, const PrefillAppend& append, int head_dim, hipStream_t stream) {
    AppendParams ap;
    ap.upd = append.upd;
    ap.k = p.k_new;
    ap.v = p.v_new;
    ap.k_tok_stride = ap.v_tok_stride = p.new_tok_stride;
    ap.k_head_stride = ap.v_head_stride = p.new_head_stride;
    ap.S = p.S;
    ap.Hkv = p.Hkv;
    ap.pos0 = p.new_from;
    ap.nkv_tasks = (p.Hkv + 7) / 8;
    ap.k_pool = p.k_pool_w;
    ap.v_pool = p.v_pool_w;
    ap.page_elems = p.page_elems;
    ap.k_ids = p.k_ids_w;
    ap.v_ids = p.v_ids_w;
    ap.max_blocks = append.max_blocks;
    return launch_kv_append(ap, head_dim, stream);
}

template <bool kNew>
int launch_prefill(const AttnParams& p, const PrefillGrid& gr, const AppendArg<kNew>& pa, int head_dim, hipStream_t stream) {
    if (head_dim == 128)
        return p.f16 ? launch_prefill_d<128, true, kNew>(p, gr, pa, stream) : launch_prefill_d<128, false, kNew>(p, gr, pa, stream);
    return p.f16 ? launch_prefill_d<256, true, kNew>(p, gr, pa, stream) : launch_prefill_d<256, false, kNew>(p, gr, pa, stream);
}

int resident_workgroups(int head_dim) { return device_cu_count() * (head_dim == 128 ? 2 : 1); }

// The terms of prefill_splits' estimate.
struct SplitCost {
    double tile_us, split_tile_us;  // a 64-key tile in the unsplit kernel, in the split kernel
    static constexpr double kPairTileUs = 1.25;  // ... with two workgroups on a CU
    static constexpr double kMergeUs = 6.0, kMergeUsPerMB = 0.46;
    static constexpr double kUnsplit = 0.85;  // less where the keys are still in the caches
    explicit SplitCost(int head_dim) : tile_us(head_dim == 128 ? 0.8 : 1.45), split_tile_us(head_dim == 128 ? 0.85 : 1.45) {}
    double unsplit(int64_t tiles) const { return kUnsplit * double(tiles) * tile_us; }
};

}  // namespace

// The most partials any chunk of a layer of max_tokens may hand over: every
// split launch keeps its workgroups resident at once, 64 rows each (17 MB at
// either head_dim), and over few keys only launches whose merge costs less than
// the split saves are split (none up to 10 key tiles at head_dim 128, 6 at 256;
// the whole 17 MB from 22 and 13 tiles on).
size_t prefill_workspace_bytes(int head_dim, int64_t max_tokens) {
    if (head_dim != 128 && head_dim != 256) return 0;
    const SplitCost cost(head_dim);
    const double cap = double(resident_workgroups(head_dim)) * QT * (head_dim + 2) * sizeof(float);
    double most = 0.0;
    const int64_t last = (max_tokens + 63) / 64;
    for (int64_t tiles = 2; tiles <= last && most < cap; ++tiles)
        for (int64_t ns = 2; ns <= std::min<int64_t>(tiles, kMaxPrefillSplits); ++ns) {
            const double gain = cost.unsplit(tiles) - double((tiles + ns - 1) / ns) * cost.split_tile_us - cost.kMergeUs;
            most = std::max(most, std::min(gain / cost.kMergeUsPerMB * 1e6, cap));
        }
    return size_t(most);
}

// Key splits of a launch of `rows` rows for each of `units` (batch entry, kv
// head) pairs: the count with the least estimated time among those whose
// workgroups are all resident at once.  Unsplit, a chunk of few rows leaves
// most CUs idle while each of its workgroups walks all key tiles in turn.
// Estimate, in us (fitted to kernel traces on MI355X): a workgroup's longest
// chain of 64-key tiles at tile_us each (split_tile_us in the split kernel, or
// kPairTileUs where two workgroups share a CU), and for a split launch the
// hand-over and the merge kernel, kMergeUs plus kMergeUsPerMB of partials
// written and read back.  Measured, both kernels against one unsplit 8-wave
// kernel (q / kv heads, head_dim, queries at the end of N keys):
//   32/8, 128,   8 of 8200: 19.2 against 148.6 us (26 splits)
//   32/8, 128,  64 of 8256: 30.6 against 138.6 us (8)
//   32/8, 128, 256 of 4096: 33.7 against  65.1 us (4)
//   32/8, 128, 512 of 8192: 89.9 against 131.6 us (2; 114.0 with 16 waves)
//   32/8, 128, 512 of 4096: 54.8 against  66.3 us (2; 58.2 with 16 waves, and
//     faster than split where the keys are still in L2: left unsplit)
//   16/8, 128,  64 of 1024: 12.6 against  22.2 us (8)
//   8/2,  256, 128 of 1128: 18.5 against  29.8 us (6)
//   8/2,  256,  64 of 8192: 24.0 against 186.2 us (26)
int prefill_splits(int64_t units, int64_t rows, int n_cached, int head_dim, size_t ws_bytes) {
    const SplitCost cost(head_dim);
    const int64_t cus = device_cu_count(), wgs = (rows + QT - 1) / QT * units;
    const int64_t tiles = (int64_t(n_cached) + 63) / 64;
    const int64_t most = std::min<int64_t>({resident_workgroups(head_dim) / wgs, tiles, kMaxPrefillSplits});
    int best = 1;
    double best_us = cost.unsplit(tiles);
    for (int64_t ns = 2; ns <= most; ++ns) {
        const double bytes = double(ns * units * rows) * (head_dim + 2) * sizeof(float);
        if (bytes > double(ws_bytes)) break;
        const double us = double((tiles + ns - 1) / ns) * (wgs * ns <= cus ? cost.split_tile_us : cost.kPairTileUs) +
                          cost.kMergeUs + bytes * 1e-6 * cost.kMergeUsPerMB;
        if (us < best_us) best = int(ns), best_us = us;
    }
    return best;
}

// Whether out overlaps the rows of a batch (out that is q itself aside: a
// workgroup writes the rows it read).  An entry's output may then lie over
// another entry's inputs, which is sound only one entry after another.
static bool out_over_entries(const AttnParams& p, const PrefillBatch& b, int head_dim) {
    if (b.n <= 1) return false;
    const auto bytes = [&](int64_t stride, int64_t heads, int64_t head_stride, int64_t tok_stride) {
        return size_t(((b.n - 1) * stride + (heads - 1) * head_stride + (p.S - 1) * tok_stride + head_dim) * 2);
    };
    const uintptr_t o = reinterpret_cast<uintptr_t>(p.out);
    const size_t o_bytes = bytes(b.o_stride, p.Hq, p.o_head_stride, p.o_tok_stride);
    const auto meets = [&](const uint16_t* x, size_t n) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(x);
        return o < a + n && a < o + o_bytes;
    };
    const bool in_place = p.out == p.q && b.o_stride == b.q_stride && p.o_head_stride == p.q_head_stride &&
                          p.o_tok_stride == p.q_tok_stride;
    if (!in_place && meets(p.q, bytes(b.q_stride, p.Hq, p.q_head_stride, p.q_tok_stride))) return true;
    if (b.kv_stride == 0) return false;  // the pages of a cache
    const size_t kv = bytes(b.kv_stride, p.Hkv, p.kv_head_stride, p.kv_row);
    return meets(p.k_pool, kv) || meets(p.v_pool, kv);
}

int launch_paged_prefill(const AttnParams& p, int head_dim, hipStream_t stream, const PrefillBatch& b, float* ws,
                         size_t ws_bytes, const PrefillAppend* append) {
    if (head_dim != 128 && head_dim != 256) return fail(GENLLM_ERR_UNSUPPORTED, "paged prefill: head_dim must be 128 or 256");
    if (p.S <= 0 || p.n_pages <= 0 || b.n <= 0) return GENLLM_OK;
    const int64_t rows = int64_t(p.S) * p.G;
    // entries per launch: a grid of about 2^21 workgroups at most (HIP takes up to 2^32 threads)
    const int64_t per = out_over_entries(p, b, head_dim)
                            ? 1
                            : std::max<int64_t>(1, (int64_t(1) << 21) / ((rows + QT - 1) / QT * p.Hkv));
    for (int64_t b0 = 0; b0 < b.n; b0 += per) {
        AttnParams pb = p;
        pb.q += b0 * b.q_stride;
        pb.out += b0 * b.o_stride;
        pb.k_pool += b0 * b.kv_stride;
        pb.v_pool += b0 * b.kv_stride;
        PrefillGrid gr;
        gr.batch = int32_t(std::min<int64_t>(per, b.n - b0));
        gr.q_batch = b.q_stride;
        gr.o_batch = b.o_stride;
        gr.kv_batch = b.kv_stride;
        gr.partial = ws;
        gr.n_splits = ws ? prefill_splits(int64_t(gr.batch) * p.Hkv, rows, p.n_cached, head_dim, ws_bytes) : 1;
        // A split launch packs the q heads of a kv head into its row tiles, as
        // does any chunk whose single heads would leave a twentieth more tiles.
        // Otherwise each q head has its own (D = 256, 16 / 4 heads, 814 tokens
        // 23.0 against 24.1 us; D = 128, 32 / 8, 700 tokens 14.1 against 14.4).
        const bool own = gr.n_splits == 1 && (int64_t(p.S) + QT - 1) / QT * p.G * 20 <= (rows + QT - 1) / QT * 21;
        gr.pack = own ? 1 : p.G;
        gr.units = gr.batch * (own ? p.Hq : p.Hkv);
        const int64_t unit_rows = own ? p.S : rows;
        // Where CUs would stay idle, smaller row tiles spread the rows over more
        // of them, fewer row blocks each (tiles of 16, 32 and 64 rows, us: 16 q
        // / 8 kv heads, 100 of 700 11.4, 11.5, 11.8; 500 of 1030 15.1, 15.3,
        // 15.6; 64 of 4000 37.5, 38.1, 39.0).
        if (gr.n_splits == 1)
            for (int r = QT / 2; r >= QW && (unit_rows + r - 1) / r * gr.units <= device_cu_count(); r /= 2) gr.tile_rows = r;
        gr.n_rt = int32_t((unit_rows + gr.tile_rows - 1) / gr.tile_rows);
        gr.by_pack = FastDiv(uint32_t(gr.pack));
        gr.by_units = FastDiv(uint32_t(gr.units));
        gr.by_heads = FastDiv(uint32_t(own ? p.Hq : p.Hkv));
        gr.by_groups = FastDiv(uint32_t(own ? p.G : 1));
        gr.by_hkv = FastDiv(uint32_t(p.Hkv));
        gr.by_splits = FastDiv(uint32_t(gr.n_splits));
        // The first launch appends, where that pays (append_in_launch); the rows
        // are in their pages before a further one.
        int rc = GENLLM_OK;
        if (append && b0 == 0 && append_in_launch(pb, gr, head_dim)) {
            rc = launch_prefill<true>(pb, gr, *append, head_dim, stream);
        } else {
            if (append && b0 == 0) rc = append_before(p, *append, head_dim, stream);
            pb.k_new = pb.v_new = nullptr;
            pb.new_from = INT32_MAX;
            if (rc == GENLLM_OK) rc = launch_prefill<false>(pb, gr, NoAppend{}, head_dim, stream);
        }
        if (rc) return rc;
    }
    return GENLLM_OK;
}

}  // namespace genllm
