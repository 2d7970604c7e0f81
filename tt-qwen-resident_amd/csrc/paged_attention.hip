// Paged GQA decode attention on gfx950 (HD 256, block 64): split-K over block-table pages, online softmax,
// an ordered merge of the splits, optional fused append of the step's new K/V rows (and the mixer edges).
//
// Grid: one workgroup per (user, KV head, split); a split is `pps` (<= 64) consecutive block-table entries.
// Every K/V byte is loaded once for all G query heads of the KV head (GQA reuse) and, in a verify step, for
// all query tokens of the step. Two kernels walk the pages:
//   attn_wave_kernel  up to 16 query rows per KV head (every one-token decode): MFMA scores and P V, each
//                     wave on its own 16-row slices with no barrier in the page loop, one or two pages in
//                     flight per workgroup;
//   attn_rows_kernel  more query rows (verify steps): MFMA, 4 waves on a page, each wave owning a quarter of the
//                     head dims in P V, one or two pages in flight, blocks of up to 64 query rows.
// The step's new rows are loaded with the query rows and attended without a round trip through the pool:
// the one-token kernel (up to two tokens) holds them in registers and patches them over the page rows they
// replace (K through a one-row LDS copy when the page goes straight into the score operand), the rows kernel,
// and with the mixer the one-token kernel, stages them in LDS; both store them to the pool after the page loop. The
// one-token kernel appends more than two tokens first, by the wave that reads them back from the pool.
// The splits' partials (m, l, unnormalised O per query row) go to the workspace and are merged in split order
// (the leader side of the reference: global max, rescale, sum, normalise, kernels/attn_leader_writer.cpp:
// 86-106 and kernels/attn_leader_compute.cpp:42-79) by the last workgroup of the (user, KV head) to finish
// when the one-token kernel's splits are few (merge_here), else by a separate merge launch, so results are identical run
// to run. Splits past a user's pages take no part (split_live).
#include <algorithm>
#include <type_traits>

#include "qs_common.h"

namespace {

constexpr int HD = 256;
constexpr int BLK = 64;
// cache policy of the K / V page loads: nontemporal (each page is read once per step; measured ~5% faster
// than the default policy at batch 8 / 4096 positions and at batch 1 / 32768)
constexpr int NT = 2;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct AttnArgs {
    const uint16_t *q;                  // [B, T, NQ, HD]
    const uint16_t *k_new, *v_new;      // nullable [B, T, NKV, HD]
    uint16_t *k_cache, *v_cache;        // [num_blocks, NKV, BLK, HD]
    const int *block_table;             // [B, max_blocks]
    const int *seq_lens;                // [B]
    uint16_t *o;                        // [B, T, NQ, HD]
    float *part_o;                      // [B, NKV, nsplit, T G, HD]: split partials (unnormalised O)
    float *part_ml;                     // [B, NKV, nsplit, T G, 2]: their (max, sum), log2 domain
    int *cnt;                           // [B, NKV] arrival counters of the in-launch merge (kept zero)
    int *status;                        // nullable: QS_STATUS_* bits of invalid lengths / table entries
    int B, T, NQ, NKV, max_blocks, num_blocks, pps, nsplit;
    int merge;                          // the splits are merged inside the attention launch
    float scale;
    // mixer edges (qs_attn_mixer_decode; null / 0 for plain attention): q and the new k rows are
    // RMS-normalised times wq / wk [HD] and rotated on their first rot dims with rcos / rsin
    // [B, T, rot / 2]; the output is multiplied by sigmoid(gate [B, T, NQ, HD])
    const uint16_t *gate;
    const float *wq, *wk, *rcos, *rsin;
    int rot;
    float eps;
};

// The mixer's tables for one 8-element chunk, requested ahead of the page loads: read where they are used they
// queue behind the launch's first page burst (B 1 / 8192 positions / T 4, stamps: query and new rows staged 12500
// cycles after the length, 5500 without the mixer). With the new rows attended from LDS too, per layer: B 1 / 8192 /
// T 4 / pps 2 21.0 -> 19.8 us, B 1 / 4096 / one page per split 15.9 -> 13.2, B 4 / 2000 / T 3 / pps 4 30.3 -> 22.5,
// B 8 / 4096 / pps 8 29.5 -> 28.7, B 1 / 200 13.2 -> 11.9.
struct MixChunk {
    f32x4_t w[2], c[2], s[2];
};
// norm weights of dims 8 ch .. + 7
__device__ __forceinline__ void mix_weights(const float *w, int ch, MixChunk &m) {
    const auto r = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(const_cast<float *>(w)), (short)0, HD * 4, 0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h)
        m.w[h] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, ch * 32, h * 16, 0));
}
// cos / sin of the chunk's dims (halves paired) for row `row` of the tables [rows, rot / 2]; zeros where the chunk
// is not rotated. Buffer loads: the tables need no more than their 4-byte alignment.
__device__ __forceinline__ void mix_angles(const AttnArgs &a, int row, int ch, MixChunk &m) {
    const int half = a.rot / 2, hc = half / 8, bytes = a.B * a.T * half * 4;
    const auto rc = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(const_cast<float *>(a.rcos)), (short)0, bytes, 0x00020000);
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(const_cast<float *>(a.rsin)), (short)0, bytes, 0x00020000);
    const int off = ch < 2 * hc ? (row * half + (ch < hc ? ch : ch - hc) * 8) * 4 : 0x7fffffe0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        m.c[h] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rc, off, h * 16, 0));
        m.s[h] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off, h * 16, 0));
    }
}
// Mixer prologue of one 8-element chunk (raw bf16 bits, chunk ch of a 256-dim row whose 32 chunks sit in 32
// consecutive, fully active lanes): y = x * rsqrt(mean(x^2) + eps) * w, then the rotary embedding on the
// first rot dims with the halves paired as at model.py:135-140 (d < rot/2 with d + rot/2:
// y_d c - y_{d+h} s and y_{d+h} c + y_d s). fp32 throughout (model.py:86-89, :237-238).
__device__ __forceinline__ void mixer_chunk(const uint4 raw, int ch, const MixChunk &m, int rot, float eps, float y[8]) {
    const uint32_t wd[4] = {raw.x, raw.y, raw.z, raw.w};
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        y[2 * e] = qs::bf_lo(wd[e]);
        y[2 * e + 1] = qs::bf_hi(wd[e]);
        ss = fmaf(y[2 * e], y[2 * e], ss);
        ss = fmaf(y[2 * e + 1], y[2 * e + 1], ss);
    }
    ss += qs::dpp<0xB1>(ss);
    ss += qs::dpp<0x4E>(ss);
    ss += qs::dpp<0x124>(ss);
    ss += qs::dpp<0x128>(ss);
    ss = qs::xor16_sum(ss);  // the 32 lanes of the row
    const float r = rsqrtf(ss * (1.0f / HD) + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = y[i] * r * m.w[i / 4][i % 4];
    if (rot > 0) {
        const int hc = rot / 16;  // chunks per half
        float yp[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) yp[i] = __shfl_xor(y[i], hc, 64);
        if (ch < 2 * hc) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float c = m.c[i / 4][i % 4], s = m.s[i / 4][i % 4];
                y[i] = ch < hc ? y[i] * c - yp[i] * s : y[i] * c + yp[i] * s;
            }
        }
    }
}
__device__ __forceinline__ uint4 pack8(const float y[8]) {
    return make_uint4(qs::cvt_pk_bf16(y[0], y[1]), qs::cvt_pk_bf16(y[2], y[3]), qs::cvt_pk_bf16(y[4], y[5]),
                      qs::cvt_pk_bf16(y[6], y[7]));
}
// The rounding residues y - bf16(y) of 8 values as bf16 (hi = pack8(y)): hi + lo carries y to ~2^-17 relative,
// so products against exact bf16 operands (K rows) keep the fp32 value of a normalised, rotated q.
__device__ __forceinline__ uint4 pack8_lo(const float y[8], uint4 hi) {
    const uint32_t h[4] = {hi.x, hi.y, hi.z, hi.w};
    uint32_t lo[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) lo[e] = qs::cvt_pk_bf16(y[2 * e] - qs::bf_lo(h[e]), y[2 * e + 1] - qs::bf_hi(h[e]));
    return make_uint4(lo[0], lo[1], lo[2], lo[3]);
}
__device__ __forceinline__ float sigm(float g) { return 1.0f / (1.0f + expf(-g)); }

// A user's length n (positions valid after this step's T rows) is usable when T <= n <= max_blocks * BLK.
// n < T marks an idle slot (nothing appended or attended, zero output); n past the block table is an error
// (reported in the status word) and the user is treated as idle, never clamped onto other positions.
__device__ __forceinline__ bool user_active(const AttnArgs &a, int n, bool report) {
    if (n > a.max_blocks * BLK) {
        if (report && a.status) atomicOr(a.status, QS_STATUS_LENGTH);
        return false;
    }
    return n >= a.T;
}
// Whether split sp of a user of length n holds pages. A table is as wide as its longest user may get: a shorter user's
// other splits have nothing to do. Their workgroups request no page, write no partial and leave, and the merges count and
// read only those that hold pages. At 8 pages a split and a 512-page table, with every split requesting its first pages,
// storing partials and being merged -> this: 200 positions, batch 8, one token 66.2 -> 22.6 us a layer, four 84.4 -> 34.8,
// batch 1, one token 16.3 -> 13.2; 64-page table, batch 4 at 200, one token 16.1 -> 13.5.
__device__ __forceinline__ bool split_live(const AttnArgs &a, int n, int sp) { return sp * a.pps * BLK < n; }
// How many do (whole waves; FEW: at most 64 splits, counted without a division)
template <bool FEW>
__device__ __forceinline__ int live_splits(const AttnArgs &a, int n, int lane) {
    if constexpr (FEW) return __builtin_popcountll(__ballot(lane < a.nsplit && split_live(a, n, lane)));
    return ((n + BLK - 1) / BLK + a.pps - 1) / a.pps;
}
__device__ __forceinline__ void report_page(const AttnArgs &a) {
    if (a.status) atomicOr(a.status, QS_STATUS_PAGE);
}
// Zero output rows of an inactive user for KV head g (all T G query rows; threads of one workgroup).
__device__ __forceinline__ void zero_rows(const AttnArgs &a, int G, int b, int g, int tid, int nth) {
    for (int idx = tid; idx < a.T * G * 32; idx += nth) {
        const int qr = idx >> 5, ch = idx & 31;
        *reinterpret_cast<uint4 *>(a.o + (((size_t)b * a.T + qr / G) * a.NQ + g * G + qr % G) * HD + ch * 8) =
            make_uint4(0, 0, 0, 0);
    }
}

// Workspace layout (bytes): arrival counters | part_ml | part_o, each 256-byte aligned. The counters sit in
// a fixed block at the head, so a workspace reused for another shape never finds partial data where its
// counters are (they must read zero).
constexpr size_t CNT_BYTES = 65536;  // room for B NKV <= 16384 counters
struct WsLayout {
    size_t cnt, ml, po, total;
};
__host__ __device__ inline WsLayout ws_layout(int B, int T, int NKV, int G, int nsplit) {
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    WsLayout l;
    l.cnt = 0;
    l.ml = CNT_BYTES;
    l.po = l.ml + up((size_t)B * T * NKV * nsplit * G * 2 * 4);
    l.total = l.po + up((size_t)B * T * NKV * nsplit * G * HD * 4);
    return l;
}
// Row of the partial of query row qr (= t G + h) of split sp for user b, KV head g: one workgroup's rows
// are contiguous.
__device__ __forceinline__ size_t prow(const AttnArgs &a, int G, int b, int g, int sp, int qr) {
    return (((size_t)b * a.NKV + g) * a.nsplit + sp) * (size_t)(a.T * G) + qr;
}

// The MFMA kernels' first requests, each one buffer load with no branch around it (lanes outside the range
// read zeros without a memory access), so the compiler's waits stay exact: the first page's loads, issued
// next, need only the block-table entries and the user's length, and nothing waits for the query rows until they are staged.
// Block-table entry p0 + lane of user b (zero past the split or the table; only entries below
// min(max_blocks, p0 + pps) are ever read back).
__device__ __forceinline__ int split_entries(const AttnArgs &a, int b, int p0, int lane) {
    const int cnt = max(0, min(a.max_blocks, p0 + a.pps) - p0);
    const auto r = __builtin_amdgcn_make_buffer_rsrc(
        qs::uniform_ptr(const_cast<int *>(a.block_table) + (size_t)b * a.max_blocks + min(p0, a.max_blocks)), (short)0,
        cnt * 4, 0x00020000);
    return (int)__builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, 0, 0);
}
// 16-byte chunk ch of query row qr = t G + hh of user b, KV head g (zeros for qr >= T G)
__device__ __forceinline__ uint4 q_chunk(const AttnArgs &a, int G, int b, int g, int qr, int ch) {
    const int T = a.T;
    const auto r = __builtin_amdgcn_make_buffer_rsrc(
        qs::uniform_ptr(const_cast<uint16_t *>(a.q) + ((size_t)b * T * a.NQ + (size_t)g * G) * HD), (short)0,
        ((T - 1) * a.NQ + G) * HD * 2, 0x00020000);
    const int off = qr < T * G ? ((qr / G) * a.NQ + qr % G) * HD * 2 + ch * 16 : 0x7ffffff0;
    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return make_uint4(x[0], x[1], x[2], x[3]);
}
// 16-byte chunk ch of the new K or V row of token t of user b, KV head g (rows [B, T, NKV, HD]; zeros for
// t >= T, ch < 0 or a null pointer)
__device__ __forceinline__ u32x4 new_chunk(const AttnArgs &a, const uint16_t *rows, int b, int g, int t, int ch) {
    const auto r = __builtin_amdgcn_make_buffer_rsrc(
        qs::uniform_ptr(const_cast<uint16_t *>(rows ? rows : a.q) + (size_t)b * a.T * a.NKV * HD), (short)0,
        rows ? a.T * a.NKV * HD * 2 : 0, 0x00020000);
    const int off = t < a.T && ch >= 0 ? ((t * a.NKV + g) * HD + ch * 8) * 2 : 0x7ffffff0;
    return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
}

// ------------------------------------------------------------------------------ shared by the MFMA kernels
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
constexpr int QPAD = HD + 8;   // s_q row pitch (bf16): 16-byte skew between rows
constexpr int VPAD = HD + 16;  // K / V slice row pitch (bf16): 32-byte skew between rows

// Split merge inside the attention launch (AttnArgs::merge). Every workgroup of (user b, KV head g) has
// stored its partial with agent-coherent stores (sc1: written through the XCD's L2); each thread waits for
// its stores to complete, then one thread counts the workgroup in (the count wraps to zero at the last
// arrival). The workgroup that completes the count merges: wave w of NWV takes query rows w, w + NWV, ...
// (two at a time), lane l owns head dims 4 l .. 4 l + 3, and every split's partial and (m, l) are read with agent-coherent
// loads in one round trip. Global max M (log2 domain) and sum L over the splits, weights 2^(m_s - M), O = sum_s w_s O_s / L
// in split order, so the result does not depend on which workgroup finished last. No L2-wide writeback or
// invalidate is needed because only sc1 accesses touch the shared data. (The leader side of the
// reference: kernels/attn_leader_writer.cpp:86-106, kernels/attn_leader_compute.cpp:42-79.)
// merge_here says which calls are merged so; the others, and every step of the rows kernel, in a launch of their own.
constexpr int MERGE_ANY = 4, MERGE_MAX = 8, MERGE_MOST = 16;
template <int NWV>
__device__ __forceinline__ void merge_in_launch(const AttnArgs &a, int G, int b, int g, int tid, int n) {
    __shared__ int s_last;
    const int ns = live_splits<true>(a, n, tid & 63);
    qs::wait_vmem();
    __syncthreads();
    if (tid == 0) {
        // an increment modulo the splits that arrive (those holding pages): the last one leaves the count at zero for
        // the next launch
        unsigned *c = reinterpret_cast<unsigned *>(a.cnt) + (size_t)b * a.NKV + g;
        const unsigned ns1 = (unsigned)ns - 1;
        s_last = __builtin_amdgcn_atomic_inc32(c, ns1, __ATOMIC_RELAXED, "agent") == ns1;
    }
    __syncthreads();
    if (!s_last) return;
    asm volatile("" ::: "memory");
    const int lane = tid & 63, w = tid >> 6;
    const int T = a.T, R = T * G;
    const auto ro = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(a.part_o + prow(a, G, b, g, 0, 0) * HD),
                                                      (short)0, ns * R * HD * 4, 0x00020000);
    const auto rm = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(a.part_ml + prow(a, G, b, g, 0, 0) * 2),
                                                      (short)0, ns * R * 8, 0x00020000);
    // ROWS query rows of a wave at a time, MOST splits
    auto merge = [&](auto rows, auto most) {
        constexpr int ROWS = decltype(rows)::value, MOST = decltype(most)::value;
        for (int r0 = w; r0 < R; r0 += ROWS * NWV) {
            f32x4_t x[ROWS][MOST];
            float2 ml[ROWS];
            uint2 gw[ROWS];
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                const int qr = r0 + NWV * j;
                if (qr >= R) continue;
#pragma unroll
                for (int sp = 0; sp < MOST; ++sp)
                    if (sp < ns)
                        x[j][sp] = __builtin_bit_cast(
                            f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ro, ((sp * R + qr) * HD + 4 * lane) * 4, 0,
                                                                            qs::CP_SC1));
                ml[j] = make_float2(-INFINITY, 0.f);
                if (lane < ns) {
                    const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(rm, (lane * R + qr) * 8, 0, qs::CP_SC1);
                    ml[j] = make_float2(__uint_as_float(u[0]), __uint_as_float(u[1]));
                }
                if (a.gate)
                    gw[j] = *reinterpret_cast<const uint2 *>(
                        a.gate + (((size_t)b * T + qr / G) * a.NQ + g * G + qr % G) * HD + 4 * lane);
            }
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                const int qr = r0 + NWV * j;
                if (qr >= R) continue;
                const float M = qs::wave_max_bcast(ml[j].x);
                const float e = ml[j].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[j].x - M);
                const float L = qs::wave_sum_dpp(e * ml[j].y);
                f32x4_t O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int sp = 0; sp < MOST; ++sp)
                    if (sp < ns) O += qs::lane_val(e, sp) * x[j][sp];
                O *= 1.0f / L;
                if (a.gate) {
                    O[0] *= sigm(qs::bf_lo(gw[j].x)), O[1] *= sigm(qs::bf_hi(gw[j].x));
                    O[2] *= sigm(qs::bf_lo(gw[j].y)), O[3] *= sigm(qs::bf_hi(gw[j].y));
                }
                *reinterpret_cast<uint2 *>(a.o + (((size_t)b * T + qr / G) * a.NQ + g * G + qr % G) * HD + 4 * lane) =
                    make_uint2(qs::cvt_pk_bf16(O[0], O[1]), qs::cvt_pk_bf16(O[2], O[3]));
            }
        }
    };
    if (ns <= MERGE_MAX)
        merge(std::integral_constant<int, 2>{}, std::integral_constant<int, MERGE_MAX>{});
    else
        merge(std::integral_constant<int, 1>{}, std::integral_constant<int, MERGE_MOST>{});
}

// ------------------------------------------------------------------------------ MFMA kernel (verify rows)
// For T query tokens the T G query rows of a KV head form a dense [T G x 256] x [256 x rows] product. One
// workgroup per (user, KV head, split of pps pages, block of 16 QT query rows) with WPP groups of 4 waves: group
// ph walks pages p0 + ph, p0 + ph + WPP, ... (WPP pages in flight), every group in step. Per page, two barriers:
//   scores  wave w takes rows 16 w .. + 15 of the page: S^T [16 rows x 16 q] = K Q^T on 8
//           v_mfma_f32_16x16x32_bf16 per query tile (lane l holds K row l % 16, dims 32 j + 8 (l / 16) .. + 7,
//           loaded in that layout), its rows' max per query row into LDS;                            barrier
//   softmax the page's max per query row from the 4 waves; the running max M (log2 domain, the same in all 4
//           waves) moves only when the page exceeds it by 2^8 (the accumulators are then rescaled); P^T =
//           2^(s - M) as bf16 hi + lo into LDS beside the page's V rows, the fp32 values summed per wave;
//                                                                                                    barrier
//   P V     every wave adds the page to O^T [its 64 head dims x 16 q]: four v_mfma_f32_16x16x32_bf16 per tile,
//           V^T read with the transposing ds_read_b64_tr_b16, accumulated by the MFMA itself.
// With one max per page fixed before P is formed, P V is a plain accumulation: no per-slice products to scale
// and add, no branch between the slices' LDS reads. The V rows and P^T are written after the first barrier and
// read after the second, so one buffer of each serves every page. P keeps its rounding residue: with bf16 alone
// and no row of the page exactly 1 it is off by 1.6e-3 of the output (0.8e-3 against each 16-row slice's own max),
// and the second product costs 3% (B 4 / 4100 positions / T 8 / pps 8: 33.7 against 32.5 us a layer).
// Bound by the chain of a page: about 7000 cycles a page pair (stamps: K requests and scores 2000, maxima and
// barrier 1500, V and P into LDS 2000, P V 1400), both waves of a SIMD in the same phase; the scores of pages
// without new rows skip the masks. Measured per layer, G 6, with the pages a workgroup walks and their groups as they
// are now chosen: B 4 / 4100 positions ragged / T 8 / pps 8 163 -> 30 us against VALU dot products with two tokens a
// pass; B 1 / 8192 / T 4 / pps 2 24.9 -> 18.8 us with the mixer, 17.4 -> 15.9 without, against the pages one at a time with
// a scaled product per 16-row slice.
// The step's new rows (mixer: k normalised and rotated) are requested with the query rows and staged in LDS by
// the workgroups whose split holds their pages; they take the place of the pool's rows as the page is used (K in
// the score operand's registers, V as it is staged) and go to the pool after the page loop, so nothing waits for
// a store, no page is read twice, and the other row blocks of the split never depend on those stores.
// At the end the WPP groups' O meet in LDS, each group finishing its share of the query tiles.
constexpr int PP = BLK + 8;  // s_p row pitch (bf16)
// TN: the most new tokens a call brings, 8 or 16 (8: half the requests and LDS for the new rows)
template <int QT, bool MIX, int WPP, int TN>
struct RowsLds {
    static constexpr int NQR = 16 * QT, NW = 4 * WPP;
    static constexpr int Q = NQR * QPAD * 2, QL = MIX ? Q : 0, V = NW * 16 * VPAD * 2, P = 2 * WPP * NQR * PP * 2;
    static constexpr int NEW = TN * 2 * HD * 2, ML = NW * NQR * 4;
    static constexpr int bytes = Q + QL + V + P + NEW + 2 * ML;
    static_assert(bytes <= 163840, "LDS");
    static_assert(NQR * HD * 4 <= V || WPP == 1, "the groups' O exchange reuses the V rows");
};
template <int QT, bool MIX, int WPP, int TN>
__global__ __launch_bounds__(256 * WPP, 2) void attn_rows_kernel(AttnArgs a, int G, int nrb) {
    using S = RowsLds<QT, MIX, WPP, TN>;
    constexpr int NQR = S::NQR, NTH = 256 * WPP;
    // Q^T fragments in registers for the split where they fit beside the page's rows and the accumulators; else
    // read from LDS per page (the mixer's residues always)
    constexpr bool QREG = QT == 2;
    const int nwg = a.B * a.NKV * a.nsplit * nrb;
    const int lid = qs::xcd_logical(blockIdx.x, nwg);
    const int rb = lid % nrb;  // the row blocks of a split are neighbours: its pages come from L2 for all but one
    const int split = (lid / nrb) % a.nsplit;
    const int g = (lid / (nrb * a.nsplit)) % a.NKV;
    const int b = lid / (nrb * a.nsplit * a.NKV);
    // the wave index through readfirstlane: the compiler then knows the wave's page and row tests are uniform
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int w = wv & 3, ph = wv >> 2;
    const int l16 = lane & 15, lg = lane >> 4;
    const int T = a.T, R = T * G, r0 = rb * NQR;

    __shared__ __align__(16) unsigned char s_raw[S::bytes];
    auto s_q = reinterpret_cast<uint16_t (*)[QPAD]>(s_raw);
    auto s_ql = reinterpret_cast<uint16_t (*)[QPAD]>(s_raw + S::Q);
    auto s_v = reinterpret_cast<uint16_t (*)[VPAD]>(s_raw + S::Q + S::QL) + 64 * ph;  // the group's page of V rows
    auto s_p = reinterpret_cast<uint16_t (*)[PP]>(s_raw + S::Q + S::QL + S::V) + 2 * NQR * ph;  // hi rows, lo rows
    auto s_new = reinterpret_cast<uint16_t (*)[2][HD]>(s_raw + S::Q + S::QL + S::V + S::P);
    auto s_m = reinterpret_cast<float (*)[4]>(s_raw + S::Q + S::QL + S::V + S::P + S::NEW) + NQR * ph;  // [row][wave]
    auto s_l = reinterpret_cast<float (*)[NQR]>(s_raw + S::Q + S::QL + S::V + S::P + S::NEW + S::ML);
    auto s_o = reinterpret_cast<f32x4_t *>(s_raw + S::Q + S::QL);

    // Issued first, in this order: the split's block-table entries, the user's length, the query rows and the
    // new rows. The first page's K / V loads then wait only for the table entries and the length.
    const int p0 = split * a.pps;
    const int bt_pre = split_entries(a, b, p0, lane);
    const int n = a.seq_lens[b];
    constexpr int QCH = NQR * 32 / NTH, NCH = TN * 64 / NTH;
    uint4 qreg[QCH];
#pragma unroll
    for (int k = 0; k < QCH; ++k) {
        const int idx = tid + NTH * k;
        qreg[k] = q_chunk(a, G, b, g, r0 + (idx >> 5), idx & 31);
    }
    // the new rows of tokens wv, wv + 4 WPP, ...: chunk lane % 32 of the K row (lanes < 32) or the V row (zeros past T)
    u32x4 nk[NCH], nv[NCH];
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        nk[k] = new_chunk(a, a.k_new, b, g, wv + 4 * WPP * k, lane < 32 ? lane : -1);
        nv[k] = new_chunk(a, a.v_new, b, g, wv + 4 * WPP * k, lane < 32 ? -1 : lane - 32);
    }
    MixChunk mq[MIX ? QCH : 1], mk[MIX ? NCH : 1];
    if constexpr (MIX) {
        mix_weights(a.wq, lane & 31, mq[0]);
        mix_weights(a.wk, lane & 31, mk[0]);
#pragma unroll
        for (int k = 0; k < QCH; ++k) {
            if (k > 0) mq[k].w[0] = mq[0].w[0], mq[k].w[1] = mq[0].w[1];
            mix_angles(a, b * T + min((r0 + ((tid + NTH * k) >> 5)) / G, T - 1), lane & 31, mq[k]);
        }
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
            if (k > 0) mk[k].w[0] = mk[0].w[0], mk[k].w[1] = mk[0].w[1];
            mix_angles(a, b * T + min(wv + 4 * WPP * k, T - 1), lane & 31, mk[k]);
        }
    }
    auto page_at = [&](int pi) {
        const int pg = __builtin_amdgcn_readlane(bt_pre, pi - p0);
        return (pg >= 0 && pg < a.num_blocks) ? pg : -1;
    };
    const size_t pstride = (size_t)a.NKV * BLK * HD;  // elements per page
    // a page of -1 is an empty range: the loads still issue (no branch around them, so the compiler's waits
    // stay exact) and read zeros without touching memory
    auto load_k = [&](int pg, u32x4 (&kb)[8]) {
        const auto rk = __builtin_amdgcn_make_buffer_rsrc(
            qs::uniform_ptr(const_cast<uint16_t *>(a.k_cache + (size_t)max(pg, 0) * pstride + (size_t)g * BLK * HD)),
            (short)0, pg >= 0 ? BLK * HD * 2 : 0, 0x00020000);
        const int off = (16 * w + l16) * HD * 2 + lg * 16;
#pragma unroll
        for (int j = 0; j < 8; ++j) kb[j] = __builtin_amdgcn_raw_buffer_load_b128(rk, off, j * 64, NT);
    };
    auto load_v = [&](int pg, u32x4 (&vb)[8]) {
        const auto rv = __builtin_amdgcn_make_buffer_rsrc(
            qs::uniform_ptr(const_cast<uint16_t *>(a.v_cache + (size_t)max(pg, 0) * pstride + (size_t)g * BLK * HD)),
            (short)0, pg >= 0 ? BLK * HD * 2 : 0, 0x00020000);
        const int off = (16 * w + (lane >> 5)) * HD * 2 + (lane & 31) * 16;
#pragma unroll
        for (int k = 0; k < 8; ++k) vb[k] = __builtin_amdgcn_raw_buffer_load_b128(rv, off, k * 1024, NT);
    };

    // the group's first page, if the user's length reaches it (the length was requested with the table's entries)
    u32x4 kb[8], vb[8];
    const int pf = p0 + ph;
    const int pg0 = pf < min(a.max_blocks, p0 + a.pps) && pf * BLK < n ? page_at(pf) : -1;
    load_k(pg0, kb);
    load_v(pg0, vb);

    if (!user_active(a, n, split == 0 && g == 0 && rb == 0 && tid == 0)) {  // uniform over the user's workgroups
        if (split == 0 && rb == 0) zero_rows(a, G, b, g, tid, NTH);
        return;
    }
    if (!split_live(a, n, split)) return;
    const int base = n - T;  // first new position
    const int p1 = min((n + BLK - 1) / BLK, p0 + a.pps);
    // an entry of the split's pages outside the pool (lane pi - p0 checks entry pi) is reported after the
    // page loop: an atomic here, inside a branch, would make the compiler wait for every load at the next use
    const bool bad_pages = __any(lane < p1 - p0 && (bt_pre < 0 || bt_pre >= a.num_blocks));
    const bool fresh = a.k_new && base / BLK < p1 && (n - 1) / BLK >= p0;  // new rows in this split (uniform)

    // query rows (and the mixer's residues) and new rows into LDS
#pragma unroll
    for (int k = 0; k < QCH; ++k) {
        const int idx = tid + NTH * k, row = idx >> 5, ch = idx & 31;
        uint4 u = qreg[k];
        if constexpr (MIX) {  // normalised and rotated q (all lanes take part in the row reductions)
            float y[8];
            mixer_chunk(u, ch, mq[k], a.rot, a.eps, y);
            u = pack8(y);
            *reinterpret_cast<uint4 *>(&s_ql[row][ch * 8]) = pack8_lo(y, u);
        }
        *reinterpret_cast<uint4 *>(&s_q[row][ch * 8]) = u;
    }
    if (fresh)
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
            const int t = wv + 4 * WPP * k;
            if (t >= T) break;
            const u32x4 x = lane < 32 ? nk[k] : nv[k];
            uint4 u = make_uint4(x[0], x[1], x[2], x[3]);
            if constexpr (MIX) {  // k rows normalised and rotated; the V lanes take part in the shuffles only
                float y[8];
                mixer_chunk(u, lane & 31, mk[k], a.rot, a.eps, y);
                if (lane < 32) u = pack8(y);
            }
            *reinterpret_cast<uint4 *>(&s_new[t][lane >> 5][(lane & 31) * 8]) = u;
        }
    __syncthreads();
    bf16x8_t qr[QREG ? QT : 1][QREG ? 8 : 1];
    if constexpr (QREG)
#pragma unroll
        for (int nt = 0; nt < QT; ++nt)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                qr[nt][j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(&s_q[16 * nt + l16][32 * j + 8 * lg]));

    const float sl2 = a.scale * 1.4426950408889634f;  // log2 domain
    int lim[QT];           // the lane's causal limit per query tile: token qr / G sees positions <= base + token
    f32x4_t oacc[QT][4];   // O^T of head dims 64 w + 16 dd + 4 lg + i (dd < 4), query row r0 + 16 nt + l16
    float M[QT], L[QT];    // running max (the same in the group's 4 waves) and this wave's rows' sum
#pragma unroll
    for (int nt = 0; nt < QT; ++nt) {
        const int row = r0 + 16 * nt + l16;
        lim[nt] = row < R ? base + row / G : -1;
        M[nt] = -INFINITY;
        L[nt] = 0.f;
#pragma unroll
        for (int dd = 0; dd < 4; ++dd) oacc[nt][dd] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // every group takes the same number of steps (the barriers are the workgroup's); a group past its last page
    // works on an empty one
    for (int s0 = p0; s0 < p1; s0 += WPP) {
        const int pi = s0 + ph;
        const int pgn = pi + WPP < p1 ? page_at(pi + WPP) : -1;
        const bool ok = pi < p1 && page_at(pi) >= 0;
        const int r0w = pi * BLK + 16 * w;  // first position of this wave's rows
        // new rows among this wave's rows (uniform): token pos - base at row pos - r0w
        const bool has_new = fresh && ok && r0w + 16 > base && r0w < n;
        if (has_new) {  // the new K row at this lane's row over the pool's (dims 32 j + 8 lg)
            const int t = r0w + l16 - base;
            const bool kp = t >= 0 && t < T;
            u32x4 x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = *reinterpret_cast<const u32x4 *>(&s_new[min(max(t, 0), T - 1)][0][32 * j + 8 * lg]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) kb[j][e] = kp ? x[j][e] : kb[j][e];
        }
        f32x4_t sacc[QT];
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) sacc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bf16x8_t ak = __builtin_bit_cast(bf16x8_t, kb[j]);
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) {
                bf16x8_t bq;
                if constexpr (QREG)
                    bq = qr[nt][j];
                else
                    bq = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(&s_q[16 * nt + l16][32 * j + 8 * lg]));
                sacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak, bq, sacc[nt], 0, 0, 0);
                if constexpr (MIX) {
                    const bf16x8_t bl = __builtin_bit_cast(
                        bf16x8_t, *reinterpret_cast<const uint4 *>(&s_ql[16 * nt + l16][32 * j + 8 * lg]));
                    sacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak, bl, sacc[nt], 0, 0, 0);
                }
            }
        }
        load_k(pgn, kb);
        // every row of the page lies before the step's new rows: no masks, no patches (uniform; query rows past R
        // then take part unmasked, into outputs that are never stored)
        const bool full = ok && (pi + 1) * BLK <= base;
        // the scores in the log2 domain, -inf where masked, and their max over this wave's 16 rows
        float mx[QT];
        if (full) {
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) {
                sacc[nt] *= sl2;
                mx[nt] = fmaxf(fmaxf(sacc[nt][0], sacc[nt][1]), fmaxf(sacc[nt][2], sacc[nt][3]));
            }
        } else {
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) {
                mx[nt] = -INFINITY;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sacc[nt][i] = ok && r0w + 4 * lg + i <= lim[nt] ? sacc[nt][i] * sl2 : -INFINITY;
                    mx[nt] = fmaxf(mx[nt], sacc[nt][i]);
                }
            }
        }
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) mx[nt] = qs::xor32_max(qs::xor16_max(mx[nt]));
        if (lg == 0)
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) s_m[16 * nt + l16][w] = mx[nt];
        __syncthreads();  // the page's maxima are in LDS, and the previous page's V and P are no longer read
        f32x4_t pm[QT];
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) pm[nt] = *reinterpret_cast<const f32x4_t *>(&s_m[16 * nt + l16][0]);
        // V rows (zero where the page is invalid or past the user's length: a stale row times a zero
        // probability could be NaN), the new ones over the pool's
        if (full) {
#pragma unroll
            for (int k = 0; k < 8; ++k) *reinterpret_cast<u32x4 *>(&s_v[16 * w + 2 * k + (lane >> 5)][(lane & 31) * 8]) = vb[k];
        } else {
            u32x4 x[8] = {};
            if (has_new)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int t = r0w + 2 * k + (lane >> 5) - base;
                    x[k] = *reinterpret_cast<const u32x4 *>(&s_new[min(max(t, 0), T - 1)][1][(lane & 31) * 8]);
                }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int row = 2 * k + (lane >> 5), pos = r0w + row;
                const bool live = ok && pos < n, patch = has_new && live && pos >= base;
                u32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = patch ? x[k][e] : live ? vb[k][e] : 0u;
                *reinterpret_cast<u32x4 *>(&s_v[16 * w + row][(lane & 31) * 8]) = v;
            }
        }
        load_v(pgn, vb);
        float Mn[QT];
        bool move = false;
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) {
            const float m4 = fmaxf(fmaxf(pm[nt][0], pm[nt][1]), fmaxf(pm[nt][2], pm[nt][3]));
            Mn[nt] = m4 > M[nt] + 8.0f ? m4 : M[nt];  // from -inf: to any finite maximum
            move |= Mn[nt] != M[nt];
        }
        if (__any(move))
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) {
                const float alpha = M[nt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M[nt] - Mn[nt]);
                L[nt] *= alpha;
#pragma unroll
                for (int dd = 0; dd < 4; ++dd) oacc[nt][dd] *= alpha;
                M[nt] = Mn[nt];
            }
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) {
            const float Ms = M[nt] == -INFINITY ? 0.f : M[nt];  // nothing visible yet: every 2^(-inf - 0) is 0
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = __builtin_amdgcn_exp2f(sacc[nt][i] - Ms);
            const uint32_t p01 = qs::cvt_pk_bf16(e[0], e[1]), p23 = qs::cvt_pk_bf16(e[2], e[3]);
            const uint32_t l01 = qs::cvt_pk_bf16(e[0] - qs::bf_lo(p01), e[1] - qs::bf_hi(p01));
            const uint32_t l23 = qs::cvt_pk_bf16(e[2] - qs::bf_lo(p23), e[3] - qs::bf_hi(p23));
            *reinterpret_cast<uint2 *>(&s_p[16 * nt + l16][16 * w + 4 * lg]) = make_uint2(p01, p23);
            *reinterpret_cast<uint2 *>(&s_p[NQR + 16 * nt + l16][16 * w + 4 * lg]) = make_uint2(l01, l23);
            L[nt] += (e[0] + e[1]) + (e[2] + e[3]);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            bf16x8_t pb[2][QT];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int nt = 0; nt < QT; ++nt)
                    pb[h][nt] = __builtin_bit_cast(
                        bf16x8_t, *reinterpret_cast<const uint4 *>(&s_p[h * NQR + 16 * nt + l16][32 * kk + 8 * lg]));
#pragma unroll
            for (int dd = 0; dd < 4; ++dd) {
                i16x4_t av[2];  // V^T: head dim l16 of the tile, page rows 32 kk + 8 lg + 4 h .. + 3
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    av[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t *)&s_v[32 * kk + 8 * lg + 4 * h + (l16 >> 2)][64 * w + 16 * dd + 4 * (l16 & 3)]);
                const u32x2 a0 = __builtin_bit_cast(u32x2, av[0]), a1 = __builtin_bit_cast(u32x2, av[1]);
                const bf16x8_t va = __builtin_bit_cast(bf16x8_t, u32x4{a0[0], a0[1], a1[0], a1[1]});
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int nt = 0; nt < QT; ++nt)
                        oacc[nt][dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb[h][nt], oacc[nt][dd], 0, 0, 0);
            }
        }
    }

    if (bad_pages && rb == 0 && tid == 0) report_page(a);
    if (fresh && rb == 0)  // the new rows into the pool (lanes < 32 the K row, the others the V row)
        for (int t = wv; t < T; t += 4 * WPP) {
            const int pos = base + t, pi = pos / BLK;
            if (pi < p0 || pi >= p1) continue;
            const int pg = page_at(pi);
            if (pg < 0) continue;  // reported with the split's pages
            const size_t row = (((size_t)pg * a.NKV + g) * BLK + pos % BLK) * HD + (lane & 31) * 8;
            *reinterpret_cast<u32x4 *>((lane < 32 ? a.k_cache : a.v_cache) + row) =
                *reinterpret_cast<const u32x4 *>(&s_new[t][lane >> 5][(lane & 31) * 8]);
        }

    // the waves' row sums and the groups' maxima
#pragma unroll
    for (int nt = 0; nt < QT; ++nt) {
        const float ls = qs::xor32_sum(qs::xor16_sum(L[nt]));
        if (lg == 0) {
            s_l[wv][16 * nt + l16] = ls;
            if (w == 0) s_m[16 * nt + l16][0] = M[nt];
        }
    }
    __syncthreads();
    auto mine = [&](int nt) { return WPP == 1 || (nt < (QT + 1) / 2) == (ph == 0); };  // tiles this group finishes
    float sc[QT], Mx[QT], Lx[QT];  // this group's scale, and the split's max and sum of each row
#pragma unroll
    for (int nt = 0; nt < QT; ++nt) {
        const int row = 16 * nt + l16;
        const float lo = ((s_l[4 * ph][row] + s_l[4 * ph + 1][row]) + s_l[4 * ph + 2][row]) + s_l[4 * ph + 3][row];
        Mx[nt] = M[nt], Lx[nt] = lo, sc[nt] = 1.f;
        if constexpr (WPP == 2) {
            const int po = 4 * (1 - ph);
            const float mo = s_m[(1 - 2 * ph) * NQR + row][0];  // s_m is based at the own group's rows
            const float l2 = ((s_l[po][row] + s_l[po + 1][row]) + s_l[po + 2][row]) + s_l[po + 3][row];
            Mx[nt] = fmaxf(M[nt], mo);
            sc[nt] = M[nt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M[nt] - Mx[nt]);
            Lx[nt] = sc[nt] * lo + (mo == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mo - Mx[nt])) * l2;
            if (!mine(nt))
#pragma unroll
                for (int dd = 0; dd < 4; ++dd) s_o[((nt * 4 + w) * 4 + dd) * 64 + lane] = oacc[nt][dd] * sc[nt];
        }
    }
    if constexpr (WPP == 2) __syncthreads();

    // this wave's head dims of the group's tiles of the split's partial (or of the output); the partials are
    // written through to the agent-coherent level (sc1), where the merge launch reads them
    const auto rpo = __builtin_amdgcn_make_buffer_rsrc(a.part_o + prow(a, G, b, g, split, 0) * HD, (short)0,
                                                       R * HD * 4, 0x00020000);
    const auto rpm = __builtin_amdgcn_make_buffer_rsrc(a.part_ml + prow(a, G, b, g, split, 0) * 2, (short)0,
                                                       R * 8, 0x00020000);
#pragma unroll
    for (int nt = 0; nt < QT; ++nt) {
        const int row = r0 + 16 * nt + l16;
        if (!mine(nt) || row >= R) continue;
        f32x4_t v[4];
#pragma unroll
        for (int dd = 0; dd < 4; ++dd) {
            v[dd] = oacc[nt][dd] * sc[nt];
            if constexpr (WPP == 2) v[dd] += s_o[((nt * 4 + w) * 4 + dd) * 64 + lane];
        }
        if (a.nsplit == 1) {
            const float inv = 1.0f / Lx[nt];
            const size_t oi = (((size_t)b * T + row / G) * a.NQ + g * G + row % G) * HD + 64 * w + 4 * lg;
#pragma unroll
            for (int dd = 0; dd < 4; ++dd) {
                v[dd] *= inv;
                if (a.gate) {
                    const uint2 gw = *reinterpret_cast<const uint2 *>(a.gate + oi + 16 * dd);
                    v[dd][0] *= sigm(qs::bf_lo(gw.x)), v[dd][1] *= sigm(qs::bf_hi(gw.x));
                    v[dd][2] *= sigm(qs::bf_lo(gw.y)), v[dd][3] *= sigm(qs::bf_hi(gw.y));
                }
                *reinterpret_cast<uint2 *>(a.o + oi + 16 * dd) =
                    make_uint2(qs::cvt_pk_bf16(v[dd][0], v[dd][1]), qs::cvt_pk_bf16(v[dd][2], v[dd][3]));
            }
        } else {
#pragma unroll
            for (int dd = 0; dd < 4; ++dd)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[dd]), rpo,
                                                       (row * HD + 64 * w + 16 * dd + 4 * lg) * 4, 0, qs::CP_SC1);
            if (w == 0 && lg == 0)
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(Mx[nt]), __float_as_uint(Lx[nt])}, rpm,
                                                      row * 8, 0, qs::CP_SC1);
        }
    }
}

// ------------------------------------------------------------------- MFMA kernel, independent waves
// Up to 16 query rows per KV head (every one-token decode, and verify steps with T G <= 16). One workgroup per
// (user, KV head, split of pps pages) with 4 WPP waves: wave w owns rows
// 16 (w % 4) .. + 15 of pages p0 + w / 4, p0 + w / 4 + WPP, ... of the split (WPP pages in flight per
// workgroup) and walks them on its own, with no workgroup barrier inside the page loop:
//   scores  S^T [16 rows x 16 q] = K Q^T on 8 v_mfma_f32_16x16x32_bf16 (K rows loaded as whole 512-byte rows
//           and turned into the A operand through the wave's LDS slice; with one page per workgroup, whose
//           chain nothing overlaps, loaded straight in the operand's layout; Q^T held in registers);
//   softmax per query row against the wave's running max M (log2 domain): P = 2^(s - M) rounded to bf16
//           lands, lane for lane, in the B-operand layout of the P V product, so P never leaves the
//           registers; M moves only when a slice max exceeds it by 2^8 (the accumulators are then rescaled),
//           so P <= 2^8;
//   P V     O^T [256 dims x 16 q] += V^T P on 16 v_mfma_f32_16x16x16_bf16, accumulated by the MFMA itself,
//           V^T read from the same LDS slice (now holding the page's 16 V rows) with the transposing
//           ds_read_b64_tr_b16.
// Each wave keeps one page of K and V in flight (refilled as soon as consumed). At the end of the split the
// waves' (max, sum) meet in LDS and their O, scaled to the common max, is summed through LDS in a fixed order
// ((w + 4) pairs first when WPP = 2), every wave summing and storing a share of the head dims; the split's
// partial, or with one split the output, has the layout the in-launch and separate merges read.
constexpr int OPAD = HD + 4;  // fp32 row pitch of the waves' O rows in LDS
template <int G, int WPP, bool MIX>
__global__ __launch_bounds__(256 * WPP, WPP == 1 ? 2 : 1) void attn_wave_kernel(AttnArgs a) {
    constexpr int QT = 1, NQR = 16;
    constexpr int NWV = 4 * WPP, NTH = 64 * NWV;
    const int nwg = a.B * a.NKV * a.nsplit;
    const int lid = qs::xcd_logical(blockIdx.x, nwg);
    const int split = lid % a.nsplit;
    const int g = (lid / a.nsplit) % a.NKV;
    const int b = lid / (a.nsplit * a.NKV);
    // the wave index through readfirstlane: the compiler then knows every page index and page address
    // derived from it is uniform over the wave (else each page load becomes a loop over the lanes' addresses)
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sl = w & 3, ph = w >> 2;  // the wave's 16-row slice and page phase
    const int l16 = lane & 15, lg = lane >> 4;
    const int T = a.T;

    // LDS: the q rows (and the mixer's residues) and the waves' K / V slices during the page loop; after it
    // the same bytes hold 4 waves' scaled O rows
    constexpr int QB = NQR * QPAD * 2, QLB = (MIX ? NQR : 1) * QPAD * 2, KVB = NWV * 16 * VPAD * 2;
    constexpr int OB = 4 * NQR * OPAD * 4;
    constexpr int LB = QB + QLB + KVB > OB ? QB + QLB + KVB : OB;
    __shared__ __align__(16) unsigned char s_raw[LB];
    auto s_q = reinterpret_cast<uint16_t (*)[QPAD]>(s_raw);
    auto s_ql = reinterpret_cast<uint16_t (*)[QPAD]>(s_raw + QB);
    auto s_kv = reinterpret_cast<uint16_t (*)[16][VPAD]>(s_raw + QB + QLB);
    auto s_o = reinterpret_cast<float (*)[NQR][OPAD]>(s_raw);
    __shared__ float s_ml[NWV][NQR][2];
    // the step's new K / V rows: every one with the mixer (k normalised and rotated), the K rows for the score
    // operand with WPP = 1
    __shared__ __align__(16) uint16_t s_nw[MIX || WPP == 1 ? 2 : 1][2][HD];

    const int p0 = split * a.pps;
    const int *bt = a.block_table + (size_t)b * a.max_blocks;
    const int bt_pre = split_entries(a, b, p0, lane);
    const int n = a.seq_lens[b];
    constexpr int QCH = (NQR * 32 + NTH - 1) / NTH;
    uint4 qreg[QCH];
#pragma unroll
    for (int k = 0; k < QCH; ++k) {
        const int idx = tid + NTH * k;
        qreg[k] = q_chunk(a, G, b, g, idx >> 5, idx & 31);  // rows past NQR are never staged
    }
    // The step's new K / V rows (up to TN tokens; more go through the pool below): chunk lane % 32 of the K row
    // (lanes < 32) or of the V row, requested before the pages like the query rows. Every wave holds all of them
    // in registers; with the mixer, which leaves none, wave t turns token t's K row and puts both rows in LDS.
    constexpr int TN = 2, NTK = MIX ? 1 : TN;
    u32x4 nk[NTK], nv[NTK];  // vector types (not uint4): selects stay in registers
#pragma unroll
    for (int t = 0; t < NTK; ++t) {
        const int tok = MIX ? (w < TN ? w : T) : t;
        nk[t] = new_chunk(a, a.k_new, b, g, tok, lane < 32 ? lane : -1);
        nv[t] = new_chunk(a, a.v_new, b, g, tok, lane < 32 ? -1 : lane - 32);
    }
    MixChunk mq[MIX ? QCH : 1], mk;
    if constexpr (MIX) {
        mix_weights(a.wq, lane & 31, mq[0]);
        mix_weights(a.wk, lane & 31, mk);
#pragma unroll
        for (int k = 0; k < QCH; ++k) {
            if (k > 0) mq[k].w[0] = mq[0].w[0], mq[k].w[1] = mq[0].w[1];
            mix_angles(a, b * T + min(((tid + NTH * k) >> 5) / G, T - 1), lane & 31, mq[k]);
        }
        mix_angles(a, b * T + min(w, T - 1), lane & 31, mk);
    }
    auto page_at = [&](int pi) {
        const int pg = __builtin_amdgcn_readlane(bt_pre, pi - p0);
        return (pg >= 0 && pg < a.num_blocks) ? pg : -1;
    };
    const size_t pstride = (size_t)a.NKV * BLK * HD;
    // K and V rows load alike, two whole 512-byte rows per instruction (lane: row 2 k + lane / 32, 16 bytes at
    // (lane % 32) 16): a gather of 16-byte pieces of 16 rows per instruction streams ~20% slower
    // (a page of -1 is an empty range: the loads still issue, with no branch around them, so the compiler's
    // waits stay exact, and read zeros without touching memory)
    auto load_rows = [&](const uint16_t *pool, int pg, uint4 (&rb)[8]) {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(
            qs::uniform_ptr(const_cast<uint16_t *>(pool + (size_t)max(pg, 0) * pstride + (size_t)g * BLK * HD)),
            (short)0, pg >= 0 ? BLK * HD * 2 : 0, 0x00020000);
        const int off = (16 * sl + (lane >> 5)) * HD * 2 + (lane & 31) * 16;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, off, k * 1024, NT);
            rb[k] = make_uint4(x[0], x[1], x[2], x[3]);
        }
    };
    // one page per workgroup (WPP = 1): K straight into the score operand's layout (lane: row 16 sl + l16,
    // dims 32 j + 8 lg .. + 7), no staging through LDS
    auto load_kfrag = [&](int pg, uint4 (&rb)[8]) {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(
            qs::uniform_ptr(const_cast<uint16_t *>(a.k_cache + (size_t)max(pg, 0) * pstride + (size_t)g * BLK * HD)),
            (short)0, pg >= 0 ? BLK * HD * 2 : 0, 0x00020000);
        const int off = (16 * sl + l16) * HD * 2 + lg * 16;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, off, j * 64, NT);
            rb[j] = make_uint4(x[0], x[1], x[2], x[3]);
        }
    };
    uint4 KA[8], VA[8];
    const int pf = p0 + ph;  // this wave's first page, if the user's length reaches it
    const int pg0 = pf < min(a.max_blocks, p0 + a.pps) && pf * BLK < n ? page_at(pf) : -1;
    if constexpr (WPP == 1)
        load_kfrag(pg0, KA);
    else
        load_rows(a.k_cache, pg0, KA);
    load_rows(a.v_cache, pg0, VA);

    if (!user_active(a, n, split == 0 && g == 0 && tid == 0)) {  // uniform over the user's workgroups
        if (split == 0) zero_rows(a, G, b, g, tid, NTH);
        return;
    }
    if (!split_live(a, n, split)) return;
    const int base = n - T;
    const int npages = (n + BLK - 1) / BLK;
    const int p1 = min(npages, p0 + a.pps);
    // an entry of the split's pages outside the pool (lane pi - p0 checks entry pi) is reported after the
    // page loop: an atomic here, inside a branch, would make the compiler wait for every load at the next use
    const bool bad_pages = __any(lane < p1 - p0 && (bt_pre < 0 || bt_pre >= a.num_blocks));

    // Fused append. Up to TN tokens: the new rows stay in registers (or LDS), the page loop writes them over
    // the staged rows of this wave's slices, and they go to the pool after the loop, so no store is in flight
    // while pages load (the compiler would then wait for every load at each use), nothing waits for the
    // stores, and no page is read twice. More tokens: each wave writes the new rows of its own slices to the
    // pool and waits for them before its pages are read (it alone reads them back).
    const bool fresh = a.k_new && T <= TN;
    auto owned = [&](int pos) {  // a new row this wave attends: in one of its pages and in its slice
        const int pi = pos / BLK;
        return pi >= p0 && pi < p1 && (pos % BLK) / 16 == sl && (pi - p0) % WPP == ph;
    };
    if (a.k_new && !fresh && p0 < p1 && base / BLK < p1 && (n - 1) / BLK >= p0) {
        for (int idx = lane; idx < T * 64; idx += 64) {
            const int t = idx >> 6, kv = (idx >> 5) & 1, ch = idx & 31;
            const int pos = base + t, pi = pos / BLK;
            const size_t src = (((size_t)b * T + t) * a.NKV + g) * HD + ch * 8;
            uint4 u = *reinterpret_cast<const uint4 *>((kv ? a.v_new : a.k_new) + src);
            if constexpr (MIX) {
                float y[8];
                mix_angles(a, b * T + t, ch, mk);
                mixer_chunk(u, ch, mk, a.rot, a.eps, y);
                if (!kv) u = pack8(y);
            }
            if (!owned(pos)) continue;
            const int pg = bt[pi];
            if (pg < 0 || pg >= a.num_blocks) continue;  // reported with the split's pages above
            const size_t dst = (((size_t)pg * a.NKV + g) * BLK + (pos % BLK)) * HD + ch * 8;
            *reinterpret_cast<uint4 *>((kv ? a.v_cache : a.k_cache) + dst) = u;
        }
        qs::wait_vmem();
        if (pg0 >= 0 && base / BLK <= pf) {  // new rows landed in this wave's first page: read it again
            if constexpr (WPP == 1)
                load_kfrag(pg0, KA);
            else
                load_rows(a.k_cache, pg0, KA);
            load_rows(a.v_cache, pg0, VA);
        }
    }

    // q rows (normalised and rotated for the mixer) through LDS into B-operand registers, kept for the split
#pragma unroll
    for (int k = 0; k < QCH; ++k) {
        const int idx = tid + NTH * k, qr = idx >> 5, ch = idx & 31;
        if (qr >= NQR) continue;
        uint4 u = qreg[k];
        if constexpr (MIX) {
            float y[8];
            mixer_chunk(u, ch, mq[k], a.rot, a.eps, y);
            u = pack8(y);
            *reinterpret_cast<uint4 *>(&s_ql[qr][ch * 8]) = pack8_lo(y, u);
        }
        *reinterpret_cast<uint4 *>(&s_q[qr][ch * 8]) = u;
    }
    if constexpr (MIX) {
        if (fresh && w < T) {
            uint4 u = make_uint4(nk[0][0], nk[0][1], nk[0][2], nk[0][3]);
            float y[8];
            mixer_chunk(u, lane & 31, mk, a.rot, a.eps, y);
            if (lane < 32) u = pack8(y);
            *reinterpret_cast<u32x4 *>(&s_nw[w][lane >> 5][(lane & 31) * 8]) = lane < 32 ? u32x4{u.x, u.y, u.z, u.w} : nv[0];
        }
    } else if constexpr (WPP == 1) {
        if (w == 0 && lane < 32)
#pragma unroll
            for (int t = 0; t < TN; ++t) *reinterpret_cast<u32x4 *>(&s_nw[t][0][lane * 8]) = nk[t];
    }
    __syncthreads();
    // token t's new K row (kv 0, lanes < 32) or V row (kv 1, lanes >= 32), this lane's chunk
    auto new_row = [&](int t, int kv) -> u32x4 {
        if constexpr (MIX)
            return *reinterpret_cast<const u32x4 *>(&s_nw[t][kv][(lane & 31) * 8]);
        else
            return kv ? nv[t] : nk[t];
    };
    // Q^T fragments, held in registers for the split
    bf16x8_t qb[QT][8], qlo[QT][MIX ? 8 : 1];
#pragma unroll
    for (int nt = 0; nt < QT; ++nt)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            qb[nt][j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(&s_q[16 * nt + l16][32 * j + 8 * lg]));
            if constexpr (MIX)
                qlo[nt][j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(&s_ql[16 * nt + l16][32 * j + 8 * lg]));
        }

    const float sl2 = a.scale * 1.4426950408889634f;
    int lim[QT];  // this lane's query row of tile nt sees positions <= lim[nt]
    f32x4_t oacc[QT][16];  // O^T of head dims 16 t + 4 lg + i, query row 16 nt + l16
    float M[QT], L[QT];
#pragma unroll
    for (int nt = 0; nt < QT; ++nt) {
        const int qr = 16 * nt + l16;
        lim[nt] = qr < T * G ? base + qr / G : -1;
        M[nt] = -INFINITY;
        L[nt] = 0.f;
#pragma unroll
        for (int t = 0; t < 16; ++t) oacc[nt][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    for (int pi = pf; pi < p1; pi += WPP) {
        const int pgn = pi + WPP < p1 ? page_at(pi + WPP) : -1;
        const bool ok = page_at(pi) >= 0;
        const int r0w = pi * BLK + 16 * sl;
        f32x4_t sacc[QT];
        if constexpr (WPP == 1) {  // K already in the operand's layout; the new rows patched from LDS
            if (fresh && base + T > r0w && base < r0w + 16) {  // new rows in this slice (uniform)
                const int t = r0w + l16 - base;
                const bool kp = t >= 0 && t < T;
                u32x4 x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    x[j] = *reinterpret_cast<const u32x4 *>(&s_nw[min(max(t, 0), TN - 1)][0][32 * j + 8 * lg]);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    KA[j].x = kp ? x[j][0] : KA[j].x;
                    KA[j].y = kp ? x[j][1] : KA[j].y;
                    KA[j].z = kp ? x[j][2] : KA[j].z;
                    KA[j].w = kp ? x[j][3] : KA[j].w;
                }
            }
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) {
                sacc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const bf16x8_t kb = __builtin_bit_cast(bf16x8_t, KA[j]);
                    sacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb, qb[nt][j], sacc[nt], 0, 0, 0);
                    if constexpr (MIX)
                        sacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb, qlo[nt][j], sacc[nt], 0, 0, 0);
                }
            }
            load_kfrag(pgn, KA);
        } else {
        // K rows through the wave's LDS slice into the A operand (row l16, dims 32 j + 8 lg .. + 7); the next
        // page's K is requested as soon as the rows are in LDS. Scores of masked rows are replaced below.
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
            *reinterpret_cast<uint4 *>(&s_kv[w][2 * kk + (lane >> 5)][(lane & 31) * 8]) = KA[kk];
        if (fresh)  // the step's new K rows over the staged ones (whatever the pool held there)
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (t < T && base + t >= r0w && base + t < r0w + 16 && lane < 32)
                    *reinterpret_cast<u32x4 *>(&s_kv[w][base + t - r0w][lane * 8]) = new_row(t, 0);
        load_rows(a.k_cache, pgn, KA);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // K fragments (row l16, dims 32 j + 8 lg .. + 7), each used by every query tile
        constexpr int KG = 8;
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) sacc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j0 = 0; j0 < 8; j0 += KG) {
            bf16x8_t kb[KG];
#pragma unroll
            for (int j = 0; j < KG; ++j)
                kb[j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(&s_kv[w][l16][32 * (j0 + j) + 8 * lg]));
#pragma unroll
            for (int nt = 0; nt < QT; ++nt)
#pragma unroll
                for (int j = 0; j < KG; ++j) {
                    sacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[j], qb[nt][j0 + j], sacc[nt], 0, 0, 0);
                    if constexpr (MIX)
                        sacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[j], qlo[nt][j0 + j], sacc[nt], 0, 0, 0);
                }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the K reads are done before V overwrites the slice
        }
        // this page's V rows into the slice (zero where invalid or past the length: a stale row times a zero
        // probability could be NaN), then the next page's V into the registers
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            const int row = 2 * kk + (lane >> 5);
            const uint4 v = ok && r0w + row < n ? VA[kk] : make_uint4(0, 0, 0, 0);
            *reinterpret_cast<uint4 *>(&s_kv[w][row][(lane & 31) * 8]) = v;
        }
        if (fresh && ok)  // the new V rows
#pragma unroll
            for (int t = 0; t < TN; ++t)
                if (t < T && base + t >= r0w && base + t < r0w + 16 && lane >= 32)
                    *reinterpret_cast<u32x4 *>(&s_kv[w][base + t - r0w][(lane - 32) * 8]) = new_row(t, 1);
        load_rows(a.v_cache, pgn, VA);
        i16x4_t pb[QT];
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) {
            float sc[4], mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[i] = ok && r0w + 4 * lg + i <= lim[nt] ? sacc[nt][i] : -INFINITY;
                mx = fmaxf(mx, sc[i]);
            }
            mx = qs::xor32_max(qs::xor16_max(mx));
            const float ms = mx * sl2;  // -inf when no row of the slice is visible to this query row
            const bool move = M[nt] == -INFINITY ? ms != -INFINITY : ms > M[nt] + 8.0f;
            if (__any(move)) {
                const float Mn = move ? ms : M[nt];
                const float alpha = M[nt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M[nt] - Mn);
                L[nt] *= alpha;
#pragma unroll
                for (int t = 0; t < 16; ++t) oacc[nt][t] *= alpha;
                M[nt] = Mn;
            }
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = sc[i] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(fmaf(sc[i], sl2, -M[nt]));
            const uint32_t p01 = qs::cvt_pk_bf16(e[0], e[1]), p23 = qs::cvt_pk_bf16(e[2], e[3]);
            float ls = (qs::bf_lo(p01) + qs::bf_hi(p01)) + (qs::bf_lo(p23) + qs::bf_hi(p23));
            L[nt] += qs::xor32_sum(qs::xor16_sum(ls));
            pb[nt] = __builtin_bit_cast(i16x4_t, make_uint2(p01, p23));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the V staging has landed in LDS
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const i16x4_t av = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4_t *)&s_kv[w][4 * lg + (l16 >> 2)][16 * t + 4 * (l16 & 3)]);
#pragma unroll
            for (int nt = 0; nt < QT; ++nt)
                oacc[nt][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, pb[nt], oacc[nt][t], 0, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads are done before the next page's staging
    }

    if (bad_pages && tid == 0) report_page(a);
    if (fresh)  // the new rows this wave attended into the pool (lanes < 32 the K row, the others the V row)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int pos = base + t;
            if (t >= T || !owned(pos)) continue;
            const int pg = page_at(pos / BLK);
            if (pg < 0) continue;  // reported with the split's pages
            const size_t dst = (((size_t)pg * a.NKV + g) * BLK + (pos % BLK)) * HD + (lane & 31) * 8;
            *reinterpret_cast<u32x4 *>((lane < 32 ? a.k_cache : a.v_cache) + dst) = lane < 32 ? new_row(t, 0) : new_row(t, 1);
        }
    // the waves' (max, sum) per query row; the barrier also frees the q and K / V bytes for the O rows
    if (lg == 0)
#pragma unroll
        for (int nt = 0; nt < QT; ++nt) {
            s_ml[w][16 * nt + l16][0] = M[nt];
            s_ml[w][16 * nt + l16][1] = L[nt];
        }
    __syncthreads();
    auto row_ml = [&](int r, float &Mr, float &Lr) {
        Mr = -INFINITY;
#pragma unroll
        for (int ww = 0; ww < NWV; ++ww) Mr = fmaxf(Mr, s_ml[ww][r][0]);
        Lr = 0.f;
#pragma unroll
        for (int ww = 0; ww < NWV; ++ww) {
            const float mw = s_ml[ww][r][0];
            Lr += (mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - Mr)) * s_ml[ww][r][1];
        }
    };
    const int R = T * G;  // live query rows
    // each wave's O scaled to the common max: waves 4 .. 7 store theirs, then waves 0 .. 3 add their own
    // (WPP = 2); with WPP = 1 every wave stores
#pragma unroll
    for (int stage = 0; stage < WPP; ++stage) {
        if (ph == WPP - 1 - stage) {
#pragma unroll
            for (int nt = 0; nt < QT; ++nt) {
                const int qr = 16 * nt + l16;
                if (qr >= R) continue;
                float Ms, Ls;
                row_ml(qr, Ms, Ls);
                const float sw = M[nt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M[nt] - Ms);
                f32x4_t *dst = reinterpret_cast<f32x4_t *>(&s_o[sl][qr][4 * lg]);  // + 4 t: head dims 16 t + ..
                if (stage == 0) {
#pragma unroll
                    for (int t = 0; t < 16; ++t) dst[4 * t] = oacc[nt][t] * sw;
                } else {  // every read first, then every write: one LDS round trip, not one per piece
                    f32x4_t prev[16];
#pragma unroll
                    for (int t = 0; t < 16; ++t) prev[t] = dst[4 * t];
#pragma unroll
                    for (int t = 0; t < 16; ++t) dst[4 * t] = oacc[nt][t] * sw + prev[t];
                }
            }
        }
        __syncthreads();
    }
    // wave w: head dims (64 / WPP) w .. of every live row summed over the 4 slots in order
    constexpr int DPW = HD / NWV;      // head dims per wave
    constexpr int PPR = DPW / 4 / 4;   // 16-byte pieces per lane per row (4 lanes per row of a 16-row tile)
    const auto rpo = __builtin_amdgcn_make_buffer_rsrc(a.part_o + prow(a, G, b, g, split, 0) * HD, (short)0,
                                                       R * HD * 4, 0x00020000);
#pragma unroll
    for (int nt = 0; nt < QT; ++nt) {
        const int qr = 16 * nt + l16;
        if (qr >= R) continue;
        const int tt = qr / G, hh = qr % G;
        float Ls = 0.f;
        if (a.nsplit == 1) {
            float Ms;
            row_ml(qr, Ms, Ls);
        }
#pragma unroll
        for (int k = 0; k < PPR; ++k) {
            const int d = DPW * w + 4 * (lg + 4 * k);
            f32x4_t v = *reinterpret_cast<const f32x4_t *>(&s_o[0][qr][d]);
            v += *reinterpret_cast<const f32x4_t *>(&s_o[1][qr][d]);
            v += *reinterpret_cast<const f32x4_t *>(&s_o[2][qr][d]);
            v += *reinterpret_cast<const f32x4_t *>(&s_o[3][qr][d]);
            if (a.nsplit == 1) {
                const size_t oi = (((size_t)b * T + tt) * a.NQ + g * G + hh) * HD + d;
                v *= 1.0f / Ls;
                if (a.gate) {
                    const uint2 gw = *reinterpret_cast<const uint2 *>(a.gate + oi);
                    v[0] *= sigm(qs::bf_lo(gw.x)), v[1] *= sigm(qs::bf_hi(gw.x));
                    v[2] *= sigm(qs::bf_lo(gw.y)), v[3] *= sigm(qs::bf_hi(gw.y));
                }
                *reinterpret_cast<uint2 *>(a.o + oi) = make_uint2(qs::cvt_pk_bf16(v[0], v[1]), qs::cvt_pk_bf16(v[2], v[3]));
            } else {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rpo, (qr * HD + d) * 4, 0,
                                                       qs::CP_SC1);
            }
        }
    }
    if (a.nsplit > 1 && tid < R) {
        const auto rpm = __builtin_amdgcn_make_buffer_rsrc(a.part_ml + prow(a, G, b, g, split, 0) * 2, (short)0,
                                                           R * 8, 0x00020000);
        float Mr, Lr;
        row_ml(tid, Mr, Lr);
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(Mr), __float_as_uint(Lr)}, rpm, tid * 8, 0,
                                              qs::CP_SC1);
    }
    if (a.merge) merge_in_launch<NWV>(a, G, b, g, tid, n);
}

// Merge of the splits of one output row (user, token, query head) in one memory round trip: wave w sums
// splits w, w + 4, w + 8, ... (lane l owns head dims 4 l .. 4 l + 3), and every wave finds the global max M
// (log2 domain, as the partials store it) and the sum L from all splits' (m, l), whose loads are in flight
// together with the partials. The 4 waves' sums are added in wave order through LDS; every reduction runs
// in a fixed order, so the result is identical run to run. (The leader side of the reference: global max,
// rescale, sum, normalise, kernels/attn_leader_writer.cpp:86-106, kernels/attn_leader_compute.cpp:42-79.)
constexpr int MAX_SPLITS = 1024;
constexpr int MCH = 16;  // splits per wave per batch of loads (64 splits in one round trip)
// MLR: 64-split groups of (m, l) pairs read. Up to 64 splits take 1, whose maxima also weight the partials: 31 fewer
// loads per wave (two layers at batch 1 / 32768, 64 splits: 61.9 -> 61.0 us).
template <int MLR>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnArgs a, int G) {
    __shared__ float4 s_part[4][64];
    const int rowh = blockIdx.x;  // ((b * T + t) * NKV + g) * G + h
    const int h = rowh % G, row = rowh / G;
    const int g = row % a.NKV, bt = row / a.NKV;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ns = a.nsplit, R = a.T * G;
    const int n = a.seq_lens[bt / a.T], live = live_splits<MLR == 1>(a, n, lane);
    // The row's partials are requested before the length is checked: their addresses do not depend on it and
    // lie in the workspace either way, so the launch waits for one round trip, not two. Buffer loads, with a
    // wave's split offset in a scalar register and the lane's 16 bytes as the vector offset, need no per-load
    // address arithmetic; the (m, l) of splits past ns lie past the descriptor's range and read zeros.
    const size_t pr = prow(a, G, bt / a.T, g, 0, (bt % a.T) * G + h);
    const int sbytes = R * HD * 4;  // bytes between consecutive splits of one row's O
    const auto rpo = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(a.part_o + pr * HD), (short)0, ns * sbytes,
                                                       0x00020000);
    const auto rml = __builtin_amdgcn_make_buffer_rsrc(qs::uniform_ptr(a.part_ml + pr * 2), (short)0, ns * R * 8,
                                                       0x00020000);
    auto load_split = [&](int sp, float4 &v, float &m) {  // sp wave-uniform, < ns
        const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(rpo, lane * 16, sp * sbytes, 0);
        v = make_float4(__uint_as_float(u[0]), __uint_as_float(u[1]), __uint_as_float(u[2]), __uint_as_float(u[3]));
        if constexpr (MLR > 1) m = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rml, 0, sp * R * 8, 0));
    };
    float4 x[MCH];
    float mw[MCH];
#pragma unroll
    for (int k = 0; k < MCH; ++k) load_split(min(w + 4 * k, ns - 1), x[k], mw[k]);
    // global max and sum over all splits: lane l covers splits l, l + 64, ...
    float M = -INFINITY;
    float2 mg[MLR];
#pragma unroll
    for (int j = 0; j < MLR; ++j) {
        const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(rml, (lane + 64 * j) * R * 8, 0, 0);
        mg[j] = lane + 64 * j < live ? make_float2(__uint_as_float(u[0]), __uint_as_float(u[1]))
                                   : make_float2(-INFINITY, 0.f);
        M = fmaxf(M, mg[j].x);
    }
    if (n < a.T || n > a.max_blocks * BLK) {  // inactive user (reported by the attention launch): zero row
        if (w == 0)
            *reinterpret_cast<uint2 *>(a.o + ((size_t)bt * a.NQ + g * G + h) * HD + 4 * lane) = make_uint2(0, 0);
        return;
    }
    M = qs::wave_max_bcast(M);
    float L = 0.f;
#pragma unroll
    for (int j = 0; j < MLR; ++j)
        if (mg[j].x != -INFINITY) L += __builtin_amdgcn_exp2f(mg[j].x - M) * mg[j].y;
    L = qs::wave_sum_dpp(L);
    float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
    auto acc = [&](int sp, const float4 &v, float m) {
        if (sp < live && m != -INFINITY) {
            const float e = __builtin_amdgcn_exp2f(m - M);
            O.x += e * v.x, O.y += e * v.y, O.z += e * v.z, O.w += e * v.w;
        }
    };
#pragma unroll
    for (int k = 0; k < MCH; ++k) acc(w + 4 * k, x[k], MLR > 1 ? mw[k] : qs::lane_val(mg[0].x, w + 4 * k));
    if constexpr (MLR > 1) {
        for (int s0 = 4 * MCH; s0 < live; s0 += 4 * MCH) {  // further splits, a batch of loads at a time
#pragma unroll
            for (int k = 0; k < MCH; ++k) load_split(min(s0 + w + 4 * k, ns - 1), x[k], mw[k]);
#pragma unroll
            for (int k = 0; k < MCH; ++k) acc(s0 + w + 4 * k, x[k], mw[k]);
        }
    }
    s_part[w][lane] = O;
    __syncthreads();
    if (w != 0) return;
    const float4 p1 = s_part[1][lane], p2 = s_part[2][lane], p3 = s_part[3][lane];
    const float inv = 1.0f / L;
    const float r0 = (((O.x + p1.x) + p2.x) + p3.x) * inv, r1 = (((O.y + p1.y) + p2.y) + p3.y) * inv;
    const float r2 = (((O.z + p1.z) + p2.z) + p3.z) * inv, r3 = (((O.w + p1.w) + p2.w) + p3.w) * inv;
    const size_t oi = ((size_t)bt * a.NQ + g * G + h) * HD + 4 * lane;
    float o0 = r0, o1 = r1, o2 = r2, o3 = r3;
    if (a.gate) {
        const uint2 gw = *reinterpret_cast<const uint2 *>(a.gate + oi);
        o0 *= sigm(qs::bf_lo(gw.x)), o1 *= sigm(qs::bf_hi(gw.x)), o2 *= sigm(qs::bf_lo(gw.y)), o3 *= sigm(qs::bf_hi(gw.y));
    }
    *reinterpret_cast<uint2 *>(a.o + oi) = make_uint2(qs::cvt_pk_bf16(o0, o1), qs::cvt_pk_bf16(o2, o3));
}

// The rows kernel's query tiles per block for R rows: the fewest that cover them in as few blocks as 4 tiles would.
int rows_tiles(int R) {
    const int nrb = (R + 63) / 64;
    return (R + 16 * nrb - 1) / (16 * nrb);
}
// Whether its LDS holds two page groups: the mixer's residues leave no room for the second with 3 tiles and more than 8
// new tokens, or with 4 tiles.
bool rows_pairs(int R, int T, bool mixer) { return !mixer || rows_tiles(R) == 2 || (rows_tiles(R) == 3 && T <= 8); }

int nsplit_of(int max_blocks, int pps) { return (max_blocks + pps - 1) / pps; }
// Pages a workgroup is best given to walk: the caller's, or as few as keep the whole launch within one workgroup per CU
// (an even number past one, for the two pages in flight). A page takes its waves ~2 us of dependent latency (load, scores,
// softmax, P V), so a grid that leaves CUs idle is cut finer; past 256 workgroups the partials cost more than the shorter
// walks save. Per layer with the mixer, the caller's pages -> the rule's: batch 1, 8 pages: 200 positions 13.0 -> 11.4 us (4
// workgroups -> 16), 1000 19.1 -> 12.3, 4096 19.7 -> 13.2; 16 pages, 2000: 26.4 -> 11.0; batch 4, 8 pages, ragged
// 1000: 19.3 -> 13.7; batch 1 / 4 tokens, 8 pages, 1000: 29.5 -> 15.2. One step finer than the rule: batch 1 / 8192
// 18.6 against 16.1, batch 4 / 4096 26.4 against 20.4, batch 8 / 2048 27.7 against 18.6. Only sizes known to the host
// enter the rule, so a user's result depends on no other user's length.
// A table of few pages stays whole (if the caller's pages allow it): without a second split there is no merge. One split
// against a page per split: one token, batch 1, 2 / 3 / 4 pages 7.8, 8.7, 9.5 against 8.8, 8.9, 8.8 us, 3 pages at batch 8
// 9.8 against 9.4, with the mixer 10.6 against 10.4; two tokens, batch 1, 2 / 3 / 4 pages 7.9, 8.9, 9.7 against 9.8, 9.9,
// 10.0, 4 pages at batch 8 10.9 against 10.5; the rows kernel, four tokens, 2 / 3 pages 9.2, 11.0 against 11.0, 11.1, eight
// 12.0, 14.9 against 13.3, 13.5; where its LDS has no room for two page groups (rows_pairs), 11 tokens with the mixer, 2
// pages 20.8 against 18.4.
constexpr int FINE_WGS = 256;
int walk_pages(int B, int T, int NKV, int G, int max_blocks, int pps, bool mixer) {
    const int R = T * G;
    const bool few = B * NKV <= 16;
    const int whole = R <= 8 ? (few && !mixer ? 3 : 2) : R <= 16 ? (few ? 4 : 3) : rows_pairs(R, T, mixer) ? 2 : 1;
    if (max_blocks <= std::min(whole, pps)) return max_blocks;
    const int nrb = (R + 63) / 64;  // row blocks of attn_rows_kernel (1 in attn_wave_kernel)
    const long most = FINE_WGS / ((long)B * NKV * nrb);  // splits per user and KV head
    if (most == 0) return pps;
    const int p = (int)((max_blocks + most - 1) / most);
    return std::min(pps, p > 1 ? (p + 1) & ~1 : 1);
}
// Whether the rows kernel walks a few pages one at a time though it could two: its workgroups then share a CU by twos, one's
// loads and merge of waves beside the other's pages, where the pair of groups is alone on it. One against two groups, us a
// layer: 4 tokens (24 rows, 2 tiles) at 2 pages a split, batch 1 / 8192 15.9 against 17.3, batch 8 / 4000 42.8, 51.6, at 4
// pages batch 8 / 4000 36.1, 39.1; 8 tokens (3 tiles) at 2 pages, batch 4 / 4000 35.7, 37.4, at 4 batch 4 / 8000 46.7, 46.5, at
// 8 38.8, 37.4; with the mixer, 4 tokens at 2 pages, batch 4 / 8000 55.7, 57.6, batch 16 / 2000 60.2, 59.0, a whole table of 2
// 14.7, 12.5, 4 pages batch 4 / 8000 43.0, 42.2, 8 tokens at 2 pages batch 8 / 4000 74.6, 73.4.
bool rows_one(int tiles, int pps, int ns, bool mixer) {
    return mixer ? tiles == 2 && pps == 2 && ns > 1 : pps <= 2 || (tiles == 2 && pps <= 4);
}
// Pages a workgroup of the independent-wave kernel walks at once (4 waves each): two when the split has more
// than one page (batch 8 at 4096 positions: 26.8 against 27.7 us; batch 1 at 32768: 29.8 against 30.4). pps is at most the
// table's width: a one-page table is walked by 4 waves whatever the caller allows (batch 1 at 60 positions, three tokens
// 9.0 -> 7.5 us, one 7.4 -> 6.5).
int attn_wpp(int pps) { return pps >= 2 ? 2 : 1; }
// Whether the splits of a call of R <= 16 query rows per KV head, wgs workgroups of 4 wpp waves, are merged inside the
// launch. Up to 4 splits, or 8 where 2 rows per wave cover the rows, always: one token (6 rows), a page per workgroup (4
// waves), in the launch against in its own, us a layer, 2 / 4 / 8 splits at batch 1 8.8, 9.0, 9.5 against 9.7, 9.7, 10.0 and
// at batch 4 9.2, 9.4, 10.5 against 10.2, 10.1, 10.3; two tokens (12 rows) at batch 1 9.8, 10.1, 10.8 against 9.9, 9.9, 10.0
// and 4 splits at batch 8 10.5 against 10.9; two pages (8 waves), 8 splits 11.2 against 11.2. 9 to 16 splits where few
// workgroups do so at a time: 4 rows, batch 1, 9 / 16 splits 9.2, 9.6 against 10.4, 10.6, batch 2 16 splits 10.5 against
// 10.7, batch 4 9 / 12 / 16 splits 10.4, 11.1, 12.1 against 10.7, 10.9, 11.1; 6 rows (two to a wave, one after the other)
// batch 1 9 / 12 / 16 splits 9.7, 10.1, 10.8 against 10.3, 10.3, 10.4. And with one row per wave, where the calls are longer:
// three or more tokens, which store their rows first (4 tokens of one head, batch 4, 9 / 16 splits 12.5, 13.6 against 13.7,
// 14.2), and more than one workgroup per CU (4 rows, batch 8, 16 splits 13.6 against 14.8).
bool merge_here(int T, int R, int wpp, int ns, long wgs) {
    if (ns <= MERGE_ANY) return true;
    if (R > 8 * wpp || ns > MERGE_MOST) return false;
    const int rows = (R + 4 * wpp - 1) / (4 * wpp);  // rows per wave of the merging workgroup
    return ns <= MERGE_MAX || wgs * rows * rows <= 192 || (rows == 1 && (T > 2 || (wpp == 1 && wgs > 256)));
}

}  // namespace

extern "C" size_t qs_paged_attention_workspace_bytes(int B, int T, int NQ, int NKV, int HDa, int max_blocks,
                                                     int pages_per_split) {
    if (B <= 0 || T <= 0 || NKV <= 0 || NQ % NKV || HDa != HD || max_blocks <= 0 || pages_per_split <= 0) return 0;
    const int G = NQ / NKV, ns = nsplit_of(max_blocks, walk_pages(B, T, NKV, G, max_blocks, pages_per_split, false));
    // at least FINE_WGS partials, which no smaller call of the same T exceeds (a smaller batch, a narrower table or the
    // mixer's call may be cut finer): a workspace sized for the largest call serves them all
    return ws_layout(std::max(B * NKV * ns, FINE_WGS), T, 1, G, 1).total;
}

extern "C" int qs_paged_attention_walk_pages(int B, int T, int NQ, int NKV, int max_blocks, int pages_per_split,
                                             int mixer) {
    if (B <= 0 || T <= 0 || NKV <= 0 || NQ <= 0 || NQ % NKV || max_blocks <= 0 || pages_per_split <= 0 ||
        pages_per_split > 64 || nsplit_of(max_blocks, pages_per_split) > MAX_SPLITS)
        return pages_per_split;  // not a call that qs_paged_gqa_decode takes: it says so
    return walk_pages(B, T, NKV, NQ / NKV, max_blocks, pages_per_split, mixer);
}

static int attn_launch(AttnArgs a, void *workspace, int HDa, int block, const char *who, void *stream) {
    const int B = a.B, T = a.T, NQ = a.NQ, NKV = a.NKV, max_blocks = a.max_blocks;
    int pages_per_split = a.pps;
    QS_REQUIRE(a.q && a.k_cache && a.v_cache && a.block_table && a.seq_lens && a.o, "%s: null pointer", who);
    QS_REQUIRE((a.k_new == nullptr) == (a.v_new == nullptr), "%s: give both k_new and v_new or neither", who);
    QS_REQUIRE(HDa == HD, "%s: HD must be %d (got %d)", who, HD, HDa);
    QS_REQUIRE(block == BLK, "%s: block must be %d (got %d)", who, BLK, block);
    QS_REQUIRE(B > 0 && T >= 1 && T <= 16, "%s: need B > 0 and 1 <= T <= 16", who);
    QS_REQUIRE(NKV > 0 && NQ > 0 && NQ % NKV == 0, "%s: NQ (%d) must be a multiple of NKV (%d)", who, NQ, NKV);
    QS_REQUIRE(max_blocks > 0 && a.num_blocks > 0, "%s: bad page counts", who);
    QS_REQUIRE(pages_per_split > 0 && pages_per_split <= 64, "%s: pages_per_split must be in [1, 64] (got %d)", who,
               pages_per_split);
    const int G = NQ / NKV;
    const int ns = nsplit_of(max_blocks, pages_per_split);
    QS_REQUIRE(ns == 1 || workspace, "%s: %d splits need a workspace", who, ns);
    QS_REQUIRE(ns <= MAX_SPLITS, "%s: %d splits exceed %d (raise pages_per_split)", who, ns, MAX_SPLITS);
    QS_REQUIRE((long)B * NKV * ns < (1L << 31), "%s: grid too large", who);
    QS_REQUIRE((size_t)B * NKV * sizeof(int) <= CNT_BYTES, "%s: B NKV = %d exceeds %d", who, B * NKV,
               (int)(CNT_BYTES / sizeof(int)));
    a.nsplit = ns;
    pages_per_split = a.pps = std::min(pages_per_split, max_blocks);
    const int wpp = attn_wpp(pages_per_split), R = T * G;
    a.merge = ns > 1 && R <= 16 && merge_here(T, R, wpp, ns, (long)B * NKV * ns);
    if (ns > 1) {  // one split leaves the workspace alone
        const WsLayout L = ws_layout(B, T, NKV, G, ns);
        char *ws = static_cast<char *>(workspace);
        a.cnt = reinterpret_cast<int *>(ws + L.cnt);
        a.part_ml = reinterpret_cast<float *>(ws + L.ml);
        a.part_o = reinterpret_cast<float *>(ws + L.po);
    }
    const dim3 grid(B * NKV * ns);
    hipStream_t st = QS_STREAM(stream);
    QS_REQUIRE(G == 1 || G == 2 || G == 4 || G == 6 || G == 8, "%s: group size NQ/NKV = %d not in {1, 2, 4, 6, 8}", who, G);
    if (R <= 16) {  // every one-token decode
#define QS_WAVE(GG)                                                              \
    if (a.wq) {                                                                  \
        if (wpp == 1) attn_wave_kernel<GG, 1, true><<<grid, 256, 0, st>>>(a);    \
        else attn_wave_kernel<GG, 2, true><<<grid, 512, 0, st>>>(a);             \
    } else {                                                                     \
        if (wpp == 1) attn_wave_kernel<GG, 1, false><<<grid, 256, 0, st>>>(a);   \
        else attn_wave_kernel<GG, 2, false><<<grid, 512, 0, st>>>(a);            \
    }
        switch (G) {
            case 1: QS_WAVE(1) break;
            case 2: QS_WAVE(2) break;
            case 4: QS_WAVE(4) break;
            case 6: QS_WAVE(6) break;
            default: QS_WAVE(8) break;
        }
#undef QS_WAVE
    } else {
        const int nrb = (R + 63) / 64, QT = rows_tiles(R);  // query rows in blocks of 16 QT
        QS_REQUIRE((long)grid.x * nrb < (1L << 31), "%s: grid too large", who);
        const dim3 rgrid(grid.x * nrb);
        const bool two = pages_per_split >= 2 && rows_pairs(R, T, a.wq) && !rows_one(QT, pages_per_split, ns, a.wq);
        // A call is given the form for up to 8 new tokens where it can be (batch 1 / 3 tokens / 60 positions 7.7 -> 7.5 us,
        // 4 tokens with the mixer 13.2 -> 12.8)
#define QS_ROWS(Q, MX, W, TN) attn_rows_kernel<Q, MX, W, TN><<<rgrid, 256 * W, 0, st>>>(a, G, nrb)
#define QS_ROWS_T(Q, MX, W) if (T <= 8) QS_ROWS(Q, MX, W, 8); else QS_ROWS(Q, MX, W, 16)
        if (a.wq) {
            if (QT == 2) { if (two) { QS_ROWS_T(2, true, 2); } else { QS_ROWS_T(2, true, 1); } }
            else if (QT == 3) { if (two) QS_ROWS(3, true, 2, 8); else { QS_ROWS_T(3, true, 1); } }
            else { QS_ROWS_T(4, true, 1); }
        } else {
            if (QT == 2) { if (two) { QS_ROWS_T(2, false, 2); } else { QS_ROWS_T(2, false, 1); } }
            else if (QT == 3) { if (two) { QS_ROWS_T(3, false, 2); } else { QS_ROWS_T(3, false, 1); } }
            else { if (two) { QS_ROWS_T(4, false, 2); } else { QS_ROWS_T(4, false, 1); } }
        }
#undef QS_ROWS_T
#undef QS_ROWS
    }
    if (int e = qs::launch_status(who)) return e;
    if (ns > 1 && !a.merge) {
        if (ns <= 64)
            attn_merge_kernel<1><<<B * T * NKV * G, 256, 0, st>>>(a, G);
        else
            attn_merge_kernel<MAX_SPLITS / 64><<<B * T * NKV * G, 256, 0, st>>>(a, G);
        return qs::launch_status(who);
    }
    return QS_OK;
}

extern "C" int qs_paged_gqa_decode(const uint16_t *q, const uint16_t *k_new, const uint16_t *v_new,
                                   uint16_t *k_cache, uint16_t *v_cache, const int *block_table, const int *seq_lens,
                                   uint16_t *o, void *workspace, int B, int T, int NQ, int NKV, int HDa, int block,
                                   int max_blocks, int num_blocks, int pages_per_split, float scale, int *status,
                                   void *stream) {
    AttnArgs a{};
    a.status = status;
    a.q = q, a.k_new = k_new, a.v_new = v_new, a.k_cache = k_cache, a.v_cache = v_cache;
    a.block_table = block_table, a.seq_lens = seq_lens, a.o = o;
    a.B = B, a.T = T, a.NQ = NQ, a.NKV = NKV, a.max_blocks = max_blocks, a.num_blocks = num_blocks;
    a.pps = pages_per_split, a.scale = scale;
    return attn_launch(a, workspace, HDa, block, "qs_paged_gqa_decode", stream);
}

extern "C" int qs_attn_mixer_decode(const uint16_t *q, const uint16_t *k_new, const uint16_t *v_new,
                                    const uint16_t *gate, const float *wq, const float *wk, const float *rope_cos,
                                    const float *rope_sin, int rot, uint16_t *k_cache, uint16_t *v_cache,
                                    const int *block_table, const int *seq_lens, uint16_t *o, void *workspace, int B,
                                    int T, int NQ, int NKV, int HDa, int block, int max_blocks, int num_blocks,
                                    int pages_per_split, float eps, int *status, void *stream) {
    QS_REQUIRE(k_new && v_new && gate && wq && wk, "qs_attn_mixer_decode: null pointer");
    QS_REQUIRE(rot == 0 || (rope_cos && rope_sin), "qs_attn_mixer_decode: rot > 0 needs rope_cos and rope_sin");
    QS_REQUIRE(rot == 0 || rot == 16 || rot == 32 || rot == 64 || rot == 128 || rot == 256,
               "qs_attn_mixer_decode: rot must be 0, 16, 32, 64, 128 or 256 (got %d)", rot);
    QS_REQUIRE(eps > 0.f, "qs_attn_mixer_decode: eps must be positive");
    QS_REQUIRE(((uintptr_t)wq | (uintptr_t)wk) % 16 == 0, "qs_attn_mixer_decode: wq and wk must be 16-byte aligned");
    AttnArgs a{};
    a.q = q, a.k_new = k_new, a.v_new = v_new, a.k_cache = k_cache, a.v_cache = v_cache;
    a.block_table = block_table, a.seq_lens = seq_lens, a.o = o;
    a.B = B, a.T = T, a.NQ = NQ, a.NKV = NKV, a.max_blocks = max_blocks, a.num_blocks = num_blocks;
    a.pps = pages_per_split, a.scale = 1.0f;  // the softmax scale is folded into wq (model.py:237)
    a.gate = gate, a.wq = wq, a.wk = wk, a.rcos = rope_cos, a.rsin = rope_sin, a.rot = rot, a.eps = eps;
    a.status = status;
    return attn_launch(a, workspace, HDa, block, "qs_attn_mixer_decode", stream);
}
