// Prefill / extend attention over the lane-grouped paged tiles (TQ_TILE_KEYS / TQ_TILE_VALUES) for
// gfx950: the Sq > 1 tiled path of kernels/attention.py:146-196 with the causal limit of an extend
// step.  The kernel for every other layout, and for a separate q_proj, is prefill_kernel.
//
// A row is one (new token, query head of the GQA group) pair, rows token-major; a segment is one
// (sequence, KV head, block of 48 rows) with the keys its rows see, walked in steps of 32 keys (two
// 16-token tiles A and B).  A wave works on its own: it looks its tiles' packed indices up in LDS
// tables straight into MFMA operands (no staging of dequantised tiles, no barriers after the tables
// are built), and one lookup feeds the MFMAs of three 16-row tiles.  MFMA layout: lane l, n = l % 16,
// g = l / 16; a 32-dim slice cc of a product covers the dims 32g + 8cc + (0..7) of lane group g, so
// the lane's chunk of a keys tile (dims 32g..32g+31 of token n) holds exactly its A operands and q
// stays in registers as the B operand:
//   S^T [16 tok x 16 rows] = K . Q^T      4 x mfma_f32_16x16x32_f16 per tile and row tile
//   T^T = signs . Q^T                      the same (QJL keys), sign byte -> 8 fp16 +-1
//   lane (n, g) holds tokens 4g + r of row n: s = norm S + rnorm c T, masked; online softmax
//   per row; fp16(p vnorm) of tokens 4g..4g+3 of both tiles is the B operand (k = 8g + i) of
//   O^T[8m + a][row] += V^T . P^T          8 x mfma_f32_16x16x32_f16 per step and row tile; field group
//                                          a of the lane's values chunk is its A operand (dim 8n + a)
// so lane (n, g) ends with dims 32g..32g+31 of row n.
//
// Work: the device's resident waves (workers, 8 per CU) share the segments' key tokens equally.  The
// segments form one stream (sequences in order, a sequence's KV heads after each other, row blocks
// ascending); a row block counts u = a + b rb tokens, the keys its last row sees rounded up to that
// form (u is linear in rb so that positions are found without a search).  Of P tokens in all, worker
// w takes positions [floor(w P / R), floor((w + 1) P / R)), and of a segment the 32-key steps that
// begin there.  A segment inside one worker is written directly; the pieces of a cut one (at most the
// first and the last of a worker, slots 2w and 2w + 1) go to the workspace and prefill_merge_kernel
// combines them.  Segments that are no more than the workers and all short are taken whole, one by a
// worker (16 sequences of 128 tokens: 55 -> 39 us).  Without a workspace, and for short block tables
// (snap), a worker takes the whole segments that begin in its range.
// Where a row block is cut follows from all lengths of the call and the number of workers, so a row's
// fp32 sums are added in an order that depends on the rest of the batch (and on whether there was a
// workspace): the same row in another batch may differ by fp32 rounding, single outputs by one step of a
// 16-bit output type.  The same call gives the same bits.
//
// Bound: VALU issue (a step: table addresses, softmax) and MFMA (busy 33 %) at two waves per SIMD (256
// registers: 96 of accumulators and 48 of q for three row tiles), and the LDS: bank conflicts of the
// lookups take about a fifth of the time of a compute unit (183 of 860 cycles per step, 3-bit keys with QJL).
// All instances spill; with QJL keys 7 to 12 values are reloaded in each step, and the wait of a reload
// behind the next step's key loads also waits for those.  Before / after against prefill_kernel, 48 query
// heads on 8 KV heads, 4 x 4096 new tokens: 3-bit keys with QJL 2627 -> 1663 us (744 TFLOP/s of products),
// 4 bits 2207 -> 1350; six sequences of 37..512 new after 1000..16000 earlier tokens (32 on 8): 986 -> 142 us.
#include "tq_common.h"
#include "tq_prefill_internal.h"

#include <cmath>

namespace {

constexpr float kNegInf = -__builtin_huge_valf();
constexpr float kWhtH = 0.08838834764831845f;  // 1 / sqrt(128)

constexpr int kRT = 3;             // 16-row MFMA tiles per wave
constexpr int kRows = 16 * kRT;    // rows of a segment
constexpr int kWaves = 8;          // waves of a workgroup (one workgroup per CU shares the tables)
// Table lookups are written kAhead slices ahead of the products that use them (0: 3-bit keys with QJL 6 %
// slower, the others equal).
constexpr int kAhead = 1;
constexpr int kMinTokens = 128;    // stream tokens a worker takes at least (32 or more: see the merge)
constexpr int kSegTokens = 96;     // a segment's set-up (query loads, output) in tokens
constexpr int kMergeTokens = 384;  // the cut pieces' set-up and their merge in tokens (192: 4 x 512 tokens
                                   // 70 -> 79 us, one of 512 unchanged)
// The exponent base lies up to this far above a row's largest score (log2), so that it moves seldom (each
// move rescales a row tile's 32 accumulators).  At 4 the largest workload gains 1 %, but fp16(p vnorm)
// loses precision: rms error against float64 1.5e-4 of the outputs' rms at 1500 tokens, 1.13e-4 at 1.
constexpr float kHeadroom = 1.0f;
constexpr float kNone = -1e30f;    // exponent base of a row that has seen no key
static_assert(kRows == kTqPrefillStreamRows && kWaves == kTqPrefillStreamWaves, "host sizing");

typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const uint8_t* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, 0x7fffffff, 0x00020000);
}
// N dwords at base + v + s
template <int N>
__device__ __forceinline__ void load_words(__amdgpu_buffer_rsrc_t r, uint32_t v, int s, uint32_t* w) {
    if constexpr (N == 2) {
        const tq_u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0);
        w[0] = x[0];
        w[1] = x[1];
    } else if constexpr (N == 3) {
        const u32x3 x = __builtin_amdgcn_raw_buffer_load_b96(r, v, s, 0);
        w[0] = x[0];
        w[1] = x[1];
        w[2] = x[2];
    } else {
        const tq_u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0);
        w[0] = x[0];
        w[1] = x[1];
        w[2] = x[2];
        w[3] = x[3];
    }
}
typedef __attribute__((address_space(3))) const uint32_t lds_u32;
typedef __attribute__((address_space(3))) const tq_u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) const tq_u32x4 lds_u32x4;

__device__ __forceinline__ float half_at(const uint32_t* w, int r) {
    const uint32_t b = (r & 1) ? (w[r >> 1] >> 16) : (w[r >> 1] & 0xffffu);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
}
// half2 of (vn.lo * p0, vn.hi * p1) for a word vn of two fp16 norms (the added zero keeps the product,
// the sum and the conversion one instruction).  No inline assembly on these operands: the compiler counts
// the wait states between MFMAs, exponentials and their readers only for its own instructions.
__device__ __forceinline__ uint32_t scale_to_half2(uint32_t vn, float p0, float p1) {
    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
    const half2_t h = {(_Float16)__builtin_fmaf(half_at(&vn, 0), p0, 0.0f), (_Float16)__builtin_fmaf(half_at(&vn, 1), p1, 0.0f)};
    return __builtin_bit_cast(uint32_t, h);
}

// ---- LDS lookup tables ----
// The lane, computed where it is written.
__device__ __forceinline__ uint32_t fresh_lane() {
    uint32_t ones;
    asm volatile("s_mov_b32 %0, -1" : "=s"(ones));
    return __builtin_amdgcn_mbcnt_hi(ones, __builtin_amdgcn_mbcnt_lo(ones, 0u));
}

template <int R>
struct Int {
    static constexpr int value = R;
};

// 3-bit fields: quads (a 12-bit field -> 4 fp16 centroids, 8 bytes), 32 KB, K at 0 and V after it
// (at 0 when K has none).  Row tables, indexed by one byte e of a word: 2-bit quads (8 bytes), 4-bit pairs (half2, 4
// bytes), signs (8 fp16 +-1, 16 bytes), entry e at region + 256 e + column, replicated over a
// 256-byte row or half of one; the address is one byte permute of the word and the lane's word (column and
// replica in byte 0, region in byte 2), and the lanes that one LDS cycle serves read different banks.
__device__ __forceinline__ uint32_t row_addr(uint32_t w, int k, uint32_t lw) {
    return __builtin_amdgcn_perm(lw, w, 0x0c060004u | ((uint32_t)k << 8));
}
template <int N>
__device__ __forceinline__ uint32_t quad3_addr(const uint32_t (&w)[N], int pos) {
    const int wi = pos >> 5, sh = pos & 31;
    uint32_t f;
    if (sh + 12 <= 32 || wi + 1 >= N)
        f = sh >= 3 ? (w[wi] >> (sh - 3)) : (w[wi] << (3 - sh));
    else
        f = __builtin_amdgcn_alignbit(w[wi + 1], w[wi], sh - 3);
    return f & 0x7ff8u;
}
// Four fp16 of field group a (4 B-bit fields from bit 4 B a) of the word array w.
template <int B, uint32_t QUAD, int N>
__device__ __forceinline__ tq_u32x2 four(const uint32_t (&w)[N], int a, uint32_t lw) {
    if constexpr (B == 3) {
        return *(lds_u32x2*)(uintptr_t)(quad3_addr(w, 12 * a) + QUAD);
    } else if constexpr (B == 2) {
        return *(lds_u32x2*)(uintptr_t)row_addr(w[a >> 2], a & 3, lw);
    } else {
        const uint32_t x = w[a >> 1];
        return tq_u32x2{*(lds_u32*)(uintptr_t)row_addr(x, 2 * (a & 1), lw),
                        *(lds_u32*)(uintptr_t)row_addr(x, 2 * (a & 1) + 1, lw)};
    }
}
__device__ __forceinline__ tq_half8 join(const tq_u32x2& a, const tq_u32x2& b) {
    return __builtin_bit_cast(tq_half8, tq_u32x4{a[0], a[1], b[0], b[1]});
}

// ---- the stream of segments ----
struct Seq {
    int q0, nq, L, nrb;
    int step;      // tokens between row blocks (causal)
    int64_t a, U;  // tokens of row block rb: a + step rb; of all row blocks
};
// (whole: every segment counts the same, so that a worker's share is one of them)
__device__ __forceinline__ Seq seq_of(const TqPrefillStream& p, int s, bool whole) {
    Seq q;
    q.q0 = p.cu_q[s];
    const int nq = p.cu_q[s + 1] - q.q0;
    q.nq = nq > 0 ? nq : 0;
    const int computed = q.nq < p.max_q ? q.nq : p.max_q;  // (positions count all new tokens)
    int L = p.seq_lens[s];
    const int cap = p.max_blocks * p.block_size;
    L = L < cap ? L : cap;
    q.L = L > 0 ? L : 0;
    q.nrb = (int)(((uint32_t)computed * (uint32_t)p.group + kRows - 1) / kRows);
    const int past = q.L > q.nq ? q.L - q.nq : 0;
    q.a = whole ? kMinTokens : (p.causal ? past + p.grow : q.L) + kSegTokens;
    q.step = whole ? 0 : p.step;
    q.U = q.nrb * q.a + (int64_t)q.step * q.nrb * (q.nrb - 1) / 2;
    return q;
}
// keys that some row of row block rb sees
__device__ __forceinline__ int visible(const TqPrefillStream& p, const Seq& q, int rb) {
    if (!p.causal) return q.L;
    int i = (int)tq_udiv_apply((uint32_t)(rb * kRows + kRows - 1), p.group_div);
    i = i < q.nq - 1 ? i : q.nq - 1;
    int v = q.L - q.nq + i + 1;
    return v > 0 ? v : 0;
}
__device__ __forceinline__ int64_t before(const Seq& q, int64_t rb) {
    return rb * q.a + (int64_t)q.step * rb * (rb - 1) / 2;
}
// Tokens of the whole stream.  whole: the segments, at kMinTokens each, if they are no more than the
// workers and the longest takes no longer than a cut one's worker and the merge.
__device__ __forceinline__ int64_t stream_total(const TqPrefillStream& p, bool& whole) {
    const int lane = threadIdx.x & 63;
    int64_t P = 0, segs = 0;
    int longest = 0;
    for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
        int64_t u = 0;
        int n = 0, L = 0;
        if (s0 + lane < p.num_seqs) {
            const Seq q = seq_of(p, s0 + lane, false);
            u = q.U * p.hkv;
            n = q.nrb < 65536 ? q.nrb : 65536;  // (more than the workers either way)
            L = q.nrb ? q.L : 0;
        }
        for (int d = 32; d >= 1; d >>= 1) {
            u += __shfl_xor(u, d, 64);
            const int ln = __shfl_xor(L, d, 64);
            L = L > ln ? L : ln;
            n += __shfl_xor(n, d, 64);
        }
        P += u;
        segs += (int64_t)n * p.hkv;
        longest = longest > L ? longest : L;
    }
    whole = segs <= p.n_workers && (int64_t)(longest - kMergeTokens) * p.n_workers <= P;
    return whole ? segs * kMinTokens : P;
}
// The workers' ranges: floor(w P / R) = w (P / R) + floor(w (P mod R) / R), R workers in use.
struct Share {
    int64_t each;
    uint32_t rest, R;
    __device__ __forceinline__ int64_t at(int64_t w) const { return w * each + (uint32_t)w * rest / R; }
};
__device__ __forceinline__ Share share_of(const TqPrefillStream& p, int64_t P) {
    const int64_t m = P / kMinTokens;
    Share h;
    h.R = m < 1 ? 1u : (uint32_t)(m < p.n_workers ? m : (int64_t)p.n_workers);
    // (P < 2^53: the quotient of the doubles is off by at most one)
    h.each = (int64_t)((double)P / (double)h.R);
    while (h.each * h.R > P) --h.each;
    while ((h.each + 1) * h.R <= P) ++h.each;
    h.rest = (uint32_t)(P - h.each * h.R);
    return h;
}
struct Place {
    int s, kh, rb;
    int64_t seg;  // stream position of the segment's start
};
// The segment that holds stream position pos (below the stream's total).
__device__ __forceinline__ Place find(const TqPrefillStream& p, int64_t pos, bool whole, Seq& q) {
    const int lane = threadIdx.x & 63;
    int64_t P = 0;
    Place at = {0, 0, 0, 0};
    for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
        const int64_t u = s0 + lane < p.num_seqs ? seq_of(p, s0 + lane, whole).U * p.hkv : 0;
        int64_t in = u;
        for (int d = 1; d < 64; d <<= 1) {
            const int64_t x = __shfl_up(in, d, 64);
            if (lane >= d) in += x;
        }
        in += P;
        const uint64_t over = __builtin_amdgcn_ballot_w64(in > pos);
        if (over) {
            const int l = __builtin_ctzll(over);
            at.s = s0 + l;
            at.seg = __shfl(in - u, l, 64);
            break;
        }
        P = __shfl(in, 63, 64);
    }
    at.s = __builtin_amdgcn_readfirstlane(at.s);
    q = seq_of(p, at.s, whole);
    int64_t off = pos - at.seg;
    // (estimates in double, put right in whole numbers)
    int kh = (int)((double)off / (double)q.U);
    kh = kh < p.hkv ? kh : p.hkv - 1;
    while (kh > 0 && kh * q.U > off) --kh;
    while (kh + 1 < p.hkv && (kh + 1) * q.U <= off) ++kh;
    off -= kh * q.U;
    const double h = (double)q.a - 0.5 * q.step;
    int rb = q.step ? (int)((__builtin_sqrt(h * h + 2.0 * q.step * (double)off) - h) / q.step) : (int)((double)off / h);
    rb = rb < 0 ? 0 : (rb < q.nrb ? rb : q.nrb - 1);
    while (rb > 0 && before(q, rb) > off) --rb;
    while (rb + 1 < q.nrb && before(q, rb + 1) <= off) ++rb;
    at.kh = __builtin_amdgcn_readfirstlane(kh);
    at.rb = __builtin_amdgcn_readfirstlane(rb);
    at.seg += at.kh * q.U + before(q, at.rb);
    return at;
}
// The steps [j0, j1) of a segment (stream position seg, u tokens, n steps) that begin in [p0, p1).
__device__ __forceinline__ void piece_of(int64_t seg, int64_t u, int n, int64_t p0, int64_t p1, int& j0, int& j1) {
    const int64_t a = p0 > seg ? p0 - seg : 0, e = p1 - seg < u ? p1 - seg : u;
    j0 = (int)((a + 31) >> 5);
    const int64_t je = (e + 31) >> 5;
    j1 = (int)(je < n ? je : n);
}

template <int KB, bool KQJL, int VB>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_stream_kernel(TqPrefillStream p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];
    constexpr uint32_t kVQuad = KB == 3 && VB == 3 ? 32768u : 0u;  // LDS address of the 3-bit V table
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int g = lane >> 4;

    // ---- this worker's part of the stream ----
    // consecutive workers share a workgroup, and consecutive workgroups an XCD (dispatched to the 8
    // XCDs in turn), so that an XCD's L2 holds few sequences' keys; with fewer workers than waves
    // the workers spread over all workgroups
    bool whole;
    const int64_t P = stream_total(p, whole);
    if (P == 0) {
        if (!p.snap && blockIdx.x == 0 && tid == 0) p.plan[0].rb = 0;  // no workers: nothing to merge
        return;
    }
    const Share share = share_of(p, P);
    const int nwg = (int)gridDim.x;
    const int wg = (nwg & 7) ? (int)blockIdx.x : (int)((blockIdx.x & 7) * (nwg >> 3) + (blockIdx.x >> 3));
    const int w0 = (int)(share.R * (uint32_t)wg / (uint32_t)nwg), w1 = (int)(share.R * (uint32_t)(wg + 1) / (uint32_t)nwg);
    if (w0 == w1) return;  // workgroup-uniform
    const int w = w0 + wave;
    const bool active = w < w1;  // (at most kWaves: R <= kWaves nwg)

    // ---- tables ----
    {
        // (lane l holds the pair of centroids l of the table being filled)
        auto fill = [&](auto bits_c, const float* c, float cs, uint32_t quad, uint32_t row) {
            constexpr int bits = decltype(bits_c)::value;
            const uint32_t mine = lane < (1 << bits) ? tq_f32_to_f16_bits(c[lane] * cs) : 0u;
            auto pair = [&](int lo, int hi) { return (uint32_t)__shfl((int)mine, lo, 64) | (uint32_t)__shfl((int)mine, hi, 64) << 16; };
            auto uniform = [](uint32_t x, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)x, l); };
            if (bits == 3) {
                const uint32_t lo = pair(lane & 7, lane >> 3);
#pragma unroll 1
                for (int h = wave; h < 64; h += kWaves)
                    *reinterpret_cast<tq_u32x2*>(s_lds + quad + 512 * h + 8 * lane) = tq_u32x2{lo, uniform(lo, h)};
            } else if (bits == 2) {
                const uint32_t lo = pair(lane & 3, (lane >> 2) & 3);
                const int at = 8 * (lane & 31);
#pragma unroll 1
                for (int e = 2 * wave; e < 256; e += 2 * kWaves) {
                    // entry e + (lane >> 5)
                    const uint32_t x = lane < 32 ? uniform(lo, e & 15) : uniform(lo, (e & 15) + 1);
                    if (at < (int)p.row_bytes)
                        *reinterpret_cast<tq_u32x2*>(s_lds + row + 256 * (e + (lane >> 5)) + at) = tq_u32x2{x, uniform(lo, e >> 4)};
                }
            } else {
                const int at = 4 * lane;
#pragma unroll 1
                for (int e = wave; e < 256; e += kWaves) {
                    const uint32_t v = uniform(mine, e & 15) | uniform(mine, e >> 4) << 16;
                    if (at < (int)p.row_bytes) *reinterpret_cast<uint32_t*>(s_lds + row + 256 * e + at) = v;
                }
            }
        };
        fill(Int<KB>{}, p.k_cent, p.k_cs, 0u, p.k_row);
        if (!p.share) fill(Int<VB>{}, p.v_cent, p.v_cs, kVQuad, p.v_row);
        if (KQJL) {
#pragma unroll 1
            for (int i = tid; i < 256 * 16; i += 64 * kWaves) {
                const int e = i >> 4, at = 16 * (i & 15);
                tq_u32x4 h;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    h[k] = (((e >> (2 * k)) & 1) ? 0x3c00u : 0xbc00u) | ((((e >> (2 * k + 1)) & 1) ? 0x3c00u : 0xbc00u) << 16);
                if (at < (int)p.row_bytes) *reinterpret_cast<tq_u32x4*>(s_lds + p.s_row + 256 * e + at) = h;
            }
        }
    }
    __syncthreads();
    if (!active) return;

    // the lane's replica: (row bytes / entry bytes) replicas of each entry
    const uint32_t klw = p.k_row + ((KB == 2 ? 8u : 4u) * lane & (p.row_bytes - 1));
    const uint32_t vlw = p.v_row + ((VB == 2 ? 8u : 4u) * lane & (p.row_bytes - 1));
    const uint32_t slw = p.s_row + (16u * lane & (p.row_bytes - 1));

    constexpr int KP = 16 * KB + (KQJL ? 16 : 0), VP = 16 * VB;  // payload bytes per token
    constexpr int KC = 4 * KB + (KQJL ? 4 : 0);                   // bytes of a keys chunk

    const int64_t p0 = share.at(w), p1 = share.at(w + 1);
    Seq q;
    Place at = find(p, p0, whole, q);
    int s = at.s, kh = at.kh, rb = at.rb;
    int64_t seg = at.seg;
    if (!p.snap) {
        // for the merge: the segment this worker's range begins inside of, if the worker before holds
        // its start and steps are left here (w0 = -1: none); worker 0 leaves the number of workers
        TqPrefillCut cut = {0, 0, 0, (int)share.R, 0, -1, 0};
        if (w > 0 && !whole) {
            const int nsteps = (visible(p, q, rb) + 31) >> 5;
            const int64_t before_this = share.at(w - 1), last = seg + 32 * (int64_t)(nsteps - 1);
            if (p0 > seg && before_this <= seg && nsteps > 0 && last >= p0) {
                int w1 = w;
                while (share.at(w1 + 1) <= last) ++w1;
                cut = {q.q0, q.nq, kh, rb, 2 * (w - 1) + (seg > before_this ? 1 : 0), w - 1, w1};
            }
        }
        if (lane == 0) p.plan[w] = cut;
    }

    while (seg < p1) {
        const int64_t u = q.a + (int64_t)q.step * rb;
        const int vis = visible(p, q, rb);
        const int nsteps = (vis + 31) >> 5;
        int j0, j1;
        bool mine;
        if (p.snap || whole) {
            mine = seg >= p0;
            j0 = 0;
            j1 = nsteps;
        } else {
            piece_of(seg, u, nsteps, p0, p1, j0, j1);
            mine = j0 < j1 || (nsteps == 0 && seg >= p0);
        }
        j0 = __builtin_amdgcn_readfirstlane(j0);
        j1 = __builtin_amdgcn_readfirstlane(j1);
        if (mine) {
            // ---- rows 48 rb + 16 rt + n: (token, query head of the group) ----
            auto row_of = [&](int rt, int& i, int& head) {
                const uint32_t row = (uint32_t)(rb * kRows + 16 * rt + n);
                i = (int)tq_udiv_apply(row, p.group_div);
                head = kh * p.group + (int)(row - (uint32_t)i * (uint32_t)p.group);
            };
            // keys that every row sees
            const int all = p.causal ? q.L - q.nq + (int)tq_udiv_apply((uint32_t)(rb * kRows), p.group_div) + 1 : q.L;

            // ---- loads ----
            const int32_t* bt_row = p.bt + (int64_t)s * p.bt_stride;
            const int last_tile = (q.L - 1) >> 4;
            // block entries of step j: lane parity = tile
            auto entries = [&](int j) -> int {
                int ti = 2 * j + (lane & 1);
                ti = ti < last_tile ? ti : last_tile;
                ti = ti > 0 ? ti : 0;
                return bt_row[tq_udiv_apply((uint32_t)ti, p.tpb_div)];
            };
            struct Where {
                uint32_t blk[2];
                int row0[2], nv[2];
            };
            auto where = [&](int j, int e) -> Where {
                Where o;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    int ti = 2 * j + h;
                    int nv = q.L - 16 * ti;
                    nv = nv < 16 ? (nv > 0 ? nv : 0) : 16;
                    ti = ti < last_tile ? ti : last_tile;
                    ti = ti > 0 ? ti : 0;
                    uint32_t blk = (uint32_t)__builtin_amdgcn_readlane(e, h);
                    if (blk >= p.num_blocks) {  // also negative entries
                        blk = 0;
                        nv = 0;
                    }
                    o.blk[h] = blk;
                    o.row0[h] = 16 * (ti - p.tpb * (int)tq_udiv_apply((uint32_t)ti, p.tpb_div));
                    o.nv[h] = nv;
                }
                return o;
            };
            const uint8_t* kb = p.kptr + (int64_t)kh * p.k_sh;
            const uint8_t* vb = p.vptr + (int64_t)kh * p.v_sh;
            // kw: the keys chunk (index words, then the sign word with QJL)
            constexpr int KW = KB + (KQJL ? 1 : 0);
            uint32_t kw[2][KW], kn[2][2], kr[2][2], vw[2][VB], vn[2][2];
            // The lane's offsets are worked out anew for each step: kept, they are spilled, and a reload waits
            // for every tile load before it (48 query heads on 8 KV heads, 4 x 4096 tokens: 4 bits 5 % faster,
            // 2 bits with QJL 9 %; but 3 bits with QJL, which has other spills, 6 % slower).
            constexpr bool kFresh = !(KB == 3 && KQJL);
            auto load_keys = [&](const Where& o) {
                const uint32_t l = kFresh ? fresh_lane() : lane, o_k = ((l & 15) * 4 + (l >> 4)) * KC, o_n = 8 * (l >> 4);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const auto r = rsrc(kb + (uint64_t)o.blk[h] * p.k_sb);
                    load_words<(KW > 4 ? 4 : KW)>(r, o_k, o.row0[h] * KP, kw[h]);
                    if (KW > 4) kw[h][KW - 1] = __builtin_amdgcn_raw_buffer_load_b32(r, o_k + 16u, o.row0[h] * KP, 0);
                    load_words<2>(r, o_n, (int)p.d_kn + 2 * o.row0[h], kn[h]);
                    if (KQJL) load_words<2>(r, o_n, (int)p.d_kr + 2 * o.row0[h], kr[h]);
                }
            };
            auto load_values = [&](const Where& o) {
                const uint32_t l = kFresh ? fresh_lane() : lane, o_v = l * (4 * VB), o_n = 8 * (l >> 4);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const auto r = rsrc(vb + (uint64_t)o.blk[h] * p.v_sb);
                    load_words<VB>(r, o_v, o.row0[h] * VP, vw[h]);
                    load_words<2>(r, o_n, (int)p.d_vn + 2 * o.row0[h], vn[h]);
                }
            };


            tq_half8 qop[kRT][4];
            // (one row tile per turn, the operands moved up, so that the code stays small)
#pragma unroll 1
            for (int rt = 0; rt < kRT; ++rt) {
                int i, head;
                row_of(rt, i, head);
                const bool rv = i < q.nq;
                float x[32];
                const int64_t off = (int64_t)(q.q0 + (rv ? i : 0)) * p.q_st + (int64_t)head * p.q_sh + 32 * g;
                if (p.q_dtype == TQ_F32) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) tq_load8(p.q, off + 8 * c, TQ_F32, &x[8 * c]);
                } else {
                    tq_u32x4 raw[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        raw[c] = *reinterpret_cast<const tq_u32x4*>(static_cast<const uint16_t*>(p.q) + off + 8 * c);
#pragma unroll
                    for (int k = 0; k < 32; ++k) {
                        const uint32_t b = (raw[k >> 3][(k >> 1) & 3] >> (16 * (k & 1))) & 0xffffu;
                        x[k] = p.q_dtype == TQ_BF16 ? tq_bf16_to_f32(b) : tq_f16_to_f32(b);
                    }
                }
                if (p.rot) tq_wht_row_g4(x, kWhtH);
#pragma unroll
                for (int cc = 0; cc < 4; ++cc) {
                    qop[0][cc] = qop[1][cc];
                    qop[1][cc] = qop[2][cc];
#pragma unroll
                    for (int j = 0; j < 8; ++j) qop[2][cc][j] = rv ? (_Float16)x[8 * cc + j] : (_Float16)0.f;
                }
            }
            // M: exponent base per row, log2 units (kNone while no key was seen); lsum: this lane's tokens
            float M[kRT], lsum[kRT];
            tq_floatx4 acc[kRT][8];
#pragma unroll
            for (int rt = 0; rt < kRT; ++rt) {
                M[rt] = kNone;
                lsum[rt] = 0.f;
#pragma unroll
                for (int a = 0; a < 8; ++a) acc[rt][a] = tq_floatx4{0.f, 0.f, 0.f, 0.f};
            }

            if (j0 < j1) {
                int e_next = entries(j0);
                Where cur = where(j0, e_next);
                load_keys(cur);
                load_values(cur);
                e_next = entries(j0 + 1);
                for (int j = j0; j < j1; ++j) {
                    // ---- scores of both tiles: tokens 4g + r of row n ----
                    // operands of slice i & 3 of tile i >> 2, looked up one slice ahead of its products
                    float sv[kRT][8];
                    tq_floatx4 sc[kRT], tj[kRT];
                    auto key_op = [&](int i, tq_half8& a, tq_half8& b) {
                        const int h = i >> 2, cc = i & 3;
                        a = join(four<KB, 0>(kw[h], 2 * cc, klw), four<KB, 0>(kw[h], 2 * cc + 1, klw));
                        if (KQJL) b = __builtin_bit_cast(tq_half8, *(lds_u32x4*)(uintptr_t)row_addr(kw[h][KW - 1], cc, slw));
                    };
                    tq_half8 ka[kAhead + 1], kb2[kAhead + 1];
#pragma unroll
                    for (int i = 0; i < kAhead; ++i) key_op(i, ka[i], kb2[i]);
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int h = i >> 2, cc = i & 3;
                        if (i + kAhead < 8) key_op(i + kAhead, ka[(i + kAhead) % (kAhead + 1)], kb2[(i + kAhead) % (kAhead + 1)]);
                        const tq_half8 a = ka[i % (kAhead + 1)], b = kb2[i % (kAhead + 1)];
                        if (cc == 0) {
#pragma unroll
                            for (int rt = 0; rt < kRT; ++rt) sc[rt] = tj[rt] = tq_floatx4{0.f, 0.f, 0.f, 0.f};
                        }
#pragma unroll
                        for (int rt = 0; rt < kRT; ++rt)
                            sc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qop[rt][cc], sc[rt], 0, 0, 0);
                        if (KQJL) {
#pragma unroll
                            for (int rt = 0; rt < kRT; ++rt)
                                tj[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, qop[rt][cc], tj[rt], 0, 0, 0);
                        }
                        if (cc == 3) {
                            // s = norm S + rnorm (c2 / c1) T, raw units: c1 s is in log2 units.  Done before
                            // the other tile's products begin: both tiles' sums at once do not fit
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const float k1 = half_at(kn[h], r);
                                const float k2 = KQJL ? half_at(kr[h], r) * p.c21 : 0.f;
#pragma unroll
                                for (int rt = 0; rt < kRT; ++rt)
                                    sv[rt][4 * h + r] = KQJL ? __builtin_fmaf(k1, sc[rt][r], k2 * tj[rt][r]) : k1 * sc[rt][r];
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                    // The lane's largest score per row tile.  Worked out here, where the scores are products
                    // fresh from the fused multiply-add: the compiler quiets the operands of a maximum that
                    // come from another basic block, one more instruction each (24 a step: 4-bit, 4 x 4096
                    // tokens 1343 -> 1380 us; here 1348).  With 2- and 4-bit keys with QJL, which spill more,
                    // the quieting is cheaper (1612 -> 1651 us; here 1686).
                    constexpr bool kEarlyMax = !KQJL || KB == 3;
                    float mx[kRT];
                    auto lane_max = [&](int rt) {
                        return fmaxf(fmaxf(fmaxf(sv[rt][0], sv[rt][1]), fmaxf(sv[rt][2], sv[rt][3])),
                                     fmaxf(fmaxf(sv[rt][4], sv[rt][5]), fmaxf(sv[rt][6], sv[rt][7])));
                    };
#pragma unroll
                    for (int rt = 0; rt < kRT; ++rt) mx[rt] = kEarlyMax ? lane_max(rt) : 0.f;
                    // the next step's keys (the current ones are used up)
                    Where nxt = cur;
                    if (j + 1 < j1) {
                        nxt = where(j + 1, e_next);
                        load_keys(nxt);
                        e_next = entries(j + 2);
                    }
                    // tokens that some row does not see, or that hold no data: masked, their value norms zeroed
                    if (32 * (j + 1) > all || cur.nv[0] + cur.nv[1] != 32) {
#pragma unroll
                        for (int rt = 0; rt < kRT; ++rt) {
                            int i, head;
                            row_of(rt, i, head);
                            const int lim = (p.causal ? q.L - q.nq + i + 1 : q.L) - 32 * j - 4 * g;
#pragma unroll
                            for (int r = 0; r < 8; ++r) {
                                const int tok = (r & 3) + 16 * (r >> 2);
                                sv[rt][r] = tok < lim && 4 * g + (r & 3) < cur.nv[r >> 2] ? sv[rt][r] : kNegInf;
                            }
                            mx[rt] = lane_max(rt);
                        }
#pragma unroll
                        for (int h = 0; h < 2; ++h)
#pragma unroll
                            for (int r = 0; r < 2; ++r) {
                                vn[h][r] &= (4 * g + 2 * r < cur.nv[h] ? 0xffffu : 0u) |
                                            (4 * g + 2 * r + 1 < cur.nv[h] ? 0xffff0000u : 0u);
                            }
                    }
                    auto value_op = [&](int a) {
                        return join(four<VB, kVQuad>(vw[0], a, vlw), four<VB, kVQuad>(vw[1], a, vlw));
                    };
                    tq_half8 va[kAhead + 1];
#pragma unroll
                    for (int a = 0; a < kAhead; ++a) va[a] = value_op(a);
                    // ---- online softmax ----
                    tq_half8 bop[kRT];
#pragma unroll
                    for (int rt = 0; rt < kRT; ++rt) {
                        float mt = kEarlyMax ? mx[rt] : lane_max(rt);
                        // M moves only when some row's score passes it, and then kHeadroom above the largest:
                        // p = exp2(c1 s - M) <= 1, and acc and lsum carry the same factor
                        if (__builtin_amdgcn_ballot_w64(__builtin_fmaf(mt, p.c1, -M[rt]) > 0.f)) {
                            mt = tq_max_over_groups(mt);
                            const float Mn = fmaxf(M[rt], __builtin_fmaf(mt, p.c1, kHeadroom));
                            const float alpha = __builtin_amdgcn_exp2f(M[rt] - Mn);
                            lsum[rt] *= alpha;
#pragma unroll
                            for (int a = 0; a < 8; ++a) acc[rt][a] *= alpha;
                            M[rt] = Mn;
                        }
                        float pr[8];
#pragma unroll
                        for (int r = 0; r < 8; ++r) pr[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[rt][r], p.c1, -M[rt]));
                        lsum[rt] += ((pr[0] + pr[1]) + (pr[2] + pr[3])) + ((pr[4] + pr[5]) + (pr[6] + pr[7]));
                        const tq_u32x4 bw = {scale_to_half2(vn[0][0], pr[0], pr[1]), scale_to_half2(vn[0][1], pr[2], pr[3]),
                                             scale_to_half2(vn[1][0], pr[4], pr[5]), scale_to_half2(vn[1][1], pr[6], pr[7])};
                        bop[rt] = __builtin_bit_cast(tq_half8, bw);
                    }
                    // ---- O^T += V^T . P^T, the operands looked up ahead in the same way ----
#pragma unroll
                    for (int a = 0; a < 8; ++a) {
                        if (a + kAhead < 8) va[(a + kAhead) % (kAhead + 1)] = value_op(a + kAhead);
#pragma unroll
                        for (int rt = 0; rt < kRT; ++rt)
                            acc[rt][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[a % (kAhead + 1)], bop[rt], acc[rt][a], 0, 0, 0);
                    }
                    if (j + 1 < j1) load_values(nxt);
                    cur = nxt;
                }
            }

            // ---- the piece's rows: acc[a][r] is dim 32g + 8r + a ----
            const bool complete = j0 == 0 && j1 == nsteps;
#pragma unroll 1
            for (int rt = 0; rt < kRT; ++rt) {
                const float l = tq_sum_over_groups(lsum[0]);
                float o[32];
#pragma unroll
                for (int a = 0; a < 8; ++a)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[8 * r + a] = acc[0][a][r];
                if (complete) {
                    const float inv = l > 0.f ? p.v_cinv / l : 0.f;
#pragma unroll
                    for (int i = 0; i < 32; ++i) o[i] *= inv;
                    if (p.rot) tq_wht_row_g4(o, kWhtH);
                    int i, head;
                    row_of(rt, i, head);
                    if (i < q.nq) {
                        const int64_t ob = (int64_t)(q.q0 + i) * p.out_st + (int64_t)head * p.out_sh + 32 * g;
                        if (p.out_dtype == TQ_F32) {
                            float4* d = reinterpret_cast<float4*>(static_cast<float*>(p.out) + ob);
#pragma unroll
                            for (int k = 0; k < 8; ++k) d[k] = make_float4(o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]);
                        } else {
                            tq_u32x4* d = reinterpret_cast<tq_u32x4*>(static_cast<uint16_t*>(p.out) + ob);
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                tq_u32x4 x;
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    x[k] = p.out_dtype == TQ_BF16
                                               ? (tq_f32_to_bf16_bits(o[8 * r + 2 * k]) | (tq_f32_to_bf16_bits(o[8 * r + 2 * k + 1]) << 16))
                                               : tq_pack_half2(o[8 * r + 2 * k], o[8 * r + 2 * k + 1]);
                                d[r] = x;
                            }
                        }
                    }
                } else {
                    const int64_t row = (int64_t)(2 * w + (seg > p0 ? 1 : 0)) * kRows + 16 * rt + n;
                    float4* d = reinterpret_cast<float4*>(p.ws_acc + row * TQ_HEAD_DIM + 32 * g);
#pragma unroll
                    for (int i = 0; i < 8; ++i) d[i] = make_float4(o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]);
                    if (g == 0) {
                        p.ws_ml[2 * row] = M[0] == kNone ? kNegInf : M[0];
                        p.ws_ml[2 * row + 1] = l;
                    }
                }
#pragma unroll
                for (int a = 0; a < 8; ++a) {
                    acc[0][a] = acc[1][a];
                    acc[1][a] = acc[2][a];
                }
                lsum[0] = lsum[1];
                lsum[1] = lsum[2];
                M[0] = M[1];
                M[1] = M[2];
            }
        }
        // next segment
        seg += u;
        if (++rb == q.nrb) {
            rb = 0;
            if (++kh == p.hkv) {
                kh = 0;
                do {
                    ++s;
                    if (s >= p.num_seqs) return;
                    q = seq_of(p, s, whole);
                } while (q.nrb == 0);
            }
        }
    }
}

// Combines the pieces of the segments that several workers share: workgroup (w - 1, y) takes the segment
// that worker w's plan names; 32 lanes per row (4 dims each), 8 rows per workgroup, 8 pieces requested
// together.  Every piece holds at least one step: a worker's range is at least kMinTokens long.
// out = sum_p 2^(m_p - M) acc_p / sum_p 2^(m_p - M) l_p (kernels/attention.py:121-140).
__global__ __launch_bounds__(256) void prefill_merge_kernel(TqPrefillStream p) {
    const int w = (int)blockIdx.x + 1;
    if (w >= p.plan[0].rb) return;
    const TqPrefillCut cut = p.plan[w];
    if (cut.w0 < 0) return;
    const int l32 = threadIdx.x & 31;
    {
        const int r0 = 8 * (int)blockIdx.y + (int)(threadIdx.x >> 5);
        const uint32_t row = (uint32_t)(cut.rb * kRows + r0);
        const int i = (int)tq_udiv_apply(row, p.group_div);
        if (i >= cut.nq) return;  // uniform over the row's 32 lanes
        float M = kNegInf, den = 0.f;
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int wb = cut.w0; wb <= cut.w1; wb += 8) {
            float mp[8], lp[8];
            float4 v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int wk = wb + k;
                mp[k] = kNegInf;
                lp[k] = 0.f;
                v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (wk <= cut.w1) {
                    const int64_t x = (int64_t)(wk == cut.w0 ? cut.slot0 : 2 * wk) * kRows + r0;
                    // (a row without a score to follow, also one whose scores are all NaN: its sums, zero or
                    // NaN, must reach the output.  Here and not where the piece is stored: without the
                    // select there the loop's registers fall otherwise, 4 x 4096 tokens 10 % slower)
                    mp[k] = fmaxf(p.ws_ml[2 * x], kNone);
                    lp[k] = p.ws_ml[2 * x + 1];
                    v[k] = *reinterpret_cast<const float4*>(p.ws_acc + x * TQ_HEAD_DIM + 4 * l32);
                }
            }
            float Mn = M;
#pragma unroll
            for (int k = 0; k < 8; ++k) Mn = fmaxf(Mn, mp[k]);
            const float f = M == kNegInf ? 0.f : __builtin_amdgcn_exp2f(M - Mn);
            den *= f;
            a.x *= f;
            a.y *= f;
            a.z *= f;
            a.w *= f;
            M = Mn;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float wk = mp[k] == kNegInf ? 0.f : __builtin_amdgcn_exp2f(mp[k] - M);
                den = __builtin_fmaf(wk, lp[k], den);
                a.x = __builtin_fmaf(wk, v[k].x, a.x);
                a.y = __builtin_fmaf(wk, v[k].y, a.y);
                a.z = __builtin_fmaf(wk, v[k].z, a.z);
                a.w = __builtin_fmaf(wk, v[k].w, a.w);
            }
        }
        const float inv = den > 0.f ? p.v_cinv / den : 0.f;
        float o[4] = {a.x * inv, a.y * inv, a.z * inv, a.w * inv};
        if (p.rot) {
            // element 4 l32 + i: bits 0-1 in registers, 2-6 over the row's lanes (half a wave)
            tq_wht_regs(o);
            for (int x = 1; x < 32; x <<= 1) {
#pragma unroll
                for (int k = 0; k < 4; ++k) o[k] = tq_wht_lane(o[k], x);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] *= kWhtH;
        }
        const int64_t ob = (int64_t)(cut.q0 + i) * p.out_st +
                           (int64_t)(cut.kh * p.group + (int)(row - (uint32_t)i * (uint32_t)p.group)) * p.out_sh + 4 * l32;
        if (p.out_dtype == TQ_F32) {
            *reinterpret_cast<float4*>(static_cast<float*>(p.out) + ob) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
            tq_u32x2 x;
#pragma unroll
            for (int k = 0; k < 2; ++k)
                x[k] = p.out_dtype == TQ_BF16 ? (tq_f32_to_bf16_bits(o[2 * k]) | (tq_f32_to_bf16_bits(o[2 * k + 1]) << 16))
                                              : tq_pack_half2(o[2 * k], o[2 * k + 1]);
            *reinterpret_cast<tq_u32x2*>(static_cast<uint16_t*>(p.out) + ob) = x;
        }
    }
}

const void* stream_kernel_ptr(int kb, bool kq, int vb) {
#define TQ_PS(KB, KQ, VB) \
    if (kb == KB && kq == KQ && vb == VB) return (const void*)prefill_stream_kernel<KB, KQ, VB>;
#define TQ_PS_V(KB, KQ) TQ_PS(KB, KQ, 2) TQ_PS(KB, KQ, 3) TQ_PS(KB, KQ, 4)
    TQ_PS_V(2, false) TQ_PS_V(2, true) TQ_PS_V(3, false) TQ_PS_V(3, true) TQ_PS_V(4, false) TQ_PS_V(4, true)
#undef TQ_PS_V
#undef TQ_PS
    return nullptr;
}

}  // namespace

int tq_prefill_stream_launch(TqPrefillStream p, int kb, bool kq, int vb, int cus, hipStream_t stream) {
    const void* kern = stream_kernel_ptr(kb, kq, vb);
    if (!kern) return TQ_ERR_BITS;
    // LDS (one workgroup per CU, up to 128 KB): 3-bit quad tables in [0, 64 KB) (K first), then 64 KB
    // regions of 256-byte rows: a region for each row table, or two tables per region, one per 128-byte
    // half row, where the regions do not suffice
    p.c21 = p.c2 / p.c1;
    p.group_div = tq_make_udiv((uint32_t)p.group);
    p.step = p.causal ? (kRows + p.group - 1) / p.group : 0;
    p.grow = (kRows - 1) / p.group + 1;
    if (kb == 3 && vb == 3) p.share = 0;  // (two tables at fixed addresses, also for one codebook)
    const uint32_t quads = (kb == 3 || vb == 3) ? 65536u : 0u;
    const int tables = (kb != 3) + (vb != 3 && !p.share) + (kq ? 1 : 0);
    p.row_bytes = quads + 65536u * tables <= 131072u ? 256u : 128u;
    int slot = 0;
    auto row_table = [&]() -> uint32_t {
        const uint32_t at = quads + (p.row_bytes == 256u ? 65536u * slot : 65536u * (slot >> 1) + 128u * (slot & 1));
        ++slot;
        return at;
    };
    if (kb != 3) p.k_row = row_table();
    if (vb != 3) p.v_row = p.share ? p.k_row : row_table();
    if (kq) p.s_row = row_table();
    const uint32_t used = quads + 65536u * (p.row_bytes == 256u ? slot : (slot + 1) / 2);
    hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)used);
    if (e != hipSuccess) return (int)e;
    void* args[] = {&p};
    e = hipLaunchKernel(kern, dim3((unsigned)cus), dim3(64 * kWaves), args, used, stream);
    if (e != hipSuccess) return (int)e;
    if (!p.snap && p.n_workers > 1) {
        e = hipLaunchKernel((const void*)prefill_merge_kernel, dim3((unsigned)p.n_workers - 1, kRows / 8), dim3(256),
                            args, 0, stream);
        if (e != hipSuccess) return (int)e;
    }
    e = hipGetLastError();
    return e == hipSuccess ? TQ_OK : (int)e;
}
