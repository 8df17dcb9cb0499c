// sjk_prefill.hip - attention of many query rows per KV head (prefill ubatches): every record and staged row is
// decoded once for 32 query rows.
//
// The 16-row kernels of sjk_attend3.hip read and decode the whole context once per 16 query rows, which is right for a
// decode step (one tile) and wrong for a ubatch (128 tiles of a 512-position ubatch at GQA 4:1). Here a tile is 32 query
// rows of a KV head and a wavefront keeps all of it: scores, P and O of 32 rows x D channels stay in its registers.
// 32x32x16 products are taken transposed (tokens or channels as rows, queries as columns), so that a query row is one
// lane pair's column throughout: maxima, sums and the rescaling of O need no exchange but one between the wavefront's
// halves, and a score tile's registers are, in their order, the k-slots of the P operand (the token order of the V
// operands follows from that).
//
// Work: a tile's context is a list of steps, 32 staged positions (sink, then tail) or one sealed record each; the tiles
// of all heads put end to end are cut into one equal share per CU by the steps' costs, and a share's part of a tile
// (a segment) into one part per wavefront. A wavefront is on its own from the query rows' staging to the segment's merge.
// A tile cut over several workgroups is put together by prefill_combine; the first segment's O waits in the output.
//
// Numerics as the 16-row kernels. Records enter as exact codes (fp16 subnormals c x 2^-24); Q' = Q x Kscale is split into
// fp16 hi + lo parts from the 32-bit query's exact product, zero points and sums are fp32, P' = P x Vscale x 2^k is rounded to
// fp16 once (against the record's own maximum, where those take the running one). Staged rows: the query enters as fp16
// hi + lo parts (times a power of two per row, so that a large row does not overflow and a small one does not lose its low
// part), a tq6_0 value as the hi + lo parts of its centroid, the K block norm multiplies the fp32 sum of its block, the V
// block norm the weight P, which is split hi + lo: three products each. Error against float64 at 7K-20K positions 0.91-1.0 of
// the 16-row kernels' on values of unit variance, 0.73-1.06 on queries, keys or zero points 2^5-2^10 off. Q' from a query
// cut to fp16 parts first took 1% less time, but was off by 8e-3 on rows whose channels are 2^20 apart and up to 1.1x
// further off than now with Kscale near 2^-9.
//
// What bounds it (D = 256): vector issue. A record is 128 + 64 products of 32 cycles, 6,100 cycles of a SIMD's matrix
// core, and about 2,300 vector instructions; 32 staged positions 96 products and 1,050 (tq6_0 rows). Two wavefronts per SIMD
// (O alone is 128 of their 256 registers) overlap the two only in part: counted over a call, a SIMD issues vector
// instructions 62% of the time and its matrix core is busy 35%. 512 positions x 16 heads at 32K, D = 256: 640-665 us by card
// against 1,315-1,330 us with the 16-row kernels (6.8K staged positions; 273 GFLOP of products at one pass, 0.41-0.43
// PFLOP/s).
#include "sjk_mfma.h"

#include <type_traits>
#include <utility>

namespace sjk {

constexpr int PF_ROWS = 32;                      // query rows of a tile: the columns of the 32x32 MFMA tiles
constexpr int PF_NW = 8, PF_NT = 64 * PF_NW;
constexpr int PF_CH = 32;                        // staged positions per step
constexpr int PF_MSTR = 68;                      // floats per query row of a merge slice (64 channels, 16-byte rows)
constexpr int PF_WAVE = PF_CH * 200;             // LDS bytes per wavefront: staged V rows and K norms

// cost of 32 staged positions and of a sealed record: 3 : 4 was the fastest (7 : 10 took 0-1% longer, 2 : 3 1-3%, 5 : 9 5-8%
// on 512-position ubatches at 16K and 32K, D = 128 and 256)
constexpr int PF_COST_CH = 3, PF_COST_REC = 4;

// Calls with fewer query rows per KV head take the 16-row kernels. Past 256 rows, where those take a third launch, this
// kernel is the faster one at every length and head count measured (100-33K positions, 1-16 KV heads, D = 128 and 256):
// 260 rows of 1 head, D = 256, 39.5 against 49.0 us at 1,500 positions, 59 against 77 at 33K; of 2 heads, D = 128, 27.2
// against 36.8 at 700. At 256 rows, two launches there, it needs 8 KV heads to win or to draw: D = 128, 27.9 against 27.5 us
// at 300 positions, 34.4 against 44.6 at 1,500, 112 against 273 at 33K (16 heads: 1.2-2.8x); with 4 heads and D = 256
// it takes 38.1 against 35.3 us at 600 positions, with 1 head 38.5 against 32.0 at 1,500. At 128 rows it takes up to twice as
// long on short contexts. The line is on rows and heads alone: a captured call does not know its context.
constexpr int PF_MIN_ROWS = 256, PF_MIN_ROWS_HEADS = 8;

struct PreArgs {
    sjk_hip_view v;
    const int32_t * desc;                        // B, N, qpos0 from the device descriptor (sjk_hip_attend_dyn), or null
    uint32_t B, N, qpos0, n_max;
    int n_q, n_head, gq;
    int rows, n_tile;                            // query rows per KV head, their 32-row tiles
    int n_wg;
    float sc2;                                   // scale * log2(e)
    const float * q;
    float * out;
    float * part;                                // [n_wg][32][D]: O of a workgroup's first segment if it starts inside a
                                                 // tile; then [2][n_wg][32] (m, l): of that segment, and of one that starts a
                                                 // tile and does not end it (its O is in out)
};

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) uint8_t * gptr;
template <typename T> SJK_DEV T gload(gptr p) { return *(const __attribute__((address_space(1))) T *) p; }
typedef uint32_t u4_a2 __attribute__((ext_vector_type(4), aligned(2)));

template <int D> struct PreLds {
    u2 pt[4096];                                 // tq6_0 pair table (fp16 hi, lo pairs)
    union {
        struct {                                 // (row strides 16 bytes off the banks' period)
            alignas(16) float qf[PF_ROWS][D + 4];          // Q, for the records
            alignas(16) uint16_t q[2][PF_ROWS][D + 8];     // Q hi / lo, for the staged rows
            alignas(16) uint8_t wv[PF_NW][PF_WAVE];        // per wavefront: record scales, staged V rows
        };
        alignas(16) float mg[PF_NW][PF_ROWS * PF_MSTR];    // merge slices: the segment's rows are done with
    };
    float wm[PF_NW][PF_ROWS], wl[PF_NW][PF_ROWS];
    float rs[PF_ROWS];                           // what takes a staged row's scores back to log2 units
    uint32_t see[PF_ROWS];                       // the visible end of a query row (0: none for a dead row)
    float cent[64];
};

SJK_DEV f16v mfma3216(const u4 & a, const u4 & b, const f16v & c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}
SJK_DEV uint32_t pk16(float a, float b) {        // v_cvt_pk_f16_f32: both rounded to nearest even
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2v{a, b}, h2v));
}
SJK_DEV u2 split_pk(float a, float b) {          // (a, b) as fp16 pairs {hi, lo}
    const uint32_t hi = pk16(a, b);
    const h2v h = __builtin_bit_cast(h2v, hi);
    return u2{hi, pk16(a - (float) h[0], b - (float) h[1])};
}
// fp32 times the low / high fp16 half of h: plus 0, so that it is one v_fma_mix (else a conversion and a product)
SJK_DEV float mix_lo(float a, uint32_t h) { return __builtin_fmaf(a, h2f(h & 0xFFFFu), 0.0f); }
SJK_DEV float mix_hi(float a, uint32_t h) { return __builtin_fmaf(a, h2f(h >> 16), 0.0f); }

// over the wavefront's halves, the same value in both (never of an MFMA's result itself, see swap32)
SJK_DEV float half_sum(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    swap32(a, b);
    return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}
SJK_DEV float half_max(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    swap32(a, b);
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
// the largest over 16 lanes (a DPP row)
SJK_DEV float row_max(float v) {
    v = fmaxf(v, dpp<0x128>(v));                 // row_ror 8, 4, 2, 1
    v = fmaxf(v, dpp<0x124>(v));
    v = fmaxf(v, dpp<0x122>(v));
    return fmaxf(v, dpp<0x121>(v));
}

// the context of a tile of query rows, whose last row is row `last`
struct PreCtx {
    uint32_t N, qpos0, sink_end, body_end, pend;
    int n_sc, n_ch, n_rec;                       // steps of staged rows (n_sc of the sink, then the tail), records
    uint32_t cost;
    bool ok;
};
SJK_DEV PreCtx pre_ctx(const PreArgs & a, int tile) {
    uint32_t B = a.B, N = a.N, q0 = a.qpos0;
    PreCtx c;
    c.ok = true;
    const uint32_t S = a.v.S;
    if (a.desc) {                                // the test of the 16-row path: NaN rows if the view cannot hold it
        const int32_t iB = a.desc[SJK_DESC_B], iN = a.desc[SJK_DESC_N], iQ = a.desc[SJK_DESC_QPOS0];
        B = (uint32_t) iB; N = (uint32_t) iN; q0 = (uint32_t) iQ;
        const uint32_t end = q0 + (uint32_t) a.n_q, pend = N < end ? N : end, bend = B < S ? S : B;
        c.ok = iB >= 0 && iN >= 0 && iQ >= 0 && B <= N && N <= a.n_max && (B <= S || (B - S) % 128u == 0u) &&
               (pend <= bend || (a.v.ring && a.v.cap >= 16u && pend - bend <= a.v.cap));
        if (!c.ok) { B = 0; N = 0; q0 = 0; }
    }
    const int last = PF_ROWS * tile + PF_ROWS < a.rows ? PF_ROWS * tile + PF_ROWS - 1 : a.rows - 1;
    const uint32_t end = q0 + (uint32_t) (last / a.gq) + 1u;
    c.N = N; c.qpos0 = q0;
    c.pend = N < end ? N : end;
    c.sink_end = c.pend < S ? c.pend : S;
    uint32_t Bb = B < S ? S : B;
    // sealed groups up to the one holding the last visible position
    const uint32_t pend_g = c.pend <= S ? S : S + (c.pend - S + 127u) / 128u * 128u;
    if (Bb > pend_g) Bb = pend_g;
    c.body_end = Bb;
    c.n_sc = (int) ((c.sink_end + PF_CH - 1u) / PF_CH);
    c.n_rec = (int) ((Bb - S) / 128u);
    const uint32_t tail = c.pend > Bb ? c.pend - Bb : 0u;
    c.n_ch = c.n_sc + (int) ((tail + PF_CH - 1u) / PF_CH);
    c.cost = (uint32_t) (c.n_ch * PF_COST_CH + c.n_rec * PF_COST_REC);
    if (c.cost == 0) c.cost = 1;
    return c;
}

// Costs of the tiles before `tile` and of all tiles of a KV head (every head has the same): computed by each wavefront,
// 64 tiles at a time. With find, `tile` is instead the tile whose cost range holds y, and before its start.
struct PrePos { uint64_t before, total; int tile; };
SJK_DEV PrePos pre_scan(const PreArgs & a, int tile, bool find, uint64_t y) {
    const int lane = threadIdx.x & 63;
    PrePos r = {0, 0, tile};
    uint64_t run = 0;
    bool done = false;
    for (int t0 = 0; t0 < a.n_tile; t0 += 64) {
        const uint32_t cost = t0 + lane < a.n_tile ? pre_ctx(a, t0 + lane).cost : 0u;
        uint64_t inc = cost;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {
            const uint32_t lo = __shfl_up((uint32_t) inc, s, 64), hi = __shfl_up((uint32_t) (inc >> 32), s, 64);
            if (lane >= s) inc += lo | ((uint64_t) hi << 32);
        }
        if (find && !done) {
            const uint64_t m = __ballot(cost != 0u && y < run + inc);
            if (m) { r.tile = t0 + __ffsll((unsigned long long) m) - 1; done = true; }
        }
        const int k = r.tile - t0;
        if ((!find || done) && k >= 0 && k < 64) {
            const uint64_t ex = inc - cost;
            r.before = run + ((uint64_t) (uint32_t) __shfl((uint32_t) ex, k, 64) | ((uint64_t) (uint32_t) __shfl((uint32_t) (ex >> 32), k, 64) << 32));
        }
        run += (uint64_t) (uint32_t) __shfl((uint32_t) inc, 63, 64) | ((uint64_t) (uint32_t) __shfl((uint32_t) (inc >> 32), 63, 64) << 32);
    }
    r.total = run;
    return r;
}

SJK_DEV uint64_t uni64(uint64_t v) {
    return (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) v) | ((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (v >> 32)) << 32);
}
#define SJK_FENCE() __builtin_amdgcn_sched_barrier(0)
// the value is made here: the compiler would move sums to where they are used next and keep their terms till then
SJK_DEV void pin(float & v) { asm volatile("" : "+v"(v)); }
// v, in a way that nothing computed from it can be moved to before this point and kept in registers from there
SJK_DEV int fresh(int v) { asm volatile("" : "+v"(v)); return v; }
SJK_DEV void pin(f16v & v) { asm volatile("" : "+v"(v)); }
SJK_DEV void pin(uint32_t & v) { asm volatile("" : "+v"(v)); }
// (a0 * s.lo, a1 * s.hi) as fp16 pairs {hi, lo}: hi = RN16(x), lo = RN16(x - hi) of the exact products x, by v_fma_mixlo /
// mixhi. Plain code, not the asm of the 16-row kernels: the compiler places the wait states
// before the MFMAs that read the pairs, and moves other instructions into them
SJK_DEV u2 mul_split(float a0, float a1, uint32_t s) {
    uint32_t h = __builtin_bit_cast(uint32_t, h2v{(_Float16) mix_lo(a0, s), (_Float16) mix_hi(a1, s)});
    pin(h);                                      // one register: its halves are read in place
    return u2{h, __builtin_bit_cast(uint32_t, h2v{(_Float16) fma_lo(a0, s, -h2f(h & 0xFFFFu)), (_Float16) fma_hi(a1, s, -h2f(h >> 16))})};
}

// bit 15 / 31: the low / high half is an infinity or a NaN
SJK_DEV uint32_t nonfinite_halves(uint32_t w) { return ((w & 0x7FFF7FFFu) + 0x04000400u) & 0x80008000u; }
// HBM -> LDS without registers: lane l's word to dst + size x l
SJK_DEV void dma4(gptr src, uint8_t * dst) {
    __builtin_amdgcn_global_load_lds((const void *) src, (__attribute__((address_space(3))) void *) dst, 4, 0, 0);
}
SJK_DEV void dma16(gptr src, uint8_t * dst) {
    __builtin_amdgcn_global_load_lds((const void *) src, (__attribute__((address_space(3))) void *) dst, 16, 0, 0);
}
SJK_DEV void vm_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int D>
__global__ __launch_bounds__(PF_NT) __attribute__((amdgpu_waves_per_eu(2))) void prefill_kernel(const PreArgs a) {
    static_assert(D == 128 || D == 256, "head dimension of the prefill kernel");
    constexpr int NB = D / 128, NT = D / 32, NC = D / 16;        // tq6_0 blocks of a row, O tiles, K steps
    using RL4 = RecLay<4, 4, D>;
    constexpr int SC_BYTES = RL4::BYTES - RL4::KSC;              // a record's scale tables
    static_assert(2 * SC_BYTES <= PF_WAVE && PF_CH * 196 + PF_CH * 2 * NB <= PF_WAVE, "a wavefront's LDS");
    __shared__ PreLds<D> L;
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const sjk_hip_view & V = a.v;
    const int H = V.n_head_kv;
    uint8_t * wv = L.wv[w];

    // this workgroup's range of the call's cost: workgroups of one head on one XCD where the counts allow it
    const int lw = (a.n_wg & 7) ? (int) blockIdx.x : ((int) blockIdx.x & 7) * (a.n_wg >> 3) + ((int) blockIdx.x >> 3);
    const uint64_t per_head = uni64(pre_scan(a, 0, false, 0).total), total = per_head * (uint64_t) H;
    const uint64_t share = uni64((total + (uint64_t) a.n_wg - 1) / (uint64_t) a.n_wg);
    uint64_t x = share * (uint64_t) lw;
    const uint64_t xe = x + share < total ? x + share : total;
    if (x >= xe) return;
    if (!pre_ctx(a, 0).ok) return;               // the combine writes NaN rows
    int head = (int) uni64(x / per_head);
    const PrePos pos = pre_scan(a, 0, true, x % per_head);
    int tile = __builtin_amdgcn_readfirstlane(pos.tile);
    uint32_t from = (uint32_t) (uni64(x) - uni64(per_head) * (uint64_t) head - uni64(pos.before));

    if (tid < 64) L.cent[tid] = tq6_cent(tid);
    __syncthreads();
    for (int e = tid; e < 4096; e += PF_NT) {
        const int c0 = (e & 15) | (((e >> 8) & 3) << 4), c1 = ((e >> 4) & 15) | (((e >> 10) & 3) << 4);
        L.pt[e] = split2(L.cent[c0], L.cent[c1]);
    }

    while (x < xe) {
        const PreCtx c = pre_ctx(a, tile);
        const uint32_t left = (uint32_t) (xe - x < (uint64_t) (c.cost - from) ? xe - x : (uint64_t) (c.cost - from));
        const uint32_t to = from + left;
        const int r0 = PF_ROWS * tile, nr = a.rows - r0 < PF_ROWS ? a.rows - r0 : PF_ROWS;
        // the query rows: as they are for the records (a negative scale negates the row, a zero one clears it, so that the
        // largest score is the largest product), and for the staged rows as fp16 hi + lo parts of the row times the power
        // of two that takes its largest value to [2^14, 2^15): channels down to 2^-28 of it keep 22 bits, as every channel
        // of the records' 32-bit rows keeps its own
        __syncthreads();
        if (tid < PF_ROWS) {
            const uint32_t e = c.qpos0 + (uint32_t) ((r0 + tid) / a.gq) + 1u;
            L.see[tid] = tid < nr ? (e < c.N ? e : c.N) : 0u;
        }
        {
            const int tid = fresh((int) threadIdx.x);
            constexpr int PT = D / 16;           // values per thread, 16 threads a row
            const int r = tid >> 4, c0 = (tid & 15) * PT;
            const int rq = r0 + (r < nr ? r : 0), iq = rq / a.gq, hq = head * a.gq + rq % a.gq;
            const float * src = a.q + ((size_t) iq * a.n_head + hq) * D + c0;
            float xv[PT], mx = 0.0f;
#pragma unroll
            for (int k = 0; k < PT; k += 4) *(float4 *) &xv[k] = *(const float4 *) (src + k);
#pragma unroll
            for (int k = 0; k < PT; ++k) {
                if (r >= nr || a.sc2 == 0.0f) xv[k] = 0.0f;
                if (a.sc2 < 0.0f) xv[k] = -xv[k];
                mx = fmaxf(mx, fabsf(xv[k]));
            }
            mx = row_max(mx);
            const int e = mx > 0.0f && mx < __builtin_inff() ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
#pragma unroll
            for (int k = 0; k < PT; k += 4) *(float4 *) &L.qf[r][c0 + k] = *(const float4 *) &xv[k];
#pragma unroll
            for (int k = 0; k < PT; k += 2) {
                const u2 hl = split_pk(__builtin_amdgcn_ldexpf(xv[k], e), __builtin_amdgcn_ldexpf(xv[k + 1], e));
                *(uint32_t *) &L.q[0][r][c0 + k] = hl.x;
                *(uint32_t *) &L.q[1][r][c0 + k] = hl.y;
            }
            if ((tid & 15) == 0) {
                // never 0, which would make a NaN of a masked score (0 x -inf): a row so small that its factor is below the
                // smallest normal number has scores below 2^-80 with that number too, and weights of exactly 1
                const float f = a.sc2 == 0.0f ? 1.0f : __builtin_amdgcn_ldexpf(fabsf(a.sc2), -e);
                L.rs[r] = f < 0x1p-126f ? 0x1p-126f : f;
            }
        }
        __syncthreads();
        uint32_t qend_min = c.qpos0 + (uint32_t) (r0 / a.gq) + 1u;   // visible to every live row
        if (qend_min > c.N) qend_min = c.N;

        // the wavefront's part: the steps whose first cost unit lies in [ca, cb)
        const uint32_t ca = from + (uint32_t) ((uint64_t) left * (uint32_t) w / PF_NW);
        const uint32_t cb = from + (uint32_t) ((uint64_t) left * (uint32_t) (w + 1) / PF_NW);
        auto ch_at = [&](uint32_t p) {
            const int k = (int) ((p + PF_COST_CH - 1) / PF_COST_CH);
            return k < c.n_ch ? k : c.n_ch;
        };
        auto rec_at = [&](uint32_t p) {
            const uint32_t s = (uint32_t) (c.n_ch * PF_COST_CH);
            const int k = p <= s ? 0 : (int) ((p - s + PF_COST_REC - 1) / PF_COST_REC);
            return k < c.n_rec ? k : c.n_rec;
        };
        const int k0 = ch_at(ca), k1 = ch_at(cb), g0 = rec_at(ca), g1 = rec_at(cb);

        f16v O[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i) O[j][i] = 0.0f;
        float m_run = -__builtin_inff(), l_run = 0.0f;
        auto rescale = [&](float alpha) {
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int i = 0; i < 16; ++i) O[j][i] *= alpha;
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) pin(O[j]);
        };

        // ---- staged rows: 32 positions a step. K operand: lane (m, h) = token m, channels 64 h .. 64 h + 63 of each
        // 128-block; scores C row r = token r. V operand: lane (m, h) = channels 128 b + 4 m + jj, tokens in the order
        // of the lane's scores. O tile 4 b + jj, C row r = channel 128 b + 4 r + jj.
        if (k0 < k1) {
            const bool st16 = V.staging == SJKVARN_STAGING_F16;
            const uint32_t vo = (uint32_t) V.stage_bytes;
            const size_t es = 2 * (size_t) vo;   // bytes per (position, head) of a staged entry
            auto range = [&](int k, uint32_t & p0, uint32_t & p1) {
                const bool sink = k < c.n_sc;
                p0 = sink ? (uint32_t) (PF_CH * k) : c.body_end + (uint32_t) (PF_CH * (k - c.n_sc));
                const uint32_t pe = sink ? c.sink_end : c.pend;
                p1 = p0 + PF_CH < pe ? p0 + PF_CH : pe;
            };
            // steps [k0, k16) are of fp16 rows, the others of tq6_0 rows
            const int e16 = st16 ? c.n_ch : V.sink_type == SJKVARN_SINK_F16 ? c.n_sc : 0;
            const int k16 = e16 < k0 ? k0 : e16 < k1 ? e16 : k1;
            auto row = [&](uint32_t p) -> gptr {
                if (p < V.S) return (gptr) V.sink + ((size_t) p * H + head) * (V.sink_type == SJKVARN_SINK_F16 ? (size_t) 4 * D : es);
                return (gptr) V.ring + ((size_t) ((p - V.S) % V.cap) * H + head) * es;
            };
            u4 kq[NB][3];                        // per block: 32 bytes of low bits, 16 of high bits
            uint16_t kn[NB];
            auto fetch = [&](int k) {
                const int lane = fresh(tid) & 63, m = lane & 31, h = lane >> 5;
                uint32_t p0, p1;
                range(k, p0, p1);
                const bool sink = k < c.n_sc;
                uint32_t sl = (uint32_t) __builtin_amdgcn_readfirstlane((int) (sink ? p0 : (p0 - V.S) % V.cap));
                if (p0 + (uint32_t) m < p1) sl += (uint32_t) m;
                if (!sink) {                     // 16 <= cap: at most two turns
                    if (sl >= V.cap) sl -= V.cap;
                    if (sl >= V.cap) sl -= V.cap;
                }
                const gptr kr = (sink ? (gptr) V.sink : (gptr) V.ring) + (size_t) head * es + (size_t) sl * ((size_t) H * es);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    kn[b] = gload<uint16_t>(kr + 98 * b);
                    kq[b][0] = gload<u4_a2>(kr + 98 * b + 2 + 32 * h);
                    kq[b][1] = gload<u4_a2>(kr + 98 * b + 18 + 32 * h);
                    kq[b][2] = gload<u4_a2>(kr + 98 * b + 66 + 16 * h);
                }
            };
            // the V rows (D = 128: K and V, 49 words either way) into the wavefront's LDS, row addresses wave-uniform
            constexpr int VS = 196, VO = NB == 2 ? 0 : 98;
            auto stage = [&](int k) {
                const int lane = fresh(tid) & 63;
                uint32_t p0, p1;
                range(k, p0, p1);
                const bool sink = k < c.n_sc;
                const size_t rowb = (size_t) H * es;
                const gptr base = (sink ? (gptr) V.sink : (gptr) V.ring) + (size_t) head * es + (NB == 2 ? vo : 0u);
                const uint32_t slot0 = (uint32_t) __builtin_amdgcn_readfirstlane((int) (sink ? p0 : (p0 - V.S) % V.cap)), nrow = p1 - p0;
                const gptr first = base + (size_t) slot0 * rowb;
                uint32_t sl = slot0;
                gptr cur = first;
                if (lane < 49) {
#pragma unroll 4
                    for (int r = 0; r < PF_CH; ++r) {
                        dma4(((uint32_t) r < nrow ? cur : first) + 4 * lane, wv + r * VS);
                        ++sl;
                        cur += rowb;
                        if (!sink && sl == V.cap) { sl = 0; cur = base; }
                    }
                }
            };
            uint16_t * nk = (uint16_t *) (wv + PF_CH * VS);        // K norms [b][32]
            auto run = [&](auto kind, int ka, int kb) {
                constexpr bool F16 = decltype(kind)::value;
                if (ka >= kb) return;
                wave_sync();
                if (!F16) { stage(ka); fetch(ka); }
                for (int k = ka; k < kb; ++k) {
                    const int lane = fresh(tid) & 63, m = lane & 31, h = lane >> 5;
                    uint32_t p0, p1;
                    range(k, p0, p1);
                    wave_sync();
                    if (!F16) {
                        if (h == 0) {
#pragma unroll
                            for (int b = 0; b < NB; ++b) nk[32 * b + m] = kn[b];
                        }
                    }
                    wave_sync();
                    const gptr kr = F16 ? row(p0 + (uint32_t) m < p1 ? p0 + (uint32_t) m : p0) : (gptr) nullptr;
                    f16v acc[NB];
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[b][i] = 0.0f;
                        // the products with a low part sum up beside: rounded at their own size, and a third of the roundings in
                        // the sum itself (error of all-staged calls against float64 4.5e-7 -> 4.2e-7; 16-row kernels 4.5e-7)
                        f16v acl = acc[b];
#pragma unroll
                        for (int kk = 0; kk < 8; ++kk) {
                            const u4 Bh = *(const u4 *) &L.q[0][m][128 * b + 64 * h + 8 * kk];
                            const u4 Bl = *(const u4 *) &L.q[1][m][128 * b + 64 * h + 8 * kk];
                            if (F16) {
                                const u4 A = gload<u4_a2>(kr + 2 * (128 * b + 64 * h + 8 * kk));
                                acc[b] = mfma3216(A, Bh, acc[b]);
                                acl = mfma3216(A, Bl, acl);
                            } else {
                                const uint32_t qs = kq[b][kk >> 2][kk & 3], qh = kq[b][2][kk >> 1];
                                // bytes [qh0, qh0, qh1, qh1] of this half-word, then byte u = its nibble u
                                const uint32_t bb = __builtin_amdgcn_perm(qh, qh, (kk & 1) ? 0x03030202u : 0x01010000u);
                                const uint32_t z = (bb & 0x000F000Fu) | ((bb >> 4) & 0x0F000F00u);
                                u4 Ah, Al;
#pragma unroll
                                for (int u = 0; u < 4; ++u) {
                                    const uint32_t idx = __builtin_amdgcn_perm(z, qs, 0x0C0C0000u | ((uint32_t) (4 + u) << 8) | (uint32_t) u);
                                    const u2 e = L.pt[idx];
                                    Ah[u] = e.x;
                                    Al[u] = e.y;
                                }
                                acc[b] = mfma3216(Ah, Bh, acc[b]);
                                acl = mfma3216(Ah, Bl, acl);
                                acl = mfma3216(Al, Bh, acl);
                            }
                            SJK_FENCE();
                        }
                        acc[b] += acl;
                    }
                    float sc[16];
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        u2 n0 = {0, 0}, n1 = {0, 0};
                        if (!F16) {
                            n0 = *(const u2 *) &nk[8 * i4 + 4 * h];
                            n1 = *(const u2 *) &nk[32 * (NB - 1) + 8 * i4 + 4 * h];
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int i = 4 * i4 + e;
                            float raw;
                            if (F16) raw = NB == 2 ? acc[0][i] + acc[NB - 1][i] : acc[0][i];
                            else {
                                raw = h2f((e & 1) ? n0[e >> 1] >> 16 : n0[e >> 1] & 0xFFFFu) * acc[0][i];
                                if (NB == 2) raw = __builtin_fmaf(h2f((e & 1) ? n1[e >> 1] >> 16 : n1[e >> 1] & 0xFFFFu), acc[NB - 1][i], raw);
                            }
                            sc[i] = raw;
                            pin(sc[i]);
                        }
                    }
                    const float rs = L.rs[m];
                    // positions that the row does not see: no score, and nothing of their values, whose infinities and NaNs
                    // would make a NaN with a weight of zero (dead: a bit per score)
                    const bool edge = p1 - p0 < PF_CH || p1 > qend_min;
                    uint32_t dead = 0;
                    if (edge) {
                        const uint32_t qend = L.see[m];
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const uint32_t p = p0 + (uint32_t) (8 * (i >> 2) + 4 * h + (i & 3));
                            if (p >= p1 || p >= qend) {
                                sc[i] = -__builtin_inff();
                                dead |= 1u << i;
                            }
                        }
                    }
                    float mx = sc[0];
#pragma unroll
                    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, sc[i]);
                    mx = half_max(mx);
                    const float m_new = fmaxf(m_run, mx * rs);
                    const bool any = m_new != -__builtin_inff();
                    const float alpha = any ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
                    const float m_sub = any ? m_new : 0.0f;
                    float ps = 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        sc[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], rs, -m_sub));
                        pin(sc[i]);
                        ps += sc[i];
                    }
                    pin(ps);
                    m_run = m_new;
                    l_run = l_run * alpha + ps;  // this lane's half of the tokens
                    rescale(alpha);
                    SJK_FENCE();
                    if (!F16) vm_done();         // the V rows are in LDS
                    SJK_FENCE();
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        // P, times the V block norm of the token, as hi + lo parts; slot t of the step = token tok(t)
                        if (!F16 && s == 1) fetch(k + 1 < kb ? k + 1 : k);
                        auto tok = [&](int t) { return 16 * s + 4 * h + (t & 3) + 8 * (t >> 2); };
#pragma unroll
                        for (int b = 0; b < NB; ++b) {
                            u4 Ph, Pl;
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                float y[2];
#pragma unroll
                                for (int e = 0; e < 2; ++e) {
                                    float nv = 1.0f;
                                    if (!F16) nv = h2f(*(const uint16_t *) (wv + tok(2 * u + e) * VS + VO + 98 * b));
                                    y[e] = sc[8 * s + 2 * u + e] * nv;
                                }
                                const u2 hl = split_pk(y[0], y[1]);
                                Ph[u] = hl.x;
                                Pl[u] = hl.y;
                            }
                            if (!F16 && edge) {
#pragma unroll
                                for (int u = 0; u < 4; ++u) {
                                    const uint32_t d = dead >> (8 * s + 2 * u);
                                    const uint32_t live = ((d & 1u) ? 0u : 0xFFFFu) | ((d & 2u) ? 0u : 0xFFFF0000u);
                                    Ph[u] &= live;
                                    Pl[u] &= live;
                                }
                            }
                            // per token the pair-table indices of channels 4 m, 4 m + 1 and 4 m + 2, 4 m + 3 (or the halves)
                            u2 ix[8];
#pragma unroll
                            for (int t = 0; t < 8; ++t) {
                                if (F16) {
                                    const uint32_t p = p0 + (uint32_t) tok(t);
                                    ix[t] = gload<u2>(row(p < p1 ? p : p0) + 2 * D + 2 * (128 * b + 4 * m));
                                } else {
                                    const uint8_t * r = wv + tok(t) * VS + VO + 98 * b;
                                    const uint32_t qs = *(const uint16_t *) (r + 2 + 2 * m), qh = r[66 + m];
                                    const uint32_t z = (qh | (qh << 4)) & 0x0F0Fu;
                                    ix[t].x = __builtin_amdgcn_perm(z, qs, 0x05010400u);
                                }
                            }
                            // fp16 values are shared by the rows of a product: in a step that not every row sees whole, those
                            // that are not finite leave it, and are added to the rows that see them (their weights go
                            // through LDS, -1 for the others)
                            if (F16 && edge) {
                                h2v nf = {(_Float16) 0.0f, (_Float16) 0.0f};
#pragma unroll
                                for (int t = 0; t < 8; ++t)
#pragma unroll
                                    for (int k2 = 0; k2 < 2; ++k2)       // 0 x value: a NaN if it is not finite
                                        nf = __builtin_elementwise_fma(__builtin_bit_cast(h2v, (uint32_t) ix[t][k2]), h2v{(_Float16) 0.0f, (_Float16) 0.0f}, nf);
                                if (__builtin_expect(__any(nonfinite_halves(__builtin_bit_cast(uint32_t, nf)) != 0u), 0)) {
                                    float * pw = (float *) wv + m;
#pragma unroll
                                    for (int t = 0; t < 8; ++t) {
                                        ix[t].x &= ~((nonfinite_halves(ix[t].x) >> 15) * 0xFFFFu);
                                        ix[t].y &= ~((nonfinite_halves(ix[t].y) >> 15) * 0xFFFFu);
                                        pw[32 * (tok(t) - 16 * s)] = (dead >> (8 * s + t) & 1u) ? -1.0f : sc[8 * s + t];
                                    }
                                    wave_sync();
#pragma unroll 1
                                    for (uint32_t t = 0; t < 16u && p0 + 16u * s + t < p1; ++t) {
                                        const float pt = pw[32 * t];
                                        const gptr vr = row(p0 + 16u * s + t) + 2 * D + 2 * (128 * b + 16 * h);
#pragma unroll
                                        for (int i = 0; i < 16; ++i) {
                                            const u2 x = gload<u2>(vr + 8 * (8 * (i >> 2) + (i & 3)));
#pragma unroll
                                            for (int jj = 0; jj < 4; ++jj) {
                                                const uint32_t v = (x[jj >> 1] >> (16 * (jj & 1))) & 0xFFFFu;
                                                if (nonfinite_halves(v) && !(pt < 0.0f)) O[4 * b + jj][i] += pt * h2f(v);
                                            }
                                        }
                                    }
#pragma unroll
                                    for (int jj = 0; jj < 4; ++jj) pin(O[4 * b + jj]);
                                    wave_sync();
                                }
                            }
                            SJK_FENCE();
#pragma unroll
                            for (int pr = 0; pr < 2; ++pr) {
                                u2 ee[8];        // the pair's values as fp16 hi, lo pairs
#pragma unroll
                                for (int t = 0; t < 8; ++t) {
                                    if (F16) ee[t] = u2{ix[t][pr], 0};
                                    else ee[t] = L.pt[pr ? ix[t].x >> 16 : ix[t].x & 0xFFFFu];
                                }
#pragma unroll
                                for (int jj = 0; jj < 2; ++jj) {
                                    const uint32_t sel = jj ? 0x07060302u : 0x05040100u;
                                    u4 Ah, Al;
#pragma unroll
                                    for (int u = 0; u < 4; ++u) {
                                        Ah[u] = __builtin_amdgcn_perm(ee[2 * u + 1].x, ee[2 * u].x, sel);
                                        Al[u] = __builtin_amdgcn_perm(ee[2 * u + 1].y, ee[2 * u].y, sel);
                                    }
                                    f16v & o = O[4 * b + 2 * pr + jj];
                                    o = mfma3216(Ah, Ph, o);
                                    o = mfma3216(Ah, Pl, o);
                                    if (!F16) o = mfma3216(Al, Ph, o);
                                    pin(o);
                                }
                                SJK_FENCE();
                            }
                        }
                    }
                    wave_sync();
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // the V rows are read
                    if (!F16 && k + 1 < kb) stage(k + 1);
                }
            };
            run(std::true_type{}, k0, k16);
            run(std::false_type{}, k16, k1);
            // O to the records' order: tile 2 p + e, C row r = channel 64 p + 16 (r / 8) + 8 e + r % 8. The two orders differ
            // by which half of the wavefront holds a channel: a register pair swaps halves. (The product with an opaque 1
            // puts a VALU result, not an MFMA's, into the swap.)
            float one = 1.0f;
            asm volatile("" : "+v"(one));
            f16v P[NT];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int jj = 0; jj < 4; ++jj) {
                            uint32_t xl = __builtin_bit_cast(uint32_t, O[4 * b + jj][4 * k4 + 2 * e] * one);
                            uint32_t yl = __builtin_bit_cast(uint32_t, O[4 * b + jj][4 * k4 + 2 * e + 1] * one);
                            swap32(xl, yl);
                            const int p = 2 * b + (k4 >> 1), i = 8 * (k4 & 1) + jj;
                            P[2 * p + e][i] = __builtin_bit_cast(float, xl);
                            P[2 * p + e][i + 4] = __builtin_bit_cast(float, yl);
                        }
#pragma unroll
            for (int j = 0; j < NT; ++j) O[j] = P[j];
        }

        // ---- sealed 4/4 records, one per step. K operand: lane (m, h) = token 16 (m / 8) + m % 8 (+ 8 in the second tile)
        // of a 64-token half, channels {4 h .. + 3, 4 h + 8 .. + 11} of a 16-channel step: two fragment words, one mask
        // per two codes. V operand: the same words with tokens and channels exchanged.
        if (g0 < g1) {
            // byte offset of this lane's two fragment words inside a row of tiles
            auto lofs = [&]() {
                const int l = fresh(tid) & 63, ml = l & 31;
                return (uint32_t) (16 * (ml & 7) + 8 * (l >> 5));
            };
            auto lblk = [&]() { return (uint32_t) ((fresh(tid) & 31) >> 3); };
            auto rec_of = [&](int g) -> gptr {
                const uint32_t blk = (uint32_t) __builtin_amdgcn_readfirstlane((int) (V.blocks ? V.blocks[g] : (uint32_t) g));
                return (gptr) V.body + ((size_t) blk * H + head) * RL4::BYTES;
            };
            constexpr int KZE = RL4::KZE - RL4::KSC, KTK = RL4::KTOK - RL4::KSC, VCH = RL4::VCH - RL4::KSC,
                          VSC = RL4::VSC - RL4::KSC, VZE = RL4::VZE - RL4::KSC;
            // a record's scale tables go to the wavefront's LDS a record ahead, its codes to registers: K words KD steps
            // ahead, V words one 64-channel part ahead
            constexpr int KD = 2;
            auto scales = [&](gptr rec, uint8_t * dst) {
                const int lane = fresh(tid) & 63;
#pragma unroll
                for (int k = 0; k < (SC_BYTES + 1023) / 1024; ++k)
                    if (64 * k + 64 <= SC_BYTES / 16 || 64 * k + lane < SC_BYTES / 16) dma16(rec + RL4::KSC + 1024 * k + 16 * lane, dst + 1024 * k);
            };
            u2 kw[KD][2], vw[8];
            auto kload = [&](gptr rec, int ck, uint32_t koff) {
#pragma unroll
                for (int u = 0; u < 2; ++u) kw[ck % KD][u] = gload<u2>(rec + (u * 4 * NC * 128 + 128 * ck) + koff);
            };
            auto vload1 = [&](gptr rec, int p, int s, uint32_t voff) { vw[s] = gload<u2>(rec + (s * NC * 128 + 512 * p) + voff); };
            gptr rec = rec_of(g0);
            wave_sync();
            scales(rec, wv);
#pragma unroll
            for (int ck = 0; ck < KD; ++ck) kload(rec, ck, lblk() * (uint32_t) (NC * 128) + lofs());
            for (int g = g0; g < g1; ++g) {
                uint32_t M0 = 0x000F000Fu, M1 = 0x00F000F0u;     // in registers: an AND with a constant takes twice as long
                pin(M0); pin(M1);
                const int lane = fresh(tid) & 63, m = lane & 31, h = lane >> 5;
                const uint32_t p0 = V.S + 128u * (uint32_t) g;
                const uint8_t * sc0 = wv + ((g - g0) & 1) * SC_BYTES;
                const gptr next = g + 1 < g1 ? rec_of(g + 1) : rec;
                vm_done();                       // this record's scale tables
                wave_sync();
                if (g + 1 < g1) scales(next, wv + ((g - g0 + 1) & 1) * SC_BYTES);
                SJK_FENCE();
                __builtin_amdgcn_s_setprio(1);
                f16v S[2][2];
                const uint32_t koff = lblk() * (uint32_t) (NC * 128) + lofs();
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int i = 0; i < 16; ++i) S[u][e][i] = 0.0f;
                float corr = 0.0f;               // sum over this lane's channels of Q x Kzero
#pragma unroll
                for (int ck = 0; ck < NC; ++ck) {
                    u4 Bh, Bl;
                    {
                        const f4 x0 = *(const f4 *) &L.qf[m][16 * ck + 4 * h], x1 = *(const f4 *) &L.qf[m][16 * ck + 8 + 4 * h];
                        const uint8_t * kp = sc0 + 2 * (2 * h * (D / 4) + 4 * ck);
                        const u2 s0 = *(const u2 *) kp, s1 = *(const u2 *) (kp + D / 2);
                        const u2 z0 = *(const u2 *) (kp + KZE), z1 = *(const u2 *) (kp + KZE + D / 2);
                        const float q[8] = {x0[0], x0[1], x1[0], x1[1], x0[2], x0[3], x1[2], x1[3]};
                        const uint32_t ks[4] = {s0.x, s0.y, s1.x, s1.y}, kz[4] = {z0.x, z0.y, z1.x, z1.y};
                        // Q' = Q x Kscale as hi + lo parts of the exact product
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const u2 hl = mul_split(q[2 * i], q[2 * i + 1], ks[i]);
                            Bh[i] = hl.x;
                            Bl[i] = hl.y;
                            corr = fma_lo(q[2 * i], kz[i], corr);
                            corr = fma_hi(q[2 * i + 1], kz[i], corr);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const u2 k2 = kw[ck % KD][u];
                        const uint32_t x0 = k2.x, x1 = k2.x >> 8, y0 = k2.y, y1 = k2.y >> 8;
                        const u4 A[2] = {u4{x0 & M0, x1 & M0, y0 & M0, y1 & M0}, u4{x0 & M1, x1 & M1, y0 & M1, y1 & M1}};
#pragma unroll
                        for (int e = 0; e < 2; ++e) S[u][e] = mfma3216(A[e], Bh, S[u][e]);
                        if (u == 1 && ck + KD < NC) kload(rec, ck + KD, koff);
#pragma unroll
                        for (int e = 0; e < 2; ++e) S[u][e] = mfma3216(A[e], Bl, S[u][e]);
                        if (u == 0) SJK_FENCE();
                    }
                    SJK_FENCE();
                }
                __builtin_amdgcn_s_setprio(0);
                const float ck = half_sum(corr);
                // scores; token of S[u][e][i]: 64 u + 16 (i / 4) + 8 e + 4 h + i % 4
                float mx = -__builtin_inff();
                const bool edge = p0 + 128u > qend_min;
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int i4 = 0; i4 < 4; ++i4) {
                            const int t0 = 64 * u + 16 * i4 + 8 * e + 4 * h;
                            const u2 kt = *(const u2 *) (sc0 + KTK + 2 * t0);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const float y = __builtin_fmaf(S[u][e][4 * i4 + i], e ? 0x1p20f : 0x1p24f, ck);
                                const float s = (i & 1) ? mix_hi(y, kt[i >> 1]) : mix_lo(y, kt[i >> 1]);
                                S[u][e][4 * i4 + i] = s;
                                mx = fmaxf(mx, s);
                            }
                            if (i4 & 1) SJK_FENCE();
                        }
                const float rs = a.sc2 == 0.0f ? 1.0f : fabsf(a.sc2);
                if (edge) {
                    const uint32_t qend = L.see[m];
                    const int n_see = (int) (qend - p0);         // of the record's tokens
                    mx = -__builtin_inff();
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int e = 0; e < 2; ++e)
#pragma unroll
                            for (int i = 0; i < 16; ++i) {
                                if (64 * u + 16 * (i >> 2) + 8 * e + 4 * h + (i & 3) >= n_see) S[u][e][i] = -__builtin_inff();
                                mx = fmaxf(mx, S[u][e][i]);
                            }
                }
                mx = half_max(mx);
                // P is taken against the record's own maximum, so that its heaviest token's weight is exactly 1 (P' is rounded
                // to fp16); O, l and the zero-point sum take it to the running one by f
                const float m_rec = mx * rs, m_new = fmaxf(m_run, m_rec);
                const bool any = m_rec != -__builtin_inff();
                const float alpha = any ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
                const float f = any ? __builtin_amdgcn_exp2f(m_rec - m_new) : -0.0f;
                const float m_sub = any ? m_rec : 0.0f;
                float pinv, ps = 0.0f, cv = 0.0f;
                const float psc = pv_scale(sc0 + VSC, lane, pinv);
                // P' = P x Vscale x 2^k as fp16; k-step st4 = 4 u + i4: slots {e = 0: 0, 1; e = 1: 0, 1; e = 0: 2, 3; e = 1: 2, 3}
                u4 Pa[8];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if (u == 1) {
                        const uint32_t voff = (uint32_t) RL4::VPAY + lblk() * 128u + lofs();
#pragma unroll
                        for (int s = 0; s < 8; ++s) vload1(rec, 0, s, voff);
                    }
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int i4 = 0; i4 < 4; ++i4) {
                            const int t0 = 64 * u + 16 * i4 + 8 * e + 4 * h;
                            u2 vs = *(const u2 *) (sc0 + VSC + 2 * t0), vz = *(const u2 *) (sc0 + VZE + 2 * t0);
                            if (edge) {          // no scale of a token that the row does not see: it may not be finite
                                const int k = (int) (L.see[m] - p0) - t0;
                                const u2 live = {(k > 0 ? 0xFFFFu : 0u) | (k > 1 ? 0xFFFF0000u : 0u), (k > 2 ? 0xFFFFu : 0u) | (k > 3 ? 0xFFFF0000u : 0u)};
                                vs &= live;
                                vz &= live;
                            }
                            float y[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(S[u][e][4 * i4 + i], rs, -m_sub));
                                ps += pr;
                                const float px = pr * psc;
                                cv = (i & 1) ? fma_hi(px, vz[i >> 1], cv) : fma_lo(px, vz[i >> 1], cv);
                                y[i] = (i & 1) ? mix_hi(px, vs[i >> 1]) : mix_lo(px, vs[i >> 1]);
                            }
                            uint32_t pa = pk16(y[0], y[1]), pb = pk16(y[2], y[3]);
                            pin(ps); pin(cv); pin(pa); pin(pb);
                            Pa[4 * u + i4][e] = pa;
                            Pa[4 * u + i4][2 + e] = pb;
                            SJK_FENCE();
                        }
                }
                m_run = m_new;
                l_run = l_run * alpha + ps * f;
                cv = half_sum(cv);
                rescale(alpha);
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int p = 0; p < NT / 2; ++p) {
                    if (p + 1 == NT / 2) {           // the last record loads its own again
#pragma unroll
                        for (int ck = 0; ck < KD; ++ck) kload(next, ck, lblk() * (uint32_t) (NC * 128) + lofs());
                    }
                    const uint32_t voff = (uint32_t) RL4::VPAY + lblk() * 128u + lofs();
                    // one tile after the other: with both, D = 256 would need more registers than there are
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        f16v t;
#pragma unroll
                        for (int i = 0; i < 16; ++i) t[i] = 0.0f;
                        const float cs = cv * (e ? 0x1p-20f : 0x1p-24f), pe = f * pinv * (e ? 0x1p20f : 0x1p24f);
#pragma unroll
                        for (int s = 0; s < 8; ++s) {
                            const u2 v2 = vw[s];
                            if (e && p + 1 < NT / 2) vload1(rec, p + 1, s, voff);
                            const uint32_t M = e ? M1 : M0;
                            t = mfma3216(u4{v2.x & M, (v2.x >> 8) & M, v2.y & M, (v2.y >> 8) & M}, Pa[s], t);
                            SJK_FENCE();
                        }
                        // channel of C row 4 h + i + 8 i4: 64 p + 16 i4 + 8 e + 4 h + i, its Vch at (4 h + i) D/8 + 8 p + 2 i4 + e;
                        // rows that see nothing of the record take nothing, whatever its channel scales are
                        if ((int) f_bits(f) >= 0) {              // not the -0 of such a row
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const u4 vc = *(const u4 *) (sc0 + VCH + 2 * ((4 * h + i) * (D / 8) + 8 * p));
#pragma unroll
                                for (int i4 = 0; i4 < 4; ++i4) {
                                    const float vcs = e ? mix_hi(pe, vc[i4]) : mix_lo(pe, vc[i4]);
                                    O[2 * p + e][4 * i4 + i] = __builtin_fmaf(t[4 * i4 + i] + cs, vcs, O[2 * p + e][4 * i4 + i]);
                                }
                            }
                        }
                        pin(O[2 * p + e]);
                        SJK_FENCE();
                    }
                }
                rec = next;
            }
        }

        // ---- the segment's merge: 64 channels at a time through the wavefronts' LDS, thread = (query row, 4 channels)
        l_run = half_sum(l_run);
        wave_sync();
        {
        const int tid = fresh((int) threadIdx.x), lane = tid & 63, m = lane & 31, h = lane >> 5;
        if (h == 0) { L.wm[w][m] = m_run; L.wl[w][m] = l_run; }
        __syncthreads();
        {
            const int r = tid >> 4, c4 = tid & 15;
            float M = L.wm[0][r], fac[PF_NW], ls = 0.0f;
#pragma unroll
            for (int k = 1; k < PF_NW; ++k) M = fmaxf(M, L.wm[k][r]);
#pragma unroll
            for (int k = 0; k < PF_NW; ++k) {
                fac[k] = M == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(L.wm[k][r] - M);
                ls = __builtin_fmaf(fac[k], L.wl[k][r], ls);
            }
            const bool whole = from == 0 && to == c.cost;
            const int rq = r0 + r, iq = rq / a.gq, hq = head * a.gq + rq % a.gq;
            float * dst = from == 0 ? a.out + ((size_t) iq * a.n_head + hq) * D
                                    : a.part + ((size_t) lw * PF_ROWS + r) * D;
            const float inv = whole ? (ls == 0.0f ? 0.0f : 1.0f / ls) : 1.0f;
#pragma unroll
            for (int p = 0; p < NT / 2; ++p) {
                float * my = L.mg[w] + m * PF_MSTR + 4 * h;
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4)
                        *(f4 *) (my + 16 * i4 + 8 * e) = f4{O[2 * p + e][4 * i4], O[2 * p + e][4 * i4 + 1], O[2 * p + e][4 * i4 + 2], O[2 * p + e][4 * i4 + 3]};
                __syncthreads();
                f4 y = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < PF_NW; ++k) {
                    const f4 z = *(const f4 *) (L.mg[k] + r * PF_MSTR + 4 * c4);
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] = __builtin_fmaf(fac[k], z[i], y[i]);
                }
                if (r < nr) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) dst[64 * p + 4 * c4 + i] = y[i] * inv;
                }
                __syncthreads();
            }
            if (c4 == 0 && !whole) {
                float * ml = a.part + (size_t) a.n_wg * PF_ROWS * D + (((size_t) (from == 0 ? a.n_wg : 0) + lw) * PF_ROWS + r) * 2;
                ml[0] = M;
                ml[1] = ls;
            }
        }
        }
        x += left;
        from = 0;
        if (++tile == a.n_tile) { tile = 0; ++head; }
    }
}

// The tiles that several workgroups took: grid (tiles, KV heads, D / 64), thread = (query row, 4 channels); eight
// segments' loads at a time go out together (one after the other they were most of the call's fixed cost, 12 us at 9
// segments a tile)
template <int D> __global__ __launch_bounds__(PF_NT) void prefill_combine(const PreArgs a) {
    constexpr int NS = 8;
    const int tid = threadIdx.x, r = tid >> 4, ch = 64 * (int) blockIdx.z + 4 * (tid & 15);
    const int tile = (int) blockIdx.x, head = (int) blockIdx.y, H = a.v.n_head_kv;
    const int rq = PF_ROWS * tile + r, iq = rq / a.gq, hq = head * a.gq + rq % a.gq;
    const PreCtx c = pre_ctx(a, tile);
    float * o = a.out + ((size_t) iq * a.n_head + hq) * D + ch;
    if (!c.ok) {
        if (rq < a.rows)
            for (int i = 0; i < 4; ++i) o[i] = __builtin_nanf("");
        return;
    }
    const PrePos pos = pre_scan(a, tile, false, 0);
    const uint64_t total = pos.total * (uint64_t) H, share = (total + (uint64_t) a.n_wg - 1) / (uint64_t) a.n_wg;
    const uint64_t x0 = pos.total * (uint64_t) head + pos.before;
    const int w0 = (int) (x0 / share), w1 = (int) ((x0 + c.cost - 1) / share);
    if (w0 == w1 || rq >= a.rows) return;
    const float * mls = a.part + (size_t) a.n_wg * PF_ROWS * D + 2 * r;
    const float * ml0 = mls + ((size_t) a.n_wg + w0) * PF_ROWS * 2;
    float M = ml0[0], ls = ml0[1];
    f4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = o[i];
    for (int k0 = w0 + 1; k0 <= w1; k0 += NS) {
        float mk[NS], lk[NS], Mn = M;
        f4 z[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int kk = k0 + k <= w1 ? k0 + k : w1;
            mk[k] = mls[(size_t) kk * PF_ROWS * 2];
            lk[k] = mls[(size_t) kk * PF_ROWS * 2 + 1];
            z[k] = *(const f4 *) (a.part + ((size_t) kk * PF_ROWS + r) * D + ch);
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (k0 + k > w1) mk[k] = -__builtin_inff();
            Mn = fmaxf(Mn, mk[k]);
        }
        if (Mn == -__builtin_inff()) continue;   // nothing visible so far
        const float f0 = __builtin_amdgcn_exp2f(M - Mn);
        M = Mn;
        ls *= f0;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] *= f0;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (k0 + k > w1) continue;
            const float f = __builtin_amdgcn_exp2f(mk[k] - M);
            ls = __builtin_fmaf(f, lk[k], ls);
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = __builtin_fmaf(f, z[k][i], y[i]);
        }
    }
    const float inv = ls == 0.0f ? 0.0f : 1.0f / ls;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = y[i] * inv;
}

// The kernel takes 4/4 bodies whose workspace holds one partial per CU and whose rows are not written where another
// workgroup still reads queries (a call with out over q takes the 16-row kernels, which write after all reads). Staged
// tq6_0 rows are copied to LDS by words, so that a hand-built view with them at odd halves keeps the 16-row kernels too.
bool sjk_prefill_takes(const sjk_hip_view & v, int body, int n_q, int n_head, const float * d_q, const float * d_out) {
    const size_t row = (size_t) n_q * (size_t) n_head * (size_t) v.lay.D, W = (size_t) n_cus(), sf = ws_slot_floats(v.lay.D);
    const int rows = n_q * (n_head / v.n_head_kv);
    if (rows < PF_MIN_ROWS || (rows == PF_MIN_ROWS && v.n_head_kv < PF_MIN_ROWS_HEADS)) return false;
    if (body != 44 || v.work_bytes < WS_PLAN_BYTES + ws_stage_bytes(v.lay.D, v.n_head_kv)) return false;
    if (d_q < d_out + row && d_out < d_q + row) return false;
    if (v.staging != SJKVARN_STAGING_F16 && (((uintptr_t) v.sink | (uintptr_t) v.ring) & 3u)) return false;
    return W * PF_ROWS * (size_t) v.lay.D + W * PF_ROWS * 4 <= ws_part_slots(v) * sf;
}

template <int D> static int launch_d(const PreArgs & a, hipStream_t st) {
    hipLaunchKernelGGL(prefill_kernel<D>, dim3((unsigned) a.n_wg), dim3(PF_NT), 0, st, a);
    hipLaunchKernelGGL(prefill_combine<D>, dim3((unsigned) a.n_tile, (unsigned) a.v.n_head_kv, (unsigned) (D / 64)), dim3(PF_NT), 0, st, a);
    return SJK_CHECK_LAUNCH();
}

int sjk_prefill(const sjk_hip_view & v, const int32_t * desc, uint32_t n_max, uint32_t B, uint32_t N, uint32_t qpos0,
                int n_q, int n_head, const float * d_q, float scale, float * d_out, hipStream_t st) {
    PreArgs a = {};
    a.v = v; a.desc = desc; a.n_max = n_max; a.B = B; a.N = N; a.qpos0 = qpos0;
    a.n_q = n_q; a.n_head = n_head; a.gq = n_head / v.n_head_kv;
    a.rows = n_q * a.gq;
    a.n_tile = (a.rows + PF_ROWS - 1) / PF_ROWS;
    a.n_wg = n_cus();
    a.sc2 = scale * 1.4426950408889634f;
    a.q = d_q; a.out = d_out; a.part = ws_part(v);   // 256-byte aligned
    return v.lay.D == 128 ? launch_d<128>(a, st) : launch_d<256>(a, st);
}

}  // namespace sjk
