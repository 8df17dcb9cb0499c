// sjk_rows.hip - row kernels: Hadamard rotation, tq6_0 / fp16 staging (the append path), unstaging,
// and record decode.
//
// Row kernels run one wavefront per row of D = 64*V values; lane l holds values V*l .. V*l+V-1.
//   * Hadamard (sj_kvarn.h:735-752): stages h < V inside a lane, stages h >= V between lanes l and
//     l ^ (h/V); the lower partner keeps a+b, the upper a-b (a = lower value), then one multiply by
//     1/sqrt(D). Same stage order and operations as the reference, so bit-identical.
//   * tq6_0 (sj_kvarn.h:1221-1247): the two per-block sums (x^2, then centroid^2) must be sequential
//     fp32 sums over the 128 values in index order. The squares are formed in parallel, written to
//     LDS and walked in order: in a small call by every lane of the block with broadcast reads, in a
//     large one by one lane per block, the workgroup's blocks side by side in one wavefront. The level
//     search, packing and stores are parallel over lanes.
#include "sjk_dev.h"

namespace sjk {

// Wavefronts (rows) per workgroup. A walk takes 32 16-byte LDS reads whatever the number of lanes that use it, so
// with a walk per row (ROW_WAVES) a large tq6_0 call is bound by them; with the walks of a workgroup's rows in one
// wavefront's lanes (ROW_WAVES_BIG) the others wait at a barrier, which costs a small call its latency. Appends at
// D = 128 / 256, walk per row against one wavefront's: 2,048 rows 4.5 / 4.9 against 5.6 / 6.4 us, 4,096 rows 5.8 / 6.4
// against 5.8 / 6.5, 8,192 rows 8.2 / 9.5 against 7.4 / 8.7, 16,384 rows 13.5 / 15.9 against 12.4 / 15.1: the line is
// at a large workgroup per CU (past it a second, partly filled round of them costs 6,144 rows 2-6%: 7.1 / 8.0 against
// 7.2 / 8.5). Rows that are no tq6_0 leave before the walks; among them the small workgroups are the faster at every size
// (8,192 fp16 rows 4.1 / 5.0 against 4.9 / 6.0 us, with the walks 9.0 / 11.0).
constexpr int ROW_WAVES = 4, ROW_WAVES_BIG = 16;
enum { OUT_F32 = 0, OUT_F16 = 1, OUT_TQ6 = 2 };

struct RowJob {
    int kind;            // 0: plain rows (stage/rotate), 1: layer store
    int D;
    int n_rows;
    int rotate;
    float rot_scale;     // RN(1/sqrt(D)), computed on the host (IEEE, same as sqrtf then /)
    // kind 0
    const float * x;
    uint8_t * dst;
    size_t dst_row_bytes;
    int out_mode;
    // kind 1 (sj_kvarn_layer_store, sj_kvarn.h:1475-1492)
    const float * k;
    const float * v;
    uint8_t * sink;
    uint8_t * ring;
    uint32_t pos0, S, cap;
    int H, sink_type, staging;
    size_t stage_bytes;
    const int32_t * pos_desc;   // sjk_hip_layer_store_dyn: pos0 = pos_desc[SJK_DESC_QPOS0], read when the kernel runs
};

SJK_DEV void job_row(const RowJob & j, int r, const float *& src, uint8_t *& dst, int & mode) {
    if (j.kind == 0) {
        src = j.x + (size_t) r * j.D;
        dst = j.dst + (size_t) r * j.dst_row_bytes;
        mode = j.out_mode;
        return;
    }
    const int side = r & 1, hh = (r >> 1) % j.H, ip = (r >> 1) / j.H;
    const uint32_t pos = (j.pos_desc ? (uint32_t) j.pos_desc[SJK_DESC_QPOS0] : j.pos0) + (uint32_t) ip;
    src = (side ? j.v : j.k) + ((size_t) ip * j.H + hh) * j.D;
    if (pos < j.S && j.sink_type == SJKVARN_SINK_F16) {
        dst = j.sink + ((size_t) pos * j.H + hh) * 4 * j.D + (size_t) side * 2 * j.D;
        mode = OUT_F16;
        return;
    }
    uint8_t * e = pos < j.S ? j.sink + ((size_t) pos * j.H + hh) * 2 * j.stage_bytes
                            : j.ring + ((size_t) ((pos - j.S) % j.cap) * j.H + hh) * 2 * j.stage_bytes;
    dst = e + (size_t) side * j.stage_bytes;
    mode = j.staging == SJKVARN_STAGING_F16 ? OUT_F16 : OUT_TQ6;
}

// up to ROW_MAXJ jobs per launch: rows [row_base[k], row_base[k+1]) of the grid belong to job k
constexpr int ROW_MAXJ = 16;
struct RowBatch {
    RowJob job[ROW_MAXJ];
    int row_base[ROW_MAXJ + 1];
    int n_jobs;
};

static_assert(sizeof(RowBatch) <= 4096, "the job table travels in the kernel arguments");

// Hadamard of one row held V values per lane (sj_kvarn.h:735-752): stages h < V inside the lane, stages h >= V
// between lanes l and l ^ (h / V) (the lower partner keeps a + b, the upper a - b, a = the lower value), then one
// multiply by 1/sqrt(D). XN: the host's NaN rule (a row holding an infinity or a NaN).
template <int V, bool XN>
SJK_DEV void hadamard_row(float (&x)[V], int lane, float scale) {
#pragma unroll
    for (int h = 1; h < V; h *= 2)
#pragma unroll
        for (int m = 0; m < V; ++m)
            if (!(m & h)) {
                const float a = x[m], b = x[m + h];
                x[m] = XN ? xadd(a, b) : a + b;
                x[m + h] = XN ? xsub(a, b) : a - b;
            }
    if (XN) {
#pragma unroll
        for (int lm = 1; lm < 64; lm *= 2) {
            const bool upper = (lane & lm) != 0;
#pragma unroll
            for (int m = 0; m < V; ++m) {
                const float o = __shfl_xor(x[m], lm, 64);
                x[m] = upper ? xsub(o, x[m]) : xadd(x[m], o);
            }
        }
    } else {
        // the partners' values by DPP inside a 16-lane row, then by row swaps: none of a lane shuffle's LDS round trips
        // (six one after the other; appends of 8 rows at D = 256 4.5 -> 4.3 us, of 8,192 9.2 -> 8.7, fp16 rows 2.85 -> 2.63
        // and 5.1 -> 4.95)
        auto stage = [&](int lm, auto && partner) {
            const bool upper = (lane & lm) != 0;
#pragma unroll
            for (int m = 0; m < V; ++m) {
                const float o = partner(x[m]);
                x[m] = upper ? o - x[m] : x[m] + o;
            }
        };
        stage(1, [](float v) { return dpp<0xB1>(v); });                 // quad_perm 1 0 3 2
        stage(2, [](float v) { return dpp<0x4E>(v); });                 // quad_perm 2 3 0 1
        stage(4, [](float v) { return dpp<0x1B>(dpp<0x141>(v)); });     // 7 - l (row_half_mirror), then quad_perm 3 2 1 0
        stage(8, [](float v) { return dpp<0x128>(v); });                // row_ror 8
#pragma unroll
        for (int lm = 16; lm < 64; lm *= 2) {
            const bool upper = (lane & lm) != 0;
#pragma unroll
            for (int m = 0; m < V; ++m) {
                uint32_t lo = f_bits(x[m]), hi = lo;                    // the lower and the upper partner's value
                if (lm == 16) swap16(lo, hi);
                else swap32(lo, hi);
                const float p = __builtin_bit_cast(float, lo), q = __builtin_bit_cast(float, hi);
                x[m] = upper ? p - q : p + q;
            }
        }
    }
#pragma unroll
    for (int m = 0; m < V; ++m) x[m] = XN ? xmul(x[m], scale) : x[m] * scale;
}

// the sum of 128 values in index order; XN: the host's NaN rule
template <bool XN> SJK_DEV float walk(const float * sq) {
    const float4 * p = (const float4 *) sq;
    float s = 0.0f;
    if (XN) {
        for (int i = 0; i < 32; ++i) {
            const float4 q = p[i];
            s = xadd(s, q.x); s = xadd(s, q.y); s = xadd(s, q.z); s = xadd(s, q.w);
        }
    } else {
#pragma unroll 8
        for (int i = 0; i < 32; ++i) {
            const float4 q = p[i];
            s = s + q.x; s = s + q.y; s = s + q.z; s = s + q.w;
        }
    }
    return s;
}

template <int V, int NW>
__global__ __launch_bounds__(64 * NW) void rows_kernel(const RowBatch bt) {
    constexpr bool BIG = NW > ROW_WAVES;   // one wavefront walks the blocks of all rows
    constexpr int NB = V / 2;              // 128-value blocks of a row
    constexpr int BS = 132;                // floats from block to block: the walking lanes' reads are in different banks
    static_assert(NW * NB <= 64, "a lane per block");
    __shared__ alignas(16) float s_sq[NW * NB * BS];
    __shared__ float s_mid[64], s_cent[64], s_sum[BIG ? NW * NB : 1];
    __shared__ bool s_xn[BIG ? NW : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x < 64) {
        s_mid[threadIdx.x] = threadIdx.x < 63 ? tq6_mid(threadIdx.x) : __builtin_inff();
        s_cent[threadIdx.x] = tq6_cent(threadIdx.x);
    }
    const int rg = blockIdx.x * NW + wave;                    // wave-uniform
    int ji = 0;
    for (int k = 1; k < bt.n_jobs; ++k) ji += rg >= bt.row_base[k] ? 1 : 0;
    ji = __builtin_amdgcn_readfirstlane(ji);
    const RowJob & j = bt.job[ji];
    const int r = rg - bt.row_base[ji];
    const bool live = rg < bt.row_base[bt.n_jobs] && !(j.pos_desc && j.pos_desc[SJK_DESC_QPOS0] < 0);
    const float * src = nullptr;
    uint8_t * dst = nullptr;
    int mode = OUT_F32;
    float x[V];
#pragma unroll
    for (int m = 0; m < V; ++m) x[m] = 0.0f;
    if (live) {
        job_row(j, r, src, dst, mode);
#pragma unroll
        for (int m = 0; m < V; ++m) x[m] = src[V * lane + m];
    }
    // a row holding an infinity or a NaN takes the rotation and the tq6_0 sums with the host's NaN rule (wave-uniform)
    bool nf = false;
#pragma unroll
    for (int m = 0; m < V; ++m) nf |= (f_bits(x[m]) & 0x7F800000u) == 0x7F800000u;
    const bool xn = __any(nf);
    if (live && j.rotate) {
        if (xn) hadamard_row<V, true>(x, lane, j.rot_scale);
        else hadamard_row<V, false>(x, lane, j.rot_scale);
    }
    const bool tq = live && mode == OUT_TQ6;
    bool any_tq = tq;
    if (BIG) any_tq = __syncthreads_or(tq) != 0;
    else __syncthreads();
    if (live && mode == OUT_F32) {
        float * o = (float *) dst;
#pragma unroll
        for (int m = 0; m < V; ++m) o[V * lane + m] = x[m];
    }
    if (live && mode == OUT_F16) {
        uint16_t * o = (uint16_t *) dst;
#pragma unroll
        for (int m = 0; m < V; ++m) o[V * lane + m] = f32_to_f16(x[m]);
    }
    if (!any_tq) return;                   // a small call's row, or a workgroup without a tq6_0 row
    // tq6_0: every wave of a large call's workgroup takes part in the barriers; only tq6 rows use the results
    constexpr int LPB = 128 / V;           // lanes per 128-value block
    const int b = lane / LPB;              // block of this lane
    float * blk_sq = s_sq + (wave * NB + b) * BS, * sq = blk_sq + V * (lane % LPB);
    auto sync = [] {
        if (BIG) __syncthreads();
        else wave_sync();
    };
    if (BIG && lane == 0) s_xn[wave] = xn;
#pragma unroll
    for (int m = 0; m < V; ++m) sq[m] = xn ? xmul(x[m], x[m]) : x[m] * x[m];
    sync();
    float nsq;
    if (BIG) {
        if (threadIdx.x < NW * NB) {
            const float * p = s_sq + (int) threadIdx.x * BS;
            s_sum[threadIdx.x] = s_xn[threadIdx.x / NB] ? walk<true>(p) : walk<false>(p);
        }
        __syncthreads();
        nsq = s_sum[wave * NB + b];
    } else {
        nsq = xn ? walk<true>(blk_sq) : walk<false>(blk_sq);
    }
    const float norm = nsq != nsq ? nan_of(nsq) : __builtin_sqrtf(nsq);
    const bool big = norm > 1e-10f;
    const float inv = big ? 1.0f / norm : 0.0f;
    int code[V];
#pragma unroll
    for (int m = 0; m < V; ++m) code[m] = tq6_level(big ? x[m] * inv : 0.0f, s_mid);
    if (!BIG) wave_sync();                 // (the barrier after the large call's walk)
#pragma unroll
    for (int m = 0; m < V; ++m) { const float c = s_cent[code[m]]; sq[m] = c * c; }
    sync();
    float rsq;
    if (BIG) {
        if (threadIdx.x < NW * NB) {
            const float s = walk<false>(s_sq + (int) threadIdx.x * BS);
            s_sum[threadIdx.x] = s;        // nsq was read before the last barrier
        }
        __syncthreads();
        rsq = s_sum[wave * NB + b];
    } else {
        rsq = walk<false>(blk_sq);
    }
    const float rn = __builtin_sqrtf(rsq);
    if (!tq) return;
    uint8_t * blk = dst + (size_t) b * SJKVARN_TQ6_BLOCK_BYTES;
    const int i0 = V * (lane % LPB);       // index of this lane's first value inside its block
    if (lane % LPB == 0) *(uint16_t *) blk = f32_to_f16(rn > 1e-10f ? xdiv(norm, rn) : norm);
    // low nibbles: qs[i/2] bit 4*(i%2); high pairs: qh[i/4] bit 2*(i%4)
    uint32_t qs = 0, qh = 0;
#pragma unroll
    for (int m = 0; m < V; ++m) {
        qs |= (uint32_t) (code[m] & 15) << (4 * m);
        qh |= (uint32_t) ((code[m] >> 4) & 3) << (2 * m);
    }
    if (V == 2) {
        // two lanes share one qh byte
        const uint32_t other = (uint32_t) __shfl_xor((int) qh, 1, 64);
        blk[2 + i0 / 2] = (uint8_t) qs;
        if (!(lane & 1)) blk[66 + i0 / 4] = (uint8_t) (qh | (other << 4));
    } else if (V == 4) {
        *(uint16_t *) (blk + 2 + i0 / 2) = (uint16_t) qs;
        blk[66 + i0 / 4] = (uint8_t) qh;
    } else {
        *(uint16_t *) (blk + 2 + i0 / 2) = (uint16_t) qs;
        *(uint16_t *) (blk + 2 + i0 / 2 + 2) = (uint16_t) (qs >> 16);
        *(uint16_t *) (blk + 66 + i0 / 4) = (uint16_t) qh;
    }
}

static int launch_batch(RowBatch & bt, hipStream_t st) {
    bt.row_base[0] = 0;
    for (int k = 0; k < bt.n_jobs; ++k) bt.row_base[k + 1] = bt.row_base[k] + (bt.job[k].n_rows > 0 ? bt.job[k].n_rows : 0);
    const int n_rows = bt.row_base[bt.n_jobs];
    if (n_rows <= 0) return 0;
    bool tq = false;
    for (int k = 0; k < bt.n_jobs; ++k)
        tq |= bt.job[k].kind == 0 ? bt.job[k].out_mode == OUT_TQ6 : bt.job[k].staging != SJKVARN_STAGING_F16;
    const int nw = tq && n_rows >= ROW_WAVES_BIG * n_cus() ? ROW_WAVES_BIG : ROW_WAVES;
    const dim3 grid((unsigned) ((n_rows + nw - 1) / nw)), block((unsigned) (64 * nw));
#define SJK_ROWS(V) \
    if (nw == ROW_WAVES) hipLaunchKernelGGL((rows_kernel<V, ROW_WAVES>), grid, block, 0, st, bt); \
    else hipLaunchKernelGGL((rows_kernel<V, ROW_WAVES_BIG>), grid, block, 0, st, bt);
    switch (bt.job[0].D) {
    case 128: SJK_ROWS(2) break;
    case 256: SJK_ROWS(4) break;
    case 512: SJK_ROWS(8) break;
    default: return SJK_ERR_UNSUPPORTED;
    }
#undef SJK_ROWS
    return SJK_CHECK_LAUNCH();
}

static int launch_rows(const RowJob & j, hipStream_t st) {
    RowBatch bt = {};
    bt.job[0] = j;
    bt.n_jobs = 1;
    return launch_batch(bt, st);
}

static float rot_scale(int D) { return 1.0f / __builtin_sqrtf((float) D); }

// ---- unstage: one thread per value (sj_kvarn.h:1249-1260, 1276-1284) ----
__global__ void unstage_kernel(int staging, const uint8_t * src, size_t src_row_bytes, float * x, int D, int n_rows) {
    const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t) n_rows * D) return;
    const size_t r = i / (size_t) D;
    const int e = (int) (i % (size_t) D);
    const uint8_t * row = src + r * src_row_bytes;
    if (staging == SJKVARN_STAGING_F16) {
        x[i] = f16_to_f32((uint16_t) (row[2 * e] | (row[2 * e + 1] << 8)));
        return;
    }
    const uint8_t * blk = row + (size_t) (e >> 7) * SJKVARN_TQ6_BLOCK_BYTES;
    const int jx = e & 127;
    const int code = ((blk[2 + (jx >> 1)] >> (4 * (jx & 1))) & 15) | (((blk[66 + (jx >> 2)] >> (2 * (jx & 3))) & 3) << 4);
    x[i] = xmul(tq6_cent(code), f16_to_f32((uint16_t) (blk[0] | (blk[1] << 8))));
}

// ---- decode: one thread per (record, token, channel) (sj_kvarn.h:1178-1207) ----
SJK_DEV float code_value(const sj_kvarn_layout & l, const uint8_t * rec, int t, int d, int is_v) {
    const int bits = is_v ? l.bits_v : l.bits_k;
    const uint8_t * payload = rec + (is_v ? l.v_payload : l.k_payload);
    if (l.body == SJKVARN_BODY_TRELLIS) return f16_to_f32(codebook(bits, is_v)[trellis_window(payload, bits, d, t)]);
    return (float) get_code(payload, code_bit(l, t, d, is_v), bits);
}

__global__ void decode_kernel(sj_kvarn_layout l, const uint8_t * body, int n_rec, float * out_k, float * out_v) {
    const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t) n_rec * l.G * l.D) return;
    const int d = (int) (i % (size_t) l.D);
    const size_t rt = i / (size_t) l.D;
    const int t = (int) (rt % (size_t) l.G);
    const uint8_t * rec = body + (rt / (size_t) l.G) * l.bytes;
    const uint32_t ci = (uint32_t) k_ch_idx(l, d);
    out_k[i] = dequant_x(code_value(l, rec, t, d, 0), get_half(rec, l.k_scale + 2u * ci), get_half(rec, l.k_zero + 2u * ci),
                         get_half(rec, l.k_tok + 2u * (uint32_t) t));
    out_v[i] = dequant_x(code_value(l, rec, t, d, 1), get_half(rec, l.v_scale + 2u * (uint32_t) t),
                         get_half(rec, l.v_zero + 2u * (uint32_t) t), get_half(rec, l.v_ch + 2u * (uint32_t) v_ch_idx(l, d)));
}

// Decode of records with a layer's own geometry (D = 128 or 256, G = 128) whose words are aligned. The kernel above is
// bound by its byte loads and address arithmetic, ~60 instructions a value (41 us for 64 3/2 trellis records at D = 256:
// 18.2 MB, 16.8 of them written). Here a thread makes 4 consecutive channels x 8 tokens of one side: whole words of codes
// in (four 8-byte reads of the 4-bit order, a channel's 8 codes and history as one 32-bit window of a trellis), one
// 16-byte store per token out; the trellis codebook sits in LDS as floats. 9.3 us for the
// same records, of which the launch is ~4; a first form of 12 us converted the halves with f16_to_f32's branches.
// The values are those of dequant_x: the plain products and sum unless the result is a NaN, whose sign dequant_x gives
// (a NaN made on the way stays one, so checking the result is enough).
SJK_DEV float dequant_fast(float q, float scale, float zero, float col) {
    const float r = (q * scale + zero) * col;
    return r == r ? r : dequant_x(q, scale, zero, col);
}

typedef uint16_t half4_t __attribute__((ext_vector_type(4), aligned(2)));

template <int D>
__global__ __launch_bounds__(256) void decode_tile_kernel(const sj_kvarn_layout l, const uint8_t * body, float * out_k,
                                                          float * out_v) {
    constexpr int NQ = D / 4, WGS = D / 64;      // channel quads; workgroups per record and side
    __shared__ float cb[512];
    const int is_v = blockIdx.y, bits = is_v ? l.bits_v : l.bits_k;
    const bool trellis = l.body == SJKVARN_BODY_TRELLIS, frag = frag_side(l, bits);
    const size_t r = blockIdx.x / WGS;
    const int u = (int) (blockIdx.x % WGS) * 256 + (int) threadIdx.x;
    const int d0 = 4 * (u % NQ), tb = u / NQ >> 1, hf = u / NQ & 1;    // 16-token block, its half
    const uint8_t * rec = body + r * l.bytes, * pay = rec + (is_v ? l.v_payload : l.k_payload);
    // this thread's tokens, t0 .. + 3 and t1 .. + 3: in the 4-bit order the halves of a block interleave by fours
    const int t0 = 16 * tb + (frag ? 4 : 8) * hf, t1 = t0 + (frag ? 8 : 4);

    // everything read is asked for before the codebook's barrier
    auto halves = [&](uint32_t off) { return *(const half4_t *) (rec + off); };
    half4_t ts[2], tz[2], ca, cz = {};           // per token: V scale and zero, or the K column scale; per channel
    ts[0] = halves((is_v ? l.v_scale : l.k_tok) + 2u * (uint32_t) t0);
    ts[1] = halves((is_v ? l.v_scale : l.k_tok) + 2u * (uint32_t) t1);
    tz[0] = halves((is_v ? l.v_zero : l.k_tok) + 2u * (uint32_t) t0);
    tz[1] = halves((is_v ? l.v_zero : l.k_tok) + 2u * (uint32_t) t1);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint32_t ci = 2u * (uint32_t) (is_v ? v_ch_idx(l, d0 + c) : k_ch_idx(l, d0 + c));
        ca[c] = *(const uint16_t *) (rec + (is_v ? l.v_ch : l.k_scale) + ci);
        if (!is_v) cz[c] = *(const uint16_t *) (rec + l.k_zero + ci);
    }
    uint32_t x[8] = {};
    if (trellis) {
        // channel d's bits from 6 before its token t0 on (from its start where that lies before it): token t0 + k's
        // window is the 6 + bits bits ending with its code
        const int at = t0 ? t0 * bits - 6 : 0, w0 = at >> 5, w1 = w0 + 1 < 4 * bits ? w0 + 1 : w0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t * w = (const uint32_t *) pay + (d0 + c) * 4 * bits;
            x[c] = __builtin_amdgcn_alignbit(w[w1], w[w0], (uint32_t) at & 31u) << (t0 ? 0 : 6);
        }
        const uint16_t * t = codebook(bits, is_v);
        for (int i = (int) threadIdx.x; i < (64 << bits); i += 256) cb[i] = f16_to_f32(t[i]);
        __syncthreads();
    } else if (frag && !is_v) {
        // 16-token x 16-channel tiles of 32 words, a = token, b = channel: 4 channels in two words
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t * w = (const uint32_t *) pay + (tb * (D / 16) + (d0 >> 4)) * 32 + 4 * (4 * hf + k) + ((d0 >> 1) & 3);
            x[2 * k] = w[0];
            x[2 * k + 1] = w[1];
        }
    } else if (frag) {
        // a = channel, b = token: a channel's tokens t0 .. + 3 and t1 .. + 3 in two words
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int d = d0 + c;
            const uint32_t * w = (const uint32_t *) pay + (tb * (D / 16) + (d >> 4)) * 32 + 4 * (d & 7) + 2 * hf;
            x[2 * c] = w[0];
            x[2 * c + 1] = w[1];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {            // token-major: 4 codes of 2 or 3 bits from bit 0 or 4 of a byte
            const uint32_t bit = ((uint32_t) ((k < 4 ? t0 : t1 - 4) + k) * D + (uint32_t) d0) * (uint32_t) bits;
            x[k] = (pay[bit >> 3] | ((bits > 2 ? (uint32_t) pay[(bit >> 3) + 1] : 0u) << 8)) >> (bit & 7u);
        }
    }

    // halves by the hardware's conversion: it quiets a NaN and keeps its sign, which is all that dequant_x keeps
    float a[4], b[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) { a[c] = f16_to_f32_fast(ca[c]); b[c] = f16_to_f32_fast(cz[c]); }
    float * out = (is_v ? out_v : out_k) + r * 128u * D + d0;
    auto emit = [&](auto && code) {              // code(k, c): the code's value, token k, channel c
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float s = f16_to_f32_fast(ts[k >> 2][k & 3]), z = f16_to_f32_fast(tz[k >> 2][k & 3]);
            float4 y;
            float * yc = &y.x;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                yc[c] = dequant_fast(code(k, c), is_v ? s : a[c], is_v ? z : b[c], is_v ? a[c] : s);
            *(float4 *) (out + (size_t) ((k < 4 ? t0 : t1 - 4) + k) * D) = y;
        }
    };
    const uint32_t mask = (1u << bits) - 1u;
    if (trellis) emit([&](int k, int c) { return cb[(x[c] >> (k * bits)) & ((64u << bits) - 1u)]; });
    else if (frag && !is_v) emit([&](int k, int c) { return (float) ((x[2 * (k & 3) + (c >> 1)] >> (4 * (k >> 2) + 16 * (c & 1) + (d0 & 8))) & 15u); });
    else if (frag) emit([&](int k, int c) { return (float) ((x[2 * c + ((k >> 1) & 1)] >> (4 * (((d0 + c) >> 3) & 1) + 16 * (k & 1) + 8 * (k >> 2))) & 15u); });
    else emit([&](int k, int c) { return (float) ((x[k] >> (c * bits)) & mask); });
}

// what decode_tile_kernel reads and writes in words: a layer's own geometry, code words at multiples of 4 bytes, halves
// at even addresses, output rows at multiples of 16
static bool decode_tiles_ok(const sj_kvarn_layout & l, const void * body, const void * out_k, const void * out_v) {
    if (!sjk_hip_supported(&l) || (l.body == SJKVARN_BODY_TRELLIS && (l.bits_k > 3 || l.bits_v > 3))) return false;
    const uint32_t half = l.k_scale | l.k_zero | l.k_tok | l.v_ch | l.v_scale | l.v_zero;
    const uintptr_t word = (uintptr_t) body | l.bytes | l.k_payload | l.v_payload;
    return !(word & 3u) && !(half & 1u) && !(((uintptr_t) out_k | (uintptr_t) out_v) & 15u);
}

// Gather / scatter of device byte runs (the sequence state stream: sink, records and ring rows of every layer
// to or from one staging buffer). Workgroups stride over the runs; the run descriptor is wave-uniform.
__global__ __launch_bounds__(256) void copy_runs_kernel(const CopyRun * runs, int n) {
    for (int r = (int) blockIdx.x; r < n; r += (int) gridDim.x) {
        const CopyRun R = runs[r];
        const uint64_t al = R.src | R.dst | R.bytes;
        if ((al & 15u) == 0) {
            const uint4 * s4 = (const uint4 *) R.src;
            uint4 * d4 = (uint4 *) R.dst;
            for (uint64_t i = threadIdx.x; i < R.bytes / 16u; i += blockDim.x) d4[i] = s4[i];
        } else if ((al & 3u) == 0) {
            const uint32_t * s1 = (const uint32_t *) R.src;
            uint32_t * d1 = (uint32_t *) R.dst;
            for (uint64_t i = threadIdx.x; i < R.bytes / 4u; i += blockDim.x) d1[i] = s1[i];
        } else {
            const uint8_t * s1 = (const uint8_t *) R.src;
            uint8_t * d1 = (uint8_t *) R.dst;
            for (uint64_t i = threadIdx.x; i < R.bytes; i += blockDim.x) d1[i] = s1[i];
        }
    }
}

int sjk_copy_runs(const CopyRun * d_runs, int n, hipStream_t stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(copy_runs_kernel, dim3((unsigned) (n < 2048 ? n : 2048)), dim3(256), 0, stream, d_runs, n);
    return SJK_CHECK_LAUNCH();
}

// Zero the dst range of every run (src unused): the truncation / reset scrub of all layers in one launch
__global__ __launch_bounds__(256) void zero_runs_kernel(const CopyRun * runs, int n) {
    for (int r = (int) blockIdx.x; r < n; r += (int) gridDim.x) {
        const CopyRun R = runs[r];
        if (((R.dst | R.bytes) & 15u) == 0) {
            uint4 * d4 = (uint4 *) R.dst;
            for (uint64_t i = threadIdx.x; i < R.bytes / 16u; i += blockDim.x) d4[i] = uint4{0u, 0u, 0u, 0u};
        } else {
            uint8_t * d1 = (uint8_t *) R.dst;
            for (uint64_t i = threadIdx.x; i < R.bytes; i += blockDim.x) d1[i] = 0;
        }
    }
}

// Words carried in the kernel arguments, so the caller's host copy may change as soon as the launch returns
__global__ __launch_bounds__(256) void set_words_kernel(uint32_t * dst, const WordBatch w) {
    for (uint32_t i = threadIdx.x; i < w.n; i += 256) dst[i] = w.v[i];
}

int sjk_set_words(uint32_t * d_dst, const uint32_t * host, uint32_t n, hipStream_t stream) {
    WordBatch w;
    for (uint32_t o = 0; o < n; o += WORD_BATCH) {
        w.n = n - o < WORD_BATCH ? n - o : WORD_BATCH;
        for (uint32_t i = 0; i < w.n; ++i) w.v[i] = host[o + i];
        hipLaunchKernelGGL(set_words_kernel, dim3(1), dim3(256), 0, stream, d_dst + o, w);
        if (hipPeekAtLastError() != hipSuccess) return SJK_ERR_DEVICE;
    }
    return 0;
}

int sjk_zero_runs(const CopyRun * d_runs, int n, hipStream_t stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(zero_runs_kernel, dim3((unsigned) (n < 2048 ? n : 2048)), dim3(256), 0, stream, d_runs, n);
    return SJK_CHECK_LAUNCH();
}

}  // namespace sjk

using namespace sjk;

namespace sjk {
// fp16 staging of rows of any width: one thread per value (sj_kvarn.h:1266-1271)
__global__ void stage_f16_kernel(const float * x, uint8_t * dst, int D, size_t dst_row_bytes, int n_rows) {
    const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t) n_rows * (size_t) D) return;
    const size_t r = i / (size_t) D, e = i % (size_t) D;
    *(uint16_t *) (dst + r * dst_row_bytes + 2 * e) = f32_to_f16(x[i]);
}
}  // namespace sjk

extern "C" int sjk_hip_stage(int staging, const float * d_x, uint8_t * d_dst, int D, size_t dst_row_bytes, int n_rows,
                             void * stream) {
    if (!d_x || !d_dst || n_rows < 0 || D <= 0 || (staging != SJKVARN_STAGING_TQ6_0 && staging != SJKVARN_STAGING_F16))
        return SJKVARN_ERR_ARG;
    if (!n_rows) return 0;
    if (D != 128 && D != 256 && D != 512) {
        hipStream_t st = (hipStream_t) stream;
        if (staging == SJKVARN_STAGING_F16) {
            const size_t n = (size_t) n_rows * (size_t) D;
            hipLaunchKernelGGL(stage_f16_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, d_x, d_dst, D,
                               dst_row_bytes, n_rows);
            return SJK_CHECK_LAUNCH();
        }
        // tq6_0: the D / 128 whole blocks of each row (the reference quantizes n / 128 blocks), as rows of 128
        const int nb = D / SJKVARN_TQ6_QK;
        if (!nb) return 0;
        for (int r = 0; r < n_rows; ++r) {
            const bool packed = dst_row_bytes == (size_t) nb * SJKVARN_TQ6_BLOCK_BYTES && D % SJKVARN_TQ6_QK == 0;
            RowJob j = {};
            j.kind = 0; j.D = SJKVARN_TQ6_QK; j.rotate = 0; j.rot_scale = rot_scale(SJKVARN_TQ6_QK);
            j.n_rows = packed ? nb * n_rows : nb;
            j.x = d_x + (size_t) r * D; j.dst = d_dst + (size_t) r * dst_row_bytes;
            j.dst_row_bytes = SJKVARN_TQ6_BLOCK_BYTES; j.out_mode = OUT_TQ6;
            const int rc = launch_rows(j, st);
            if (rc || packed) return rc;
        }
        return 0;
    }
    RowJob j = {};
    j.kind = 0; j.D = D; j.n_rows = n_rows; j.rotate = 0; j.rot_scale = rot_scale(D);
    j.x = d_x; j.dst = d_dst; j.dst_row_bytes = dst_row_bytes;
    j.out_mode = staging == SJKVARN_STAGING_F16 ? OUT_F16 : OUT_TQ6;
    return launch_rows(j, (hipStream_t) stream);
}

namespace sjk {

// Hadamard of rows of any power-of-two length n (sj_kvarn.h:735-752) outside the row kernel's widths: stage h pairs
// element j with j + h (j in the lower half of its 2h block) as a + b, a - b, stages in ascending h, then one
// multiply by s. The order of the stages, not the order of the pairs inside a stage, fixes every value, so
// these are bit-identical to the reference's loop.
constexpr int HD_LDS_MAX = 8192;          // rows up to 32 KB go through LDS, one workgroup per row

__global__ __launch_bounds__(256) void hadamard_lds_kernel(float * x, int n, float s) {
    extern __shared__ float t[];
    float * row = x + (size_t) blockIdx.x * (size_t) n;
    for (int i = (int) threadIdx.x; i < n; i += 256) t[i] = row[i];
    __syncthreads();
    for (int h = 1; h < n; h <<= 1) {
        for (int k = (int) threadIdx.x; k < n / 2; k += 256) {
            const int j = (k / h) * 2 * h + (k % h);
            const float a = t[j], b = t[j + h];
            t[j] = xadd(a, b);
            t[j + h] = xsub(a, b);
        }
        __syncthreads();
    }
    for (int i = (int) threadIdx.x; i < n; i += 256) row[i] = xmul(t[i], s);
}

// one stage of longer rows in global memory: pair k of the n_rows * n / 2 pairs
__global__ __launch_bounds__(256) void hadamard_stage_kernel(float * x, int n, int h, size_t n_pairs) {
    const size_t k = (size_t) blockIdx.x * 256u + threadIdx.x;
    if (k >= n_pairs) return;
    const size_t row = k / (size_t) (n / 2), kk = k % (size_t) (n / 2);
    const size_t j = row * (size_t) n + (kk / (size_t) h) * 2u * (size_t) h + kk % (size_t) h;
    const float a = x[j], b = x[j + (size_t) h];
    x[j] = xadd(a, b);
    x[j + (size_t) h] = xsub(a, b);
}

// one stage along the rows of a [n_blocks * n][cols] matrix (each column's n-blocks are the vectors): pair k of the
// n_blocks * n / 2 * cols pairs, column fastest (adjacent threads, adjacent columns)
__global__ __launch_bounds__(256) void hadamard_cols_stage_kernel(float * x, int n, int h, int cols, size_t n_pairs) {
    const size_t k = (size_t) blockIdx.x * 256u + threadIdx.x;
    if (k >= n_pairs) return;
    const size_t c = k % (size_t) cols, rest = k / (size_t) cols;
    const size_t blk = rest / (size_t) (n / 2), kk = rest % (size_t) (n / 2);
    const size_t j = blk * (size_t) n + (kk / (size_t) h) * 2u * (size_t) h + kk % (size_t) h;
    float * pa = x + j * (size_t) cols + c;
    float * pb = pa + (size_t) h * (size_t) cols;
    const float a = *pa, b = *pb;
    *pa = xadd(a, b);
    *pb = xsub(a, b);
}

__global__ __launch_bounds__(256) void scale_kernel(float * x, size_t n, float s) {
    const size_t i = (size_t) blockIdx.x * 256u + threadIdx.x;
    if (i < n) x[i] = xmul(x[i], s);
}

}  // namespace sjk

// Rotation folded into projection weights. Output side (W_q, W_k, W_v, their biases): [n_heads * D][cols], each
// column's head blocks rotated, i.e. the per-head rotation applied from the left, W' = blockdiag(R) W. Input side
// (W_o): [rows][n_heads * D], each row's head segments rotated, W' = W blockdiag(R) (R = H / sqrt(D) is
// symmetric and its own inverse) - sjk_hip_rotate over rows x n_heads segments of D.
extern "C" int sjk_hip_fold_rotation_out(float * d_w, int n_heads, int D, int cols, void * stream) {
    if (!d_w || n_heads < 0 || cols < 0 || D <= 0 || (D & (D - 1))) return SJKVARN_ERR_ARG;
    if (!n_heads || !cols) return 0;
    hipStream_t st = (hipStream_t) stream;
    const size_t pairs = (size_t) n_heads * (size_t) (D / 2) * (size_t) cols, all = (size_t) n_heads * D * (size_t) cols;
    for (int h = 1; h < D; h <<= 1) {
        hipLaunchKernelGGL(hadamard_cols_stage_kernel, dim3((unsigned) ((pairs + 255) / 256)), dim3(256), 0, st, d_w, D,
                           h, cols, pairs);
        if (SJK_CHECK_LAUNCH()) return SJK_ERR_DEVICE;
    }
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned) ((all + 255) / 256)), dim3(256), 0, st, d_w, all, rot_scale(D));
    return SJK_CHECK_LAUNCH();
}

extern "C" int sjk_hip_rotate(float * d_x, int n_rows, int D, void * stream);

extern "C" int sjk_hip_fold_rotation_in(float * d_w, int rows, int n_heads, int D, void * stream) {
    if (!d_w || rows < 0 || n_heads < 0 || D <= 0 || (D & (D - 1))) return SJKVARN_ERR_ARG;
    if ((size_t) rows * (size_t) n_heads > (size_t) 0x7fffffff) return SJKVARN_ERR_ARG;
    return sjk_hip_rotate(d_w, rows * n_heads, D, stream);
}

extern "C" int sjk_hip_rotate(float * d_x, int n_rows, int D, void * stream) {
    if (!d_x || n_rows < 0 || D <= 0 || (D & (D - 1))) return SJKVARN_ERR_ARG;
    if (!n_rows) return 0;
    hipStream_t st = (hipStream_t) stream;
    if (D == 128 || D == 256 || D == 512) {
        RowJob j = {};
        j.kind = 0; j.D = D; j.n_rows = n_rows; j.rotate = 1; j.rot_scale = rot_scale(D);
        j.x = d_x; j.dst = (uint8_t *) d_x; j.dst_row_bytes = (size_t) D * 4; j.out_mode = OUT_F32;
        return launch_rows(j, st);
    }
    const float s = rot_scale(D);
    if (D <= HD_LDS_MAX) {
        hipLaunchKernelGGL(hadamard_lds_kernel, dim3((unsigned) n_rows), dim3(256), (size_t) D * 4, st, d_x, D, s);
        return SJK_CHECK_LAUNCH();
    }
    const size_t pairs = (size_t) n_rows * (size_t) (D / 2), all = (size_t) n_rows * (size_t) D;
    for (int h = 1; h < D; h <<= 1) {
        hipLaunchKernelGGL(hadamard_stage_kernel, dim3((unsigned) ((pairs + 255) / 256)), dim3(256), 0, st, d_x, D, h, pairs);
        if (SJK_CHECK_LAUNCH()) return SJK_ERR_DEVICE;
    }
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned) ((all + 255) / 256)), dim3(256), 0, st, d_x, all, s);
    return SJK_CHECK_LAUNCH();
}

static RowJob store_job(const sjk_hip_view * v, uint32_t pos0, uint32_t n_pos, const float * d_k, const float * d_v,
                        int rotate) {
    RowJob j = {};
    j.kind = 1; j.D = v->lay.D; j.n_rows = (int) n_pos * v->n_head_kv * 2; j.rotate = rotate ? 1 : 0;
    j.rot_scale = rot_scale(v->lay.D);
    j.k = d_k; j.v = d_v; j.sink = v->sink; j.ring = v->ring;
    j.pos0 = pos0; j.S = v->S; j.cap = v->cap; j.H = v->n_head_kv; j.sink_type = v->sink_type;
    j.staging = v->staging; j.stage_bytes = v->stage_bytes;
    return j;
}

extern "C" int sjk_hip_layer_store(const sjk_hip_view * v, uint32_t pos0, uint32_t n_pos, const float * d_k,
                                   const float * d_v, int rotate, void * stream) {
    if (!v || !d_k || !d_v || !v->sink || !v->ring) return SJKVARN_ERR_ARG;
    return launch_rows(store_job(v, pos0, n_pos, d_k, d_v, rotate), (hipStream_t) stream);
}

extern "C" int sjk_hip_layer_store_dyn(const sjk_hip_view * v, const int32_t * d_desc, uint32_t n_pos, const float * d_k,
                                       const float * d_v, int rotate, void * stream) {
    if (!v || !d_desc || !d_k || !d_v || !v->sink || !v->ring) return SJKVARN_ERR_ARG;
    RowJob j = store_job(v, 0, n_pos, d_k, d_v, rotate);
    j.pos_desc = d_desc;
    return launch_rows(j, (hipStream_t) stream);
}

extern "C" int sjk_hip_store_batch(const sjk_hip_store_job * jobs, int n_jobs, uint32_t n_pos, int rotate, void * stream) {
    if (n_jobs < 0 || (n_jobs > 0 && !jobs)) return SJKVARN_ERR_ARG;
    for (int k = 0; k < n_jobs; ++k)
        if (!jobs[k].d_k || !jobs[k].d_v || !jobs[k].v.sink || !jobs[k].v.ring || jobs[k].v.lay.D != jobs[0].v.lay.D)
            return SJKVARN_ERR_ARG;
    for (int k0 = 0; k0 < n_jobs; k0 += ROW_MAXJ) {
        RowBatch bt = {};
        bt.n_jobs = n_jobs - k0 < ROW_MAXJ ? n_jobs - k0 : ROW_MAXJ;
        for (int k = 0; k < bt.n_jobs; ++k) {
            const sjk_hip_store_job & J = jobs[k0 + k];
            bt.job[k] = store_job(&J.v, J.pos0, n_pos, J.d_k, J.d_v, rotate);
        }
        const int rc = launch_batch(bt, (hipStream_t) stream);
        if (rc) return rc;
    }
    return 0;
}

extern "C" int sjk_hip_unstage(int staging, const uint8_t * d_src, size_t src_row_bytes, float * d_x, int D, int n_rows,
                               void * stream) {
    if (!d_src || !d_x || n_rows < 0 || D <= 0 || (staging == SJKVARN_STAGING_TQ6_0 && D % 128)) return SJKVARN_ERR_ARG;
    const size_t n = (size_t) n_rows * D;
    if (!n) return 0;
    hipLaunchKernelGGL(unstage_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, (hipStream_t) stream, staging,
                       d_src, src_row_bytes, d_x, D, n_rows);
    return SJK_CHECK_LAUNCH();
}

extern "C" int sjk_hip_decode(const sj_kvarn_layout * l, const uint8_t * d_body, int n_rec, float * d_out_k,
                              float * d_out_v, void * stream) {
    if (!l || !d_body || !d_out_k || !d_out_v || n_rec < 0) return SJKVARN_ERR_ARG;
    const size_t n = (size_t) n_rec * l->G * l->D;
    if (!n) return 0;
    if (decode_tiles_ok(*l, d_body, d_out_k, d_out_v)) {
        const dim3 grid((unsigned) n_rec * (unsigned) (l->D / 64), 2);
        if (l->D == 256) hipLaunchKernelGGL(decode_tile_kernel<256>, grid, dim3(256), 0, (hipStream_t) stream, *l, d_body, d_out_k, d_out_v);
        else hipLaunchKernelGGL(decode_tile_kernel<128>, grid, dim3(256), 0, (hipStream_t) stream, *l, d_body, d_out_k, d_out_v);
        return SJK_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(decode_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, (hipStream_t) stream, *l, d_body,
                       n_rec, d_out_k, d_out_v);
    return SJK_CHECK_LAUNCH();
}

namespace sjk {

// ---- record_scores / record_accum_v (sj_kvarn.h:1288-1311): sequential fp32 as in the reference ----
SJK_DEV float decode_k_at(const sj_kvarn_layout & l, const uint8_t * rec, int t, int d) {
    const uint32_t ci = (uint32_t) k_ch_idx(l, d);
    return dequant_x(code_value(l, rec, t, d, 0), get_half(rec, l.k_scale + 2u * ci), get_half(rec, l.k_zero + 2u * ci),
                     get_half(rec, l.k_tok + 2u * (uint32_t) t));
}

SJK_DEV float decode_v_at(const sj_kvarn_layout & l, const uint8_t * rec, int t, int d) {
    return dequant_x(code_value(l, rec, t, d, 1), get_half(rec, l.v_scale + 2u * (uint32_t) t),
                     get_half(rec, l.v_zero + 2u * (uint32_t) t), get_half(rec, l.v_ch + 2u * (uint32_t) v_ch_idx(l, d)));
}

__global__ void record_scores_kernel(sj_kvarn_layout l, const uint8_t * rec, const float * q, int n, float * scores) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    float s = 0.0f;
    for (int d = 0; d < l.D; ++d) s = s + q[d] * decode_k_at(l, rec, t, d);
    scores[t] = s;
}

__global__ void record_accum_kernel(sj_kvarn_layout l, const uint8_t * rec, const float * w, int n, float * acc) {
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= l.D) return;
    float a = acc[d];
    for (int t = 0; t < n; ++t) a = a + w[t] * decode_v_at(l, rec, t, d);
    acc[d] = a;
}

}  // namespace sjk

extern "C" int sjk_hip_record_scores(const sj_kvarn_layout * l, const uint8_t * d_rec, const float * d_q, int n,
                                     float * d_scores, void * stream) {
    if (!l || !d_rec || !d_q || !d_scores || n < 0 || n > l->G) return SJKVARN_ERR_ARG;
    if (!n) return 0;
    hipLaunchKernelGGL(sjk::record_scores_kernel, dim3((unsigned) ((n + 127) / 128)), dim3(128), 0, (hipStream_t) stream,
                       *l, d_rec, d_q, n, d_scores);
    return SJK_CHECK_LAUNCH();
}

extern "C" int sjk_hip_record_accum_v(const sj_kvarn_layout * l, const uint8_t * d_rec, const float * d_w, int n,
                                      float * d_acc, void * stream) {
    if (!l || !d_rec || !d_w || !d_acc || n < 0 || n > l->G) return SJKVARN_ERR_ARG;
    hipLaunchKernelGGL(sjk::record_accum_kernel, dim3((unsigned) ((l->D + 127) / 128)), dim3(128), 0, (hipStream_t) stream,
                       *l, d_rec, d_w, n, d_acc);
    return SJK_CHECK_LAUNCH();
}
