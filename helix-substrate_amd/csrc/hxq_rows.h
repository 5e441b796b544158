// Few-row GEMM: Y[M, OUT] = X[M, K] @ W^T for batched decode and short prompts,
// W in any HXQ index format (the contraction of hxq_prefill_gemm, same
// operands bit for bit; hxq_prefill.hip says which calls come here).
//
// What bounds it: the compressed weights, read once.  A 128- or 256-row tile
// spends its LDS reads, MFMAs and stores on rows that are not there (16 rows
// of an 18944 x 3584 layer: 54 us + a 6 us split-K reduce, 1.2 TB/s; here
// 24.2 us, 3.0 TB/s).  A block owns a run of NS 16-row subtiles of W over the
// whole K, and its W waves split K between them:
//   * wave w takes the 64-column steps w SP .., w SP + W SP .., so a block reads
//     W SP 64 consecutive columns of its rows at a time; it dequantises 16
//     weights per lane and subtile into the A operand of
//     v_mfma_f32_16x16x32_{bf16,f16} (fp32 X: v_mfma_f32_16x16x4_f32); X is
//     the B operand.  No barrier in the loop, loads one iteration ahead;
//   * lane (r = lane % 16, h = lane / 16) holds the physical columns
//     16h .. 16h + 15 of the step of row r; the MFMA's k order is permuted
//     alike for W and X;
//   * the waves' partial sums meet in LDS (in wave order: deterministic) and
//     leave as four consecutive outputs per thread.  No partials in memory,
//     no second launch, no workspace.
// SP steps per iteration keep about four index loads per lane in flight
// whatever NS is; NS up to five, so that a run touches two 64-row sidecar
// groups, half a wave each.  Sidecar values replace the operand registers, as
// in the prefill kernel.
#pragma once
#include <type_traits>

#include "hxq_common.h"

namespace hxq {
namespace rw {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));

constexpr int kStep = 64;    // columns per step
constexpr int kSub = 16;     // W rows per subtile
constexpr int kNrep = 64;    // uint8 codebook replicas
constexpr uint32_t kOob = 0x80000000u;

struct Args {
    const int32_t *sc_ptr;   // step pointers per 64-row group, or null
    const uint32_t *sc_key;
    const float *sc_val;
    const float *bias;
    void *y;
    int32_t n_codes, y_dtype, vec_out;
};

// Row tiles and subtiles per block, steps per iteration, grid (W, X).
struct Plan {
    int mt, ns, sp, bx, by;
};

struct Call {
    const uint8_t *idx;
    const void *x;           // [M, K]
    const float *cb;
    const float2 *ga;        // [K/G, OUT] {scale, offset} or null
    int32_t M, OUT, K, ngroups;
    uint32_t gmul;           // group of 16-column unit u: umulhi(u, gmul) (0: u itself)
    Args a;
};

// Grouped (mixture-of-experts) launches: the rows of Y are the expert-sorted
// assignment list, a block takes one row tile of one expert and one run of one
// bank's subtiles.  Eight waves a block, two blocks per CU: one's table and
// first loads pass while the other computes.
struct Bank {
    const uint8_t *idx;
    const float *cb;
    const float2 *ga;
    const int32_t *sc_ptr;
    const uint32_t *sc_key;
    const float *sc_val;
};

struct Grouped {
    Bank bank[2];            // columns [0, OUT) of Y from bank 0, [OUT, 2 OUT) from bank 1
    const int32_t *rows;     // X row of each sorted position (null: the position)
    const int32_t *seg;      // expert e owns positions [seg[e], seg[e + 1])
    int32_t n_exp, n_banks, x_rows, runs;   // runs: blocks per bank and row tile
    int64_t idx_es, ga_es, scp_es;          // per-expert strides (codebooks: 256)
};

// index bytes per 16 weights
__host__ __device__ constexpr int fmt_b16(int f) {
    return f == HXQ_FMT_SCALAR_U16 ? 32 : (f == HXQ_FMT_VQ2_P12 || f == HXQ_FMT_AF6) ? 12 : 16;
}
__host__ __device__ constexpr int fmt_table_bytes(int f) {
    return f == HXQ_FMT_SCALAR ? 256 * kNrep * 4
         : f == HXQ_FMT_SCALAR_U16 ? kPairCodes * 4
         : f == HXQ_FMT_AF6 ? 16 : kPairCodes * 8;
}

// MT: 16-row tiles of X; NS: subtiles per block (the grid's last block may own
// fewer rows: loads past OUT return 0 and nothing is stored); SP: 64-column
// steps per iteration; XT: 0 fp16, 1 bf16, 2 fp32; W: waves per block.
// The arguments that the first loads need come first, as scalars: they are
// preloaded into SGPRs, so no argument fetch precedes the stream.
template <int MT, int NS, int SP, int XT, bool AFF, int FMT, int W, bool GRP = false>
__global__ __launch_bounds__(W * 64, GRP ? 4 : 1) void rows_kernel(const uint8_t *a_idx, const void *a_x, const float *a_cb,
                                                      const float2 *a_ga, const int32_t M, const int32_t OUT,
                                                      const int32_t K, const int32_t ngroups,
                                                      const uint32_t gmul, const Args g,
                                                      const typename std::conditional<GRP, Grouped, int>::type grp) {
    constexpr bool F32 = XT == 2;
    constexpr int XB = F32 ? 4 : 2;
    constexpr int XCH = kStep * XB / 16;      // 16-byte chunks per X row and step
    constexpr int NX = XCH * kSub / 64;       // X loads per lane, step and row tile
    constexpr int B16 = fmt_b16(FMT);
    constexpr int NQ = B16 == 32 ? 2 : 1;     // index loads per lane, step and subtile
    constexpr bool PAIR = FMT == HXQ_FMT_VQ2_U16 || FMT == HXQ_FMT_VQ2_P12;
    constexpr int kTbl = fmt_table_bytes(FMT);
    constexpr int kX = kSub * kStep * XB;     // bytes of an X step tile
    constexpr int kRed = W * NS * MT * 1024;
    constexpr int kMain = kTbl + W * kX;
    typedef typename std::conditional<F32, u32x16, u32x8>::type BV;
    // lookup table first (LDS address 0), then a tile of X per wave; the
    // partial sums over them afterwards
    __shared__ __attribute__((aligned(16))) char smem[kMain > kRed ? kMain : kRed];
    float *tbl = reinterpret_cast<float *>(smem);
    if (lds_offset_of(tbl) != 0) return;  // never taken: no other LDS in this kernel

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, hq = lane >> 4;
    int n0 = blockIdx.x * (NS * kSub);
    int m0 = blockIdx.y * (MT * kSub);  // first row of X and Y
    int mend = M, ybase = 0, ywidth = OUT;
    int64_t xrows = M;
    const int32_t *sc_ptr = g.sc_ptr;
    const uint32_t *sc_key = g.sc_key;
    const float *sc_val = g.sc_val;
    int nnz = 0;
    if constexpr (GRP) {
        int e, w = blockIdx.x % (grp.runs * grp.n_banks);
        if (!expert_row_tile(grp.seg, grp.n_exp, MT * kSub, blockIdx.x / (grp.runs * grp.n_banks), e, m0, mend))
            return;  // block-uniform
        const Bank &b = grp.bank[w >= grp.runs];
        if (w >= grp.runs) {
            w -= grp.runs;
            ybase = OUT;
        }
        n0 = w * (NS * kSub);
        ywidth = OUT * grp.n_banks;
        xrows = grp.x_rows;
        a_idx = b.idx + e * grp.idx_es;
        a_cb = b.cb + e * 256;
        a_ga = b.ga + e * grp.ga_es;
        sc_key = b.sc_key;
        sc_val = b.sc_val;
        if (b.sc_ptr) {   // the lists of all experts are one: its length after the last expert's last step
            nnz = kload(b.sc_ptr[grp.n_exp * grp.scp_es - 1]);
            sc_ptr = b.sc_ptr + e * grp.scp_es;
        } else {
            sc_ptr = nullptr;
        }
    }
    const int nst = K / kStep;
    char *sx = smem + kTbl + wave * kX;

    // ---- global sources ------------------------------------------------------------
    // Loads are laid out for the cache, not for the MFMA: four lanes read a
    // row's 64 index bytes, eight (fp32: sixteen) its X columns, so that 16
    // consecutive lanes touch four (two, one) lines and not 16 -- one line a
    // clock is what the address path takes (operand-layout loads: 36 us for
    // K = 18944, 16 rows, of which X alone 16).  Indices change lanes by
    // ds_bpermute, X through the wave's LDS tile.
    const int64_t row_bytes = (int64_t)K / 16 * B16;
    const int64_t x_bytes = xrows * K * XB, q_bytes = (int64_t)OUT * row_bytes;
    const int64_t a_bytes = (int64_t)ngroups * OUT * 8;
    uint32_t x_off[MT][NX], q_off[NS];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < NX; ++q) {
            const int m = m0 + 16 * i + lane / XCH + (64 / XCH) * q;
            int row = m;
            if constexpr (GRP) row = m < mend && grp.rows ? grp.rows[m] : m;
            x_off[i][q] = m < mend ? static_cast<uint32_t>(row * K * XB + (lane % XCH) * 16) : kOob;
        }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int n = n0 + kSub * j + (lane >> 2);
        q_off[j] = n < OUT ? static_cast<uint32_t>(n * row_bytes + B16 * (lane & 3)) : kOob;
    }
    // operand lane (r16, hq) takes what lane 4 r16 + hq loaded
    const int src = (4 * r16 + hq) * 4;

    // ---- loads, one iteration (SP steps) ahead ------------------------------------------
    // The step's column offset is the scalar offset of a load (at most a row,
    // below the resource's size, as the range check wants); a step past the
    // last one reads through an empty resource: zeros, and no memory traffic.
    u32x4 xv[SP][MT][NX];
    u32x4 qv[SP][NS][NQ];
    float2 av[SP][NS];
    auto load_x = [&](int t, int s) {
        const __amdgpu_buffer_rsrc_t r = make_rsrc(a_x, t < nst ? x_bytes : 0);
        const int so = t < nst ? t * (kStep * XB) : 0;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < NX; ++q)
                xv[s][i][q] = __builtin_amdgcn_raw_buffer_load_b128(r, x_off[i][q], so, 0);
    };
    auto load_w = [&](int t, int s, int j) {
        const __amdgpu_buffer_rsrc_t r = make_rsrc(a_idx, t < nst ? q_bytes : 0);
        const int so = t < nst ? t * (4 * B16) : 0;
        if constexpr (B16 == 12) {
            const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(r, q_off[j], so, 0);
            qv[s][j][0] = u32x4{v[0], v[1], v[2], 0u};
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                qv[s][j][q] = __builtin_amdgcn_raw_buffer_load_b128(r, q_off[j] + 16u * q, so, 0);
        }
    };
    // {scale, offset}, in operand layout: rows run on past OUT into the next
    // group's factors (or past the end: zeros), whose results are not stored
    auto a_base = [&](int t) {
        const uint32_t u = static_cast<uint32_t>(4 * t + hq);  // 16-column unit
        const uint32_t gi = gmul ? __umulhi(u, gmul) : u;
        return static_cast<uint32_t>(n0 + r16) * 8u + gi * (static_cast<uint32_t>(OUT) * 8u);
    };
    auto load_a = [&](int t, int s, int j, uint32_t o) {
        if constexpr (AFF) {
            const __amdgpu_buffer_rsrc_t r = make_rsrc(a_ga, t < nst ? a_bytes : 0);
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, o + kSub * 8u * j, 0, 0);
            av[s][j] = make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
        }
    };
    // sidecar: lanes 0-31 the run's first 64-row group, 32-63 the next one;
    // the pointers of an iteration two ahead, its entries one ahead
    const bool has_sc = sc_ptr != nullptr;
    const int ngrp = (OUT + 63) >> 6;
    const int half = lane >> 5;
    const uint32_t l32 = lane & 31u;
    const int sgrp = (n0 >> 6) + half;
    const int rbase = sgrp * 64 - n0;         // row of the run of the group's first row
    const uint32_t p_off = sgrp < ngrp ? static_cast<uint32_t>(sgrp * nst) * 4u : kOob;
    const int64_t p_bytes = has_sc ? int64_t{4} * (ngrp * nst + 1) : 0;
    if constexpr (!GRP) nnz = has_sc ? kload(sc_ptr[ngrp * nst]) : 0;
    const __amdgpu_buffer_rsrc_t kr = make_rsrc(sc_key, int64_t{4} * nnz);
    const __amdgpu_buffer_rsrc_t vr = make_rsrc(sc_val, int64_t{4} * nnz);
    uint32_t pf, pl;          // first entry and end of an iteration's steps
    uint32_t se, sn;          // this lane's list index, the group's entry count
    uint32_t sk;
    float sv;
    auto load_ptr = [&](int t) {
        const __amdgpu_buffer_rsrc_t r = make_rsrc(sc_ptr, t < nst ? p_bytes : 0);
        const int so = t < nst ? t * 4 : 0;
        pf = __builtin_amdgcn_raw_buffer_load_b32(r, p_off, so, 0);
        pl = __builtin_amdgcn_raw_buffer_load_b32(r, p_off + 4u * min(SP, max(nst - t, 0)), so, 0);
    };
    auto load_entries = [&]() {
        se = pf + l32;
        sn = pl - pf;
        const uint32_t o = l32 < sn ? se * 4u : kOob;
        sk = __builtin_amdgcn_raw_buffer_load_b32(kr, o, 0, 0);
        sv = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vr, o, 0, 0));
    };

    const int t0 = wave * SP;
    load_ptr(t0);
#pragma unroll
    for (int s = 0; s < SP; ++s) {
#pragma unroll
        for (int j = 0; j < NS; ++j) load_w(t0 + s, s, j);
        const uint32_t ao = a_base(t0 + s);
#pragma unroll
        for (int j = 0; j < NS; ++j) load_a(t0 + s, s, j, ao);
        load_x(t0 + s, s);
    }

    // ---- lookup table ------------------------------------------------------------
    if constexpr (FMT == HXQ_FMT_SCALAR) {
#pragma unroll
        for (int q = 0; q < 4096 / (W * 64); ++q) {
            const int slot = tid + W * 64 * q;  // float4 slot: entry slot / 16
            const float c = a_cb[slot >> 4];
            *reinterpret_cast<float4 *>(tbl + 4 * slot) = make_float4(c, c, c, c);
        }
    } else if constexpr (FMT == HXQ_FMT_SCALAR_U16) {
        for (int j = tid; j < kPairCodes; j += W * 64) tbl[j] = j < g.n_codes ? a_cb[j] : 0.f;
    } else if constexpr (PAIR) {
        float2 *t2 = reinterpret_cast<float2 *>(tbl);
        for (int j = tid; j < kPairCodes; j += W * 64)
            t2[j] = j < g.n_codes ? make_float2(a_cb[2 * j], a_cb[2 * j + 1]) : make_float2(0.f, 0.f);
    }
    load_entries();
    load_ptr(t0 + W * SP);
    lds_barrier();

    // ---- 16 weights of one subtile into operand registers ---------------------------
    const uint32_t lane_off = static_cast<uint32_t>(lane) * 4u;
    auto perm = [&](uint32_t v) {
        return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(v)));
    };
    auto field12 = [](const u32x4 &q, int bit, int width) -> uint32_t {
        const int wi = bit >> 5, sh = bit & 31;
        const uint32_t v = sh + width <= 32 ? q[wi] >> sh : __builtin_amdgcn_alignbit(q[wi + 1], q[wi], sh);
        return v & ((1u << width) - 1u);
    };
    auto dequant = [&](int s, int j, BV &b) {
        const float sc = AFF ? av[s][j].x : 1.f, of = AFF ? av[s][j].y : 0.f;
        u32x4 q[NQ];
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            q[i] = u32x4{perm(qv[s][j][i][0]), perm(qv[s][j][i][1]), perm(qv[s][j][i][2]), 0u};
            if constexpr (B16 != 12) q[i][3] = perm(qv[s][j][i][3]);
        }
        float v[16];
        if constexpr (FMT == HXQ_FMT_SCALAR) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                v[4 * d] = tbl_lookup0<kNrep, 0>(lane_off, q[0][d]);
                v[4 * d + 1] = tbl_lookup0<kNrep, 1>(lane_off, q[0][d]);
                v[4 * d + 2] = tbl_lookup0<kNrep, 2>(lane_off, q[0][d]);
                v[4 * d + 3] = tbl_lookup0<kNrep, 3>(lane_off, q[0][d]);
            }
        } else if constexpr (FMT == HXQ_FMT_SCALAR_U16) {
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const uint32_t w = q[NQ > 1 ? d >> 2 : 0][d & 3];
                v[2 * d] = tbl[w & (kPairCodes - 1u)];
                v[2 * d + 1] = tbl[(w >> 16) & (kPairCodes - 1u)];
            }
        } else if constexpr (PAIR) {
            const float2 *t2 = reinterpret_cast<const float2 *>(tbl);
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const uint32_t id = FMT == HXQ_FMT_VQ2_P12 ? field12(q[0], 12 * d, 12)
                                                           : (q[0][d >> 1] >> (16 * (d & 1))) & (kPairCodes - 1u);
                const float2 c = t2[id];
                v[2 * d] = c.x;
                v[2 * d + 1] = c.y;
            }
        } else {  // 6-bit levels
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = static_cast<float>(field12(q[0], 6 * e, 6));
        }
        if constexpr (F32) {
#pragma unroll
            for (int e = 0; e < 16; ++e) b[e] = __float_as_uint(AFF ? affine_exact(v[e], sc, of) : v[e]);
        } else {
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                if constexpr (AFF) b[d] = pack16<XT == 1>(affine_fma(v[2 * d], sc, of), affine_fma(v[2 * d + 1], sc, of));
                else b[d] = pack16<XT == 1>(v[2 * d], v[2 * d + 1]);
            }
        }
    };
    // replace the entries set in m (one per lane: `code` = owner lane | register
    // << 8 | upper half << 16, `val` its operand bits) in b
    auto apply = [&](unsigned long long m, uint32_t code, uint32_t val, BV &b) {
        while (m) {
            const int l = __builtin_ctzll(m);
            m &= m - 1;
            const uint32_t c = __builtin_amdgcn_readlane(code, l);
            const uint32_t nv = __builtin_amdgcn_readlane(val, l);
            const int reg = __builtin_amdgcn_readfirstlane(static_cast<int>((c >> 8) & 15u));
            const uint32_t old = b[reg];
            uint32_t upd = nv;
            if constexpr (!F32)
                upd = (c >> 16) ? ((old & 0xffffu) | (nv << 16)) : ((old & 0xffff0000u) | nv);
            b[reg] = lane == static_cast<int>(c & 63u) ? upd : old;
        }
    };
    // where the entry {key, v} of this lane's group goes in the iteration that
    // starts at step t: subtile + 8 * step (255: none of this run), and for
    // apply() its code and operand bits
    auto place = [&](uint32_t key, float v, bool in, int t, uint32_t &where, uint32_t &code, uint32_t &val) {
        const int lr = rbase + static_cast<int>(key & 63u);   // row within the run
        const uint32_t c = (key >> 6) - static_cast<uint32_t>(t) * kStep;  // column within the iteration
        where = in && lr >= 0 ? static_cast<uint32_t>(lr >> 4) + 8u * (c >> 6) : 255u;
        const uint32_t owner = (lr & 15u) + (c & 48u);
        if constexpr (F32) {
            code = owner | (c & 15u) << 8;
            val = __float_as_uint(v);
        } else {
            code = owner | ((c & 15u) >> 1) << 8 | (c & 1u) << 16;
            val = pack16<XT == 1>(v, 0.f) & 0xffffu;
        }
    };
    // chunk c of row m of the wave's X tile: the same bank swizzle as the
    // prefill kernel's (16 rows of one chunk on 16 distinct 16-byte slots)
    auto x_slot = [&](int m, int c) {
        return sx + m * (kStep * XB) + ((F32 ? c ^ m : c ^ ((m >> 1) & 7)) << 4);
    };

    f32x4 acc[NS][MT];
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int t = t0; t < nst; t += W * SP) {
        const int tn = t + W * SP;
        uint32_t where, code, val;
        place(sk, sv, l32 < sn, t, where, code, val);
        const bool more = __ballot(sn > 32u) != 0;  // entries of a group beyond its 32 lanes
        const uint32_t e0 = se, en = se - l32 + sn;
        load_entries();
        load_ptr(tn + W * SP);
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            // a step past the last would add codebook entry 0 times zero: NaN where
            // that entry is infinite and no weight uses it (the exit: at most 1 %, 16 x
            // 3584 x 18944 30.7 / 30.9 us, 64 x 3584 x 18944 52.2 / 52.1)
            if (SP > 1 && t + s >= nst) break;
            // X through the wave's tile into operand layout
            u32x4 xo[MT][XCH / 4];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
#pragma unroll
                for (int q = 0; q < NX; ++q)
                    *reinterpret_cast<u32x4 *>(x_slot(lane / XCH + (64 / XCH) * q, lane % XCH)) = xv[s][i][q];
                wave_lds_order();
#pragma unroll
                for (int q = 0; q < XCH / 4; ++q)
                    xo[i][q] = *reinterpret_cast<const u32x4 *>(x_slot(r16, (XCH / 4) * hq + q));
                wave_lds_order();
            }
            load_x(tn + s, s);
            const uint32_t ao = a_base(tn + s);
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                BV b;
                dequant(s, j, b);
                load_w(tn + s, s, j);
                load_a(tn + s, s, j, ao);
                apply(__ballot(where == j + 8u * s), code, val, b);
                if (more) {  // the rest from the list (a later copy of a position wins)
                    for (uint32_t e = e0 + 32; __ballot(e < en) != 0; e += 32) {
                        const bool in = e < en;
                        uint32_t w2, c2, v2;
                        place(in ? sc_key[e] : 0u, in ? sc_val[e] : 0.f, in, t, w2, c2, v2);
                        apply(__ballot(w2 == j + 8u * s), c2, v2, b);
                    }
                }
                if constexpr (F32) {
#pragma unroll
                    for (int e = 0; e < 16; ++e)
#pragma unroll
                        for (int i = 0; i < MT; ++i)
                            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                __uint_as_float(b[e]), __uint_as_float(xo[i][e >> 2][e & 3]), acc[j][i], 0, 0, 0);
                } else {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const u32x4 w = u32x4{b[4 * h], b[4 * h + 1], b[4 * h + 2], b[4 * h + 3]};
#pragma unroll
                        for (int i = 0; i < MT; ++i) {
                            if constexpr (XT == 1)
                                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    __builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, xo[i][h]), acc[j][i], 0, 0, 0);
                            else
                                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                    __builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, xo[i][h]), acc[j][i], 0, 0, 0);
                        }
                    }
                }
            }
        }
    }

    // ---- the waves' partial sums, in wave order ----------------------------------
    lds_barrier();   // every wave is done with the table and its X tile
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) red[((wave * NS + j) * MT + i) * 64 + lane] = acc[j][i];
    lds_barrier();
    for (int it = tid; it < NS * MT * 64; it += W * 64) {
        f32x4 p[W];   // (waves without a step left zeros)
#pragma unroll
        for (int w = 0; w < W; ++w) p[w] = red[w * (NS * MT * 64) + it];
        f32x4 s = p[0];
#pragma unroll
        for (int w = 1; w < W; ++w) s += p[w];
        const int l = it & 63, i = (it >> 6) % MT, j = (it >> 6) / MT;
        const int m = m0 + 16 * i + (l & 15);
        const int n = n0 + kSub * j + 4 * (l >> 4);  // C layout: rows 4 (lane / 16) + r
        if (m >= mend || n >= OUT) continue;
        const int nv = min(4, OUT - n);
        float v[4] = {s[0], s[1], s[2], s[3]};
        if (g.bias)
            for (int r = 0; r < nv; ++r) v[r] += g.bias[n + r];
        const int64_t o = (int64_t)m * ywidth + ybase + n;
        if (g.y_dtype == HXQ_F32) {
            float *y = static_cast<float *>(g.y) + o;
            if (g.vec_out && nv == 4) *reinterpret_cast<float4 *>(y) = make_float4(v[0], v[1], v[2], v[3]);
            else for (int r = 0; r < nv; ++r) y[r] = v[r];
        } else {
            uint16_t *y = static_cast<uint16_t *>(g.y) + o;
            uint32_t p0, p1;
            if (g.y_dtype == HXQ_BF16) { p0 = pack16<true>(v[0], v[1]); p1 = pack16<true>(v[2], v[3]); }
            else { p0 = pack16<false>(v[0], v[1]); p1 = pack16<false>(v[2], v[3]); }
            if (g.vec_out && nv == 4) {
                *reinterpret_cast<uint2 *>(y) = make_uint2(p0, p1);
            } else {
                const uint32_t h[4] = {p0 & 0xffffu, p0 >> 16, p1 & 0xffffu, p1 >> 16};
                for (int r = 0; r < nv; ++r) y[r] = static_cast<uint16_t>(h[r]);
            }
        }
    }
}

constexpr int kMaxRows = 64, kMaxRowsF32 = 32;
constexpr int kWideSubs = 3;     // most subtiles per block with uint16 scalar indices (two index loads: registers)
constexpr int kGroupedSubs = 5;  // subtiles per block of a grouped launch (16-row tiles)

// Launches the kernel for XT with mt row tiles and ns subtiles per block.
template <int XT>
int launch_grouped(const Call &c, const Grouped &g, bool aff, int blocks, hipStream_t stream);
template <int XT>
int launch_rows(const Call &c, int format, bool aff, const Plan &p, hipStream_t stream);

}  // namespace rw
}  // namespace hxq
