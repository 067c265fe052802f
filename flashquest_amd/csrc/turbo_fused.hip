// Sparse GQA decode attention over the TurboQuant K3-V3 cache, one workgroup
// of 8 waves per KV group (gfx950).  Semantics of flash_attn_sparse_turbo_fwd
// (src/flashquest/kernel/sparse_turbo_fwd.py:110-251, wrapper 254-346): Q is
// rotated by the normalised WHT, a token's K / V channel value is
// codebook[(msb << 2) | lsb] * scale[token] (msb bit i of byte j is channel
// 8j + i, lsb field i of byte j is channel 4j + i; kv_quant.py:225-279), base-2
// online softmax, O rotated back.
//
// FUSED: the workgroup also scores the group's pages from the un-rotated K's
// page scale/min (K_scale_raw / K_mn_raw, bf16; criticality.py:128-163) and
// selects them, like the INT4 fused decode (one launch per decode step).
// Otherwise the pages come from the workspace lists and splits of a group
// meet in merge_splits_kernel.
//
// Layout: the page loop runs on the matrix cores (attn_turbo_fused_kernel
// below); the wave merge, the inverse rotation of O and the split merge are
// the INT4 kernels' (attn_common.h).
#include "attn_common.h"
#include "fused_common.h"

namespace fq {
namespace {

// The codebook is whole in units of 1e-4 (+-2451, 7560, 13439, 21519; its fp32
// values differ from those by their own rounding), and each value is 256 H + L
// with two int8 digits: byte tables for v_perm, codes 0-3 and 4-7.
constexpr int kTurboInt[8] = {-21519, -13439, -7560, -2451, 2451, 7560, 13439, 21519};
constexpr float kTurboUnit = 1e-4f;
constexpr int turbo_low(int v) { return v - 256 * ((v + 32768 + 128) / 256 - 128); }     // in [-128, 127]
constexpr uint32_t turbo_table(bool high, int first) {
    uint32_t t = 0;
    for (int i = 0; i < 4; ++i) {
        const int v = kTurboInt[first + i], d = high ? (v - turbo_low(v)) / 256 : turbo_low(v);
        t |= (uint32_t)(d & 0xFF) << (8 * i);
    }
    return t;
}
constexpr uint32_t kCodeHi[2] = {turbo_table(true, 0), turbo_table(true, 4)};
constexpr uint32_t kCodeLo[2] = {turbo_table(false, 0), turbo_table(false, 4)};
static_assert(turbo_low(2451) == -109 && turbo_low(-13439) == -127 && turbo_low(21519) == 15, "codebook digits");

constexpr float kFixScale = 8323071.0f;       // 2^23 - 2^16 - 1: |X| <= this has 3 balanced int8 digits
constexpr uint32_t kDigitFlip3 = 0x80808080u;
// Byte I of four values, packed (byte 0 from y0).
template <int I>
FQ_DEV uint32_t byte_of(uint32_t y0, uint32_t y1, uint32_t y2, uint32_t y3) {
    constexpr uint32_t lo = 0x0C0C0000u | ((4u + I) << 8) | I;
    constexpr uint32_t hi = ((4u + I) << 24) | ((uint32_t)I << 16) | 0x0C0Cu;
    return __builtin_amdgcn_perm(y1, y0, lo) | __builtin_amdgcn_perm(y3, y2, hi);
}

struct TurboFusedParams {
    fq_turbo_cache c;
    Int4Cache raw;          // FUSED: ksc / kmn = K_scale_raw / K_mn_raw (bf16), P, D
    QueryArgs q;
    Workspace ws;
    int splits;
    SelectArgs sel;
};

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
// One page as a lane loads it: bytes 16 lane .. + 15 of every KB of its planes
// (k[0] / v[0]: the 64 MSB rows of 16 bytes; k[1], k[2] / v[1], v[2]: the 64 LSB
// rows of 32), and the K and V scale of token `lane` (2-byte loads: rows of any
// token count, and exact at a partial last page).
struct TurboPage {
    uint4 k[3], v[3];
    uint32_t ks, vs;
};

// A wave's page in LDS, as its operands are read (lane = (n16 = lane & 15, lg = lane >> 4)):
//   q.k: K row dwords of token 16 T + n16 (MSB dword lg, LSB dwords 2 lg, 2 lg + 1);
//   p.v: V columns, transposed, of tokens 16 byte + 4 jd + lg: 64 (MSB) / 128 (LSB)
//   bytes of padding per 16 tokens keep the four bytes' rows on different banks.
struct TurboLds {
    uint8_t k[3][1024];
    uint8_t vm[1024 + 3 * 64], vl[2048 + 3 * 128];
};

struct TurboRsrc {
    __amdgpu_buffer_rsrc_t km, kl, ks, vm, vl, vs;
    int km_t, kl_t, vm_t, vl_t, ks_t, vs_t;     // token strides in bytes
};

// Token rows are dense (16-byte MSB, 32-byte LSB rows, 2-byte scales).
FQ_DEV void load_turbo_page(TurboPage& b, const TurboRsrc& r, int lane, int p) {
    const int row = 16 * lane + p * 1024, row2 = 16 * lane + p * 2048, sc = 2 * lane + p * 128;
    b.k[0] = ld128(r.km, row);
    b.k[1] = ld128(r.kl, row2);
    b.k[2] = ld128(r.kl, row2 + 1024);
    b.ks = ld16(r.ks, sc);
    b.v[0] = ld128(r.vm, row);
    b.v[1] = ld128(r.vl, row2);
    b.v[2] = ld128(r.vl, row2 + 1024);
    b.vs = ld16(r.vs, sc);
}
FQ_DEV void stage_turbo_page(TurboLds& s, const TurboPage& b, int lane) {
#pragma unroll
    for (int u = 0; u < 3; ++u) *(uint4*)&s.k[u][16 * lane] = b.k[u];
    *(uint4*)&s.vm[16 * lane + 64 * (lane >> 4)] = b.v[0];
    *(uint4*)&s.vl[16 * lane + 128 * (lane >> 5)] = b.v[1];
    *(uint4*)&s.vl[1024 + 16 * lane + 128 * (2 + (lane >> 5))] = b.v[2];
}
// out[T]: v of lane 16 T + (lane & 15), for every lane.
FQ_DEV void spread_rows(uint32_t v, uint32_t (&out)[4]) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);       // rows 0 1 0 1, rows 2 3 2 3
    const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
    out[0] = a[0]; out[1] = a[1]; out[2] = c[0]; out[3] = c[1];
}

// Transposing LDS reads (ds_read_b64_tr_b8 / _tr_b16).  In each group of 16
// lanes: tr8, lanes 2r and 2r + 1 address the two halves of row r of an 8 x 16 byte
// matrix and lane i gets column i, one byte per row; tr16, lanes 4r .. 4r + 3
// address row r of a 4 x 16 matrix of 16-bit values and lane i gets column i.
typedef int v2i __attribute__((ext_vector_type(2)));
typedef short v4s __attribute__((ext_vector_type(4)));
FQ_DEV uint2 read_tr8(const void* lds) {
    const v2i r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)lds);
    return make_uint2((uint32_t)r[0], (uint32_t)r[1]);
}
FQ_DEV uint2 read_tr16(const void* lds) {
    const v4s r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)lds);
    return __builtin_bit_cast(uint2, r);
}

// Sparse decode attention over the TurboQuant cache on the matrix cores
// (v_mfma_i32_16x16x64_i8): both products contract 24-bit fixed-point values X
// (three balanced int8 digits a2 a1 a0) with the codebook's two digits H L, all
// int32 exact.  Query head r owns rows 4r .. 4r + 3, of weights 2^24, 2^16, 2^8
// and 1: against H the A operand's rows are a2 a1 a0 0, against L they are 0 a2
// a1 a0, into the same accumulator, so a lane ends with its head's four rows of
// one column.  The codebook bytes come from 3-bit codes with one v_perm per
// four codes and digit.
//
// q.k (16 tokens x 64 channels per step): X = q_rot of the head relative to its
// largest |q_rot| (rotated, pre-scaled by sm_scale * log2 e / sqrt(D)), the same
// operands for every page; logit = sum * the token's K scale.
//
// p.v (64 tokens x 16 channels): X = p * V_scale / s_run (at most 1; s_run a
// running bound of the V scales, p relative to the running maximum), so a
// product carries 2^-24 of the largest one; the sums stay integers until a page
// raises a reference, which moves them to fp32 and rescales.  Column n16 of
// channel tile j is channel 8 n16 + j.
//
// A page comes in as six 16-byte row loads and two scales per lane (48 loads of 2 to
// 4 bytes when each operand was gathered from memory) and is staged through LDS:
// K is read back as row dwords, V's columns by transposing reads.
//
// What bounds it is the instruction issue (the codes' selectors and the tables'
// v_perm): with fp16 hi + lo parts on both sides a page took 64 matrix
// instructions, 64 16-byte LDS table reads that conflict and about 720 vector
// instructions; now 32, none and about 600.  28 layers x 32768 tokens, 24 query
// heads on 8, a quarter of the pages, per query head: 137 us before; 129 on int8
// digits, 118 with V and 112 with K and V through LDS (446 MB: 4.0 TB/s).
//
// HCH (FUSED only): head chunks, sel.head_chunks virtual KV heads per cache KV
// head (virtual head h = cache head hk * HC + chunk, NREP query heads each; q,
// outputs and retention follow h, the cache pages and raw metadata hk).
// per_kv_head_sum then scores the summed query of all 2 NREP heads of the
// cache head, so every chunk selects the same pages; the chunks of a cache
// head are mapped to one XCD.
template <int NREP, bool FUSED, bool HCH = false>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_turbo_fused_kernel(TurboFusedParams a) {
    constexpr int D = 128, NW = 8, NT = 512;
    static_assert(NREP <= 4, "query heads per KV head");
    static_assert(!HCH || FUSED, "head chunks run in the fused kernel");
    // a row takes two digit products a token: |A| <= 128 against |H| <= 85 and |L| <= 128
    static_assert((int64_t)kMaxWgPages / NW * 64 * 128 * (85 + 128) < INT32_MAX, "a wave's int32 sums");
    __shared__ SplitLds<D, NREP, NW> s_split;
    __shared__ int s_ent[kMaxWgPages];
    __shared__ float s_qraw[HCH ? 2 * NREP : NREP][D];      // chunk_sum: every head of the cache head
    __shared__ float s_qrot[NREP][D];
    // p.v A digits per wave: [head][0, a2, a1, a0, 0][k-group, XOR head][16 bytes]; the H operand reads rows
    // 1 .. 4 of a head, the L operand rows 0 .. 3
    __shared__ uint32_t s_apv[NW][4][5][4][4];
    __shared__ __attribute__((aligned(16))) TurboLds s_page[NW];      // each wave's current page

    const fq_turbo_cache& c = a.c;
    const QueryArgs& q = a.q;
    const int gy = blockIdx.y, GY = gridDim.y, split = blockIdx.x;
    const int g = (HCH && gridDim.x == 1 && GY % 8 == 0) ? (gy % 8) * (GY / 8) + gy / 8 : gy;
    const int h = g % c.H_kv, b = (g / c.H_kv) % c.B, l = g / (c.H_kv * c.B);
    const int HC = HCH ? a.sel.head_chunks : 1;
    const int hk = HCH ? h / HC : h;
    const bool chunk_sum = HCH && a.sel.mode == FQ_SELECT_PER_KV_HEAD_SUM;
    const int tid = threadIdx.x, L = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
    const int n16 = L & 15, lg = L >> 4;
    const int S = c.S;

    // q (raw basis): element tid of the group's NREP heads.  Branch-free (two
    // 16-bit loads, the high one masked off for 16-bit q types), so the
    // metadata loads below go out before the first wait.
    // chunk_sum: all 2 NREP heads of the cache head (two elements per
    // thread; rows chunk * NREP .. are this workgroup's own)
    const int q_rows = chunk_sum ? 2 * NREP : NREP;
    const int q_row0 = chunk_sum ? (h - hk * HC) * NREP : 0;
    const int64_t qb = l * q.q_s[0] + b * q.q_s[1] + (int64_t)(chunk_sum ? hk * 2 * NREP : h * NREP) * q.q_s[2];
    const int qi = min(tid, q_rows * D - 1);
    const int qi1 = min(tid + NT, q_rows * D - 1);
    const bool q32 = q.q_dtype == FQ_F32;
    const int esz = q32 ? 4 : 2;
    uint32_t hi_mask = (0u - (uint32_t)q32) & 0xFFFF0000u;
    asm volatile("" : "+s"(hi_mask));
    uint32_t ql, qh, ql1 = 0u, qh1 = 0u;
    {
        const char* qc = (const char*)q.q + (qb + (qi >> 7) * q.q_s[2] + (qi & 127) * q.q_s[3]) * esz;
        ql = *(const uint16_t*)qc;
        qh = *(const uint16_t*)(qc + esz - 2);
        if constexpr (HCH) {
            const char* qc1 = (const char*)q.q + (qb + (qi1 >> 7) * q.q_s[2] + (qi1 & 127) * q.q_s[3]) * esz;
            ql1 = *(const uint16_t*)qc1;
            qh1 = *(const uint16_t*)(qc1 + esz - 2);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    float ret_l = 0.f;
    ScoreRegs<NT> sr;
    ScoreRowRegs<NREP, NT> srow;        // kSelectOnly: the group's scores from the scoring launch
    const bool from_scores = FUSED && a.sel.enabled == kSelectOnly;
    const int score_rows = a.sel.mode == FQ_SELECT_PER_KV_HEAD_SUM ? 1 : NREP;
    if constexpr (FUSED) {
        if (chunk_sum)      // uniform: the k of the summed row is the cache head's largest retention
            ret_l = wave_max(a.sel.retention[l * q.ret_ls + hk * 2 * NREP + min(L, 2 * NREP - 1)]);
        else
            ret_l = a.sel.retention[l * q.ret_ls + h * NREP + min(L, NREP - 1)];
        if (from_scores)      // per_kv_head_sum with head chunks: the cache head's one summed row
            scores_load<NREP, NT>(srow, a.ws.scores + (int64_t)(chunk_sum ? g - (h - hk * HC) : g) * NREP * c.P,
                                  score_rows, c.P, tid);
        else score_group_load<bf16, NT>(sr, a.raw, tid, l, b, hk);
    }
    auto q_value = [&](uint32_t lo, uint32_t hi) {
        const uint32_t u = (lo & ~hi_mask) | ((hi << 16) & hi_mask);
        const float fh = f16_bits_to_f(u), fb = bf16_bits_to_f(u);
        return q32 ? __uint_as_float(u) : (q.q_dtype == FQ_BF16 ? fb : fh);
    };
    const float qv_raw = q_value(ql, qh);
    for (int i = tid; i < NW * 4 * 5 * 16; i += NT) (&s_apv[0][0][0][0][0])[i] = 0u;      // the zero rows, and heads past NREP
    if constexpr (HCH) {
        if (tid < q_rows * D) s_qraw[qi >> 7][qi & 127] = qv_raw;
        if (tid + NT < q_rows * D) s_qraw[qi1 >> 7][qi1 & 127] = q_value(ql1, qh1);
    } else if (tid < NREP * D) {
        s_qraw[qi >> 7][qi & 127] = qv_raw;
    }
    __syncthreads();
    // q_rot = WHT(q) / sqrt(D) (Sylvester order), pre-scaled by sm_scale * log2(e);
    // wave r rotates head r (row q_row0 + r of s_qraw)
    if (w < NREP) {
        float v0 = s_qraw[q_row0 + w][L], v1 = s_qraw[q_row0 + w][L + 64];
        wave_hadamard128(v0, v1);
        const float sc = q.qk_scale / sqrtf((float)D);
        s_qrot[w][L] = v0 * sc;
        s_qrot[w][L + 64] = v1 * sc;
    }

    TurboRsrc rs;
    {
        const int64_t bl = l;
        const uint8_t* km = c.k_msb + bl * c.kmsb_strides[0] + b * c.kmsb_strides[1] + hk * c.kmsb_strides[2];
        const uint8_t* kl = c.k_lsb + bl * c.klsb_strides[0] + b * c.klsb_strides[1] + hk * c.klsb_strides[2];
        const uint8_t* vm = c.v_msb + bl * c.vmsb_strides[0] + b * c.vmsb_strides[1] + hk * c.vmsb_strides[2];
        const uint8_t* vl = c.v_lsb + bl * c.vlsb_strides[0] + b * c.vlsb_strides[1] + hk * c.vlsb_strides[2];
        const uint16_t* ks = (const uint16_t*)c.k_scale + bl * c.kst_strides[0] + b * c.kst_strides[1] + hk * c.kst_strides[2];
        const uint16_t* vs = (const uint16_t*)c.v_scale + bl * c.vst_strides[0] + b * c.vst_strides[1] + hk * c.vst_strides[2];
        rs.km_t = (int)c.kmsb_strides[3]; rs.kl_t = (int)c.klsb_strides[3];
        rs.vm_t = (int)c.vmsb_strides[3]; rs.vl_t = (int)c.vlsb_strides[3];
        rs.km = make_rsrc(km, (int64_t)S * rs.km_t);
        rs.kl = make_rsrc(kl, (int64_t)S * rs.kl_t);
        rs.vm = make_rsrc(vm, (int64_t)S * rs.vm_t);
        rs.vl = make_rsrc(vl, (int64_t)S * rs.vl_t);
        rs.ks_t = (int)c.kst_strides[3] * 2; rs.vs_t = (int)c.vst_strides[3] * 2;
        rs.ks = make_rsrc(ks, (int64_t)S * rs.ks_t);
        rs.vs = make_rsrc(vs, (int64_t)S * rs.vs_t);
    }
    auto issue_page = [&](TurboPage& bf, int p) {
        __builtin_amdgcn_sched_barrier(0);
        load_turbo_page(bf, rs, L, p);
        __builtin_amdgcn_sched_barrier(0);
    };
    TurboPage nb;          // the page after the one in LDS
    bool first_issued = false;

    int e0, e1, ent_base = 0;          // this split's entries are s_ent[ent_base ..]
    if constexpr (FUSED) {
        // scores (this workgroup's own, or the scoring launch's), then the
        // selection; every split of a group selects the same list and takes
        // the balanced slice [e0, e1) of it
        __shared__ uint32_t s_key[NREP * 64 * kSelC];
        __shared__ BlockSelectLds s_bsel;
        if (from_scores) scores_to_keys<NREP, NT>(srow, s_key, score_rows, c.P, tid);
        else if (chunk_sum) score_group_regs<bf16, HCH ? 2 * NREP : NREP, NT, true>(sr, s_qraw, s_key, tid, c.P);
        else if (a.sel.mode == FQ_SELECT_PER_KV_HEAD_SUM) score_group_regs<bf16, NREP, NT, true>(sr, s_qraw, s_key, tid, c.P);
        else score_group_regs<bf16, NREP, NT, false>(sr, s_qraw, s_key, tid, c.P);
        const ForcedPages fp = forced_pages(c.P, a.sel.num_sinks, a.sel.window);
        if (S > 0 && split == 0 && w < fp.count) {   // split 0's first entries are the forced pages
            issue_page(nb, fp.page(w));
            first_issued = true;
        }
        __syncthreads();
        const int total = block_select_group<kSelC, NW, NREP>(s_key, c.P, a.sel.mode, ret_l, a.sel.k_max,
                                                              a.sel.num_sinks, a.sel.window, s_ent, s_bsel);
        if (a.sel.mask_out && split == 0)            // uniform: the caller asked for the selection
            block_write_mask<NT, NREP>(s_ent, total, c.P, (uint8_t*)s_key, a.sel.mask_out + (int64_t)g * NREP * c.P,
                                       tid);
        e0 = (int)((int64_t)total * split / a.splits);
        e1 = (int)((int64_t)total * (split + 1) / a.splits);
        ent_base = e0;
    } else {
        const int n_sel = a.ws.n_sel[g];
        e0 = (int)((int64_t)n_sel * split / a.splits);
        e1 = (int)((int64_t)n_sel * (split + 1) / a.splits);
        for (int i = tid; i < e1 - e0; i += NT) s_ent[i] = a.ws.entries[(int64_t)g * c.P + e0 + i];
        __syncthreads();
    }
    const int n_mine = S > 0 && w < e1 - e0 ? (e1 - e0 - w + NW - 1) / NW : 0;

    // q.k A operands: lane (row n16 = 4 r + i, k-group lg); k = 16 lg + 4 jd + byte of
    // step s is channel 32 lg + 8 byte + 4 s + jd.  aqh: digits a2 a1 a0 0 in rows i,
    // aql: 0 a2 a1 a0.  unscale: of head lg, the logits' factor (NaN where the
    // head's query has a NaN or an infinity: those have no digits).
    v4i aqh[2], aql[2];
    float unscale;
    {
        const int r = min(n16 >> 2, NREP - 1), i = n16 & 3;
        float am = 0.f, bad = 0.f;
        for (int d = lg; d < D; d += 4) {                  // 4 lanes per row
            am = fmaxf(am, fabsf(s_qrot[r][d]));
            bad = fmaf(s_qrot[r][d], 0.f, bad);
        }
        am = fmaxf(am, __shfl_xor(am, 16, 64));
        am = fmaxf(am, __shfl_xor(am, 32, 64));
        bad += __shfl_xor(bad, 16, 64);
        bad += __shfl_xor(bad, 32, 64);
        const float inv = am > 0.f ? kFixScale / am : 0.f;
        const float un = fmaf(am, kTurboUnit / kFixScale, bad);
        unscale = __shfl(un, 4 * min(lg, NREP - 1), 64);
        const bool mine = (n16 >> 2) < NREP;
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int jd = 0; jd < 4; ++jd) {
                uint32_t Y[4];
#pragma unroll
                for (int by = 0; by < 4; ++by)        // X + 0x808080, rounded by the fp32 add itself
                    Y[by] = (uint32_t)fmaf(s_qrot[r][32 * lg + 8 * by + 4 * st + jd], inv, 8421504.0f);
                const uint32_t a2 = byte_of<2>(Y[0], Y[1], Y[2], Y[3]) ^ kDigitFlip3;
                const uint32_t a1 = byte_of<1>(Y[0], Y[1], Y[2], Y[3]) ^ kDigitFlip3;
                const uint32_t a0 = byte_of<0>(Y[0], Y[1], Y[2], Y[3]) ^ kDigitFlip3;
                const uint32_t hi = i == 0 ? a2 : i == 1 ? a1 : i == 2 ? a0 : 0u;
                const uint32_t lo = i == 0 ? 0u : i == 1 ? a2 : i == 2 ? a1 : a0;
                aqh[st][jd] = mine ? (int)hi : 0;
                aql[st][jd] = mine ? (int)lo : 0;
            }
    }

    auto entry_of = [&](int k) { return __builtin_amdgcn_readfirstlane(s_ent[ent_base + w + NW * k]); };

    float m_run[NREP];
#pragma unroll
    for (int r = 0; r < NREP; ++r) m_run[r] = -INFINITY;
    float s_run = 0.f, fix_s = 0.f;          // running bound of the V scales, kFixScale / s_run
    float m_lane = 0.f;                      // m_run[lg], or 0 while head lg has no logit yet
    v4i pacc[8];                             // [channel tile]: head lg's digit rows since the references last moved
    float facc[8];                           // and what came before
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        pacc[t] = (v4i){0, 0, 0, 0};
        facc[t] = 0.f;
    }
    float l_acc = 0.f, bad_v = 0.f;          // bad_v: NaN once a p * V_scale is one or infinite (no digits either)
    auto& W = s_apv[w];
    auto& WP = s_page[w];
    // the lane's addresses: K rows (tile T 16 tokens on); the transposed reads' V rows: MSB read u, row r = 0..7 is
    // token 16 (r & 3) + 4 (2 u + (r >> 2)) + lg, LSB read jd, row r = 0..3 token 16 r + 4 jd + lg
    const uint8_t* const kmp = &WP.k[0][0] + 16 * n16 + 4 * lg;
    const uint8_t* const klp = &WP.k[1][0] + 32 * n16 + 8 * lg;
    const int trr = (n16 >> 1) & 3;
    const uint8_t* const trm = WP.vm + (16 * trr + 4 * (n16 >> 3) + lg) * 16 + 64 * trr + 8 * (n16 & 1);
    const uint8_t* const trl = WP.vl + (16 * (n16 >> 2) + lg) * 32 + 128 * (n16 >> 2) + 8 * (n16 & 3);

    // the idle partner-wave priority rule of the INT4 fused decode: two waves
    // share a SIMD; the one with more pages left (on a tie the younger) takes
    // the higher priority
    __shared__ int s_left[NW];
    auto balance = [&](int k) {
        s_left[w] = n_mine - k;
        const int other = __builtin_amdgcn_readfirstlane(s_left[w ^ 4]);
        if (n_mine - k > other || (n_mine - k == other && w >= 4)) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
    };

    auto compute = [&](uint32_t scales, int k) {       // scales: K and V scale of token `lane`
        balance(k);
        const int ent = entry_of(k);
        const int p = ent & 0xFFFF, qm = ent >> 16;
        const int tok0 = p * 64;
        uint32_t sc[4];
        spread_rows(scales, sc);
        // ---- q.k: tile T is tokens 16 T + n16
        float lg4[4], mp = -INFINITY;
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            // LSB bytes of channels 8 byte + 0..3 / 4..7
            const uint2 kl = *(const uint2*)(klp + 512 * T);
            const uint32_t km = *(const uint32_t*)(kmp + 256 * T);
            const uint32_t le = __builtin_amdgcn_perm(kl.y, kl.x, 0x06040200u);
            const uint32_t lo = __builtin_amdgcn_perm(kl.y, kl.x, 0x07050301u);
            v4i acc = {0, 0, 0, 0};
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                v4i bh, bl;
#pragma unroll
                for (int jd = 0; jd < 4; ++jd) {
                    const int i = 4 * st + jd;                 // byte: channel 8 byte + i, its MSB at bit i
                    const uint32_t m = i >= 2 ? km >> (i - 2) : km << (2 - i);
                    const uint32_t sel = (m & 0x04040404u) | (((st ? lo : le) >> (2 * jd)) & 0x03030303u);
                    bh[jd] = (int)__builtin_amdgcn_perm(kCodeHi[1], kCodeHi[0], sel);
                    bl[jd] = (int)__builtin_amdgcn_perm(kCodeLo[1], kCodeLo[0], sel);
                }
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(aqh[st], bh, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(aql[st], bl, acc, 0, 0, 0);
            }
            const float lgt = digit_rows(acc) * unscale * bf16_bits_to_f(sc[T] & 0xFFFFu);
            const bool ok = lg < NREP && ((qm >> lg) & 1) && tok0 + 16 * T + n16 < S;
            lg4[T] = ok ? lgt : -INFINITY;
            mp = fmaxf(mp, lg4[T]);
        }
        // ---- page maxima, running references
        float vs_t[4], sp = 0.f;
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            vs_t[T] = __uint_as_float(sc[T] & 0xFFFF0000u);
            sp = fmaxf(sp, vs_t[T]);
        }
        mp = row16_max(mp);
        sp = lane_value(row16_max(sp), 0);
        bool grow = sp > s_run;
        float mp_r[NREP];
#pragma unroll
        for (int r = 0; r < NREP; ++r) {
            mp_r[r] = lane_value(mp, 16 * r);
            grow |= mp_r[r] > m_run[r];
        }
        if (grow) {      // wave-uniform
            float am[NREP];
#pragma unroll
            for (int r = 0; r < NREP; ++r) {
                const float mn = fmaxf(mp_r[r], m_run[r]);
                am[r] = mn == m_run[r] ? 1.0f : exp2_fast(m_run[r] - mn);
                m_run[r] = mn;
            }
            const float sn = fmaxf(sp, s_run);
            const float as = sn > 0.f ? s_run / sn : 1.0f;
            s_run = sn;
            fix_s = sn > 0.f ? kFixScale / sn : 0.f;
            float am_lg = am[0], ml = m_run[0];
#pragma unroll
            for (int r = 1; r < NREP; ++r) {
                am_lg = lg == r ? am[r] : am_lg;
                ml = lg == r ? m_run[r] : ml;
            }
            m_lane = ml == -INFINITY ? 0.f : ml;
            l_acc *= am_lg;
            const float f = am_lg * as;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                facc[t] = (facc[t] + digit_rows(pacc[t])) * f;
                pacc[t] = (v4i){0, 0, 0, 0};
            }
        }
        // ---- p.v A: the digits of p * V_scale / s_run; operand k = 16 kg + 4 jd + byte
        // is token 16 byte + 4 jd + kg, so the lane's four tokens are one dword
        uint32_t Y[4];
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            const float pr = exp2_fast(lg4[T] - m_lane);
            l_acc += pr;
            const float x = pr * vs_t[T];
            bad_v = fmaf(x, 0.f, bad_v);
            Y[T] = (uint32_t)fmaf(x, fix_s, 8421504.0f);
        }
        if (lg < NREP) {
            uint32_t* dst = &W[lg][1][(n16 & 3) ^ lg][n16 >> 2];
            dst[0] = byte_of<2>(Y[0], Y[1], Y[2], Y[3]) ^ kDigitFlip3;
            dst[16] = byte_of<1>(Y[0], Y[1], Y[2], Y[3]) ^ kDigitFlip3;
            dst[32] = byte_of<0>(Y[0], Y[1], Y[2], Y[3]) ^ kDigitFlip3;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int hr = n16 >> 2;
        const v4i aph = *(const v4i*)&W[hr][(n16 & 3) + 1][lg ^ hr][0];
        const v4i apl = *(const v4i*)&W[hr][n16 & 3][lg ^ hr][0];
        // ---- p.v B: codes of channel 8 n16 + j, dword jd = tokens 16 byte + 4 jd + lg
        uint32_t m4[4], ll[4], lh[4];        // the 4 tokens' MSB bytes; LSB fields of channels 0-3 / 4-7
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint2 m = read_tr8(trm + 128 * u);
            m4[2 * u] = m.x;
            m4[2 * u + 1] = m.y;
        }
#pragma unroll
        for (int jd = 0; jd < 4; ++jd) {
            const uint2 x = read_tr16(trl + 128 * jd);      // two tokens' LSB halves a dword
            ll[jd] = __builtin_amdgcn_perm(x.y, x.x, 0x06040200u);
            lh[jd] = __builtin_amdgcn_perm(x.y, x.x, 0x07050301u);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v4i bh, bl;
#pragma unroll
            for (int jd = 0; jd < 4; ++jd) {
                const uint32_t m = j >= 2 ? m4[jd] >> (j - 2) : m4[jd] << (2 - j);
                const uint32_t sel = (m & 0x04040404u) | (((j < 4 ? ll[jd] : lh[jd]) >> (2 * (j & 3))) & 0x03030303u);
                bh[jd] = (int)__builtin_amdgcn_perm(kCodeHi[1], kCodeHi[0], sel);
                bl[jd] = (int)__builtin_amdgcn_perm(kCodeLo[1], kCodeLo[0], sel);
            }
            pacc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(aph, bh, pacc[j], 0, 0, 0);
            pacc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(apl, bl, pacc[j], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    };

    // A page is loaded in whole rows (8 loads), one page ahead, and goes to LDS
    // when the page before it is done; a wave's LDS accesses are in order, so its one
    // page buffer needs no barrier.
    {
        s_left[w] = n_mine;
        if (!first_issued) issue_page(nb, n_mine > 0 ? entry_of(0) & 0xFFFF : 0);
        for (int k = 0; k < n_mine; ++k) {
            stage_turbo_page(WP, nb, L);
            const uint32_t scales = (nb.ks & 0xFFFFu) | (nb.vs << 16);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            issue_page(nb, entry_of(min(k + 1, n_mine - 1)) & 0xFFFF);
            compute(scales, k);
        }
        __builtin_amdgcn_s_setprio(0);
    }

    // ---- wave state -> LDS: head lg's sums (over its lane group's 16 token columns)
    // and its outputs of channels 8 n16 + j, in units of s_run / kFixScale * 1e-4
    l_acc = row_sum<16>(l_acc);
    bad_v = row_sum<16>(bad_v);
    const float pv_unscale = s_run * (kTurboUnit / kFixScale);
    if (lg < NREP) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            s_split.acc[w][lg][8 * n16 + j] = fmaf(facc[j] + digit_rows(pacc[j]), pv_unscale, bad_v);
        if (n16 == 0) {
            float m = m_run[0];
#pragma unroll
            for (int r = 1; r < NREP; ++r) m = lg == r ? m_run[r] : m;
            s_split.m[w][lg] = m;
            s_split.l[w][lg] = l_acc;
        }
    }
    __syncthreads();
    merge_waves_and_store<D, NREP, true, NW>(s_split, q, a.ws, g, l, b, h, split, a.splits > 1);
}

template <bool FUSED>
hipError_t launch_turbo_fused_nrep(const TurboFusedParams& a, dim3 grid, hipStream_t st) {
    switch (a.q.nrep) {
#define FQ_CASE(N)                                                                                          \
    case N:                                                                                                 \
        timer_before_launch(st);                                                                            \
        if (FUSED && (N == 3 || N == 4) && a.sel.head_chunks > 1)                                           \
            hipLaunchKernelGGL((attn_turbo_fused_kernel<N, FUSED, FUSED && N >= 3>), grid, dim3(512), 0, st, a); \
        else                                                                                                \
            hipLaunchKernelGGL((attn_turbo_fused_kernel<N, FUSED>), grid, dim3(512), 0, st, a);             \
        timer_after_launch(st);                                                                             \
        if (a.splits > 1)                                                                                   \
            launch_split_merge<N, true>(a.q, a.ws, a.c.H_kv, a.c.B, grid.y, a.splits, TailArgs{}, st);         \
        break;
        FQ_CASE(1) FQ_CASE(2) FQ_CASE(3) FQ_CASE(4)
#undef FQ_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

bool turbo_fused_supported(const fq_turbo_cache& c, const QueryArgs& q) {
    if (c.D != 128 || c.page_size != 64 || q.nrep > 4 || c.P > kMaxWgPages) return false;
    if (c.kmsb_strides[4] != 1 || c.klsb_strides[4] != 1 || c.vmsb_strides[4] != 1 || c.vlsb_strides[4] != 1)
        return false;
    // dense token rows (16-byte MSB, 32-byte LSB rows, 2-byte scales), read in
    // words of 4 bytes or more
    if (c.kmsb_strides[3] != 16 || c.klsb_strides[3] != 32 || c.vmsb_strides[3] != 16 || c.vlsb_strides[3] != 32)
        return false;
    if (c.kst_strides[3] != 1 || c.vst_strides[3] != 1) return false;
    for (int i = 0; i < 3; ++i) {
        if (c.kmsb_strides[i] % 4 || c.klsb_strides[i] % 4 || c.vmsb_strides[i] % 4 || c.vlsb_strides[i] % 4) return false;
    }
    if (((uintptr_t)c.k_msb | (uintptr_t)c.k_lsb | (uintptr_t)c.v_msb | (uintptr_t)c.v_lsb) & 3) return false;
    if (((uintptr_t)c.k_scale | (uintptr_t)c.v_scale) & 1) return false;
    return true;
}

// Pages from the workspace lists (splits per group chosen like the INT4
// matrix-core kernel); with sel = kScoreSelect and raw, scored and selected in
// the kernel (one workgroup per group); with sel = kSelectOnly, selected in the
// kernel from the scores a scoring launch left in the workspace, each group
// split over workgroups like the INT4 kernel's split steps.
hipError_t launch_attn_turbo_fused(const fq_turbo_cache& c, const Int4Cache* raw, const QueryArgs& q,
                                   const Workspace& ws, int max_entries, const SelectArgs* sel, hipStream_t st) {
    TurboFusedParams a{};
    a.c = c; a.q = q; a.ws = ws;
    const int groups = c.L * c.B * c.H_kv;
    if (sel && sel->enabled == kScoreSelect && raw) {
        a.raw = *raw;
        a.sel = *sel;
        a.splits = 1;
        return launch_turbo_fused_nrep<true>(a, dim3(1, groups), st);
    }
    if (sel && sel->enabled == kSelectOnly) {
        if (c.P > 64 * kSelC) return hipErrorInvalidValue;
        a.sel = *sel;
        int s = (256 + groups - 1) / std::max(groups, 1);
        s = std::min(s, (max_entries + 7) / 8);
        a.splits = std::max(1, std::min(s, ws.s_max));
        return launch_turbo_fused_nrep<true>(a, dim3(a.splits, groups), st);
    }
    int s = groups >= 192 ? 1 : (512 + groups - 1) / groups;
    s = std::min(s, (max_entries + 7) / 8);
    s = std::max(s, (max_entries + kMaxWgPages - 1) / kMaxWgPages);
    a.splits = std::max(1, std::min(s, ws.s_max));
    return launch_turbo_fused_nrep<false>(a, dim3(a.splits, groups), st);
}

}  // namespace fq
