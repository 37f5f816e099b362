/* prefill.hip — the expert half of the MoE layer for many tokens (a prefill chunk) as MFMA
 * grouped GEMMs on gfx950.
 *
 * Reference: engine/blocks/qwen3_moe.c:199-222 runs, for each token in turn, its 8 experts'
 * gate/up GEMVs (matmul_wx_q4 / _q8, engine/kernels/kernels.c:368-396, :514-540), SwiGLU
 * (kernels.c:416) and the down GEMV, and adds wt_j * y_j into the token's output. With
 * hundreds of tokens the same expert serves tens of them, so here each expert's tokens (the
 * groups the routing step formed) are one dense product:
 *   G = X_e Wg_e^T, U = X_e Wu_e^T, H = silu(G) * U          k_pf_gemm<ENC, true>
 *   Y = H Wd_e^T                                              k_pf_gemm<ENC, false>
 *   out[t] (+)= sum_j wt_j Y[t, j]  (slot order j = 0..K-1)   k_pair_combine
 *
 * Numerics. A Q4_0 / Q8_0 weight is q * d with q a small integer (Q4: -8..7, Q8: -127..127),
 * exact in f16, and d the block's fp16 scale. Each 32-wide step of k is one block: the MFMA
 * takes the exact q values as its B operand and the activations as its A operand, and the
 * step's product is scaled by d in fp32 and added to the fp32 accumulator, so no weight is
 * ever rounded. Activations are split x = hi + lo with hi = f16(x) and lo = f16(x - hi) and
 * both halves go through the MFMA (22 significant bits), so the products differ from the fp32
 * CPU GEMVs by roughly fp32 rounding, not by f16's.
 *
 * MFMA v_mfma_f32_16x16x32_f16 operand layout (checked on the device): lane l holds
 * A[l%16][8(l/16) + j] and B[8(l/16) + j][l%16] for j = 0..7, and D[4(l/16) + i][l%16] for
 * i = 0..3. A block's 32 elements map to k-slot s = element s: a Q4 lane group g takes the low
 * (g < 2) or high (g >= 2) nibbles of payload bytes 8(g%2)..8(g%2)+7, which hold elements
 * 8g..8g+7 (byte i holds elements i and i+16).
 *
 * Work decomposition. A chunk is up to 64 tokens of one expert group (an expert with 150
 * tokens is three chunks); a workgroup of 4 wavefronts computes 128 rows of each of its
 * matrices for one chunk (gate/up: 128 rows of Wg and the same rows of Wu, so SwiGLU pairs
 * are in one lane; down: 128 rows of Wd), each wavefront 32 rows for every non-empty token
 * tile of 16 (a chunk of 20 tokens costs 2 tiles, not 4). Calls whose experts have few tokens
 * (cpg_prefill_chunk) take chunks of one token tile and use variants with 64 gate/up rows per
 * workgroup (PF_SMALL_RW_GU): there the VALU weight conversion, not the MFMAs, sets each
 * wavefront's pace, and twice the workgroups spread it over the CUs. The activations are split into
 * hi/lo f16 planes once per call (k_split_planes for xn; the gate/up epilogue writes h split).
 * Both operands reach the MFMAs through a ring of stages in LDS filled by direct
 * global-to-LDS loads (k_pf_gemm; k_dense for the dense projections).
 */
#include "cpg_internal.h"
#include "cpg_gemv.h"
#include "cpg_mfma.h"
#include <type_traits>

/* ---------------------------------------------------------------- chunk list */

/* One wavefront: the chunk list over the groups the routing step formed (pf_chunk_list), for
   routing steps that do not form it themselves; lane t takes groups 4t..4t+3 (E <= 256). */
__global__ __launch_bounds__(64) void k_chunks(const int *__restrict__ grp_cnt, int E, int ch,
                                               int max_chunks, int *__restrict__ chunk_grp,
                                               int *__restrict__ chunk_m0) {
    int cnt[4], grp[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        grp[j] = 4 * threadIdx.x + j;
        cnt[j] = grp[j] < E ? grp_cnt[grp[j]] : 0;
    }
    pf_chunk_list(cnt, grp, ch, max_chunks, chunk_grp, chunk_m0);
}

/* grid rows, 256 threads: rows of n floats (n % 4 == 0) as planes */
template <int FMT>
__global__ __launch_bounds__(256) void k_split_planes(const float *__restrict__ x, int n,
                                                      cpg_planes pl) {
    const size_t r = blockIdx.x;
    for (int c = threadIdx.x; c < n / 4; c += 256) {
        const float4 v = *(const float4 *)(x + r * n + 4 * c);
        const float o[4] = {v.x, v.y, v.z, v.w};
        planes_put<FMT>(pl, r * n + 4 * c, o);
    }
}

/* ---------------------------------------------------------------- expert GEMMs */

/* The expert GEMMs stream both operands through a ring of P stages in LDS, filled by direct
   global-to-LDS loads (global_load_lds_dwordx4: 16 bytes per lane, a wavefront's 64 lanes
   into 1 KiB of consecutive LDS), so loads in flight hold no registers and a stage is never
   copied through them. A stage is KB blocks of 32 of the k range:
     A planes     the chunk's 16 * TT activation rows, 32 * KB numbers each (64 * KB bytes per
                  token and plane, NA planes; a wavefront's 1 KiB is 16 / KB rows), rows past the
                  chunk repeating its last; 16-byte piece c of row r sits at piece apos(r, c) of its
                  row, so that the 16 rows that one MFMA operand read touches fall in distinct
                  LDS banks;
     W            NSEG 64-row segments of weight payload (the row-tiled layout keeps a
                  segment's block contiguous: 64 * PB bytes);
     Sc           their fp16 scales, 128 bytes per segment and block.
   A wavefront issues the same number of loads in every stage (Q, or Q - QA where its token tile
   is empty), so "stage s has landed" is that number times P - 2 or fewer in flight, for each
   wavefront, followed by a barrier for the others' loads. The
   barrier is s_barrier alone: __syncthreads() would wait for every load in flight. The
   workgroup (4 wavefronts) computes RW rows of each of its matrices for the chunk; a
   wavefront RW/4 rows of each (RW 128, GU: gate rows, up rows: four 16-row B tiles; down: two).
   KG > 1 (one token tile): KG groups of four wavefronts, each taking KB / KG blocks of every
   stage for all the rows; group 0 adds the groups' sums in order at the end. SUMS = 2 gives one
   group's sums the order of two groups: stages of the blocks that group 0 and group 1 would take
   in turn, into a sum each (an even number of stages). */
#define PF_NT 256
/* chunks of one token tile: rows of each matrix per workgroup (gate/up, down; measured at 16 tokens
   with rings of 4, gate/up, down us: 128 rows 38.4, 16.6; 64 rows 29.3, 20.1). Up to PF_FEW_PAIRS
   pairs there are at most a few workgroups per CU and the length of each one's chain of stages
   counts: eight wavefronts in two groups, each taking half the blocks of a stage of four, in a ring
   of two (us per layer with the routing, against four wavefronts and a ring of three: 2 tokens Q4_0
   33.6, 40.2; 4 tokens 42.3, 45.4, Q8_0 48.1, 48.8; 8 tokens 56.3, 56.8; four groups and stages of
   eight: 4 tokens 41.2, Q8_0 61.5). More pairs: four wavefronts and stages of two blocks. There a
   ring of two lets eight workgroups share a CU, where the weight conversion (Q4_0 with many experts)
   or nothing but latency (Q8_0 with few) sets the pace; a ring of three keeps more in flight where
   the loads do.
   Up to 16 tokens the one group sums in the order of two (SUMS = 2), so that a token's bits are the
   same in every batch of 2 to 16; its 78 registers leave six workgroups per CU, as many as the LDS
   of a ring of three does (Q4_0), or of two (Q8_0). Ring of two, three, with one sum: Q4_0 10
   tokens 60.0, 58.7, 16 skewed 58.4, 58.4; Q8_0 73.5, 76.6 and 69.2, 75.5; with two sums, as
   chosen, Q4_0 60.6 and 58.3, Q8_0 74.2 and 69.7.
   From 17 tokens, rings of two and three: Q4_0 20 tokens 101, 103, 45 tokens 117, 121, 96 tokens
   120, 126, 128 tokens 123, 130, skewed 137, 133, and with more than 8 tokens per expert on average
   160 tokens 138, 134, 176 tokens 140, 137, skewed 153, 150; Q8_0 20 tokens 137, 138, skewed 100,
   107, 32 tokens 164, 151, 45 tokens 167, 155, 96 skewed 165, 156, 176 tokens 183, 182 */
#define PF_SMALL_RW_GU 64
#define PF_SMALL_RW_DN 128
#define PF_FEW_PAIRS 64
#define PF_RING_Q4 128      /* pairs from which Q4_0 takes the ring of two, up to 8 tokens per expert */
#define PF_RING_Q8 160      /* pairs up to which Q8_0 does */
#define PF_SUM 4            /* pf_loop: stages whose sums are taken together, one token tile */
#define R_Q_FITS(q, p) ((q) * ((p) - 2) < 64)   /* the stage wait's vmcnt fits its field */

template <int ENC, bool GU, int TT_ = PF_CHUNK / 16, int P_ = 2, int RW_ = 128, int KB_ = 2, int KG_ = 1,
          int FMT_ = CPG_PL_F16, int SUMS_ = 1>
struct PfRing {
    static constexpr int ENCODING = ENC;
    static constexpr bool GATE_UP = GU;
    static constexpr int TT = TT_;                            /* token tiles of 16 at most */
    static constexpr int KB = KB_;                            /* blocks of 32 per stage */
    static constexpr int KG = KG_;                            /* groups of 4 wavefronts */
    static constexpr int FMT = FMT_;                          /* the activations' planes */
    static constexpr int NA = FMT_ == CPG_PL_BF16 ? 3 : 2;
    static constexpr int SUMS = SUMS_;                        /* sums, a stage in turn each */
    static constexpr int NT = 256 * KG_;                      /* threads */
    static constexpr int KBW = KB_ / KG_;                     /* blocks of a stage per group */
    static constexpr int AI = KG_ == 1 ? KB_ : 1;             /* A loads of each plane per wave */
    static constexpr int PB = ENC == CPG_ENC_Q4 ? 16 : 32;   /* payload bytes per row-block */
    static constexpr int RW = RW_;                            /* rows of each matrix */
    static constexpr int TPM = RW / 64;                       /* B tiles per matrix per wave */
    static constexpr int NSEG = GU ? 2 * TPM : TPM;           /* 64-row weight segments */
    static constexpr int NBT = NSEG;                          /* B tiles per wavefront */
    static constexpr int PP = 4 * KB;                         /* 16-byte pieces per A row */
    static constexpr int A_BYTES = TT * 16 * 32 * KB * 2;     /* one activation plane */
    static constexpr int W_BYTES = NSEG * KB * 64 * PB;
    static constexpr int S_BYTES = NSEG * KB * 128;
    static constexpr int STAGE = NA * A_BYTES + W_BYTES + S_BYTES;
    static constexpr int WB = W_BYTES / (4 * KG);             /* weight bytes per wavefront */
    static constexpr int WI = (WB + 1023) / 1024;             /* their loads */
    static constexpr int SB = S_BYTES / (4 * KG);             /* scale bytes per wavefront */
    static constexpr int QA = KG == 1 ? NA * KB : 1;          /* A loads per stage per wavefront */
    static constexpr int Q = QA + WI + 1;                     /* loads per stage per wavefront */
    /* ring depth: chunks of up to 64 tokens (TT = 4) use 2, the next stage loading while
       this one is computed. Stages of two blocks with two slots (37-52 KiB) let three
       workgroups share a CU (the register limit) and halve the barriers of one-block stages;
       measured: gate/up 134 us with one-block stages in three slots, 144 with two-block
       stages in three slots (two workgroups per CU), 125 with two in two; deeper rings were
       slower still, as fewer workgroups then hide each other's barriers and LDS latency.
       Chunks of one token tile: PF_RING_Q4, PF_RING_Q8. */
    static constexpr int P = P_;
    static_assert(RW % 64 == 0 && P >= 2 && WB % 16 == 0 && SB % 16 == 0 && SB <= 1024 && PP <= 16 &&
                      TT >= 1 && TT <= PF_CHUNK / 16 && R_Q_FITS(NA * KB + WI + 1, P) &&
                      KB % KG == 0 && (KG == 1 || (TT == 1 && NA * KB == 4 * KG)) &&
                      (SUMS == 1 || (TT == 1 && KG == 1)),
                  "ring geometry");
    /* the position of logical piece c of A row r: rows 16 * 4 / PP apart share banks, so the
       16 rows of an MFMA operand read land in distinct banks */
    __device__ static int apos(int r, int c) { return c ^ ((r / (16 / PP)) % PP); }
};

/* One lane's B operand of one block as exact f16 integers q, in natural k order: the nibble
   mask (Q4, after a shift to the lane group's nibbles) or nothing (Q8) leaves each byte u, a
   byte permute puts bytes 2i, 2i+1 under 0x64 (the f16 1024 + u), and the bias 1024 + 8 (Q4)
   or 1024 + 128 (Q8) is subtracted exactly: 12 instructions for Q4's 8 weights. */
template <int ENC>
__device__ static inline half8_t weight_q(uint2 pw, int g) {
    uint32_t src[2] = {pw.x, pw.y};
    if (ENC == CPG_ENC_Q4) {
        const int sh = (g >> 1) * 4;
        src[0] = (src[0] >> sh) & 0x0F0F0F0Fu;
        src[1] = (src[1] >> sh) & 0x0F0F0F0Fu;
    }
    const _Float16 bias = ENC == CPG_ENC_Q4 ? (_Float16)1032.0f : (_Float16)1152.0f;
    const half2_t bb = {bias, bias};
    half8_t q;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t p = __builtin_amdgcn_perm(0x64646464u, src[i >> 1],
                                                 (i & 1) ? 0x07030702u : 0x07010700u);
        const half2_t v = __builtin_bit_cast(half2_t, p) - bb;
        q[2 * i] = v.x;
        q[2 * i + 1] = v.y;
    }
    return q;
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

/* The same weights as exact bf16 integers, Q4's 16 times larger (the caller scales by 2^-4): bytes
   with their bias turned into a sign (Q4: the nibble in the byte's upper half), converted as
   signed integers of at most 8 significant bits, whose fp32 upper halves are the bf16 numbers. */
template <int ENC> __device__ static inline bf16x8_t weight_q_bf16(uint2 pw, int g) {
    uint32_t src[2] = {pw.x, pw.y};
    if (ENC == CPG_ENC_Q4) {
        const int sh = 4 - (g >> 1) * 4;
        src[0] = (src[0] << sh) & 0xF0F0F0F0u;
        src[1] = (src[1] << sh) & 0xF0F0F0F0u;
    }
    uint4 q;
    uint32_t *o = (uint32_t *)&q;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t s = src[i >> 1] ^ 0x80808080u;
        const float x = (float)(int8_t)(s >> (16 * (i & 1))), y = (float)(int8_t)(s >> (16 * (i & 1) + 8));
        o[i] = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
    }
    return __builtin_bit_cast(bf16x8_t, q);
}

/* the k loop of one chunk for NMT token tiles: per block, t = A_hi[mt] . q[n] + A_lo[mt] . q[n]
   (two MFMAs, the second accumulating onto the first) and acc[n][mt] += d[n] * t in fp32,
   blocks in order. Measured against the B operand w = q * d as an exact f16 pair hi + lo
   (three MFMAs accumulating across blocks, 22 instructions per lane to form hi and lo from
   a block's 8 weights, against 12 for q here plus 4 fused multiply-adds per token tile):
   gate/up 112.7 -> 103.5 us, down 60.2 -> 57.6 us at 512 tokens.
   CPG_PL_F16UP: the lo plane is 2^11 times larger, and is multiplied by q * 2^-11, exact in f16:
   four more instructions per B tile and block. CPG_PL_BF16: the smallest plane's product first
   (weight_q_bf16).
   x: the first plane at the chunk's first token and block, the others xs elements apart. */
template <class R, int NMT>
__device__ static void pf_loop(uint8_t *ring, int S, const uint16_t *x, size_t xs,
                               const uint32_t (&aoff)[R::AI], const uint8_t *wsrc,
                               const uint8_t *ssrc, f32x4_t (*acc)[R::TT]) {
    static_assert(NMT <= R::TT, "token tiles");
    constexpr int ENC = R::ENCODING;
    constexpr int KB = R::KB;
    const int l = threadIdx.x & 63, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   /* wavefront-uniform */
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const void __attribute__((address_space(3))) *)ring);
    /* the next stage to load: its sources (scalar pointers; a lane's part is a 32-bit offset) and
       its slot. Past the end: the last stage again, into a free slot. */
    const int w4 = w & 3, kg = w >> 2;           /* the wavefront of its group, the group */
    const uint8_t *pa[R::NA], *pw = uniform_ptr(wsrc), *ps = uniform_ptr(ssrc);
#pragma unroll
    for (int p = 0; p < R::NA; p++) pa[p] = uniform_ptr(x + (R::KG > 1 ? w / R::KB : p) * xs);
    int left = S - 1;
    uint32_t put = 0;
    auto issue = [&]() __attribute__((always_inline)) {
        const uint32_t dst = lds0 + put;
        if constexpr (R::KG > 1) {      /* one KiB of one plane per wavefront */
            lds_dma16(pa[0], aoff[0], dst + 1024 * w);
        } else if (w < NMT) {           /* empty token tiles are not loaded */
#pragma unroll
            for (int i = 0; i < KB; i++)
#pragma unroll
                for (int p = 0; p < R::NA; p++)
                    lds_dma16(pa[p], aoff[i], dst + p * R::A_BYTES + 1024 * (KB * w + i));
        }
#pragma unroll
        for (int i = 0; i < R::WI; i++)
            if (R::WB >= 1024 * (i + 1) || l * 16 < R::WB - 1024 * i)
                lds_dma16(pw, 1024 * i + 16 * l, dst + R::NA * R::A_BYTES + w * R::WB + 1024 * i);
        if (l * 16 < R::SB)
            lds_dma16(ps, 16 * l, dst + R::NA * R::A_BYTES + R::W_BYTES + w * R::SB);
        const uint32_t on = left > 0;
        left--;
#pragma unroll
        for (int p = 0; p < R::NA; p++) pa[p] += on * (64 * KB);
        pw += on * (KB * 64 * R::PB);
        ps += on * (128 * KB);
        put = put + R::STAGE == R::P * R::STAGE ? 0 : put + R::STAGE;
    };
    /* this lane's B rows: segment and row within it, per tile */
    int boff[R::NBT], soff[R::NBT];
#pragma unroll
    for (int n = 0; n < R::NBT; n++) {
        /* tile n: matrix n / TPM (GU: gate, then up), rows RW/4 * w + 16 * (n % TPM) of it;
           the workgroup's RW rows of a matrix are its segments TPM * matrix .. */
        const int r = R::RW * (n / R::TPM) + R::RW / 4 * w4 + 16 * (n % R::TPM) + (l & 15);
        const int seg = r >> 6, rs = r & 63;
        boff[n] = (seg * KB * 64 + rs) * R::PB + (ENC == CPG_ENC_Q4 ? 8 * (g & 1) : 8 * g);
        soff[n] = (seg * KB * 64 + rs) * 2;
    }
    /* one token tile: the sums are taken PF_SUM stages at a time and added up, which takes a fifth
       off the error of one chain over all blocks (a layer at 16 tokens 3.5e-7 -> 2.8e-7 against 64
       bits; more tiles have no registers for it) */
    constexpr bool PARTS = R::TT == 1;
    constexpr int NS = R::SUMS;
    f32x4_t tot[PARTS ? NS : 1][PARTS ? R::NBT : 1], odd[R::NBT][R::TT];
    if constexpr (PARTS) {
#pragma unroll
        for (int n = 0; n < R::NBT; n++) {
#pragma unroll
            for (int u = 0; u < NS; u++) tot[u][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            odd[n][0] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    for (int st = 0; st < R::P - 1; st++) issue();
    uint32_t get = 0;
    auto stage = [&](f32x4_t (*acc)[R::TT]) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        /* stage s has landed when at most the later stages' loads are in flight: Q per stage
           for a wavefront that loads A tiles, Q - QA for one that does not */
        if (R::KG > 1 || w < NMT) wait_vm_lgkm<R::Q * (R::P - 2)>();
        else wait_vm_lgkm<(R::Q - R::QA) * (R::P - 2)>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue();
        const uint8_t *slot = ring + get;
        get = get + R::STAGE == R::P * R::STAGE ? 0 : get + R::STAGE;
        const uint8_t *wl = slot + R::NA * R::A_BYTES;
        const uint16_t *sl = (const uint16_t *)(wl + R::W_BYTES);
#pragma unroll
        for (int kq = 0; kq < R::KBW; kq++) {
            const int kb = R::KG > 1 ? kg * R::KBW + kq : kq;
            uint4 a[R::NA][NMT];
#pragma unroll
            for (int mt = 0; mt < NMT; mt++) {
                const int r = mt * 16 + (l & 15);
                const int o = 2 * (r * 32 * KB + 8 * R::apos(r, 4 * kb + g));
#pragma unroll
                for (int p = 0; p < R::NA; p++) a[p][mt] = *(const uint4 *)(slot + p * R::A_BYTES + o);
            }
#pragma unroll
            for (int n = 0; n < R::NBT; n++) {
                WRaw r;
                r.w = *(const uint2 *)(wl + boff[n] + kb * 64 * R::PB);
                r.d = *(const uint16_t *)((const uint8_t *)sl + soff[n] + kb * 128);
                float d = scale_f32(r.d);
                f32x4_t t[NMT];
#pragma unroll
                for (int mt = 0; mt < NMT; mt++) t[mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (R::FMT == CPG_PL_BF16) {
                    const bf16x8_t q = weight_q_bf16<ENC>(r.w, g);
                    if (ENC == CPG_ENC_Q4) d *= 0x1p-4f;
#pragma unroll
                    for (int p = R::NA - 1; p >= 0; p--)
#pragma unroll
                        for (int mt = 0; mt < NMT; mt++)
                            t[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(bf16x8_t, a[p][mt]), q, t[mt], 0, 0, 0);
                } else {
                    const half8_t q = weight_q<ENC>(r.w, g);
                    half8_t ql = q;
                    if (R::FMT == CPG_PL_F16UP) ql *= (_Float16)0x1p-11f;
#pragma unroll
                    for (int p = 0; p < R::NA; p++)
#pragma unroll
                        for (int mt = 0; mt < NMT; mt++)
                            t[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                __builtin_bit_cast(half8_t, a[p][mt]), p ? ql : q, t[mt], 0, 0, 0);
                }
#pragma unroll
                for (int mt = 0; mt < NMT; mt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[n][mt][i] = fmaf(d, t[mt][i], acc[n][mt][i]);
            }
        }
    };
    for (int s = 0; s < S; s += NS) {
        if constexpr (PARTS) {
            if (s % (PF_SUM * NS) == 0)
#pragma unroll
                for (int n = 0; n < R::NBT; n++) {
                    tot[0][n] += acc[n][0];
                    acc[n][0] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    if constexpr (NS == 2) {
                        tot[1][n] += odd[n][0];
                        odd[n][0] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                }
        }
        stage(acc);
        if constexpr (NS == 2) stage(odd);
    }
    if constexpr (PARTS) {
#pragma unroll
        for (int n = 0; n < R::NBT; n++) {
            acc[n][0] += tot[0][n];
            if constexpr (NS == 2) acc[n][0] += odd[n][0] + tot[1][n];
        }
    }
    /* no load may still write this workgroup's LDS when it ends */
    asm volatile("" ::: "memory");
    wait_vm_lgkm<0>();
    if constexpr (R::KG > 1) {                   /* the groups' sums: group 0 adds the others in order */
        float *red = (float *)ring;
        __syncthreads();                         /* every load has landed, every stage is read */
        if (kg > 0)
#pragma unroll
            for (int n = 0; n < R::NBT; n++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    red[(((kg - 1) * R::NBT + n) * 4 + i) * 256 + 64 * w4 + l] = acc[n][0][i];
        __syncthreads();
        if (kg == 0)
#pragma unroll
            for (int q = 1; q < R::KG; q++)
#pragma unroll
                for (int n = 0; n < R::NBT; n++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[n][0][i] += red[(((q - 1) * R::NBT + n) * 4 + i) * 256 + 64 * w4 + l];
    }
}

/* grid (rows / RW, max_chunks), PF_NT threads, dynamic LDS PfRing::P * PfRing::STAGE,
   max_chunks a multiple of 8. Chunk c = (group g, tokens m0..m0+m-1) of expert e.
   GU (gate/up): rows r0..r0+RW-1 of Wg and of Wu (n_in = D) over the hi/lo planes of xn (one
     row per token id), then h = silu(g) * u (kernels.c:416) written as hi/lo f16 rows hh/hl
     at the token's position in the group list (off + m0 + i), the A operand of the down GEMM.
   down: rows r0..r0+RW-1 of Wd (n_in = F) over hh/hl at the group-list positions; y[pair]
     (row stride n_out) for the pair of each position.
   TT (a ring for TT token tiles): a chunk holds at most 16 * TT tokens, so the chunk list must have
   been formed with ch = 16 * TT: its writers and this kernel's dispatch both take
   cpg_prefill_chunk(T, K, E). With sel there is no list: there an expert's pairs are one chunk, at
   most 16 as T <= 16 and a token's K experts are distinct. */
template <int ENC, bool GU, int TT = PF_CHUNK / 16, int P = 2, int RW = 128, int KB = 2, int KG = 1, int SUMS = 1>
__global__ __launch_bounds__(PF_NT *KG) __attribute__((amdgpu_waves_per_eu(TT == 4 ? 3 : 1))) void k_pf_gemm(
    const uint8_t *__restrict__ experts, size_t exp_stride, size_t mat0, size_t mat_bytes,
    size_t payload_plane, int n_in, int n_out, const int *__restrict__ chunk_grp,
    const int *__restrict__ chunk_m0, const int *__restrict__ grp_expert,
    const int *__restrict__ grp_off, const int *__restrict__ grp_cnt,
    const int *__restrict__ list, const _Float16 *__restrict__ xh,
    const _Float16 *__restrict__ xl, _Float16 *__restrict__ hh, _Float16 *__restrict__ hl,
    float *__restrict__ y, const int *__restrict__ sel, int npairs, int K, int E,
    int *__restrict__ ngroups) {
    using R = PfRing<ENC, GU, TT, P, RW, KB, KG, CPG_PL_F16, SUMS>;
    extern __shared__ __align__(16) uint8_t ring[];
    __shared__ int arow[PF_CHUNK], orow[PF_CHUNK];
    __shared__ uint64_t tab[32];
    /* workgroup i runs on XCD i % 8: the row tiles of chunk c are placed on XCD c % 8, next
       to each other in its dispatch order, so the chunk's activations are fetched into one L2
       (gridDim.y is a multiple of 8) */
    const int nx = gridDim.x, id = blockIdx.x + nx * blockIdx.y, sidx = id >> 3;
    const int c = 8 * (sidx / nx) + (id & 7);
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, w4 = w & 3, g = l >> 4;
    const int r0 = (sidx % nx) * RW, nb = n_in / 32;
    int e, m;
    if (TT == 1 && sel) {
        /* chunk c is the c-th expert with pairs (ascending id) of the npairs <= 256 selections
           sel[t * K + j] (ids below E <= 256 count): found by wavefront 0 from sel itself, with the expert's
           pairs in ascending pair order (at most 16: one token tile); no grouping step
           before this launch. Gate/up: A rows the pairs' tokens, outputs at the pair
           indices; down: A rows and outputs at the pair indices. */
        __shared__ int used[MAX_E], pick[2];
        if (w == 0) {
            int v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v[q] = l + 64 * q < npairs ? sel[l + 64 * q] : -1;
                if ((unsigned)v[q] >= (unsigned)E) v[q] = -1;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) used[l + 64 * q] = 0;
            wave_lds_sync();
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (v[q] >= 0) used[v[q]] = 1;
            wave_lds_sync();
            const unsigned long long lt = (1ull << l) - 1ull;
            int ex = -1, before = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const unsigned long long u = __ballot(used[l + 64 * q] != 0);
                const int cc = c - before;
                const bool hit = cc >= 0 && ((u >> l) & 1ull) && __popcll(u & lt) == cc;
                const unsigned long long hb = __ballot(hit);
                if (hb) ex = 64 * q + __ffsll((long long)hb) - 1;
                before += __popcll(u);
            }
            /* the number of experts with pairs, for the caller (one workgroup writes it) */
            if (ngroups && id == 0 && l == 0) *ngroups = before;
            int n = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const bool mine = ex >= 0 && v[q] == ex;
                const unsigned long long pb = __ballot(mine);
                const int i = n + __popcll(pb & lt), pr = l + 64 * q;
                if (mine && i < 16) {
                    arow[i] = GU ? pr / K : pr;
                    orow[i] = pr;
                }
                n += __popcll(pb);
            }
            n = min(n, 16);
            wave_lds_sync();
            /* rows past the expert's pairs repeat its last one (valid addresses) */
            if (ex >= 0 && l >= n) {
                arow[l] = arow[n - 1];
                orow[l] = orow[n - 1];
            }
            if (l == 0) {
                pick[0] = ex;
                pick[1] = n;
            }
        }
        if (GU && tid < 32) tab[tid] = cpg_exp2f_tab[tid];
        __syncthreads();
        e = pick[0];
        m = pick[1];
        if (e < 0) return;
    } else {
        const int grp = chunk_grp[c];
        if (grp < 0) return;
        e = grp_expert[grp];
        const int off = grp_off[grp], m0 = chunk_m0[c];
        m = min(16 * TT, grp_cnt[grp] - m0);
        if (tid < PF_CHUNK) {
            const int i = min(tid, m - 1);
            arow[tid] = GU ? list[off + m0 + i] : off + m0 + i;
            orow[tid] = GU ? off + m0 + i : list[off + m0 + i];
        }
        if (GU && tid < 32) tab[tid] = cpg_exp2f_tab[tid];
        __syncthreads();
    }
    const int nmt = (m + 15) / 16;
    /* the sources of this lane's loads for block 0 (block st adds st * 32 halves, or one
       block's bytes): A row 16w + l/4, piece l%4; the wavefront's WB weight bytes and SB
       scale bytes of the stage */
    /* A load i of the wavefront fills rows 16w + i * 64/PP .. (PP lanes per row): this lane's
       row and the logical piece that belongs at its position */
    uint32_t aoff[R::AI];            /* bytes (T K F halves are far below 2^32 of them) */
#pragma unroll
    for (int i = 0; i < R::AI; i++) {
        const int ar = (KG > 1 ? w % KB : 16 / (64 / R::PP) * w + i) * (64 / R::PP) + l / R::PP;
        aoff[i] = 2 * ((uint32_t)arow[ar] * n_in + 8 * R::apos(ar, l % R::PP));
    }
    const uint8_t *M0 = experts + (size_t)e * exp_stride + mat0;
    const int wseg = w * R::WB / (R::KB * 64 * R::PB), wofs = w * R::WB % (R::KB * 64 * R::PB);
    const int sseg = w * R::SB / (R::KB * 128), sofs = w * R::SB % (R::KB * 128);
    /* a segment's matrix (GU: gate, then up) and 64-row tile */
    auto seg_mat = [&](int seg) { return GU ? M0 + (size_t)(seg / R::TPM) * mat_bytes : M0; };
    auto seg_tile = [&](int seg) { return (size_t)((r0 >> 6) + seg % R::TPM); };
    const uint8_t *wsrc = seg_mat(wseg) + seg_tile(wseg) * nb * 64 * R::PB + wofs;
    const uint8_t *ssrc = seg_mat(sseg) + payload_plane + seg_tile(sseg) * nb * 128 + sofs;
    f32x4_t acc[R::NBT][TT];
#pragma unroll
    for (int n = 0; n < R::NBT; n++)
#pragma unroll
        for (int mt = 0; mt < TT; mt++)
            for (int i = 0; i < 4; i++) acc[n][mt][i] = 0.0f;
    const int S = nb / R::KB;
    if constexpr (TT == 1) {
        pf_loop<R, 1>(ring, S, (const uint16_t *)xh, xl - xh, aoff, wsrc, ssrc, acc);
    } else {
        switch (nmt) {
        case 1: pf_loop<R, 1>(ring, S, (const uint16_t *)xh, xl - xh, aoff, wsrc, ssrc, acc); break;
        case 2: pf_loop<R, 2>(ring, S, (const uint16_t *)xh, xl - xh, aoff, wsrc, ssrc, acc); break;
        case 3: pf_loop<R, 3>(ring, S, (const uint16_t *)xh, xl - xh, aoff, wsrc, ssrc, acc); break;
        default: pf_loop<R, 4>(ring, S, (const uint16_t *)xh, xl - xh, aoff, wsrc, ssrc, acc); break;
        }
    }
    if (KG > 1 && w >= 4) return;                /* group 0 holds the sums */
    if constexpr (GU) {
#pragma unroll
        for (int half = 0; half < R::TPM; half++)
#pragma unroll
            for (int mt = 0; mt < TT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int r = mt * 16 + 4 * g + i;
                    if (r < m) {
                        const float hv =
                            swiglu_t(acc[half][mt][i], acc[R::TPM + half][mt][i], tab);
                        const f16pair p = split_f16(hv);
                        const size_t o = (size_t)orow[r] * n_out + r0 + RW / 4 * w4 +
                                         16 * half + (l & 15);
                        hh[o] = p.hi;
                        hl[o] = p.lo;
                    }
                }
    } else {
#pragma unroll
        for (int n = 0; n < R::NBT; n++)
#pragma unroll
            for (int mt = 0; mt < TT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int r = mt * 16 + 4 * g + i;
                    if (r < m)
                        y[(size_t)orow[r] * n_out + r0 + RW / 4 * w4 + 16 * n + (l & 15)] =
                            acc[n][mt][i];
                }
    }
}

/* ---------------------------------------------------------------- dense */

#define DENSE_RW 64         /* rows per workgroup. Measured at 64, 128 and 256 (q|k|v, output
                               projection with the sums of their parts, us): 512 tokens Q4_0 77.8,
                               80.1, 87.1; 96 tokens 38, 39, 41; 21 tokens Q8_0, two planes, 21.9, 22.7, - */

/* grid (n_out / DENSE_RW, chunks, ks), PF_NT threads, dynamic LDS PfRing::P * PfRing::STAGE: one
   row-tiled matrix W (n_out rows of n_in) times the ct <= 16 TT tokens from blockIdx.y * ct of
   the planes pl of format FMT (T rows of n_in), over the nbs blocks of 32 from
   blockIdx.z * nbs (nbs a multiple of KB); written to out[(blockIdx.z * T + t) * n_out + row],
   one part per blockIdx.z.

   The expert GEMMs' k loop over a ring of stages in LDS (pf_loop), each wavefront 16 rows for
   the chunk's token tiles. Few tokens are bound by the launch and one trip through the ring (one
   token tile a ring of four stages, all of a part's loads in flight at once; two a ring of three,
   which leaves LDS for three workgroups per CU: 21 tokens q|k|v 8.2 us, with four 10.0), many by the MFMAs
   and the LDS reads of their operands (per block and wavefront 2 token-tile operands for 2 MFMAs).
   Against a k loop through registers (weights two stages ahead, a barrier a block): q|k|v and
   output projection, Q4_0, us: 512 tokens 49.2 + 35.2 -> 36.6 + 26.8, 96 tokens 18.0 + 14.5 ->
   14.7 + 12.6; and against k_gemv's passes of four tokens: 21 tokens Q8_0 46.8 + 49.4 -> 8.3 +
   6.8, 4 tokens Q4_0 12.0 + 13.6 -> 6.2 + 5.4 (two planes of f16 instead of three of bf16: 7.6 + 6.4
   and 5.8 + 4.9, without fp32's range). */
template <int ENC, int TT, int P, int KB, int FMT>
__global__ __launch_bounds__(PF_NT) __attribute__((amdgpu_waves_per_eu(TT == 4 ? 3 : 1))) void k_dense(
    const uint8_t *__restrict__ W, size_t payload_plane, int n_in, int n_out, int T, int ct,
    int nbs, cpg_planes pl, float *__restrict__ out) {
    constexpr int RW = DENSE_RW;
    using R = PfRing<ENC, false, TT, P, RW, KB, 1, FMT>;
    extern __shared__ __align__(16) uint8_t ring[];
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, g = l >> 4;
    const int m0 = blockIdx.y * ct, m = min(ct, T - m0), nmt = (m + 15) / 16;
    const int r0 = blockIdx.x * RW, nb = n_in / 32, b0 = blockIdx.z * nbs;
    uint32_t aoff[KB];
#pragma unroll
    for (int i = 0; i < KB; i++) {
        const int ar = 16 * w + i * (64 / R::PP) + l / R::PP;
        aoff[i] = 2 * ((uint32_t)min(ar, m - 1) * n_in + 8 * R::apos(ar, l % R::PP));
    }
    const size_t a0 = (size_t)m0 * n_in + 32 * b0;
    const int wseg = w * R::WB / (KB * 64 * R::PB), wofs = w * R::WB % (KB * 64 * R::PB);
    const int sseg = w * R::SB / (KB * 128), sofs = w * R::SB % (KB * 128);
    const uint8_t *wsrc = W + ((size_t)((r0 >> 6) + wseg) * nb + b0) * 64 * R::PB + wofs;
    const uint8_t *ssrc = W + payload_plane + ((size_t)((r0 >> 6) + sseg) * nb + b0) * 128 + sofs;
    f32x4_t acc[R::NBT][TT];
#pragma unroll
    for (int n = 0; n < R::NBT; n++)
#pragma unroll
        for (int mt = 0; mt < TT; mt++)
            for (int i = 0; i < 4; i++) acc[n][mt][i] = 0.0f;
    const int S = nbs / KB;
    if constexpr (TT == 1) {
        pf_loop<R, 1>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc);
    } else if constexpr (TT == 2) {
        if (nmt == 1) pf_loop<R, 1>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc);
        else pf_loop<R, 2>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc);
    } else {
        switch (nmt) {
        case 1: pf_loop<R, 1>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc); break;
        case 2: pf_loop<R, 2>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc); break;
        case 3: pf_loop<R, 3>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc); break;
        default: pf_loop<R, 4>(ring, S, pl.p + a0, pl.stride, aoff, wsrc, ssrc, acc); break;
        }
    }
    float *o = out + ((size_t)blockIdx.z * T + m0) * n_out + r0 + RW / 4 * w + (l & 15);
#pragma unroll
    for (int n = 0; n < R::NBT; n++)
#pragma unroll
        for (int mt = 0; mt < TT; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = mt * 16 + 4 * g + i;
                if (r < m) o[(size_t)r * n_out + 16 * n] = acc[n][mt][i];
            }
}

/* grid ceil(n/512), 128 threads, n % 4 == 0: out[i] = ((part[0][i] + part[1][i]) + part[2][i]) +
   ..., ks parts of n floats, in part order; the loads of eight parts in flight together (one
   round trip each had been most of the launch with 16 parts) */
__global__ __launch_bounds__(128) void k_sum_parts(const float *__restrict__ part, int ks,
                                                   size_t n, float *__restrict__ out) {
    const size_t i = 4 * ((size_t)blockIdx.x * 128 + threadIdx.x);
    if (i >= n) return;
    float4 a = *(const float4 *)(part + i);
    for (int z0 = 1; z0 < ks; z0 += 8) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = *(const float4 *)(part + (size_t)min(z0 + u, ks - 1) * n + i);
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (z0 + u < ks)
                a = make_float4(__fadd_rn(a.x, v[u].x), __fadd_rn(a.y, v[u].y),
                                __fadd_rn(a.z, v[u].z), __fadd_rn(a.w, v[u].w));
    }
    *(float4 *)(out + i) = a;
}

/* ---------------------------------------------------------------- combine */

/* grid (ceil(D/1024), T), 256 threads, D % 4 == 0: o = mlp[t][d] + sum_j wt[t][j] *
   y[t*K + j][d] in slot order (qwen3_moe.c:221), four consecutive d per thread (float4);
   written to mlp, or with xres: xres[t][d] += attn[t][d] + o and mlp untouched (mlp must then
   be zero, the reference's calloc'ed start, cachepotato.c:157-159). KT > 0: K == KT, every
   pair's load issued before the sums. */
template <int KT>
__global__ __launch_bounds__(256) void k_pair_combine(const float *__restrict__ y,
                                                      const float *__restrict__ wt, int D, int K,
                                                      float *__restrict__ mlp,
                                                      float *__restrict__ xres,
                                                      const float *__restrict__ attn) {
    const int t = blockIdx.y, d = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (d >= D) return;
    if (KT) K = KT;
    const size_t o = (size_t)t * D + d;
    float4 acc = xres ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : *(const float4 *)(mlp + o);
    auto add = [&](float w, float4 v) {
        acc = make_float4(__fadd_rn(acc.x, __fmul_rn(w, v.x)), __fadd_rn(acc.y, __fmul_rn(w, v.y)),
                          __fadd_rn(acc.z, __fmul_rn(w, v.z)), __fadd_rn(acc.w, __fmul_rn(w, v.w)));
    };
    if constexpr (KT > 0) {
        float4 v[KT];
#pragma unroll
        for (int j = 0; j < KT; j++) v[j] = *(const float4 *)(y + ((size_t)t * KT + j) * D + d);
#pragma unroll
        for (int j = 0; j < KT; j++) add(wt[(size_t)t * KT + j], v[j]);
    } else {
        for (int j = 0; j < K; j++)
            add(wt[(size_t)t * K + j], *(const float4 *)(y + ((size_t)t * K + j) * D + d));
    }
    if (xres) {
        const float4 xr = *(const float4 *)(xres + o), ar = *(const float4 *)(attn + o);
        *(float4 *)(xres + o) = make_float4(__fadd_rn(xr.x, __fadd_rn(ar.x, acc.x)),
                                            __fadd_rn(xr.y, __fadd_rn(ar.y, acc.y)),
                                            __fadd_rn(xr.z, __fadd_rn(ar.z, acc.z)),
                                            __fadd_rn(xr.w, __fadd_rn(ar.w, acc.w)));
    } else {
        *(float4 *)(mlp + o) = acc;
    }
}

/* ---------------------------------------------------------------- host */

static int max_chunks(int T, int K, int E, int ch) {
    const int pairs = T * K;
    const int groups = pairs < E ? pairs : E;
    const int n = (pairs + ch - 1) / ch + groups;
    return (n + 7) / 8 * 8;                      /* k_pf_gemm places chunk c on XCD c % 8 */
}

/* Tokens per chunk of T tokens with K experts each: one tile of 16 while the experts have at most 11
   tokens each on average, so that most experts are one chunk: the one-tile GEMMs' smaller
   workgroups then keep more of the weights in flight (us per layer with the routing, chunks of 64 and
   of 16, 128 experts top-8: 45 tokens Q4_0 123.2, 117.0, Q8_0 skewed 145.9, 132.8; 96 tokens 126.8,
   119.7 and 168.8, 156.1; 160 tokens Q4_0 136.8, 134.3, Q8_0 185.4, 179.7; 176 tokens 138.1, 137.4
   and 187.5, 182.0). The second chunks of crowded experts read their weights again, so a skewed
   choice of experts turns earlier: 160 tokens Q4_0 145.5, 146.0, Q8_0 183.5, 184.7; 176 tokens 149.4,
   150.3 and 188.0, 191.4. Above, 192 tokens Q8_0 188.5, 184.4, skewed 185.2, 195.5, Q4_0 133.5,
   134.8; 256 tokens 142, 155. */
int cpg_prefill_chunk(int T, int K, int E) {
    return T <= 16 || T * K <= 11 * E ? 16 : PF_CHUNK;
}

/* the most chunks T tokens with K experts each over E experts can form */
int cpg_prefill_max_chunks(int T, int K, int E) {
    return max_chunks(T, K, E, cpg_prefill_chunk(T, K, E));
}

int cpg_prefill_chunks_upto(int T, int K, int E) { return max_chunks(T, K, E, 16); }

bool cpg_prefill_shape_ok(int D, int F) {
    return D % 128 == 0 && F % 128 == 0;
}

template <int ENC>
static int prefill_experts(const cpg_moe_layer *L, int T, const float *xn, const float *wt,
                           const int *grp_expert, const int *grp_off, const int *grp_cnt,
                           const int *list_tok, const int *list_pair, int *chunk_grp,
                           int *chunk_m0, void *scratch, float *y, float *mlp, float *xres,
                           const float *attn, bool prepared, const int *sel, int *ngroups) {
    const int D = L->D, F = L->F, E = L->E, K = L->K;
    /* sel: the one-tile GEMMs find their expert and pairs in the selections themselves, one
       chunk per expert with pairs */
    if (sel && !cpg_prefill_sel_ok(T, K, E)) {
        cpg_set_error("prefill_experts: selections of %d tokens x %d over %d experts", T, K, E);
        return -1;
    }
    const int mc = sel ? ((T * K < E ? T * K : E) + 7) / 8 * 8 : cpg_prefill_max_chunks(T, K, E);
    _Float16 *xh = (_Float16 *)scratch, *xl = xh + (size_t)T * D;
    _Float16 *hh = xl + (size_t)T * D, *hl = hh + (size_t)T * K * F;
    if (!prepared) {
        if (!sel)
            LAUNCH(CPG_KT_SELECT, k_chunks, dim3(1), dim3(64), 0, grp_cnt, E,
                   cpg_prefill_chunk(T, K, E), mc, chunk_grp, chunk_m0);
        LAUNCH(CPG_KT_SELECT, k_split_planes<CPG_PL_F16>, dim3(T), dim3(256), 0, xn, D,
               (cpg_planes{(uint16_t *)xh, (size_t)T * D, CPG_PL_F16}));
    }
    const uint8_t *ex = (const uint8_t *)L->experts;
    const size_t es = cpg_expert_bytes(ENC, D, F), mg = cpg_matrix_bytes(ENC, F, D);
    auto gemms = [&](int nt, auto gu_kernel, size_t ring_gu, int rw_gu, auto dn_kernel,
                     size_t ring_dn, int rw_dn) {
        if (ring_gu > 64 * 1024)
            CPG_HIP(hipFuncSetAttribute((const void *)gu_kernel,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)ring_gu));
        if (ring_dn > 64 * 1024)
            CPG_HIP(hipFuncSetAttribute((const void *)dn_kernel,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)ring_dn));
        LAUNCH(CPG_KT_GATEUP, gu_kernel, dim3(F / rw_gu, mc), dim3(nt), ring_gu, ex, es,
               (size_t)0, mg, cpg_payload_plane(ENC, F, D), D, F, chunk_grp, chunk_m0,
               grp_expert, grp_off, grp_cnt, list_tok, xh, xl, hh, hl, (float *)nullptr, sel,
               T * K, K, E, ngroups);
        LAUNCH(CPG_KT_DOWN, dn_kernel, dim3(D / rw_dn, mc), dim3(nt), ring_dn, ex, es, 2 * mg,
               mg, cpg_payload_plane(ENC, D, F), F, D, chunk_grp, chunk_m0, grp_expert, grp_off,
               grp_cnt, list_pair, hh, hl, (_Float16 *)nullptr, (_Float16 *)nullptr, y, sel,
               T * K, K, E, (int *)nullptr);
        return 0;
    };
    int rc;
    if (cpg_prefill_chunk(T, K, E) == 16) {
        /* chunks of one token tile */
        auto tile = [&](auto groups, auto ring, auto sums) {
            constexpr int KG = groups, P = ring, KB = 2 * KG, SUMS = sums;
            using RG = PfRing<ENC, true, 1, P, PF_SMALL_RW_GU, KB, KG>;
            using RD = PfRing<ENC, false, 1, P, PF_SMALL_RW_DN, KB, KG>;
            return gemms(RG::NT, k_pf_gemm<ENC, true, 1, P, PF_SMALL_RW_GU, KB, KG, SUMS>,
                         (size_t)RG::P * RG::STAGE, RG::RW,
                         k_pf_gemm<ENC, false, 1, P, PF_SMALL_RW_DN, KB, KG, SUMS>,
                         (size_t)RD::P * RD::STAGE, RD::RW);
        };
        constexpr std::integral_constant<int, 1> one;
        constexpr std::integral_constant<int, 2> two;
        constexpr std::integral_constant<int, 3> three;
        if (T * K <= PF_FEW_PAIRS) {
            rc = tile(two, two, one);
        } else if (T <= 16) {
            if constexpr (ENC == CPG_ENC_Q4) rc = tile(one, three, two);
            else rc = tile(one, two, two);
        } else if (ENC == CPG_ENC_Q4 ? T * K > PF_RING_Q4 && T * K <= 8 * E : T * K <= PF_RING_Q8) {
            rc = tile(one, two, one);
        } else {
            rc = tile(one, three, one);
        }
    } else {
        using RG = PfRing<ENC, true>;
        using RD = PfRing<ENC, false>;
        rc = gemms(PF_NT, k_pf_gemm<ENC, true>, (size_t)RG::P * RG::STAGE, RG::RW,
                   k_pf_gemm<ENC, false>, (size_t)RD::P * RD::STAGE, RD::RW);
    }
    if (rc) return rc;
    if (K == 8)
        LAUNCH(CPG_KT_COMBINE, k_pair_combine<8>, dim3((D + 1023) / 1024, T), dim3(256), 0, y,
               wt, D, K, mlp, xres, attn);
    else
        LAUNCH(CPG_KT_COMBINE, k_pair_combine<0>, dim3((D + 1023) / 1024, T), dim3(256), 0, y,
               wt, D, K, mlp, xres, attn);
    return 0;
}

/* The dense product's launch for T tokens: blocks of 32 per stage (two where the row has an
   even number), token tiles of 16 and chunks (a workgroup's tokens, spread evenly: 96 tokens are
   two chunks of 48, not 64 and 32), and the split of the k range, doubled while every part keeps
   at least 8 blocks and the grid stays within 1024 workgroups (640 with 128 and more blocks per row,
   whose many parts cost more where they are summed than their shorter loops give: output
   projection and sum of its parts at 96 tokens 13.0 + 5.3 -> 10.6 + 3.9 us with 8 parts for 16, 512
   tokens 28.4 + 5.1 and 28.8 + 4.9 with 2 for 4; q|k|v at 96 tokens 13.2 with 4 parts, 14.6 with 2). */
struct dense_geo {
    int kb, tt, tpc, chunks, ks;                 /* tt: the kernel's tiles; tpc: a chunk's */
};
/* Up to 32 tokens the activations keep fp32's bits and range, as in the GEMVs (k_gemv) that fewer
   tokens take: three planes of bf16. More take two planes of f16. */
static int dense_format(int T) { return T <= 32 ? CPG_PL_BF16 : CPG_PL_F16UP; }
static size_t dense_plane_bytes(int T, int n_in) {
    return cpg_round256((size_t)2 * cpg_plane_count(dense_format(T)) * T * n_in);
}
cpg_planes cpg_dense_planes(int T, int n_in, void *scratch) {
    return {(uint16_t *)scratch, (size_t)T * n_in, dense_format(T)};
}
static dense_geo dense_geometry(int T, int n_in, int n_out) {
    const int nb = n_in / 32, tiles = (T + 15) / 16;
    dense_geo d;
    d.kb = nb % 2 ? 1 : 2;
    d.tt = d.kb == 1 || T > 32 ? 4 : T > 16 ? 2 : 1;
    d.chunks = (tiles + d.tt - 1) / d.tt;
    d.tpc = (tiles + d.chunks - 1) / d.chunks;
    d.chunks = (tiles + d.tpc - 1) / d.tpc;
    const int base = n_out / DENSE_RW * d.chunks;
    d.ks = 1;
    while (d.ks < 16 && nb % (2 * d.ks * d.kb) == 0 && nb / (2 * d.ks) >= 8 &&
           base * 2 * d.ks <= (nb >= 128 ? 640 : 1024))
        d.ks *= 2;
    return d;
}
static int dense_ksplit(int T, int n_in, int n_out) { return dense_geometry(T, n_in, n_out).ks; }

bool cpg_dense_shape_ok(int n_in, int n_out) {
    return n_in > 0 && n_out > 0 && n_in % 32 == 0 && n_out % 64 == 0;
}

size_t cpg_dense_scratch_bytes(int T, int n_in, int n_out) {
    const int ks = dense_ksplit(T, n_in, n_out);
    return dense_plane_bytes(T, n_in) + (ks > 1 ? (size_t)4 * ks * T * n_out : 0);
}

template <int ENC, int TT, int P, int KB, int FMT> static size_t dense_lds() {
    using R = PfRing<ENC, false, TT, P, DENSE_RW, KB, 1, FMT>;
    return (size_t)R::P * R::STAGE;
}

/* the products from the planes already in scratch: out directly (ks == 1) or ks parts
   of T * n_out floats, left unsummed in *parts when sum is false */
template <int ENC>
static int dense_from_planes(const void *w, int n_in, int n_out, int T, void *scratch,
                             float *out, bool sum, const float **parts, int *ks_out) {
    const int ks = dense_ksplit(T, n_in, n_out);
    const cpg_planes pl = cpg_dense_planes(T, n_in, scratch);
    float *part = ks > 1 ? (float *)((uint8_t *)scratch + dense_plane_bytes(T, n_in)) : out;
    hipStream_t s = g_cpg.stream;
    const dense_geo d = dense_geometry(T, n_in, n_out);
    auto go = [&](auto kernel, size_t lds) {
        if (lds > 64 * 1024)
            CPG_HIP(hipFuncSetAttribute((const void *)kernel,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kernel, dim3(n_out / DENSE_RW, d.chunks, ks), dim3(PF_NT), lds, s,
                           (const uint8_t *)w, cpg_payload_plane(ENC, n_out, n_in), n_in, n_out,
                           T, 16 * d.tpc, n_in / 32 / ks, pl, part);
        CPG_LAUNCH_CHECK("k_dense");
        return 0;
    };
#define DENSE_GO(TT, DEPTH, KB, FMT) go(k_dense<ENC, TT, DEPTH, KB, FMT>, dense_lds<ENC, TT, DEPTH, KB, FMT>())
    int rc;
    if (pl.fmt == CPG_PL_F16UP)
        rc = d.kb == 1 ? DENSE_GO(4, 2, 1, CPG_PL_F16UP) : DENSE_GO(4, 2, 2, CPG_PL_F16UP);
    else if (d.kb == 1) rc = DENSE_GO(4, 2, 1, CPG_PL_BF16);
    else if (d.tt == 1) rc = DENSE_GO(1, 4, 2, CPG_PL_BF16);
    else rc = DENSE_GO(2, 3, 2, CPG_PL_BF16);
#undef DENSE_GO
    if (rc) return rc;
    if (parts) *parts = part;
    if (ks_out) *ks_out = ks;
    if (ks > 1 && sum) {
        const size_t n = (size_t)T * n_out;
        hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)((n + 511) / 512)), dim3(128), 0, s, part,
                           ks, n, out);
        CPG_LAUNCH_CHECK("k_sum_parts");
    }
    return 0;
}

template <int ENC>
static int dense_mfma(const void *w, int n_in, int n_out, const float *x, int T, void *scratch,
                      float *out) {
    const cpg_planes pl = cpg_dense_planes(T, n_in, scratch);
    hipLaunchKernelGGL(pl.fmt == CPG_PL_BF16 ? k_split_planes<CPG_PL_BF16> : k_split_planes<CPG_PL_F16UP>,
                       dim3(T), dim3(256), 0, g_cpg.stream, x, n_in, pl);
    CPG_LAUNCH_CHECK("k_split_planes");
    return dense_from_planes<ENC>(w, n_in, n_out, T, scratch, out, true, nullptr, nullptr);
}

int cpg_dense_from_planes(int enc, const void *w, int n_in, int n_out, int T, void *scratch,
                          float *out, int sum, const float **parts, int *ks) {
    if (!w || !scratch || !out || T <= 0 || !cpg_dense_shape_ok(n_in, n_out)) {
        cpg_set_error("cpg_dense_from_planes: bad arguments (n_in %d, n_out %d, T %d)", n_in,
                      n_out, T);
        return -1;
    }
    if (enc == CPG_ENC_Q4)
        return dense_from_planes<CPG_ENC_Q4>(w, n_in, n_out, T, scratch, out, sum, parts, ks);
    if (enc == CPG_ENC_Q8)
        return dense_from_planes<CPG_ENC_Q8>(w, n_in, n_out, T, scratch, out, sum, parts, ks);
    cpg_set_error("cpg_dense_from_planes: encoding %d is not row-tiled (Q4_0 or Q8_0 only)", enc);
    return -1;
}

int cpg_dense_mfma(int enc, const void *w, int n_in, int n_out, const float *x, int T,
                   void *scratch, float *out) {
    if (!w || !x || !scratch || !out || T <= 0 || !cpg_dense_shape_ok(n_in, n_out)) {
        cpg_set_error("cpg_dense_mfma: bad arguments (n_in %d, n_out %d, T %d)", n_in, n_out, T);
        return -1;
    }
    if (enc == CPG_ENC_Q4) return dense_mfma<CPG_ENC_Q4>(w, n_in, n_out, x, T, scratch, out);
    if (enc == CPG_ENC_Q8) return dense_mfma<CPG_ENC_Q8>(w, n_in, n_out, x, T, scratch, out);
    cpg_set_error("cpg_dense_mfma: encoding %d is not row-tiled (Q4_0 or Q8_0 only)", enc);
    return -1;
}

size_t cpg_prefill_scratch_bytes(int T, int D, int K, int F) {
    return (size_t)2 * 2 * ((size_t)T * D + (size_t)T * K * F);
}

bool cpg_prefill_sel_ok(int T, int K, int E) {
    return T > 0 && T <= 16 && K > 0 && T * K <= 256 && E > 0 && E <= MAX_E && MAX_E <= 256;
}

int cpg_prefill_experts(const cpg_moe_layer *L, int T, const float *xn, const float *wt,
                        const int *grp_expert, const int *grp_off, const int *grp_cnt,
                        const int *list_tok, const int *list_pair, int *chunk_grp,
                        int *chunk_m0, void *scratch, float *y, float *mlp, float *xres,
                        const float *attn, int prepared, const int *sel, int *ngroups) {
    if (L->enc == CPG_ENC_Q4)
        return prefill_experts<CPG_ENC_Q4>(L, T, xn, wt, grp_expert, grp_off, grp_cnt, list_tok,
                                           list_pair, chunk_grp, chunk_m0, scratch, y, mlp, xres,
                                           attn, prepared != 0, sel, ngroups);
    return prefill_experts<CPG_ENC_Q8>(L, T, xn, wt, grp_expert, grp_off, grp_cnt, list_tok,
                                       list_pair, chunk_grp, chunk_m0, scratch, y, mlp, xres,
                                       attn, prepared != 0, sel, ngroups);
}
