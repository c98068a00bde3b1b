// Per-block INT8 GEMMs for gfx950 (MI355X).
//
//   acc[m,n] = sum over 32-deep K blocks kb (ascending) of  (sa[kb,m/32]*sb[kb,n/32]) * d_kb[m,n]
//   d_kb     = exact INT32 dot product of the kb-th 32-wide slices of A[m,:] and B[n,:]
//
// One v_mfma_i32_32x32x32_i8 produces d_kb for a whole 32x32 output block, i.e. exactly one Jetfire
// quantisation-block product.  (Reference kernels: igemm_BlockSquare32OutputIntQuantizeBiasRowCol.cu:134-225 and
// its siblings under JetfireGEMMKernel/BlockQuantize/cpp_extension/igemm/.)
//
// Scale-accumulate.  The vector ALU is the bottleneck of this kernel, and on this part it runs plain fp32
// add/mul/fma at twice the rate of conversions (v_cvt_f32_i32 included).  So the product is not converted:
// the MFMA's accumulator input is the inline constant 0x3e22f983 (the bit pattern of 1/(2 pi)) in every
// element.  |d| <= 32*127^2 < 2^21 keeps 0x3e22f983 + d inside the binade [1/8, 1/4), whose unit in the last
// place is 2^-26, so  as_float(0x3e22f983 + d) - as_float(0x3e22f983) = d * 2^-26  exactly (one v_sub_f32),
// and  fma(sa*sb*2^26, d*2^-26, acc)  has the same exact product, hence the same rounding, as
// fma(sa*sb, float(d), acc).  The only way the two differ is an overflow of sa*sb*2^26; that is detected
// after the K loop and the wave then recomputes its blocks with the plain sequence (see there).
//
// Work decomposition (large launches; see launch_gemm_b): workgroup = 8 waves (2 x 4), tile 128x128, each wave owns 64x32 = 2 quantisation
// blocks (32 fp32 accumulators per lane); two workgroups per CU.  K is consumed in stages of 4 blocks (128
// bytes per row) through an LDS ring filled by LDS-direct loads (global_load_lds_dwordx4: no register
// staging).  LDS rows are 128 bytes with an XOR chunk swizzle, so the 16-byte MFMA operand reads are
// conflict-free.  A is K-contiguous; B is either K-contiguous ([N,K]) or [K,N], which is staged as it lies
// in memory and read with the transposing LDS read.  Scales are wave-uniform; each wave multiplies those it
// needs once per stage and reads the products from a private LDS patch.
#include "jf_device.hpp"

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#pragma clang diagnostic ignored "-Winline-asm"     // M0 appears in clobber lists on purpose

// The kernels are many instantiations of one function: a library is built from this file in JF_PARTS pieces, compiled side by side (each
// with -DJF_PART=0 .. and its share of the explicit instantiations below; the entry points are in piece 0).  Without JF_PART: all of it.
#ifdef JF_PART
#define JF_IN_PART(n) (JF_PART == (n))
#else
#define JF_IN_PART(n) 1
#endif

namespace jf {

constexpr int KB_STAGE = 4;                         // 32-deep K blocks per LDS stage (128 bytes of K per row)
constexpr int ROW_BYTES = KB_STAGE * QB;            // 128: one LDS row = one 128-byte global segment
constexpr int EPI_LD = 36;                          // floats per staged row (32 + pad, keeps 16B alignment)

// EPI_QG: EPI_Q (deterministic) followed by the GELU forward of the block just requantised: two block tensors leave
// EPI_QB: EPI_Q (stochastic: an activation gradient) followed by the GELU backward of the block just requantised against
//         the saved forward input of the GELU: only the result of the GELU backward leaves
// EPI_QD: EPI_Q followed by the dequantisation of the block just requantised (codes x stored scale), written as float /
//         binary16 / bfloat16: the requantised tensor itself is never written.
// EPI_QA: EPI_Q (deterministic) followed by the residual addition of the block just requantised: the sum, its requantisation and its
//         partial row sums leave
enum Epilogue { EPI_S32 = 0, EPI_FP = 1, EPI_Q = 2, EPI_QG = 3, EPI_QB = 4, EPI_QD = 5, EPI_QA = 6 };
// Wave-priority schemes of the main loop (launch_gemm_cfg picks one per launch)
enum Pace { PACE_HARDWARE = 0, PACE_EVEN = 1, PACE_ORDERED = 2 };

struct GemmArgs {
    const int8_t *A;      // [M, lda] (K-contiguous) or, for the AKM kernels, [K, lda] (M-contiguous rows)
    const int8_t *B;      // [N, ldb] (K-contiguous) or, for the BKN kernels, [K, ldb] (N-contiguous)
    const void *sa;       // scale of A block (mb, kb) at sa[kb * sa_ks + mb * sa_is]
    const void *sb;       // scale of B block (nb, kb) at sb[kb * sb_ks + nb * sb_is]
    int sa_ks, sa_is, sb_ks, sb_is;
    void *C;              // s32 / fp / s8 [M, N]
    void *sc;             // [M/32, N/32]   (EPI_Q)
    const float *bias;    // [N] or null   (EPI_Q)
    const float *biasmax; // [1] or null   (EPI_Q)
    uint64_t seed, offset;
    int M, N, K, lda, ldb;
    int tiles_m, tiles_n;
    int m_base;           // first row of the tiles (a launch of two tile sizes: its second part)
    int big_tiles;        // 128x128 tiles of a launch of both tile sizes, rows 0 .. m_base - 1 (the 32x128 tiles start there)
    int splits, kb_per_split;   // split-K (EPI_FP only): workgroup w works on K blocks [s*kb_per_split, ...) of tile w % tiles,
                                // s = w / tiles, and stores fp32 partial sums at C + s*M*N
    int out_dtype;        // JF_FP_*        (EPI_FP)
    int rounding;         // JF_ROUND_*     (EPI_Q)
    void *C2, *sc2;       // s8 [M, N], [M/32, N/32]: GELU of the requantised result   (EPI_QG)
    int gelu_approx;      // JF_GELU_*
    float gelu_eps;       // added to the GELU output's block absmax (the reference: 5e-5, gelu_fwd.py:93)
    const int8_t *Xq;     // s8 [M, N]: forward input of the GELU   (EPI_QB)
    const void *Xs;       // [M/32, N/32]
    uint64_t seed2, offset2;   // noise of the GELU backward's own requantisation   (EPI_QB)
    int rounding2;        // JF_ROUND_NEAREST / JF_ROUND_STOCHASTIC   (EPI_QB)
    int pace;             // PACE_*: wave priorities that order the resident workgroups of a CU (set by the launcher, see there)
    unsigned long long *phases;   // PROF kernels: 8 words per workgroup (jf_prof_igemm_block_q), first phase_capacity workgroups
    int phase_capacity;
    int fold_kb;          // K blocks after which the accumulators are added up in `fold` (a multiple of NSTAGE stages; 0: never)   (FOLD)
    float *fold;          // BM x BN values per workgroup, in an order of their own   (FOLD)
    const void *x1;       // [M, N], x1_dtype: what the requantised result is added to   (EPI_QA; rounding2: JF_ROUND_NEAREST / _TRUNC)
    int x1_dtype;
    void *y;              // [M, N], out_dtype: the sum   (EPI_QA)
    float *rowsum, *rowsq;   // [N/32, M] or null: per row and 32 columns, of the sum and its square   (EPI_QA)
};

// Position of workgroup wg in `work` pieces of work, or -1 behind the last.  Workgroups are dealt round-robin to the 8 XCDs, each with a
// private L2: every XCD gets one contiguous run of the work.
__device__ __forceinline__ int logical_workgroup(int work, int wg, bool all = false)     // (all: no workgroup lies behind the last)
{
    const int xcd = wg & 7, idx = wg >> 3;
    const int per = work >> 3, rem = work & 7;
    if (!all && idx >= per + (xcd < rem ? 1 : 0)) return -1;
    return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// Tile (and K split) at a position of a GEMM's work: tiles in groups of 8 tile-rows, so that concurrently resident workgroups
// of an XCD share A and B panels.  With K splits the order is split-major.
__device__ __forceinline__ void tile_at(int logical, int tiles_m, int tiles_n, bool has_splits, int &tm, int &tn, int &split)
{
    split = has_splits ? logical / (tiles_m * tiles_n) : 0;
    logical -= split * (tiles_m * tiles_n);
    constexpr int GROUP = 8;
    const int group_size = GROUP * tiles_n;
    const int g = logical / group_size;
    const int first_m = g * GROUP;
    const int gm = (tiles_m - first_m) < GROUP ? (tiles_m - first_m) : GROUP;
    const int in_group = logical - g * group_size;
    tm = first_m + in_group % gm;
    tn = in_group / gm;
}

// vmcnt(n), no wait on the other counters (gfx9 encoding: vmcnt = bits 3:0 and 15:14)
#define JF_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | 0x0F70)

// WGM x WGN waves, each owning WBM x WBN quantisation blocks (WBM = 2: 64x32 elements; WBM = 1: one block, for launches whose
// 128x128 tiles would leave most of the chip idle, see launch_gemm).
constexpr int WBN = 1;
// threads of a workgroup: with one block per wave, as many waves again that do nothing but load (see load_loop)
constexpr int gemm_threads(int WBM, int WGM, int WGN) { return 64 * WGM * WGN * (WBM == 1 ? 2 : 1); }
constexpr int TABLE_KB = 512;                        // K blocks a wave's table of scale products holds (WBM = 1)
// LDS of a workgroup: the operand ring; per-wave scale and product patches or tables; from gelu_lds_at on the GELU tables of the epilogue where
// they don't fit into those (WBM = 1: 1 KB per wave).  Epilogues that go through LDS use the ring.
constexpr int SPLIT_GROUP = 8 * ROW_BYTES + 64;       // SPLIT: bytes from one 8-row group of a stage to the next
constexpr int gelu_lds_at(int WBM, int WGM, int WGN, int NSTAGE)
{
    const int scales = WBM == 1 ? 4 * (TABLE_KB + KB_STAGE) * WGM * WGN : NSTAGE * WGM * WGN * 512;
    return NSTAGE * (QB * WBM * WGM + QB * WBN * WGN) * ROW_BYTES + scales;
}
// SPLIT: tables of scale products, patches, ring (it also serves as the GELU's tables)
constexpr int SPLIT_RING_AT = 2 * (4 * (TABLE_KB + KB_STAGE) + QB * EPI_LD * 4);
constexpr int SPLIT_RING = 6;                        // stages: at 0.23 us each, five on their way cover the latency of the memory behind the L2s
constexpr int SPLIT_LDS = SPLIT_RING_AT + SPLIT_RING * 12 * SPLIT_GROUP;
constexpr int gemm_lds(int EPI, int WBM, int WGM, int WGN, int NSTAGE)
{
    const int tables = WBM == 1 ? (EPI == EPI_QG || EPI == EPI_QB) * 1024 * WGM * WGN : 0;
    const int used = gelu_lds_at(WBM, WGM, WGN, NSTAGE) + tables, patch = WGM * WGN * QB * EPI_LD * (int)sizeof(float);
    return used > patch ? used : patch;
}
// NSTAGE = depth of the LDS ring (one stage being computed, NSTAGE-1 in flight); WGPC = workgroups per CU
// (the second launch bound counts waves per SIMD: WGPC workgroups of WGM*WGN waves over 4 SIMDs).
// AKM = 1: A is [K, lda] (M-contiguous rows), staged and read like a [K,N] B operand (below); lower tiles than 128 rows stage the whole lines.
// BKN = 0: B is [N, ldb] (K-contiguous rows, like A).  BKN = 1: B is [K, ldb] (N-contiguous rows); its tile is staged
// as it lies in memory and the K-contiguous MFMA operand is produced by the transposing LDS read of gfx950.
static int pace_of(long wgs, long slots, int k_per_wg);

// PROF = 1: the first wave of every workgroup also records when the workgroup's phases began and ended (wall clock) and
// how many shader cycles its main loop took: a profiling build of the same code, instantiated only in the measurement
// library (jf_prof_igemm_block_q).
// FOLD = 1: a workgroup may sum its K range in parts (p.fold_kb K blocks each, added in ascending order): the same additions as a K
// split's, without a workgroup, an epilogue and a partial result in a common buffer for every part.
// SPLIT = 2: two waves share a block, 16 rows each (split_loop, below).
template <int EPI, typename ST, int WBM, int WGM, int WGN, int NSTAGE, int WGPC, int BKN, int AKM, int PROF, int FOLD = 0, int SPLIT = 1>
__device__ __forceinline__ void igemm_body(const GemmArgs &p_in, const int logical)
{
    GemmArgs p = p_in;                                        // K-split launches narrow it to the split's K range below
    unsigned long long *const prof_buf = p_in.phases;
    const int prof_cap = p_in.phase_capacity;
    // (a macro, so that the clock is read by the one storing thread only)
#define phase(k, v) do { if (PROF && threadIdx.x == 0 && (int)blockIdx.x < prof_cap) prof_buf[(size_t)blockIdx.x * 8 + (k)] = (v); } while (0)
    if (PROF) {
        phase(0, (unsigned long long)wall_clock64());
        phase(6, (unsigned long long)__builtin_amdgcn_s_getreg((31 << 11) | 4));      // HW_ID: which CU it ran on
    }
    constexpr int NW = WGM * WGN;
    constexpr int BM = QB * WBM * WGM, BN = QB * WBN * WGN;
    constexpr int AM = AKM ? ROW_BYTES : BM;                 // rows of A that a stage holds: whole 128-byte lines of a [K,M] operand, whatever the tile's height
    constexpr int GROUP_BYTES = SPLIT > 1 ? SPLIT_GROUP : 8 * ROW_BYTES;
    constexpr int A_BYTES = AM / 8 * GROUP_BYTES;            // one stage of A
    constexpr int STAGE_BYTES = (AM + BN) / 8 * GROUP_BYTES;
    constexpr int GROUPS = (AM + BN) / 8;                    // 8-row groups (1 KiB each) per stage
    constexpr int LW = SPLIT > 1 ? 4 : NW;                   // waves that load
    constexpr int LPW = GROUPS / LW;                         // LDS-direct loads per wave per stage
    static_assert(GROUPS % LW == 0, "stage must split evenly over the waves");
    static_assert(NSTAGE >= 2 && NSTAGE <= 5, "ring depth");
    static_assert(SPLIT == 1 || (SPLIT == 2 && WBM == 1 && WGM == 1 && WGN == 2), "32x64 tiles");
    static_assert(SPLIT > 1 || !BKN || (BN == ROW_BYTES && WBN == 1), "a staged [K,N] row is one 128-byte LDS row");
    static_assert(!AKM || ROW_BYTES % BM == 0, "a staged [K,M] row is one 128-byte LDS row");
    // The epilogues that requantise want a lane to hold 16 consecutive columns of a row.  They form the transposed product (B block
    // times A block, the same integers): its registers run along the columns, see the epilogue.
    constexpr bool QUANT = EPI == EPI_Q || EPI == EPI_QG || EPI == EPI_QB || EPI == EPI_QD || EPI == EPI_QA;
    static_assert(SPLIT == 1 || QUANT, "the halves of a block meet as the transposed product");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    typedef __attribute__((address_space(3))) unsigned char lds_u8;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loader = WBM == 1 && wave_id >= NW * SPLIT;    // a wave that fetches for the others
    unsigned char *const ring_lds = smem + (SPLIT > 1 ? SPLIT_RING_AT : 0);
    const int load_wave = WBM == 1 ? wave_id % LW : wave_id;
    const int wave = SPLIT > 1 ? wave_id / SPLIT % NW : load_wave, part = wave_id % SPLIT;     // (SPLIT: the wave's block and its part of it)
    const int wm = wave % WGM, wn = wave / WGM;

    int tile_m, tile_n, split;
    tile_at(logical, p.tiles_m, p.tiles_n, EPI == EPI_FP && p.splits > 1, tile_m, tile_n, split);
    int kb_base = 0;                                          // first K block of this workgroup (scale indices count from 0)
    if (EPI == EPI_FP && p.splits > 1) {                      // uniform: the same problem on a K range, fp32 partial output
        kb_base = split * p.kb_per_split;
        const int kbn = (p.K / QB - kb_base) < p.kb_per_split ? (p.K / QB - kb_base) : p.kb_per_split;
        p.A += AKM ? (size_t)kb_base * QB * (size_t)p.lda : (size_t)kb_base * QB;
        p.B += BKN ? (size_t)kb_base * QB * (size_t)p.ldb : (size_t)kb_base * QB;
        p.K = kbn * QB;
        p.C = reinterpret_cast<float *>(p.C) + (size_t)split * (size_t)p.M * (size_t)p.N;
        p.out_dtype = JF_FP_F32;
    }
    const int m0 = p.m_base + tile_m * BM, n0 = tile_n * BN;
    const int SM = p.M / QB, SN = p.N / QB;
    const int nkb = p.K / QB;
    const int nstages = (nkb + KB_STAGE - 1) / KB_STAGE;

    // ---- global -> LDS, without passing through registers ------------------------------------
    // A stage in LDS is (BM+BN) rows of 128 bytes (A rows first).  One load instruction of one wave
    // moves 8 rows: lane l supplies the address of one 16-byte chunk and the hardware writes it to
    // LDS at (base + 16*l), i.e. row l/8, slot l%8.  To keep the later 16-byte operand reads free of
    // bank conflicts, slot c' of row r holds global chunk c' ^ ((r>>1)&7); the permutation stays
    // inside the row's 128-byte segment, so every instruction still reads 8 full 128-byte lines.
    // Address split: the 8-row group of load j is wave-uniform (scalar base pointer, advanced by 128 bytes per
    // stage on the scalar ALU); the lane contributes a fixed offset (its row of the group, its swizzled chunk).
    // The vector ALU is the bottleneck of this kernel, so the loads must not cost vector instructions.
    static_assert(NW % 2 == 0, "the chunk swizzle of a lane must not depend on the load index");
    const int lrow = lane >> 3;
    // (SPLIT: chunk c of row r of a group at slot c ^ ((r>>1)&3), groups 64 bytes apart: also free of conflicts, and a K block's
    // operands lie 64 bytes from those of the one two before)
    const int gchunk = SPLIT > 1 ? (lane & 7) ^ ((lane >> 4) & 3) : (lane & 7) ^ (((load_wave & 1) * 4 + (lane >> 4)) & 7);     // global chunk this lane fetches
    // A as [K,M]: as for B as [K,N] below (8 K rows x 128 M bytes per load, slot c' of row r holds chunk c' ^ r)
    const int m0_line = AKM ? m0 & ~(AM - 1) : m0;            // (first column of the lines)
    const int km_chunk = (m0_line + (((lane & 7) ^ lrow) << 4)) < p.M ? ((lane & 7) ^ lrow) : 0;
    const unsigned loff_a = AKM ? (unsigned)lrow * (unsigned)p.lda + km_chunk * 16
                                : (unsigned)lrow * (unsigned)p.lda + gchunk * 16;
    // B as [K,N]: a load moves 8 K rows x 128 N bytes (group g of a stage = K rows 8g .. 8g+7 of the stage).  Slot c'
    // of row r holds global chunk c' ^ r, which makes the transposing reads below conflict-free.  Chunks beyond N (partial
    // tile) fetch the tile's first chunk instead (never used).
    const int kn_chunk = (n0 + (((lane & 7) ^ lrow) << 4)) < p.N ? ((lane & 7) ^ lrow) : 0;
    // (SPLIT: rows of 64 bytes, 16 of them a group, chunk c of row r at slot c ^ ((r>>2)&3))
    constexpr int KN_ROWS = SPLIT > 1 ? 16 : 8;
    const int kn_row = SPLIT > 1 ? lane >> 2 : lrow;
    const int kn_at = SPLIT > 1 ? (n0 + (((lane & 3) ^ (lane >> 4)) << 4) < p.N ? (lane & 3) ^ (lane >> 4) : 0) : kn_chunk;
    const unsigned loff_b = BKN ? (unsigned)kn_row * (unsigned)p.ldb + kn_at * 16
                                : (unsigned)lrow * (unsigned)p.ldb + gchunk * 16;
    const int8_t *gbase[LPW];      // wave-uniform: first byte of the group's first row in the stage issued next
    bool is_a[LPW];
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        const int grp = load_wave + j * LW;
        is_a[j] = grp < AM / 8;
        if (BKN && !is_a[j]) {
            const int k0 = (grp - AM / 8) * KN_ROWS;                     // K row of the stage (redirected at issue time if beyond K)
            gbase[j] = p.B + (size_t)k0 * (size_t)p.ldb + n0;
        } else if (AKM && is_a[j]) {
            gbase[j] = p.A + (size_t)(grp * 8) * (size_t)p.lda + m0_line;
        } else {
            int r0 = (is_a[j] ? m0 : n0) + (is_a[j] ? grp : grp - AM / 8) * 8;
            if (r0 >= (is_a[j] ? p.M : p.N)) r0 = is_a[j] ? m0 : n0;   // groups of a partial tile: any valid group
            gbase[j] = (is_a[j] ? p.A : p.B) + (size_t)r0 * (size_t)(is_a[j] ? p.lda : p.ldb);
        }
    }
    // Scales.  A K block of a wave needs the NBLK products sa * sb * 2^26 (see accumulate()), wave-uniform.  They are formed once
    // per stage: lanes 0..31 fetch the A-side and lanes 32..63 the B-side scale of product l % (4 NBLK) (K block of the stage,
    // block) of a stage, LDS-direct, one stage ahead of its operands; during the stage before, each lane multiplies its pair and
    // leaves the product in a private patch, from which one broadcast read per K block returns the block's products.  Per
    // stage 2 conversions, 2 multiplications and 2 LDS operations, where multiplying the scales at every K block took 12
    // conversions and 16 multiplications, 28 of the 290 vector instructions of a stage (XL forward 8192x1600x6400, binary16
    // scales: 162 -> 154 us; 8192^3, binary32: 985 -> 966 us).  Not through registers: a load of the compiler's own makes it
    // wait for every load in flight when the value is used, the stages ahead included.
    constexpr int NBLK = WBM * WBN;
    static_assert(NBLK == 2 || NBLK == 1, "one or two products per K block and wave");
    constexpr int SC_SLOT = 256;                              // a ring slot of a wave's fetched scales; its products follow all of them
    static_assert(WBM == 1 || NSTAGE <= 3, "8-bit word offsets of the paired scale read");
    unsigned char *const scale_patch = smem + NSTAGE * STAGE_BYTES + wave * (2 * NSTAGE * SC_SLOT);
    const int s_prod = lane % (KB_STAGE * NBLK), s_blk = s_prod % NBLK, s_kb = s_prod / NBLK;
    const bool s_is_b = lane >= 32;
    const unsigned char *const s_base = reinterpret_cast<const unsigned char *>(s_is_b ? p.sb : p.sa);
    unsigned s_off, s_last, s_step;                           // byte offsets: in the stage fetched next, of the last K block, per stage
    {
        // (clamped for partial tiles: those blocks are never stored)
        int i = s_is_b ? n0 / QB + wn * WBN + s_blk % WBN : m0 / QB + wm * WBM + s_blk / WBN;
        const int lim = s_is_b ? SN : SM, ks = s_is_b ? p.sb_ks : p.sa_ks, is = s_is_b ? p.sb_is : p.sa_is;
        i = i < lim ? i : lim - 1;
        s_off = (unsigned)((s_kb + kb_base) * ks + i * is) * (unsigned)sizeof(ST);
        s_last = (unsigned)((nkb - 1 + kb_base) * ks + i * is) * (unsigned)sizeof(ST);
        s_step = (unsigned)(KB_STAGE * ks) * (unsigned)sizeof(ST);
    }
    // WBM = 1: all of a block's products at once, before the main loop, into a table of the wave: lane l those of the K blocks l,
    // l + 64, ...  (SPLIT: a table of the block, which its waves fill and read together)
    constexpr bool TABLE = WBM == 1;
    float *const table = reinterpret_cast<float *>(smem + (SPLIT > 1 ? 0 : NSTAGE * STAGE_BYTES)) + wave * ((nkb + KB_STAGE - 1) / KB_STAGE * KB_STAGE + KB_STAGE);
    auto make_table = [&] {
        const int mi = m0 / QB + wm < SM ? m0 / QB + wm : SM - 1, ni = n0 / QB + wn < SN ? n0 / QB + wn : SN - 1;
        const ST *ta = reinterpret_cast<const ST *>(p.sa) + (size_t)mi * p.sa_is, *tb = reinterpret_cast<const ST *>(p.sb) + (size_t)ni * p.sb_is;
        for (int k = lane + WAVE * part; k < nkb; k += WAVE * SPLIT) table[k] = (SPLIT > 1 ? -1.0f : 1.0f) * ((float)ta[(size_t)(k + kb_base) * p.sa_ks] * (float)tb[(size_t)(k + kb_base) * p.sb_ks]) * 67108864.0f;
    };
    // the scales of the next stage (one after the other) into ring slot `slot`; K blocks beyond the last: the last one again
    auto issue_scales = [&](auto slot_c) {
        if (EPI == EPI_S32 || TABLE) return;
        const unsigned char *const src = s_base + (s_off < s_last ? s_off : s_last);
        const unsigned dst = (unsigned)(uintptr_t)(lds_u8 *)scale_patch + decltype(slot_c)::value * SC_SLOT;
        // a binary16 scale is fetched with the 16-bit form (zero-extended into the lane's LDS word): exactly the
        // element's two bytes are read, whatever the parity of its index or the length of the array
        if (sizeof(ST) == 4)
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(dst) : "memory", "m0");
        else
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_ushort %0, off" ::"v"(src), "s"(dst) : "memory", "m0");
        s_off += s_step;
    };
    const unsigned sc_rd = (unsigned)(uintptr_t)(lds_u8 *)scale_patch + (lane & 31) * 4, sc_wr = (unsigned)(uintptr_t)(lds_u8 *)scale_patch + NSTAGE * SC_SLOT + lane * 4;
    v2i s_pair;                                               // the lane's two scales, between read_scales and put_products
    auto read_scales = [&](auto slot_c) {
        if (EPI == EPI_S32) return;
        constexpr int W = decltype(slot_c)::value * (SC_SLOT / 4);
        v2i &dst = s_pair;
        const unsigned src = sc_rd;
        asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(dst) : "v"(src), "n"(W), "n"(W + 32));
    };
    auto put_products = [&](auto slot_c) {                    // the read has been waited for
        if (EPI == EPI_S32) return;
        v2i &pair = s_pair;
        const unsigned dst = sc_wr;
        asm volatile("" : "+v"(pair));
        auto value = [](int bits) -> float {
            if (sizeof(ST) == 4) return __int_as_float(bits);
            return (float)__builtin_bit_cast(half_t, (uint16_t)bits);
        };
        const float t = (value(pair.x) * value(pair.y)) * 67108864.0f;
        asm volatile("ds_write_b32 %0, %1 offset:%2" ::"v"(dst), "v"(t), "n"(decltype(slot_c)::value * SC_SLOT) : "memory");
    };

    constexpr int A_LOADS = (AM / 8) / LW;                    // loads 0 .. A_LOADS-1 of a wave fetch A rows, the rest B rows
    static_assert((AM / 8) % LW == 0, "a load instruction fetches rows of one operand");
    // FULL: the stage has all KB_STAGE K blocks (every stage but a short last one)
    auto issue_stage_as = [&](int stage, unsigned slot, auto full_c) {       // slot: stage % NSTAGE
        constexpr bool FULL = decltype(full_c)::value;
        const unsigned slot_lds = (unsigned)(uintptr_t)(lds_u8 *)ring_lds + slot * STAGE_BYTES;
        const int kb0 = stage * KB_STAGE;
        // asm: scalar base + 32-bit lane offset is the addressing mode that costs no vector instruction, and the
        // compiler does not choose it by itself here.  M0 holds the LDS destination of an LDS-direct load.
        unsigned la = loff_a, lb = loff_b;
        if (!FULL && kb0 + (gchunk >> 1) >= nkb) {            // chunks of missing K blocks: the stage's first block again
            if (!AKM) la -= (unsigned)(gchunk >> 1) * QB;
            if (!BKN) lb -= (unsigned)(gchunk >> 1) * QB;
        }
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const int grp = load_wave + j * LW;
            const int8_t *base;                                // wave-uniform
            if (BKN && j >= A_LOADS) {
                base = gbase[j];
                gbase[j] += (size_t)(KB_STAGE * QB) * (size_t)p.ldb;
                // K rows of a missing K block: the stage's first group again
                if (!FULL && kb0 * QB + (grp - AM / 8) * KN_ROWS >= p.K) base -= (size_t)((grp - AM / 8) * KN_ROWS) * (size_t)p.ldb;
            } else if (AKM && j < A_LOADS) {
                base = gbase[j];
                gbase[j] += (size_t)(KB_STAGE * QB) * (size_t)p.lda;
                if (!FULL && kb0 * QB + grp * 8 >= p.K) base -= (size_t)(grp * 8) * (size_t)p.lda;
            } else {
                base = gbase[j];
                gbase[j] += KB_STAGE * QB;
            }
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         ::"v"(j < A_LOADS ? la : lb), "s"(base), "s"(slot_lds + (unsigned)grp * (unsigned)GROUP_BYTES) : "memory", "m0");
        }
    };
    auto issue_stage = [&](int stage, unsigned slot) {        // stage < nstages, one after the other
        if (stage < nkb / KB_STAGE) issue_stage_as(stage, slot, std::true_type{});
        else issue_stage_as(stage, slot, std::false_type{});
    };

    // ---- operand fetch addresses ----------------------------------------------------------------
    // MFMA operand layout: lane l holds row l%32 of the block and K bytes 16*(l/32) .. +15, i.e. chunk
    // 2*kb + l/32 of the stage row.  Both operands use the same mapping, so one offset per K block.
    // (Ring slot, block index and the A/B split are compile-time offsets folded into the instruction.)
    lds_u8 *const lds = (lds_u8 *)smem;
    unsigned fa_u[KB_STAGE], fb_u[KB_STAGE];          // per-lane LDS addresses (ring slot 0), fixed for the whole kernel
#pragma unroll
    for (int kb = 0; kb < KB_STAGE; ++kb) {
        const unsigned fo = (lane & 31) * ROW_BYTES + (((2 * kb + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4);
        fa_u[kb] = (unsigned)(uintptr_t)lds + fo + (wm * WBM * QB) * ROW_BYTES;
        fb_u[kb] = (unsigned)(uintptr_t)lds + A_BYTES + fo + (wn * WBN * QB) * ROW_BYTES;
    }
    // B staged as [K,N]: ds_read_b64_tr_b8 works on groups of 16 lanes; lane i of a group receives byte (i & 7) of the
    // 8-byte rows addressed by lanes (i>>3), (i>>3)+2, ... (i>>3)+14 of the group.  Lanes 2q and 2q+1 address K row q
    // of an 8-row group at N bytes 0..7 and 8..15 of a 16-column strip, so lane i gets 8 consecutive K values of
    // column i: the MFMA operand (lane l: column l%32, K bytes 16*(l/32) .. +15) is two such reads (K rows +0..7, +8..15).
    // The K block and the half are immediates, so one address register serves all of a stage.
    unsigned fb_kn = 0;
    if (BKN) {
        const int g = lane >> 4, r = lane & 15, rho = r >> 1;
        const int c = 2 * wn * WBN + (g & 1);                                    // 16-byte chunk of the N strip
        fb_kn = (unsigned)(uintptr_t)lds + A_BYTES + (g >> 1) * 2048 + ((rho * 8 + (c ^ rho)) << 4) + 8 * (r & 1);
    }
    unsigned fa_km[WBM];                                                             // A staged as [K,M]: the same, per block
#pragma unroll
    for (int i = 0; i < WBM; ++i) {
        const int g = lane >> 4, r = lane & 15, rho = r >> 1;
        const int c = 2 * ((m0 - m0_line) / QB + wm * WBM + i) + (g & 1);
        fa_km[i] = AKM ? (unsigned)(uintptr_t)lds + (g >> 1) * 2048 + ((rho * 8 + (c ^ rho)) << 4) + 8 * (r & 1) : 0u;
    }
    // product patch of this wave: a uniform address, parked in a vector register once (LDS reads take a VGPR address)
    unsigned sc_v;
    {
        const unsigned sc_u = (unsigned)(uintptr_t)(lds_u8 *)scale_patch + NSTAGE * SC_SLOT;
        asm volatile("v_mov_b32 %0, %1" : "=v"(sc_v) : "s"(sc_u));
    }

    // ---- accumulators ------------------------------------------------------------------------
    float acc[WBM][WBN][16];
    v16i iacc[WBM][WBN];
#pragma unroll
    for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j) {
#pragma unroll
            for (int v = 0; v < 16; ++v) { acc[i][j][v] = 0.0f; iacc[i][j][v] = 0; }
        }
    // block indices of this wave's scales (clamped for partial tiles: those blocks are never stored)
    int mb[WBM], nb[WBN];
#pragma unroll
    for (int i = 0; i < WBM; ++i) { mb[i] = m0 / QB + wm * WBM + i; mb[i] = mb[i] < SM ? mb[i] : SM - 1; }
#pragma unroll
    for (int j = 0; j < WBN; ++j) { nb[j] = n0 / QB + wn * WBN + j; nb[j] = nb[j] < SN ? nb[j] : SN - 1; }

    // EPI_QA: the lane's 16 elements of x1 of the wave's block i.  With one block per wave they are on their way during the main loop (the
    // waves that multiply wait for no load in it), with two each while the block before is worked on.
    v4i x1_raw[4];
    auto fetch_x1 = [&](int i) {
        const size_t at = (size_t)(m0 + (wm * WBM + i) * QB + (lane & 31)) * p.N + n0 + wn * QB + (lane >> 5) * 16;
        if (p.x1_dtype == JF_FP_F32) {
            const v4i *src = reinterpret_cast<const v4i *>(reinterpret_cast<const float *>(p.x1) + at);
#pragma unroll
            for (int k = 0; k < 4; ++k) x1_raw[k] = src[k];
        } else {
            const v4i *src = reinterpret_cast<const v4i *>(reinterpret_cast<const uint16_t *>(p.x1) + at);
            x1_raw[0] = src[0]; x1_raw[1] = src[1];
            x1_raw[2] = x1_raw[3] = v4i{0, 0, 0, 0};
        }
    };

    // ---- main loop ----------------------------------------------------------------------------
    // The whole ring is filled up front; afterwards the loads of stage s+NSTAGE are issued when the last K block
    // of stage s has been read.  Operand fragments and scales of K block k+1 are read from LDS into a second set
    // of registers BEFORE the products of K block k are issued, so the LDS pipe works while the wave multiplies
    // and accumulates; without this all waves of a SIMD queue at the LDS together and then compute together.
    constexpr int LOADS = LPW + (EPI != EPI_S32 && !TABLE ? 1 : 0);     // LDS-direct loads per wave and stage
    const int nfull = nkb / KB_STAGE;                         // stages with all KB_STAGE blocks
    const int ktail = nkb - nfull * KB_STAGE;                 // K blocks of the short last stage (0: none)
    issue_scales(std::integral_constant<int, 0>{});
    if constexpr (SPLIT > 1) {
        if (loader) {
#pragma unroll 1
            for (int s = 0; s < SPLIT_RING && s < nstages; ++s) issue_stage(s, (unsigned)s);
        }
    } else static_for<0, NSTAGE>([&](auto slot_c) {
        constexpr int SLOT = decltype(slot_c)::value;
        if (SLOT < nstages && (!TABLE || loader)) {
            issue_stage(SLOT, (unsigned)SLOT);
            // (ring slot 0 holds the first stage's scales until they are read, below)
            if (SLOT + 1 < NSTAGE) issue_scales(std::integral_constant<int, (SLOT + 1) % NSTAGE>{});
        }
    });

    // The fragment reads are written as asm so that they stay where they are and so that the wait for them can
    // name a count: the compiler, tracking them itself, waits for ALL outstanding LDS reads (the prefetch included)
    // on every other K block.  LDS reads of a wave return in order, so "at most FETCH_OPS outstanding" after issuing
    // the next K block's reads means that the current K block's have arrived.
    typedef float scale_vec __attribute__((ext_vector_type(2)));
    v4i fa_reg[2][WBM], fb_reg[2][WBN];
    scale_vec sc_raw[2];
    constexpr int FETCH_OPS = (AKM ? 2 : 1) * WBM + (BKN ? 2 : 1) * WBN + (EPI != EPI_S32 ? 1 : 0);
    static_assert(2 * FETCH_OPS <= 15, "lgkmcnt is a 4-bit counter");
    // pa/pb: this lane's fragment addresses for the K block (ring slot 0); psc: the wave's product patch;
    // slot_bytes: compile-time offset of the ring slot in the tile ring; sc_off: of the K block's products in the patch
    // kn_base: runtime offset of the ring slot for the transposing reads (0 where the slot is in the immediates)
    auto fetch = [&](const unsigned pa, const unsigned pb, const unsigned kn_base, const unsigned psc, auto slot_bytes_c,
                     auto kn_off_c, auto sc_off_c, auto buf_c) {
        constexpr int BUF = decltype(buf_c)::value;
        constexpr int SB = decltype(slot_bytes_c)::value, SC = decltype(sc_off_c)::value;
        // the instruction's offset field has 16 bits: slots beyond that are reached through the address register
        constexpr int HI = (SB + (WBM > WBN ? WBM : WBN) * QB * ROW_BYTES) > 65535 ? SB : 0;
        const unsigned pa2 = pa + HI, pb2 = pb + HI;
        constexpr int KO = decltype(kn_off_c)::value;         // slot + K block offset of a [K,N] / [K,M] staging
        constexpr int KHI = KO + 1024 > 65535 ? KO : 0;
        if (AKM) {
#pragma unroll
            for (int i = 0; i < WBM; ++i) {
                const unsigned pakm = fa_km[i] + kn_base + KHI;
                v2i lo, hi;
                asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(lo) : "v"(pakm), "n"(KO - KHI));
                asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(hi) : "v"(pakm), "n"(KO - KHI + 1024));
                fa_reg[BUF][i] = v4i{lo.x, lo.y, hi.x, hi.y};
            }
        } else {
#pragma unroll
            for (int i = 0; i < WBM; ++i)
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa_reg[BUF][i]) : "v"(pa2), "n"(SB - HI + i * (QB * ROW_BYTES)));
        }
        if (BKN) {
            const unsigned pbkn = fb_kn + kn_base + KHI;
            v2i lo, hi;
            asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(lo) : "v"(pbkn), "n"(KO - KHI));
            asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(hi) : "v"(pbkn), "n"(KO - KHI + 1024));
            fb_reg[BUF][0] = v4i{lo.x, lo.y, hi.x, hi.y};
        } else {
#pragma unroll
            for (int j = 0; j < WBN; ++j)
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb_reg[BUF][j]) : "v"(pb2), "n"(SB - HI + j * (QB * ROW_BYTES)));
        }
        if (EPI != EPI_S32) {
            scale_vec &dst = sc_raw[BUF];
            if (NBLK == 2) {
                asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(psc), "n"(SC));
            } else {
                float one;
                asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(one) : "v"(psc), "n"(SC));
                dst.x = one;
            }
        }
    };
    // wait until at most `n` LDS reads are outstanding, and tie register set BUF to that point in program order
    auto fetched = [&](auto n_c, auto buf_c) {
        constexpr int BUF = decltype(buf_c)::value, N = decltype(n_c)::value;
        __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));        // lgkmcnt(N) only
#pragma unroll
        for (int i = 0; i < WBM; ++i) asm volatile("" : "+v"(fa_reg[BUF][i]));
#pragma unroll
        for (int j = 0; j < WBN; ++j) asm volatile("" : "+v"(fb_reg[BUF][j]));
        if (EPI != EPI_S32) { scale_vec &r = sc_raw[BUF]; asm volatile("" : "+v"(r)); }
    };
    // Products and scale-accumulate of one K block (global index kbg) from register set CUR.
    // The matrix pipe and the vector ALU do not run concurrently on this part, and a product needs about 40 cycles
    // before the vector ALU can read it.  So the accumulation lags the products by one: product n is issued, THEN
    // product n-1 (long finished) is converted and accumulated.  (d_pend, sab_pend) carry the lagging product across
    // K blocks and stages; the first accumulation adds 0*0 and the last product is accumulated after the loop.
    v16i d_pend = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    float sab_pend = 0.0f;
    auto accumulate = [&](auto blk_c) {
        constexpr int i = decltype(blk_c)::value / WBN, j = decltype(blk_c)::value % WBN;
        float t[16];
#pragma unroll
        for (int v = 0; v < 16; ++v)                          // = d * 2^-26, exactly (asm: the compiler adds a 32-bit literal, twice the code bytes)
            asm("v_subrev_f32_e32 %0, 0.15915494, %1" : "=v"(t[v]) : "v"(d_pend[v]));
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_fmaf(sab_pend, t[v], acc[i][j][v]);
        // pin the accumulation here: the optimiser would otherwise postpone it past the next K blocks and keep their
        // products alive in registers it does not have
#pragma unroll
        for (int v = 0; v < 16; ++v) asm volatile("" : "+v"(acc[i][j][v]));
    };
    // the same of one block with everything as arguments
    auto compute_block = [&](const v4i &fa, const v4i &fb, const float sab_new) {
        v16i d_new;
        if constexpr (QUANT) asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0x3e22f983" : "=&v"(d_new) : "v"(fb), "v"(fa));
        else asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0x3e22f983" : "=&v"(d_new) : "v"(fa), "v"(fb));
        __builtin_amdgcn_sched_barrier(0);
        accumulate(std::integral_constant<int, 0>{});
        // (a copy of its own, made here: the register the product was read into is the target of the next read by the time it is used)
        asm volatile("v_mov_b32_e32 %0, %1" : "=v"(sab_pend) : "v"(sab_new));
        __builtin_amdgcn_sched_barrier(0);
        d_pend = d_new;
    };
    auto compute = [&](auto cur_c, const int kbg) {
        constexpr int CUR = decltype(cur_c)::value;
        if (EPI == EPI_S32) {
#pragma unroll
            for (int i = 0; i < WBM; ++i)
#pragma unroll
                for (int j = 0; j < WBN; ++j)
                    iacc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa_reg[CUR][i], fb_reg[CUR][j], iacc[i][j], 0, 0, 0);
        } else {
            static_for<0, NBLK>([&](auto n_c) {
                constexpr int n = decltype(n_c)::value, i = n / WBN, j = n % WBN;
                // asm: as a builtin operand the constant is hoisted into 16 registers instead of being encoded inline.
                // The compiler therefore does not know this is an MFMA; its result is first read by the accumulate()
                // AFTER the one below (32 vector instructions and another MFMA later), far beyond the wait states
                // a vector read of an MFMA result needs.
                v16i d_new;
                v4i &fa = fa_reg[CUR][i], &fb = fb_reg[CUR][j];
                if constexpr (QUANT) asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0x3e22f983" : "=&v"(d_new) : "v"(fb), "v"(fa));
                else asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0x3e22f983" : "=&v"(d_new) : "v"(fa), "v"(fb));
                const float sab_new = sc_raw[CUR][n];
                __builtin_amdgcn_sched_barrier(0);
                accumulate(std::integral_constant<int, (n + NBLK - 1) % NBLK>{});
                __builtin_amdgcn_sched_barrier(0);
                d_pend = d_new;
                sab_pend = sab_new;
            });
        }
    };
    // FOLD.  At the end of a part: the lagging product is accumulated, the accumulators are added to what this lane has left in p.fold
    // before (a wave's values lie block by block, 16 bytes per lane) and start from zero again.  The first K block of the next stage is on
    // its way into register set 0: it is waited for here, since the compiler may move those registers about.
    static_assert(!FOLD || (EPI == EPI_FP && WBM == 2), "weight gradients");
    int folds = 0;
    float *const fold_base = FOLD ? p.fold + ((size_t)logical * NW + wave) * (NBLK * QB * QB) : nullptr;   // (wave-uniform)
    auto fold_lane = [&]() -> unsigned {                      // this lane's first value (made anew: not a register over the main loop)
        unsigned l;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
        return l * 4;
    };
    auto add_parts = [&] {
        const float *const fold_at = fold_base + fold_lane();
#pragma unroll
        for (int i = 0; i < WBM; ++i)
#pragma unroll
            for (int j = 0; j < WBN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const v4f t = *reinterpret_cast<const v4f *>(fold_at + ((i * WBN + j) * 4 + g) * (4 * WAVE));
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[i][j][4 * g + v] = t[v] + acc[i][j][4 * g + v];
                }
    };
    auto end_part = [&] {
        fetched(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
        accumulate(std::integral_constant<int, NBLK - 1>{});
        sab_pend = 0.0f;
        if (folds > 0) add_parts();
        float *const fold_at = fold_base + fold_lane();
#pragma unroll
        for (int i = 0; i < WBM; ++i)
#pragma unroll
            for (int j = 0; j < WBN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    v4f t;
#pragma unroll
                    for (int v = 0; v < 4; ++v) { t[v] = acc[i][j][4 * g + v]; acc[i][j][4 * g + v] = 0.0f; }
                    *reinterpret_cast<v4f *>(fold_at + ((i * WBN + j) * 4 + g) * (4 * WAVE)) = t;
                }
#pragma unroll
        for (int v = 0; v < 16; ++v) d_pend[v] = 0;
        ++folds;
    };
    // Loads retire in order: a stage (and the scales of the one after it) has landed once only the loads of the Y stages
    // issued after it (up to `last`) are outstanding.  Near the end of K, with fewer stages behind it than usual, everything is waited for.
    auto wait_stage = [&](int last, auto younger_c) {
        constexpr int Y = decltype(younger_c)::value;
        if (Y == 0 || last >= nstages) JF_WAIT_VMCNT(0);
        else JF_WAIT_VMCNT(Y * LOADS);
    };
    auto wait_behind = [&](const int n) {                      // the loads of n stages may be outstanding (SPLIT)
        static_for<0, SPLIT_RING>([&](auto n_c) { if (n == decltype(n_c)::value) JF_WAIT_VMCNT(decltype(n_c)::value * LPW); });
    };
    using c0 = std::integral_constant<int, 0>;
    if constexpr (TABLE) {
        if (!loader) {
            make_table();
            if constexpr (SPLIT > 1) {                         // the waves of a block share its table: each one's part is written before the barrier
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0xC07F);
            }
        } else if (SPLIT > 1) wait_behind(SPLIT_RING < nstages ? SPLIT_RING - 1 : nstages - 1);
        else wait_stage(NSTAGE - 1, std::integral_constant<int, NSTAGE - 1>{});           // stage 0 has landed
        if constexpr (EPI == EPI_QA) { if (!loader && part == 0 && m0 + wm * QB < p.M && n0 + wn * QB < p.N) fetch_x1(0); }   // (the wave that goes on to the epilogue)
    } else {
        if (NSTAGE - 1 >= nstages) JF_WAIT_VMCNT(0);
        else JF_WAIT_VMCNT((NSTAGE - 1) * LOADS - (EPI != EPI_S32 ? 1 : 0));      // stage 0 and the scales of stage 1 have landed
        read_scales(c0{});
        __builtin_amdgcn_s_waitcnt(0xC07F);                    // lgkmcnt(0) only
        put_products(c0{});
        if (NSTAGE - 1 < nstages) issue_scales(c0{});          // stage NSTAGE, behind the operands of stage NSTAGE - 1
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();                              // bare: __syncthreads() would drain every load
    asm volatile("" ::: "memory");
    // A wave whose blocks all lie beyond M or N (the ragged edge of the tile grid: GPT-2 XL's 1600 columns are 12.5
    // tiles) keeps its part in the loads and barriers of the workgroup but neither reads operands nor multiplies: the
    // SIMD it sits on is left to the waves of the other resident workgroup.  ACTIVE = false is that walk.
    const bool wave_active = m0 + wm * (WBM * QB) < p.M && n0 + wn * (WBN * QB) < p.N;        // wave-uniform
    // which of the CU's two workgroup slots this is: the base of its LDS allocation (the low field of the LDS_ALLOC
    // register; its size field starts at bit 12)
    const bool second_slot = (__builtin_amdgcn_s_getreg((31 << 11) | 6) & 0xFFF) != 0;
    // (not QUANT, EPI_QA or SPLIT)
    float *const patch = reinterpret_cast<float *>(smem + (SPLIT > 1 ? NW * 4 * (TABLE_KB + KB_STAGE) : 0)) + wave * (QB * EPI_LD);
    long long prof_c0 = 0;
    if (PROF) { phase(1, (unsigned long long)wall_clock64()); prof_c0 = clock64(); }
    auto main_loop = [&](auto active_c, auto pace_c) {
    constexpr bool ACTIVE = decltype(active_c)::value;
    constexpr int PACE = decltype(pace_c)::value;
    if constexpr (ACTIVE) fetch(fa_u[0], fb_u[0], 0u, sc_v, c0{}, c0{}, c0{}, c0{});

    int s0 = 0;
    auto stages_to = [&](const int stop) {
    for (; s0 < stop; s0 += NSTAGE) static_for<0, NSTAGE>([&](auto slot_c) {
        constexpr int SLOT = decltype(slot_c)::value;         // ring slot of this stage, a compile-time constant
        constexpr int NEXT_SLOT = (SLOT + 1) % NSTAGE;
        const int s = s0 + SLOT;
        if (s >= nfull) return;
        static_for<0, KB_STAGE>([&](auto kb_c) {
            constexpr int kb = decltype(kb_c)::value;
            constexpr int CUR = kb & 1, NXT = CUR ^ 1;
            if constexpr (kb == KB_STAGE - 1) {
                if (s + 1 < nstages) {
                    // Stage hand-over.  This wave's LDS reads of stage s are complete (lgkmcnt 0) and stage s+1 has
                    // landed; after the barrier that holds for every wave, so (a) stage s+1 may be read and (b) the
                    // ring slot of stage s may be overwritten by the loads of stage s+NSTAGE.
                    __builtin_amdgcn_s_waitcnt(0xC07F);       // lgkmcnt(0) only
                    wait_stage(s + NSTAGE - 1, std::integral_constant<int, NSTAGE - 2>{});
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    if (s + NSTAGE < nstages) {
                        issue_stage(s + NSTAGE, (unsigned)SLOT);
                        issue_scales(std::integral_constant<int, NEXT_SLOT>{});      // of stage s + NSTAGE + 1
                    }
                }
                // unconditional: past the last stage it reads bytes of the ring that nobody uses
                if constexpr (ACTIVE)
                    fetch(fa_u[0], fb_u[0], 0u, sc_v, std::integral_constant<int, NEXT_SLOT * STAGE_BYTES>{},
                          std::integral_constant<int, NEXT_SLOT * STAGE_BYTES>{}, std::integral_constant<int, NEXT_SLOT * SC_SLOT>{},
                          std::integral_constant<int, NXT>{});
            } else {
                if constexpr (ACTIVE)
                    fetch(fa_u[kb + 1], fb_u[kb + 1], 0u, sc_v, std::integral_constant<int, SLOT * STAGE_BYTES>{},
                          std::integral_constant<int, SLOT * STAGE_BYTES + (kb + 1) * 4096>{},
                          std::integral_constant<int, SLOT * SC_SLOT + (kb + 1) * NBLK * 4>{}, std::integral_constant<int, NXT>{});
                if constexpr (ACTIVE && kb == 0) read_scales(std::integral_constant<int, NEXT_SLOT>{});
            }
            // The arbiter of a SIMD serves its oldest wave first, so the older of two resident workgroups runs about 1.4
            // times as fast as the younger one and the second wave of a workgroup on a SIMD trails the first by a quarter
            // of a stage.  PACE_EVEN: priority rises with the K block of the stage (and falls back at the next stage):
            // all four waves of a SIMD advance together.  PACE_ORDERED: the workgroup in the CU's second LDS slot always
            // goes before the one in the first, and inside a workgroup the wave that is behind goes first.
            if constexpr (PACE == PACE_EVEN) __builtin_amdgcn_s_setprio(kb);
            if constexpr (PACE == PACE_ORDERED && kb == 0) { if (second_slot) __builtin_amdgcn_s_setprio(3); else __builtin_amdgcn_s_setprio(1); }
            if constexpr (PACE == PACE_ORDERED && kb == 2) { if (second_slot) __builtin_amdgcn_s_setprio(2); else __builtin_amdgcn_s_setprio(0); }
            if constexpr (ACTIVE) {
                fetched(std::integral_constant<int, FETCH_OPS + (kb == 0 && EPI != EPI_S32 ? 1 : 0)>{}, std::integral_constant<int, CUR>{});
                __builtin_amdgcn_sched_barrier(0);            // the reads above stay above the products below,
                compute(std::integral_constant<int, CUR>{}, s * KB_STAGE + kb);
                __builtin_amdgcn_sched_barrier(0);            // and K blocks are scheduled one by one (register pressure)
                if constexpr (kb == 1) put_products(std::integral_constant<int, NEXT_SLOT>{});     // the next stage's
            }
        });
    });
    };
    if constexpr (FOLD && ACTIVE) {
        const int part = p.fold_kb > 0 ? p.fold_kb / KB_STAGE : 0x3fffffff;        // stages of a part: whole turns of the ring
        for (int end = part; s0 < nfull; end += part) {
            stages_to(end < nfull ? end : nfull);
            if (end < nfull || (end == nfull && ktail)) end_part();
        }
    } else {
        stages_to(nfull);
    }
    if (ACTIVE && ktail) {
        // short last stage (K not a multiple of 128): its first K block is already on its way to register set 0
        const unsigned slot = (unsigned)(nfull % NSTAGE);
        static_for<0, KB_STAGE - 1>([&](auto kb_c) {
            constexpr int kb = decltype(kb_c)::value;
            constexpr int CUR = kb & 1;
            if (kb < ktail) {
                if (kb > 0)
                    fetch(fa_u[kb] + slot * STAGE_BYTES, fb_u[kb] + slot * STAGE_BYTES, slot * STAGE_BYTES,
                          sc_v + slot * SC_SLOT, c0{}, std::integral_constant<int, kb * 4096>{}, std::integral_constant<int, kb * NBLK * 4>{},
                          std::integral_constant<int, CUR>{});
                fetched(c0{}, std::integral_constant<int, CUR>{});
                compute(std::integral_constant<int, CUR>{}, nfull * KB_STAGE + kb);
            }
        });
    }
    };
    // WBM = 1.  A wave that multiplies is (nearly) alone on its SIMD, so what counts is the length of its own chain: a vector
    // instruction takes 4.1 cycles there, an LDS read 15, an LDS-direct load 25 to 64 (four waves that load at once wait for each
    // other) and a branch 27 to 120, all of it in sequence.  So the loads are left to four waves of their own, the products of the
    // scales come from a table, operands are read two K blocks at a time, two ahead, and a turn of the ring has no branch.
    // 228 cycles per K block, and per launch, us, before | after: 32x768x768 6.6 | 5.7, 512x768x3072 17.7 | 12.8, 1248x768x3072
    // 17.9 | 13.0, 2048x768x768 8.4 | 7.6.
    auto load_loop = [&] {
        unsigned slot = 0;
        auto hand_over = [&](int s, auto steady_c) {
            // stage s + 1 has landed; behind the barrier every wave holds all of stage s in registers: its slot may be overwritten
            if constexpr (decltype(steady_c)::value) JF_WAIT_VMCNT((NSTAGE - 2) * LOADS);
            else wait_stage(s + NSTAGE - 1, std::integral_constant<int, NSTAGE - 2>{});
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr (decltype(steady_c)::value) issue_stage_as(s + NSTAGE, slot, std::true_type{});
            else if (s + NSTAGE < nstages) issue_stage(s + NSTAGE, slot);
            slot = slot + 1 == NSTAGE ? 0 : slot + 1;
        };
        int s = 0;
        for (; s + NSTAGE < nfull; ++s) hand_over(s, std::true_type{});
        for (; s + 1 < nstages; ++s) hand_over(s, std::false_type{});
    };
    auto table_loop = [&] {
        typedef float v2f __attribute__((ext_vector_type(2)));
        v4i fa2[2][2], fb2[2][2];
        v2f pr[2];
        const std::integral_constant<int, 0> p0;
        const std::integral_constant<int, 1> p1;
        if (!wave_active) {
            for (int s = 0; s + 1 < nstages; ++s) __builtin_amdgcn_s_barrier();
            return;
        }
        unsigned tab;                                           // products of the stage in ring slot 0
        {
            const unsigned u = (unsigned)(uintptr_t)(lds_u8 *)reinterpret_cast<unsigned char *>(table);
            asm volatile("v_mov_b32 %0, %1" : "=v"(tab) : "s"(u));
        }
        // K blocks 2 pair, 2 pair + 1 of a stage into register set `pair`; extra: run-time offsets of operands and products
        auto fetch_pair = [&](auto pair_c, auto slot_c, unsigned extra, unsigned extra_tab) {
            constexpr int PAIR = decltype(pair_c)::value, SLOT = decltype(slot_c)::value, SB = SLOT * STAGE_BYTES;
            static_assert(SPLIT > 1 || (NSTAGE - 1) * STAGE_BYTES + (BKN ? (KB_STAGE - 1) * 4096 + 1024 : 0) < 65536, "offsets of 16 bits");
            v2f &t = pr[PAIR];
            const unsigned pt = tab + extra_tab;
            asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(t) : "v"(pt), "n"(SLOT * KB_STAGE * 4 + 8 * PAIR));
            static_for<0, 2>([&](auto i_c) {
                constexpr int I = decltype(i_c)::value, kb = 2 * PAIR + I;
                v4i &a = fa2[PAIR][I], &b = fb2[PAIR][I];
                const unsigned pa = (AKM ? fa_km[0] : fa_u[kb]) + extra, pb = (BKN ? fb_kn : fb_u[kb]) + extra;
                if (AKM) {
                    v2i lo, hi;
                    asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(lo) : "v"(pa), "n"(SB + kb * 4096));
                    asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(hi) : "v"(pa), "n"(SB + kb * 4096 + 1024));
                    a = v4i{lo.x, lo.y, hi.x, hi.y};
                } else {
                    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a) : "v"(pa), "n"(SB));
                }
                if (BKN) {
                    v2i lo, hi;
                    asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(lo) : "v"(pb), "n"(SB + kb * 4096));
                    asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(hi) : "v"(pb), "n"(SB + kb * 4096 + 1024));
                    b = v4i{lo.x, lo.y, hi.x, hi.y};
                } else {
                    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(b) : "v"(pb), "n"(SB));
                }
            });
        };
        auto arrived = [&](auto pair_c) {                       // every outstanding read: the pair's
            constexpr int PAIR = decltype(pair_c)::value;
            __builtin_amdgcn_s_waitcnt(0xC07F);
            static_for<0, 2>([&](auto i_c) {
                v4i &a = fa2[PAIR][decltype(i_c)::value], &b = fb2[PAIR][decltype(i_c)::value];
                asm volatile("" : "+v"(a), "+v"(b));
            });
            v2f &t = pr[PAIR];
            asm volatile("" : "+v"(t));
        };
        // a stage that is not the last one (and therefore whole), in ring slot SLOT
        auto stage = [&](auto slot_c) {
            constexpr int NEXT_SLOT = (decltype(slot_c)::value + 1) % NSTAGE;
            arrived(p0);
            fetch_pair(p1, slot_c, 0u, 0u);
            __builtin_amdgcn_sched_barrier(0);
            compute_block(fa2[0][0], fb2[0][0], pr[0][0]);
            compute_block(fa2[0][1], fb2[0][1], pr[0][1]);
            arrived(p1);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr (NEXT_SLOT == 0) tab += NSTAGE * KB_STAGE * 4;
            fetch_pair(p0, std::integral_constant<int, NEXT_SLOT>{}, 0u, 0u);
            __builtin_amdgcn_sched_barrier(0);
            compute_block(fa2[1][0], fb2[1][0], pr[1][0]);
            compute_block(fa2[1][1], fb2[1][1], pr[1][1]);
        };
        fetch_pair(p0, p0, 0u, 0u);
        int s = 0;
        for (; s + NSTAGE < nstages; s += NSTAGE) static_for<0, NSTAGE>(stage);
        static_for<0, NSTAGE - 1>([&](auto slot_c) {
            if (s + decltype(slot_c)::value + 1 < nstages) stage(slot_c);
        });
        // the last stage: its first K blocks are on their way
        const int left = nkb - (nstages - 1) * KB_STAGE;
        const unsigned slot = (unsigned)(nstages - 1 - s);
        arrived(p0);
        if (left > 2) fetch_pair(p1, p0, slot * STAGE_BYTES, slot * (KB_STAGE * 4));
        __builtin_amdgcn_sched_barrier(0);
        compute_block(fa2[0][0], fb2[0][0], pr[0][0]);
        if (left > 1) compute_block(fa2[0][1], fb2[0][1], pr[0][1]);
        if (left > 2) {
            arrived(p1);
            compute_block(fa2[1][0], fb2[1][0], pr[1][0]);
            if (left > 3) compute_block(fa2[1][1], fb2[1][1], pr[1][1]);
        }
    };
    auto split_loads = [&] {
        int s = 0;
        auto hand_over = [&](auto behind_c) {                  // stage s + 1 has landed: at most the loads of so many stages are outstanding
            JF_WAIT_VMCNT(decltype(behind_c)::value * LPW);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        int slot = 0;
#pragma unroll 1
        for (; s + SPLIT_RING < nstages; ++s) {
            hand_over(std::integral_constant<int, SPLIT_RING - 2>{});
            issue_stage(s + SPLIT_RING, (unsigned)slot);
            slot = slot + 1 == SPLIT_RING ? 0 : slot + 1;
        }
        const int left = nstages - 2 - s;                      // stages behind stage s + 1
        static_for<0, SPLIT_RING - 1>([&](auto n_c) {
            constexpr int BEHIND = SPLIT_RING - 2 - decltype(n_c)::value;
            if (BEHIND <= left) hand_over(std::integral_constant<int, BEHIND>{});
        });
    };
    // SPLIT.  With fewer blocks than SIMDs the vector ALU idles for half of table_loop: a wave alone on its SIMD issues every 4.1 cycles,
    // and 32 vector instructions per K block in one chain are what the launch waits for.  Two waves share a block: each forms the
    // products of 16 rows and STRIPS x 16 columns (v_mfma_i32_16x16x32_i8: the same integers) and accumulates them in the same chain over
    // K, 16 vector instructions per K block.  One turn per stage, and nothing unrolled beyond two of them: code that is executed once
    // costs an instruction fetch per 64 bytes.
    constexpr int STRIPS = 2;
    auto split_loop = [&] {
        if (!wave_active) {
            for (int s = 0; s + 1 < nstages; ++s) __builtin_amdgcn_s_barrier();
            return;
        }
        // operand addresses of the current slot.  Lane l holds row (column) l%16 of its strip and K bytes 8*(l/16) .. +7 of a K block:
        // qa[i], qb[i] for K blocks i, i + 2 (a second strip: an offset); as [K,N] qb[strip] (a group of 16 lanes reads 8 K rows of
        // 16 columns, as for fb_kn)
        unsigned qa[2], qb[2], tab;
        {
            const int g = lane >> 4, r = lane & 15;
            const unsigned base = (unsigned)(uintptr_t)(lds_u8 *)ring_lds, row = (r >> 3) * GROUP_BYTES + (r & 7) * ROW_BYTES + 8 * (g & 1);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const unsigned slot = ((2 * i + (g >> 1)) ^ ((r >> 1) & 3)) << 4;
                qa[i] = base + part * 2 * GROUP_BYTES + row + slot;
                qb[i] = base + A_BYTES + wn * 4 * GROUP_BYTES + row + slot;
                if (BKN) {
                    const int k = 8 * g + (r >> 1);
                    qb[i] = base + A_BYTES + (k >> 4) * GROUP_BYTES + (k & 15) * 64 + (((2 * wn + i) ^ ((k >> 2) & 3)) << 4) + 8 * (r & 1);
                }
            }
            const unsigned u = (unsigned)(uintptr_t)(lds_u8 *)reinterpret_cast<unsigned char *>(table);
            asm volatile("v_mov_b32 %0, %1" : "=v"(tab) : "s"(u));
        }
        // operands and products of a whole stage per register set: they are read while the stage before is multiplied
        typedef float v4f_t __attribute__((ext_vector_type(4)));
        v2i fa[2][KB_STAGE], fb[2][KB_STAGE][STRIPS];
        v4f_t pr[2];
        constexpr int READS = 1 + KB_STAGE * (1 + STRIPS);     // LDS reads of a stage
        auto fetch_one = [&](auto set_c, auto n_c) {           // the n-th of them, of the current slot
            constexpr int SET = decltype(set_c)::value, N = decltype(n_c)::value, kb = (N - 1) / (1 + STRIPS), J = (N - 1) % (1 + STRIPS) - 1;
            if constexpr (N == 0) {
                v4f_t &t = pr[SET];
                const unsigned pt = tab;
                asm volatile("ds_read_b128 %0, %1" : "=v"(t) : "v"(pt));
            } else if constexpr (J < 0) {
                v2i &a = fa[SET][kb];
                const unsigned pa = qa[kb & 1];
                asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(a) : "v"(pa), "n"(64 * (kb >> 1)));
            } else {
                v2i &b = fb[SET][kb][J];
                const unsigned pb = BKN ? qb[J] : qb[kb & 1];
                if (BKN) asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(b) : "v"(pb), "n"(kb * 2 * GROUP_BYTES));
                else asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(b) : "v"(pb), "n"(64 * (kb >> 1) + J * 2 * GROUP_BYTES));
            }
        };
        auto arrived = [&](auto set_c) {
            constexpr int SET = decltype(set_c)::value;
            __builtin_amdgcn_s_waitcnt(0xC07F);
            v4f_t &t = pr[SET];
            asm volatile("" : "+v"(t));
            static_for<0, KB_STAGE>([&](auto kb_c) {
                v2i &a = fa[SET][decltype(kb_c)::value];
                asm volatile("" : "+v"(a));
                static_for<0, STRIPS>([&](auto j_c) {
                    v2i &b = fb[SET][decltype(kb_c)::value][decltype(j_c)::value];
                    asm volatile("" : "+v"(b));
                });
            });
        };
        // The products lead the accumulation by one K block.  0.15915494 - (0x3e22f983 + d) = -d * 2^-26, exactly, against a negated
        // factor: the product of accumulate() (this way round the constant is an inline one for the compiler too).
        constexpr int ONE = 0x3e22f983;
        const v4i one = {ONE, ONE, ONE, ONE};
        v4i lag[STRIPS];
        float lag_s = 0.0f, t[4 * STRIPS];
#pragma unroll
        for (int j = 0; j < STRIPS; ++j) lag[j] = one;
        auto unbias = [&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
#pragma unroll
            for (int v = 0; v < 4; ++v) t[4 * J + v] = __int_as_float(ONE) - __int_as_float(lag[J][v]);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
#pragma unroll
            for (int v = 4 * J; v < 4 * J + 4; ++v) acc[0][0][v] = __builtin_fmaf(lag_s, t[v], acc[0][0][v]);
            __builtin_amdgcn_sched_barrier(0);
        };
        // One K block.  AHEAD: with the first two K blocks of a stage go the reads of the next stage, which then have the time of the other
        // two to arrive.  (Spread evenly, one for every four vector instructions, 20 cycles more per K block: an LDS read takes 12 to 16
        // cycles of a wave that is alone on its SIMD, wherever it stands.)
        auto product = [&](auto set_c, auto kb_c, auto ahead_c) {
            constexpr int SET = decltype(set_c)::value, kb = decltype(kb_c)::value;
            static_for<0, STRIPS>([&](auto j_c) {              // (four vector instructions fill the 16 cycles of each)
                constexpr int J = decltype(j_c)::value;
                const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, fb[SET][kb][J]), __builtin_bit_cast(long, fa[SET][kb]), one, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (decltype(ahead_c)::value && kb < 2 && J == 0) {
                    constexpr int HALF = (READS + 1) / 2;
                    static_for<kb * HALF, (kb == 0 ? HALF : READS)>([&](auto n_c) { fetch_one(std::integral_constant<int, SET ^ 1>{}, n_c); });
                    __builtin_amdgcn_sched_barrier(0);
                }
                unbias(j_c);
                lag[J] = d;
            });
            static_for<0, STRIPS>(add);
            lag_s = pr[SET][kb];
        };
        int slot = 0;
        auto stage = [&](auto set_c) {                         // a stage that is not the last one (and therefore whole)
            constexpr int SET = decltype(set_c)::value;
            arrived(set_c);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            slot = slot + 1 == SPLIT_RING ? 0 : slot + 1;
            const unsigned step = slot == 0 ? (unsigned)-((SPLIT_RING - 1) * STAGE_BYTES) : (unsigned)STAGE_BYTES;
            qa[0] += step; qa[1] += step; qb[0] += step; qb[1] += step; tab += KB_STAGE * 4;
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, KB_STAGE>([&](auto kb_c) { product(set_c, kb_c, std::true_type{}); });
        };
        const std::integral_constant<int, 0> set0;
        const std::integral_constant<int, 1> set1;
        int n = nstages - 1;                                   // the last stage is in set 0
        if (n & 1) static_for<0, READS>([&](auto n_c) { fetch_one(set1, n_c); });
        else static_for<0, READS>([&](auto n_c) { fetch_one(set0, n_c); });
#pragma unroll 1
        while (n > 0) {
            if (!(n & 1)) { stage(set0); --n; }
            stage(set1);
            --n;
        }
        const int left = nkb - (nstages - 1) * KB_STAGE;
        arrived(set0);
        static_for<0, KB_STAGE>([&](auto kb_c) { if (decltype(kb_c)::value < left) product(set0, kb_c, std::false_type{}); });
        static_for<0, STRIPS>(unbias);
        static_for<0, STRIPS>(add);
        // [row][column] of the block
        float *const at = patch + (part * 16 + (lane & 15)) * EPI_LD + 4 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < STRIPS; ++j)
            *reinterpret_cast<v4f *>(at + 16 * j) = v4f{acc[0][0][4 * j], acc[0][0][4 * j + 1], acc[0][0][4 * j + 2], acc[0][0][4 * j + 3]};
    };
    if constexpr (SPLIT > 1) {
        if (loader) split_loads();
        else split_loop();
        __syncthreads();                                       // the halves meet in the patch; the first wave of a block goes on with it
        if (loader || part > 0 || !wave_active) return;
#pragma unroll
        for (int v = 0; v < 16; ++v)
            acc[0][0][v] = patch[(lane & 31) * EPI_LD + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)];
    }
    else if constexpr (TABLE) { if (loader) load_loop(); else table_loop(); }
    else if (!wave_active) main_loop(std::false_type{}, std::integral_constant<int, PACE_HARDWARE>{});
    else if (WBM == 2 && p.pace == PACE_EVEN) main_loop(std::true_type{}, std::integral_constant<int, PACE_EVEN>{});
    else if (WBM == 2 && p.pace == PACE_ORDERED) main_loop(std::true_type{}, std::integral_constant<int, PACE_ORDERED>{});
    else main_loop(std::true_type{}, std::integral_constant<int, PACE_HARDWARE>{});
    __builtin_amdgcn_s_waitcnt(0xC07F);                        // the last, unused prefetch must land before its registers are reused
    float lane_max[WBM][WBN];                                  // largest magnitude of this lane's results, per block   (QUANT)
    bool nonfinite = false;                                    // wave-uniform: some result is infinite or NaN   (QUANT)
    if constexpr (EPI == EPI_QA && WBM == 2) { if (wave_active) fetch_x1(0); }
    if (EPI != EPI_S32 && wave_active && !loader) {
        if constexpr (SPLIT == 1) accumulate(std::integral_constant<int, NBLK - 1>{});
        if constexpr (FOLD) { if (folds > 0) add_parts(); }
        // The scaled factor sa*sb*2^26 overflows when sa*sb >= 2^102.  An infinite factor leaves every accumulator
        // it touches infinite or NaN (inf*0 included), so "some accumulator of the wave is not finite" catches all such
        // cases; the wave then recomputes its blocks the plain way (operands straight from memory, zero accumulator
        // input, v_cvt_f32_i32, unscaled factor), which also reproduces results that really are infinite.
        // (A requantising epilogue needs the largest magnitude anyway: taken with the maximum that keeps a NaN, it is the check.)
        auto largest = [&](auto nan_c) {
            float all = 0.0f;
#pragma unroll
            for (int i = 0; i < WBM; ++i)
#pragma unroll
                for (int j = 0; j < WBN; ++j) {
                    float m = 0.0f;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float t = __builtin_fabsf(acc[i][j][v]);
                        m = decltype(nan_c)::value ? __builtin_elementwise_maximum(m, t) : fmaxf(m, t);
                    }
                    lane_max[i][j] = m;
                    all = __builtin_elementwise_maximum(all, m);
                }
            return all;
        };
        bool again;
        if constexpr (QUANT) {
            const float all = largest(std::true_type{});
            again = __ballot(!(all < __builtin_inff())) != 0;
        } else {
            float chk = 0.0f;
#pragma unroll
            for (int i = 0; i < WBM; ++i)
#pragma unroll
                for (int j = 0; j < WBN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) chk = __builtin_fmaf(acc[i][j][v], 0.0f, chk);
            again = __ballot(chk != chk) != 0;
        }
        if (__builtin_expect(again, 0)) {
            const ST *const sa_t = reinterpret_cast<const ST *>(p.sa), *const sb_t = reinterpret_cast<const ST *>(p.sb);
            static_for<0, NBLK>([&](auto blk_c) {              // compile-time block index: no indexed register arrays
                constexpr int blk = decltype(blk_c)::value, i = blk / WBN, j = blk % WBN;
                const size_t arow = (size_t)(mb[i] * QB + (lane & 31)), bcol = (size_t)(nb[j] * QB + (lane & 31));
                float r[16];
#pragma unroll
                for (int v = 0; v < 16; ++v) r[v] = 0.0f;
#pragma unroll 1
                for (int kb = 0; kb < nkb; ++kb) {
                    const int k0 = kb * QB + 16 * (lane >> 5);
                    v4i fa;
                    if (AKM) {
                        const int8_t *src = p.A + (size_t)k0 * (size_t)p.lda + arow;
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            unsigned w = 0;
#pragma unroll 1
                            for (int q = 0; q < 4; ++q, src += p.lda) w |= (unsigned)(uint8_t)*src << (8 * q);
                            fa[c] = (int)w;
                        }
                    } else {
                        fa = *reinterpret_cast<const v4i *>(p.A + arow * (size_t)p.lda + k0);
                    }
                    v4i fb;
                    if (BKN) {
                        const int8_t *src = p.B + (size_t)k0 * (size_t)p.ldb + bcol;
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            unsigned w = 0;
#pragma unroll 1
                            for (int q = 0; q < 4; ++q, src += p.ldb) w |= (unsigned)(uint8_t)*src << (8 * q);
                            fb[c] = (int)w;
                        }
                    } else {
                        fb = *reinterpret_cast<const v4i *>(p.B + bcol * (size_t)p.ldb + k0);
                    }
                    const v16i z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                    const v16i d = QUANT ? __builtin_amdgcn_mfma_i32_32x32x32_i8(fb, fa, z, 0, 0, 0)
                                         : __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, z, 0, 0, 0);
                    const float sab = (float)sa_t[(kb + kb_base) * p.sa_ks + mb[i] * p.sa_is] * (float)sb_t[(kb + kb_base) * p.sb_ks + nb[j] * p.sb_is];
#pragma unroll
                    for (int v = 0; v < 16; ++v) r[v] = __builtin_fmaf(sab, (float)d[v], r[v]);
                    if (FOLD && p.fold_kb > 0 && (kb + 1) % p.fold_kb == 0 && kb + 1 < nkb) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) { acc[i][j][v] = kb + 1 == p.fold_kb ? r[v] : acc[i][j][v] + r[v]; r[v] = 0.0f; }
                    }
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = FOLD && folds > 0 ? acc[i][j][v] + r[v] : r[v];
            });
            if constexpr (QUANT) { nonfinite = true; largest(std::false_type{}); }
        }
    }
    if (PROF) { phase(2, (unsigned long long)wall_clock64()); phase(7, (unsigned long long)(clock64() - prof_c0)); }
    if (p.pace != PACE_HARDWARE) __builtin_amdgcn_s_setprio(0);
    if constexpr (SPLIT == 1 && (!QUANT || (EPI == EPI_QA && WBM == 1))) __syncthreads();    // the epilogue reuses the ring as scratch
    if (loader) return;
    if (PROF) phase(3, (unsigned long long)wall_clock64());

    // ---- epilogue ------------------------------------------------------------------------------------------
    // Row layout of a block, 16 consecutive columns per lane, which is what the Philox noise (8 elements per call) and 16-byte stores
    // want.  Results are stored straight from it: 16, 32 or 64 contiguous bytes per lane, two lanes per row of the block (measured
    // 1 % faster than collecting one- and two-byte outputs in a workgroup-wide LDS image of the tile and writing that out in whole rows
    // behind a barrier).
    //   QUANT: the transposed product leaves lane l with row l%32, register v with column 8*(v/4) + 4*(l/32) + v%4; eight exchanges
    //   between the lane halves make that columns 16*(l/32) .. +15.  No LDS and no barrier: a wave requantises while others of its
    //   workgroup still multiply.  (With the product the other way round the block went through a wave-private LDS patch behind a
    //   barrier of the workgroup.  us, that | this, the check for results that are not finite and the clamps saved with it:
    //   12288x3072x768 forward with GELU 77.9 | 75.6, backward through the GELU 94.4 | 90.3; 12288x768x768 23.5 | 22.6;
    //   8192x6400x1600 forward with GELU 185.9 | 183.4, backward 209.7 | 205.0; 12288x768x3072 71.7 | 71.0.)
    //   Otherwise: one block at a time goes through a wave-private LDS patch that turns the MFMA result layout
    //     (lane l, register v  <->  row 8*(v/4) + 4*(l/32) + v%4, column l%32)
    //   into lane l <-> row l/2, columns 16*(l%2) .. +15.
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const int rrow = QUANT ? lane & 31 : lane >> 1, rcol = (QUANT ? lane >> 5 : lane & 1) * 16;
    // GELU table of the wave: its scale patch (nothing is on its way there any more) or a piece of its own.  The forward's byte table is written
    // over it: by then every lane has read its entries.
    float *const gelu_tab = SPLIT > 1 ? reinterpret_cast<float *>(ring_lds) + wave * 256
                          : TABLE ? reinterpret_cast<float *>(smem + gelu_lds_at(WBM, WGM, WGN, NSTAGE)) + wave * 256 : reinterpret_cast<float *>(scale_patch);
    int *const gelu_qtab = reinterpret_cast<int *>(gelu_tab);
    if (EPI == EPI_QG || EPI == EPI_QB) JF_WAIT_VMCNT(0);
    if constexpr (EPI == EPI_QB && WBM == 2) {
        // Read again (these kernels' first argument): held over the main loop they are scalar registers that it has to do without, and what
        // it then parks in lanes costs the 64x128 tiles four vector instructions per K block.  us, held | read again: 1600x3680x1024 24.2 | 23.4,
        // 2048x3072x768 20.4 | 20.0, 1664x3072x2048 33.6 | 32.8, 7040x768x3040 45.3 | 44.4.
        typedef const __attribute__((address_space(4))) GemmArgs *KernelArgs;
        KernelArgs again = (KernelArgs)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(again));
        p.seed = again->seed; p.offset = again->offset; p.seed2 = again->seed2; p.offset2 = again->offset2;
        p.rounding = again->rounding; p.rounding2 = again->rounding2; p.gelu_approx = again->gelu_approx;
    }
    const float biasmax = (QUANT && p.biasmax) ? p.biasmax[0] : 0.0f;
    float gelu_f0 = 0.0f;                                     // gelu(+0), evaluated on the device like every table entry
    if (EPI == EPI_QG) {
        float zero = 0.0f;
        asm volatile("" : "+v"(zero));
        gelu_f0 = p.gelu_approx == JF_GELU_TANH ? gelu<JF_GELU_TANH>(zero) : gelu<JF_GELU_ERF>(zero);
    }
    // EPI_QB: the saved forward input of this wave's blocks is requested now, so that it has arrived when the
    // requantisation of the first block is done
    v4i xq_codes[WBM][WBN];
    float xq_scale[WBM][WBN];
    if (EPI == EPI_QB) {
        float zero = 0.0f;
        asm volatile("" : "+v"(zero));
        gelu_f0 = p.gelu_approx == JF_GELU_TANH ? dgelu<JF_GELU_TANH>(zero) : dgelu<JF_GELU_ERF>(zero);
#pragma unroll
        for (int i = 0; i < WBM; ++i)
#pragma unroll
            for (int j = 0; j < WBN; ++j) {
                const int bm = m0 + (wm * WBM + i) * QB, bn = n0 + (wn * WBN + j) * QB;
                if (bm < p.M && bn < p.N) {
                    xq_codes[i][j] = *reinterpret_cast<const v4i *>(p.Xq + (size_t)(bm + rrow) * p.N + bn + rcol);
                    xq_scale[i][j] = load_scale(reinterpret_cast<const ST *>(p.Xs), (bm / QB) * SN + bn / QB);
                }
            }
    }

    // 16 consecutive results of a row as float / binary16 / bfloat16 (rounded to nearest even): 64 or 32 contiguous bytes
    auto store_fp = [&](void *out, const float (&x)[16], const size_t e0) {
        if (p.out_dtype == JF_FP_F32) {
            v4f *dst = reinterpret_cast<v4f *>(reinterpret_cast<float *>(out) + e0);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v4f t = {x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
                dst[k] = t;
            }
        } else {
            v4i lo, hi;
            if (p.out_dtype == JF_FP_F16) {
                half_t h[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) h[k] = (half_t)x[k];
                lo = *reinterpret_cast<v4i *>(&h[0]); hi = *reinterpret_cast<v4i *>(&h[8]);
            } else {
                __bf16 h[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) h[k] = (__bf16)x[k];
                lo = *reinterpret_cast<v4i *>(&h[0]); hi = *reinterpret_cast<v4i *>(&h[8]);
            }
            v4i *dst = reinterpret_cast<v4i *>(reinterpret_cast<unsigned char *>(out) + e0 * 2);   // 32 of a row's 64 bytes
            dst[0] = lo; dst[1] = hi;
        }
    };
    // A block's float results from the patch in the shape that stores best: every store instruction writes 8 whole 128-byte rows of the
    // block instead of 64 separate 16-byte pieces (3-6 us off the weight gradients of GPT-2 XL; the same for 16-bit outputs, 16 rows x
    // 64 bytes per instruction, measured slower than the two 16-byte pieces per lane of the row layout)
    auto store_patch_rows = [&](void *out, const int bm, const int bn) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const int row = 8 * h + (lane >> 3), c4 = (lane & 7) * 4;
            const v4f t = *reinterpret_cast<const v4f *>(patch + row * EPI_LD + c4);
            *reinterpret_cast<v4f *>(reinterpret_cast<float *>(out) + (size_t)(bm + row) * p.N + bn + c4) = t;
        }
        wave_sync();
    };
#pragma unroll
    for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j) {
            const int bm = m0 + (wm * WBM + i) * QB, bn = n0 + (wn * WBN + j) * QB;
            const bool valid = bm < p.M && bn < p.N;          // wave-uniform
            if (!valid) continue;
            float amax = 0.0f;
            if (QUANT) amax = wave_max(lane_max[i][j]) + biasmax;
            if constexpr (!QUANT) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int r = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                    if (EPI == EPI_S32) patch[r * EPI_LD + (lane & 31)] = __int_as_float(iacc[i][j][v]);
                    else patch[r * EPI_LD + (lane & 31)] = acc[i][j][v];
                }
                wave_sync();
            }
            if (EPI == EPI_FP && p.out_dtype == JF_FP_F32) {
                store_patch_rows(p.C, bm, bn);                // (no arithmetic follows)
                continue;
            }
            float x[16];
            if constexpr (QUANT) {
                row_halves(acc[i][j], x);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const v4f t = *reinterpret_cast<const v4f *>(patch + rrow * EPI_LD + rcol + 4 * k);
                    x[4 * k] = t.x; x[4 * k + 1] = t.y; x[4 * k + 2] = t.z; x[4 * k + 3] = t.w;
                }
                wave_sync();
            }
            const size_t e0 = (size_t)(bm + rrow) * p.N + bn + rcol;
            if (EPI == EPI_S32) {
                v4i *dst = reinterpret_cast<v4i *>(reinterpret_cast<int32_t *>(p.C) + e0);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    v4i t = {__float_as_int(x[4 * k]), __float_as_int(x[4 * k + 1]),
                             __float_as_int(x[4 * k + 2]), __float_as_int(x[4 * k + 3])};
                    dst[k] = t;
                }
            } else if (EPI == EPI_FP) {
                store_fp(p.C, x, e0);
            } else {
                v4i codes = {0, 0, 0, 0};
                float scale = 0.0f;
                if (amax > 0.0f) {
                    BlockDivisor d(amax);
                    scale = d.fast ? div_by_127_in_range(amax) : amax / 127.0f;      // (uniform)
                    float t[16];
                    if (p.bias) {
#pragma unroll
                        for (int k = 0; k < 16; ++k) x[k] = x[k] + p.bias[bn + rcol + k];
                    }
#pragma unroll
                    for (int k = 0; k < 16; ++k) x[k] = 127.0f * x[k];
                    d.div16(x, t);
                    // Without a bias no |x| exceeds amax and no quotient that of amax itself, which is 127 or, for one block in
                    // eight, the number after it; the noise stays below 1/2.  So only then (and where the quotient overflows, and
                    // for results that are not finite) does any sum leave what rounds into +-127.
                    float top;
                    {
                        const float a127 = 127.0f * amax;
                        d.divn<1>(&a127, &top);
                    }
                    const bool clamp = __builtin_amdgcn_readfirstlane((p.bias != nullptr) | nonfinite | !(top <= 127.0f)) != 0;
                    if (p.rounding == JF_ROUND_STOCHASTIC) {
                        float n[16];
                        sr_noise16(p.seed, p.offset, (uint64_t)e0, n);
#pragma unroll
                        for (int k = 0; k < 16; ++k) t[k] = t[k] + n[k];
                    }
                    if (clamp) {
#pragma unroll
                        for (int k = 0; k < 16; ++k) t[k] = __builtin_amdgcn_fmed3f(t[k], -127.0f, 127.0f);
                    }
                    codes.x = (int)round_clamp_pack4<false>(t[0], t[1], t[2], t[3]);
                    codes.y = (int)round_clamp_pack4<false>(t[4], t[5], t[6], t[7]);
                    codes.z = (int)round_clamp_pack4<false>(t[8], t[9], t[10], t[11]);
                    codes.w = (int)round_clamp_pack4<false>(t[12], t[13], t[14], t[15]);
                }
                if (EPI == EPI_QB) {
                    // GELU backward of the gradient block as a reader of the stored tensor would see it (codes x the scale
                    // rounded to ST) against the saved forward input
                    const float stored = (float)(ST)scale;
                    float scale2;
                    codes = p.gelu_approx == JF_GELU_TANH
                        ? gelu_bwd_block<JF_GELU_TANH>(xq_codes[i][j], xq_scale[i][j], codes, stored, gelu_f0, gelu_tab, lane,
                                                       p.rounding2, p.seed2, p.offset2, (uint64_t)e0, &scale2)
                        : gelu_bwd_block<JF_GELU_ERF>(xq_codes[i][j], xq_scale[i][j], codes, stored, gelu_f0, gelu_tab, lane,
                                                      p.rounding2, p.seed2, p.offset2, (uint64_t)e0, &scale2);
                    scale = scale2;
                }
                if constexpr (EPI == EPI_QA) {
                    // the sum with the block as a reader of the stored tensor would dequantise it; its partial row sums, columns 0..15
                    // and 16..31 (add_kernel's order); its own requantisation
                    float y[16];
                    unpack16(codes, (float)(ST)scale, y);
                    // (one branch per type: the compiler makes a choice per element sixteen branches)
                    if (p.x1_dtype == JF_FP_F32) {
#pragma unroll
                        for (int k = 0; k < 16; ++k) y[k] = __int_as_float(x1_raw[k / 4][k % 4]) + y[k];
                    } else if (p.x1_dtype == JF_FP_F16) {
#pragma unroll
                        for (int k = 0; k < 16; ++k) y[k] = (float)__builtin_bit_cast(half_t, (uint16_t)(x1_raw[k / 8][(k / 2) % 4] >> (16 * (k & 1)))) + y[k];
                    } else {
#pragma unroll
                        for (int k = 0; k < 16; ++k) {
                            const unsigned w = (unsigned)x1_raw[k / 8][(k / 2) % 4];
                            y[k] = __uint_as_float(k & 1 ? w & 0xffff0000u : w << 16) + y[k];
                        }
                    }
                    if (i + 1 < WBM && bm + QB < p.M) fetch_x1(i + 1);
                    if (p.out_dtype == JF_FP_F32 && WBM == 2) {
                        // whole rows without a patch of the block's size and its barrier: eight at a time through the wave's scale patch
                        static_assert(EPI != EPI_QA || WBM == 1 || 2 * NSTAGE * SC_SLOT >= 8 * 128, "eight rows of 128 bytes");
#pragma unroll
                        for (int h = 0; h < 4; ++h) {
                            if ((rrow >> 3) == h) {
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    *reinterpret_cast<v4f *>(scale_patch + (rrow & 7) * 128 + (((rcol / 4 + k) ^ (rrow & 7)) << 4)) = v4f{y[4 * k], y[4 * k + 1], y[4 * k + 2], y[4 * k + 3]};
                            }
                            wave_sync();
                            const int row = lane >> 3;
                            const v4f t = *reinterpret_cast<const v4f *>(scale_patch + row * 128 + (((lane & 7) ^ row) << 4));
                            *reinterpret_cast<v4f *>(reinterpret_cast<float *>(p.y) + (size_t)(bm + 8 * h + row) * p.N + bn + (lane & 7) * 4) = t;
                            wave_sync();
                        }
                    } else if (p.out_dtype == JF_FP_F32) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) *reinterpret_cast<v4f *>(patch + rrow * EPI_LD + rcol + 4 * k) = v4f{y[4 * k], y[4 * k + 1], y[4 * k + 2], y[4 * k + 3]};
                        wave_sync();
                        store_patch_rows(p.y, bm, bn);
                    } else {
                        store_fp(p.y, y, e0);
                    }
                    if (p.rowsum) {
                        float t1 = 0.0f, t2 = 0.0f;
#pragma unroll
                        for (int k = 0; k < 16; ++k) { t1 = t1 + y[k]; t2 = __builtin_fmaf(y[k], y[k], t2); }
                        const float o1 = __shfl_xor(t1, 32, WAVE), o2 = __shfl_xor(t2, 32, WAVE);
                        if (lane < 32) {
                            p.rowsum[(size_t)(bn / QB) * p.M + bm + lane] = t1 + o1;
                            p.rowsq[(size_t)(bn / QB) * p.M + bm + lane] = t2 + o2;
                        }
                    }
                    codes = quantize16(y, 0.0f, p.rounding2, 0, 0, 0, &scale);
                }
                if (EPI == EPI_QD) {
                    // the block as a reader of the stored tensor would dequantise it: codes x the scale rounded to ST
                    float y[16];
                    unpack16(codes, (float)(ST)scale, y);
                    store_fp(p.C, y, e0);
                } else {
                    *reinterpret_cast<v4i *>(reinterpret_cast<int8_t *>(p.C) + e0) = codes;     // 16 of a row's 32 bytes
                    if (lane == 0) store_scale(reinterpret_cast<ST *>(p.sc), (bm / QB) * SN + bn / QB, scale);
                }
                if (EPI == EPI_QG) {
                    // GELU of the block as a reader of the stored tensor would see it (codes x the scale rounded to ST)
                    const float stored = (float)(ST)scale;
                    float scale2;
                    const v4i codes2 = p.gelu_approx == JF_GELU_TANH
                        ? gelu_fwd_block<JF_GELU_TANH>(codes, stored, gelu_f0, p.gelu_eps, gelu_tab, gelu_qtab, lane, &scale2)
                        : gelu_fwd_block<JF_GELU_ERF>(codes, stored, gelu_f0, p.gelu_eps, gelu_tab, gelu_qtab, lane, &scale2);
                    *reinterpret_cast<v4i *>(reinterpret_cast<int8_t *>(p.C2) + e0) = codes2;
                    if (lane == 0) store_scale(reinterpret_cast<ST *>(p.sc2), (bm / QB) * SN + bn / QB, scale2);
                }
            }
        }

    if (PROF) phase(4, (unsigned long long)wall_clock64());
    if (PROF) phase(5, (unsigned long long)wall_clock64());
#undef phase
}

template <int EPI, typename ST, int WBM, int WGM, int WGN, int NSTAGE, int WGPC, int BKN, int AKM = 0, int PROF = 0>
__global__ __launch_bounds__(gemm_threads(WBM, WGM, WGN), WGPC * gemm_threads(WBM, WGM, WGN) / 256) void igemm_nt_kernel(GemmArgs p)
{
    p.m_base = 0;
    igemm_body<EPI, ST, WBM, WGM, WGN, NSTAGE, WGPC, BKN, AKM, PROF>(p, logical_workgroup(gridDim.x, blockIdx.x, true));
}

// 32x64 tiles, two waves per block.
template <int EPI, typename ST, int BKN> __global__ __launch_bounds__(512, 4) void igemm_split_kernel(GemmArgs p)
{
    p.m_base = 0;
    igemm_body<EPI, ST, 1, 1, 2, 2, 2, BKN, 0, 0, 0, 2>(p, logical_workgroup(gridDim.x, blockIdx.x, true));
}

// Rows 0 .. m_base - 1 in 128x128 tiles, the others in 32x128 tiles (launch_gemm_mixed).
template <int EPI, typename ST, int BKN> __global__ __launch_bounds__(512, 4) void igemm_mixed_kernel(GemmArgs p)
{
    const int first_small = (p.big_tiles + 7) & ~7;           // (both parts are dealt to the XCDs from the first one on)
    const int wg = blockIdx.x;
    if (wg < first_small) {
        const int logical = logical_workgroup(p.big_tiles, wg);
        if (logical < 0) return;
        p.tiles_m = p.m_base / (4 * QB);
        p.m_base = 0;
        igemm_body<EPI, ST, 2, 2, 4, 2, 2, BKN, 0, 0>(p, logical);
    } else {
        const int logical = logical_workgroup(p.tiles_m * p.tiles_n, wg - first_small);
        if (logical < 0) return;
        p.pace = PACE_HARDWARE;                               // (no paced instances)
        igemm_body<EPI, ST, 1, 1, 4, 3, 2, BKN, 0, 0>(p, logical);
    }
}

// Several weight gradients over the same tokens in one launch (jf_wgrad_many).  Every XCD gets one contiguous run of each problem's
// work, one problem after the other, so that the XCDs finish together although the parts of the problems differ in length.  (One
// run over all problems: GPT-2 XL's four, one of them in parts a third as long, took 60 us more than the 500 they take.)
constexpr int WGRAD_MAX = 4;
struct GemmGroup {
    GemmArgs g[WGRAD_MAX];
    int end[WGRAD_MAX];       // first workgroup behind problem k, of an XCD's: ceil(work / 8) for each problem
    int n;
};
template <typename ST, bool SMALL> __device__ __forceinline__ void wgrad_group_body(const GemmGroup &grp, const int wg)
{
    const int xcd = wg & 7, at = wg >> 3;
    int k = 0, begin = 0;
#pragma unroll
    for (int i = 1; i < WGRAD_MAX; ++i)
        if (i < grp.n && at >= grp.end[i - 1]) { k = i; begin = grp.end[i - 1]; }
    const GemmArgs &p = grp.g[k];
    const int logical = logical_workgroup(p.tiles_m * p.tiles_n * p.splits, (at - begin) * 8 + xcd);
    if (logical < 0) return;
    if constexpr (SMALL) igemm_body<EPI_FP, ST, 1, 1, 4, 2, 2, 1, 1, 0>(p, logical);
    else igemm_body<EPI_FP, ST, 2, 2, 4, 2, 2, 1, 1, 0, 1>(p, logical);
}
template <typename ST> __global__ __launch_bounds__(512, 4) void igemm_wgrad_group_kernel(GemmGroup grp) { wgrad_group_body<ST, false>(grp, blockIdx.x); }

// An activation gradient (EPI_Q or EPI_QD, B as [K,N]; 32x64, 32x128 or 128x128 tiles), then weight gradients, in one launch: both gradients of
// a linear layer, or the last one of a block with all of the block's weight gradients.
enum BackwardTile { TILE_128x128, TILE_32x128, TILE_32x64 };   // of the activation gradient
struct GemmBackward {
    GemmArgs x;
    GemmGroup w;
};
template <int EPI, typename ST, int TILE, bool SMALL_W> __global__ __launch_bounds__(512, 4) void igemm_backward_kernel(GemmBackward b)
{
    const int work_x = b.x.tiles_m * b.x.tiles_n, first_w = (work_x + 7) & ~7;      // (both parts are dealt to the XCDs from the first one on)
    const int wg = blockIdx.x;
    if (wg < first_w) {
        const int logical = logical_workgroup(work_x, wg);
        if (logical >= 0) igemm_body<EPI, ST, TILE == TILE_128x128 ? 2 : 1, TILE == TILE_128x128 ? 2 : 1, TILE == TILE_32x64 ? 2 : 4, TILE == TILE_32x128 ? 3 : 2, 2, 1, 0, 0, 0, TILE == TILE_32x64 ? 2 : 1>(b.x, logical);
    } else {
        wgrad_group_body<ST, SMALL_W>(b.w, wg - first_w);
    }
}

#if JF_IN_PART(0)
// -------------------------------------------------------------------------------------------------
// int8 transpose: out[C,R] = in[R,C].  TR_ROWS x 64 tiles through LDS: 16-byte loads, the transposing LDS read of gfx950
// (ds_read_b64_tr_b8, as for the GEMM's [K,N] operands) and 16-byte stores.  The instruction works on groups of 16 lanes:
// lanes 2k and 2k+1 of a group address the 8-byte pieces [8 columns] x 2 of tile row k (k = 0..7), and lane i receives
// byte i%8 of the pieces addressed by lanes i/8, i/8 + 2, ..., i/8 + 14: column i of the 16, rows 0..7.  Two reads (rows
// +0..7, +8..15) give a lane 16 consecutive bytes of one output row.  Wave w of the workgroup takes tile columns 16w ..
// 16w+15 (16 output rows); its four lane groups take 16 tile rows each, so a store instruction writes 64 contiguous bytes
// of each of its 16 output rows, and the passes of a tall tile continue those runs.
constexpr int TR_ROWS = 64;                        // tile rows (input rows = bytes per output-row run)
__global__ __launch_bounds__(256) void transpose_s8_kernel(const int8_t *in, int8_t *out, int R, int C)
{
    __shared__ __attribute__((aligned(16))) unsigned char tile[TR_ROWS][64 + 16];
    typedef __attribute__((address_space(3))) unsigned char lds_u8;
    const int tiles_c = (C + 63) / 64;
    // Workgroups are dealt round-robin to the 8 XCDs: with 8 consecutive workgroups on 8 consecutive row tiles of one
    // column tile, every XCD walks along the columns of its own rows, so the two 64-byte halves of a 128-byte line meet
    // in one L2 (measured at 8192x6400: 17.8 us against 24.4 us with the column tile running fastest).
    const int tiles_r = (R + TR_ROWS - 1) / TR_ROWS;
    const int per = 8 * tiles_c, grp = blockIdx.x / per, rem = blockIdx.x % per;
    const int nr = (tiles_r - grp * 8) < 8 ? (tiles_r - grp * 8) : 8;
    const int tr = grp * 8 + rem % nr, tc = rem / nr;
    const int r0 = tr * TR_ROWS, c0 = tc * 64;
    const int tid = threadIdx.x;
#pragma unroll
    for (int pass = 0; pass < TR_ROWS / 64; ++pass) {
        const int row = pass * 64 + (tid >> 2), ch = tid & 3;   // 64 rows x 4 chunks of 16 bytes per pass
        v4i v = {0, 0, 0, 0};
        if (r0 + row < R && c0 + ch * 16 < C)
            v = *reinterpret_cast<const v4i *>(in + (size_t)(r0 + row) * C + c0 + ch * 16);
        *reinterpret_cast<v4i *>(&tile[row][ch * 16]) = v;
    }
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, i = lane & 15;
    const int ocol = 16 * wave + (i & 7) + 8 * (i >> 3);        // tile column this lane receives = output row
#pragma unroll
    for (int pass = 0; pass < TR_ROWS / 64; ++pass) {
        const int trow = pass * 64 + 16 * g;                    // first of the 16 tile rows of this lane group
        const unsigned addr = (unsigned)(uintptr_t)(lds_u8 *)&tile[trow + (i >> 1)][16 * wave + 8 * (i & 1)];
        v2i lo, hi;
        asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(lo) : "v"(addr));
        asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(8 * (64 + 16)));
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(lo), "+v"(hi));
        if (c0 + ocol < C && r0 + trow < R)
            *reinterpret_cast<v4i *>(out + (size_t)(c0 + ocol) * R + r0 + trow) = v4i{lo.x, lo.y, hi.x, hi.y};
    }
}

static int launch_transpose(const int8_t *in, int R, int C, int8_t *out, hipStream_t st)
{
    const int tiles = ((R + TR_ROWS - 1) / TR_ROWS) * ((C + 63) / 64);
    hipLaunchKernelGGL(transpose_s8_kernel, dim3(tiles), dim3(256), 0, st, in, out, R, C);
    return (int)hipGetLastError();
}
#endif

// more than 64 KiB of dynamic LDS has to be opted into, per function and device: once, not on every launch
// (the reference sets its attribute on every call, igemm_BlockSquare32OutputIntQuantizeBiasRowCol.cu:418)
static int allow_lds(const void *kern, int bytes, std::atomic<bool> (&opted_in)[MAX_DEVICES])
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return JF_ERR_DEVICE;
    if (!opted_in[dev].load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return (int)e;
        opted_in[dev].store(true, std::memory_order_release);
    }
    return JF_OK;
}

// Pace of the workgroups that share a CU.  Left to the hardware, the older one runs ahead: a launch ends with every CU
// half empty while the younger workgroups finish alone, at two thirds of the shared throughput (two waves per SIMD
// meeting at a barrier).  Kept in step by wave priorities (PACE_EVEN) they finish together: 5-16 % faster for launches
// of up to two rounds of workgroups.  The exception is a launch of between 1 and 1.5 rounds: there the early finishers
// are what starts the short second round early, and an even pace is 5-9 % slower than the hardware's order.  A strict
// order with fairness inside each workgroup (PACE_ORDERED) does that job 4-6 % better than the hardware when tiles are
// long (K >= 4096) and 5-16 % worse when they are short.  Beyond two rounds the schemes are within 3 % of each other,
// either way depending on shape and data: left to the hardware.  (All measured; results do not depend on the scheme.)
static int pace_of(long wgs, long slots, int k_per_wg)
{
    if (wgs > slots && 2 * wgs < 3 * slots) return k_per_wg >= 4096 ? PACE_ORDERED : PACE_HARDWARE;      // a short second round
    return wgs <= 2 * slots ? PACE_EVEN : PACE_HARDWARE;
}

template <int EPI, typename ST, int WBM, int WGM, int WGN, int NSTAGE, int WGPC, int BKN, int AKM = 0, int PROF = 0>
static int launch_gemm_cfg(const GemmArgs &a, hipStream_t st)
{
    constexpr int BM = QB * WBM * WGM, BN = QB * WBN * WGN, NT = gemm_threads(WBM, WGM, WGN);
    constexpr int SMEM = gemm_lds(EPI, WBM, WGM, WGN, NSTAGE);
    if (!device_is_gfx950()) return JF_ERR_DEVICE;
    GemmArgs p = a;
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    auto kern = igemm_nt_kernel<EPI, ST, WBM, WGM, WGN, NSTAGE, WGPC, BKN, AKM, PROF>;
    static std::atomic<bool> opted_in[MAX_DEVICES] = {};
    if (int rc = allow_lds(reinterpret_cast<const void *>(kern), SMEM, opted_in)) return rc;
    if (EPI != EPI_FP || p.splits < 1) p.splits = 1;
    p.pace = WBM == 1 ? (int)PACE_HARDWARE                    // (no paced instances: all its workgroups are resident)
                      : pace_of((long)p.tiles_m * p.tiles_n * p.splits, (long)WGPC * cu_count(), p.splits > 1 ? p.kb_per_split * QB : p.K);
    hipLaunchKernelGGL(kern, dim3(p.tiles_m * p.tiles_n * p.splits), dim3(NT), SMEM, st, p);
    return (int)hipGetLastError();
}

// A launch of 128x128 tiles that begins a short last round (of one workgroup per CU, or of two) takes that round's part of M as 32x128
// tiles, in the same launch: tiles left alone on their CUs run at two thirds of the rate and leave most of the chip idle for the whole
// length of a tile.  Rows of 128x128 tiles if so, else 0.  The line: after two (or four) big tiles per CU up to two small ones each (all of
// them resident at once), otherwise one small one each.  us, 128x128 | mixed:
//   768 wide, K = 3072: 5504 rows (258 tiles) 39.8 | 32.0, 6144 (288) 42.2 | 33.5, 12288 (576) 72.4 | 61.9; K = 768: 2048x2304 (288)
//   15.4 | 11.5, 12288x768 23.2 | 21.6; K = 1536: 11008 rows (516) 41.2 | 32.8, 13312 (624) 38.8 | 35.3, 22016 (1032) 63.0 | 56.3;
//   11008x2304x768 (1548) 50.6 | 45.9; 4224x1024x4096 (264) 52.1 | 43.0.
// Beyond it: 13824x768x1536 (648 tiles) 38.8 | 39.0, 15360 (720) 39.4 | 42.5, 8192x768x3072 (384) 43.5 | 47.5, 24576x768x1536 (1152)
// 61.7 | 61.8, 11264x3072x768 (2112, behind eight) 63.0 | 62.3.
// After three, five and so on, where half of the slots go on with a big tile, for rows of K up to 8192 only.
// Behind three 17024x768x768 (798) 28.3 | 27.2, with the GELU backward 40.7 | 36.1, x3072 84.1 | 77.3, 7680x1600x1600 (780) 47.4 | 44.6, 8064x1600x6400
// (819, 208 small) 160.9 | 158.8, 13312x1024x4096 (832, 256 small) 111.1 | 108.9, 17408x768x8192 208 | 195, x96 12.9 | 12.3; behind five 27648x768x1536 (1296) 73.5 |
// 67.3, 5376x4096x1024 (1344, 256 small) 55.3 | 52.8; behind seven 38400x768x768 (1800) 58.7 | 54.3, 9600x3072x768 (1800)
// 56.7 | 54.4, 17920x1600x6400 (1820) 344.9 | 336.4, 18048x1600x256 (1833, 208 small) 30.2 | 28.4.  A longer row: 8064x1600x12800 313 | 322.  More than one
// small tile each: 8192x1600x1600 (832 tiles, 260 small) 49.7 | 53.2, x4800 126.6 | 130.9, 13184x1600x1600 (1339, 260) 76.9 | 76.4.
// Up to two small ones each also behind four where a small tile is long enough: 23168x768x3072 (1086, 264 small) 123.2 | 115.2, 24192x768x3072
// (1134, 456) 124.4 | 120.8, 10752x1600x1600 (1092, 312) 69.7 | 66.1, 11136x1600x6400 (1131, 468) 244.7 | 231.1, 5888x3072x1536 (1104, 384) 66.7 | 66.2; K = 768
// 24192 rows 39.8 | 41.4, 5760x3072 (288 small) 40.5 | 40.1; behind six 34560x768x1536 (336) 93.9 | 93.4, 16128x1600x1600 (416) 95.4 | 98.6.
// With more rounds the gain falls slowly: behind eight 11008x3072x768 (2064) 68.2 | 63.8, 20608x1600x6400 (2093) 409 | 405, nine 12544x3072x3072 (2352) 235 | 220,
// ten 13696x3072x1600 (2568) 146.3 | 136.6, twelve 16512x3072x768 (3096) 90.8 | 86.5, sixteen 21888x3072x3072 (4104) 401 | 382.
static int mixed_big_rows(int M, int N, int K)
{
    const int rows = (M + 127) / 128, tiles_n = (N + 127) / 128, cus = cu_count();
    if (K > TABLE_KB * QB) return 0;
    const int last = (int)((long)rows * tiles_n / cus);
    for (int rounds = last > 3 ? last - 2 : 1; rounds <= last; rounds++) {      // big tiles per CU
        if (rounds >= 3 && rounds % 2 && K > 8192) continue;
        const bool two = rounds == 2 || (rounds == 4 && K >= 1536 && K <= 8192);
        const int big = rounds * cus / tiles_n;
        const long small = (long)((M - big * 128) / QB) * tiles_n;
        if (big < rows && big * tiles_n > (rounds - 1) * cus && small <= (two ? 2L : 1L) * cus) return big;
    }
    return 0;
}

template <int EPI, typename ST, int BKN> static int launch_gemm_mixed(const GemmArgs &a, int big_rows, hipStream_t st)
{
    if (!device_is_gfx950()) return JF_ERR_DEVICE;
    GemmArgs p = a;
    p.splits = 1;
    p.tiles_n = (p.N + 127) / 128;
    p.m_base = big_rows * 128;
    p.big_tiles = big_rows * p.tiles_n;
    p.tiles_m = (p.M - p.m_base) / QB;
    p.pace = pace_of(p.big_tiles, 2L * cu_count(), p.K);
    constexpr int BIG = gemm_lds(EPI, 2, 2, 4, 2), SMALL = gemm_lds(EPI, 1, 1, 4, 3), SMEM = BIG > SMALL ? BIG : SMALL;
    static std::atomic<bool> opted_in[MAX_DEVICES] = {};
    if (int rc = allow_lds(reinterpret_cast<const void *>(igemm_mixed_kernel<EPI, ST, BKN>), SMEM, opted_in)) return rc;
    const unsigned wgs = ((p.big_tiles + 7) & ~7) + p.tiles_m * p.tiles_n;
    hipLaunchKernelGGL((igemm_mixed_kernel<EPI, ST, BKN>), dim3(wgs), dim3(512), SMEM, st, p);
    return (int)hipGetLastError();
}

template <int EPI, typename ST, int BKN> static int launch_gemm_split(const GemmArgs &a, hipStream_t st)
{
    if (!device_is_gfx950()) return JF_ERR_DEVICE;
    GemmArgs p = a;
    p.splits = 1;
    p.tiles_m = p.M / QB;
    p.tiles_n = (p.N + 63) / 64;
    p.pace = PACE_HARDWARE;
    static std::atomic<bool> opted_in[MAX_DEVICES] = {};
    if (int rc = allow_lds(reinterpret_cast<const void *>(igemm_split_kernel<EPI, ST, BKN>), SPLIT_LDS, opted_in)) return rc;
    hipLaunchKernelGGL((igemm_split_kernel<EPI, ST, BKN>), dim3(p.tiles_m * p.tiles_n), dim3(512), SPLIT_LDS, st, p);
    return (int)hipGetLastError();
}

template <typename ST> int launch_wgrad_group(const GemmGroup &grp, unsigned wgs, hipStream_t st)
{
    constexpr int SMEM = gemm_lds(EPI_FP, 2, 2, 4, 2);
    static std::atomic<bool> opted_in[MAX_DEVICES] = {};
    if (int rc = allow_lds(reinterpret_cast<const void *>(igemm_wgrad_group_kernel<ST>), SMEM, opted_in)) return rc;
    hipLaunchKernelGGL(igemm_wgrad_group_kernel<ST>, dim3(wgs), dim3(512), SMEM, st, grp);
    return (int)hipGetLastError();
}

#if JF_IN_PART(0)
// out[i] = convert(part[0][i] + part[1][i] + ... + part[S-1][i]), added in ascending split order, for the four elements at i.
__device__ __forceinline__ void reduce_splits(const float *part, size_t n, int splits, void *out, int out_dtype, size_t i)
{
    if (i >= n) return;                                        // n is a multiple of 1024
    v4f t = *reinterpret_cast<const v4f *>(part + i);
    for (int s = 1; s < splits; ++s) {
        const v4f u = *reinterpret_cast<const v4f *>(part + (size_t)s * n + i);
        t.x = t.x + u.x; t.y = t.y + u.y; t.z = t.z + u.z; t.w = t.w + u.w;
    }
    if (out_dtype == JF_FP_F32) {
        *reinterpret_cast<v4f *>(reinterpret_cast<float *>(out) + i) = t;
    } else if (out_dtype == JF_FP_F16) {
        half_t h[4] = {(half_t)t.x, (half_t)t.y, (half_t)t.z, (half_t)t.w};
        *reinterpret_cast<v2i *>(reinterpret_cast<half_t *>(out) + i) = *reinterpret_cast<v2i *>(h);
    } else {
        __bf16 h[4] = {(__bf16)t.x, (__bf16)t.y, (__bf16)t.z, (__bf16)t.w};
        *reinterpret_cast<v2i *>(reinterpret_cast<__bf16 *>(out) + i) = *reinterpret_cast<v2i *>(h);
    }
}
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *part, size_t n, int splits, void *out, int out_dtype)
{
    reduce_splits(part, n, splits, out, out_dtype, ((size_t)blockIdx.x * 256 + threadIdx.x) * 4);
}

static int launch_splitk_reduce(const float *part, size_t n, int splits, void *out, int out_dtype, hipStream_t st)
{
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)(n / 1024)), dim3(256), 0, st, part, n, splits, out, out_dtype);
    return (int)hipGetLastError();
}

// What follows the weight gradients of a block, one launch: the K splits of each (as splitk_reduce_kernel) and column sums over
// per-strip terms (the gradients of the LayerNorm weights; the order of layernorm_bwd_colsum_finish_kernel: thread (g, column)
// adds the strips g, g + 32, ... ascending, then the 32 partial sums are added ascending).
struct WgradFinish {
    const float *part[WGRAD_MAX];
    void *out[WGRAD_MAX];
    size_t count[WGRAD_MAX];  // elements of gradient k
    int end[WGRAD_MAX];       // first workgroup behind gradient k (4096 elements each)
    const float *terms[WGRAD_MAX];                             // [strips][width]
    float *sum[WGRAD_MAX];
    int width[WGRAD_MAX], cend[WGRAD_MAX];                     // first workgroup behind column sum k (32 columns each)
    int splits[WGRAD_MAX];
    int n, ncol, strips, out_dtype;
};
__global__ __launch_bounds__(1024) void wgrad_finish_kernel(WgradFinish f)
{
    __shared__ float red[32][QB + 1];
    const int wg = blockIdx.x, nred = f.n > 0 ? f.end[f.n - 1] : 0;
    int k = 0, begin = 0;
    if (wg < nred) {
#pragma unroll
        for (int i = 1; i < WGRAD_MAX; ++i)
            if (i < f.n && wg >= f.end[i - 1]) { k = i; begin = f.end[i - 1]; }
        reduce_splits(f.part[k], f.count[k], f.splits[k], f.out[k], f.out_dtype, ((size_t)(wg - begin) * 1024 + threadIdx.x) * 4);
        return;
    }
    begin = nred;
#pragma unroll
    for (int i = 1; i < WGRAD_MAX; ++i)
        if (i < f.ncol && wg >= f.cend[i - 1]) { k = i; begin = f.cend[i - 1]; }
    const float *src = f.terms[k];
    const int C = f.width[k], x = threadIdx.x & 31, c = (wg - begin) * QB + x, g = threadIdx.x >> 5;
    float acc = 0.0f;
    for (int s0 = g; s0 < f.strips; s0 += 256) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) { const int s = s0 + 32 * i; v[i] = s < f.strips ? src[(size_t)s * C + c] : 0.0f; }
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = acc + v[i];
    }
    red[g][x] = acc;
    __syncthreads();
    if (g == 0) {
        float t = red[0][x];
#pragma unroll
        for (int i = 1; i < 32; ++i) t = t + red[i][x];
        f.sum[k][c] = t;
    }
}

#endif

// K split of the fp-output GEMM.  request 1: none; request > 1: that many parts (fewer if K is short); request 0: as
// many parts as it takes to give every CU two workgroups, when the tiles alone fill less than half of them.  Parts are
// whole multiples of 4 K blocks (one LDS stage), at least 16 K blocks long.
static void splitk_plan(int M, int N, int K, int request, int &splits, int &kb_per_split)
{
    const int nkb = K / QB;
    int want = request;
    if (request == 0) {
        const int tiles = ((M + 127) / 128) * ((N + 127) / 128), slots = 2 * cu_count();
        want = 2 * tiles <= slots ? slots / tiles : 1;
        if (want > 16) want = 16;
    }
    if (want > nkb / 16) want = nkb / 16;
    if (want < 1) want = 1;
    kb_per_split = ((nkb + want - 1) / want + 3) / 4 * 4;
    splits = (nkb + kb_per_split - 1) / kb_per_split;
}

// K splits of a group of weight gradients.  First one for all of them, by time: the launch takes, on the fullest CU, as many tiles as
// fall to it times their K blocks: about 0.27 us per block for a lone tile and 0.2 us per tile beyond (GPT-2 XL and small
// gradients), 3 us of ramp and epilogue per pair of tiles; parts cost a write and a read of every partial sum at about 8 TB/s (they
// stay in the caches).  Parts are at least 8 K blocks (two stages) of at least 16.
// Then, by rounding: the squared error of the sum of p parts of kb blocks grows as kb + p (each addition rounds the partial sum it has
// reached; 1 part: kb), and no gradient is summed in an order that rounds more than its own launch would (splitk_plan).  Where the
// split of the group is such a one, its workgroups sum their K range in parts themselves (FOLD, above): q parts of f blocks in each
// of p workgroups, f + q + p.  A gradient that would take more than FOLD_MAX of them (few tiles, which then end last) keeps its own
// split.  Error against float64, 768 wide over 12288 tokens, of one chain | of the parts: 3.5e-7 | 1.2e-7 to 2.1e-7.  Launch and sums, us,
// in one chain | with parts in workgroups | with a workgroup for every part | four launches of their own: 512 wide, 4096 tokens
// 42 | 52 | 55 | 87; 1024, 8192 196 | 209 | 232 | 246; 768, 12288 171 | 183 | 199 | 235; 1600, 8192 515 | 518 | 514 | 543.
// FOLD_MAX = 4 | 6 or more: 1152 wide, 8192 tokens (6 parts of one gradient) 264 | 250; = 6 or less | 8: 1024, 8192 (8 parts) 209 | 223.
struct WgradPlan {
    int splits[WGRAD_MAX], kb_per_split[WGRAD_MAX], fold_kb[WGRAD_MAX];
};
constexpr int FOLD_MAX = 6;                                    // parts inside a workgroup
static void wgrad_group_plan(int n, const int *M, const int *N, int K, WgradPlan &plan)
{
    int splits, kb_per_split;
    const int nkb = K / QB;
    long tiles = 0;
    double elems = 0;
    for (int i = 0; i < n; ++i) {
        tiles += (long)((M[i] + 127) / 128) * ((N[i] + 127) / 128);
        elems += (double)M[i] * N[i];
    }
    double best = 0;
    splits = 1; kb_per_split = nkb;
    for (int s = 1; s <= 16 && (s == 1 || (nkb >= 16 && nkb / s >= 8)); ++s) {
        const int kb = s == 1 ? nkb : ((nkb + s - 1) / s + KB_STAGE - 1) / KB_STAGE * KB_STAGE, parts = (nkb + kb - 1) / kb;
        const long per_cu = (tiles * parts + cu_count() - 1) / cu_count();
        const double t = kb * (0.2 * per_cu + (per_cu & 1 ? 0.07 : 0.0)) + 3.0 * ((per_cu + 1) / 2) + (parts > 1 ? parts * elems * 8 / 8e6 : 0.0);
        if (s == 1 || t < best) { best = t; splits = parts; kb_per_split = kb; }
    }
    for (int i = 0; i < n; ++i) {
        const auto parts = [](int p) { return p > 1 ? p : 0; };
        int own, own_kb, fold = 0;
        splitk_plan(M[i], N[i], K, 0, own, own_kb);
        const int limit = own_kb + parts(own);
        bool keep = kb_per_split + parts(splits) <= limit;
        if (!keep) {                                           // parts inside the workgroups
            constexpr int TURN = 2 * KB_STAGE;                 // (of the kernel's ring)
            if (splits == 1 && own_kb % TURN == 0) fold = own_kb;
            else for (fold = (kb_per_split - 1) / TURN * TURN; fold > 0 && fold + (kb_per_split + fold - 1) / fold + parts(splits) > limit; fold -= TURN) {}
            keep = fold > 0 && (kb_per_split + fold - 1) / fold <= FOLD_MAX;
        }
        plan.splits[i] = keep ? splits : own;
        plan.kb_per_split[i] = keep ? kb_per_split : own_kb;
        plan.fold_kb[i] = keep ? fold : 0;
    }
}

// 32x64 tiles, two waves per block: where one per CU holds them all.  us, 32x128 tiles | these: 32x768x768 5.7 | 5.3, 64x256x256 4.1 | 3.9,
// 512x768x768 (192 of them) 5.8 | 5.5, 512x768x2304 10.3 | 8.7, 416x1120x2080 (234) 9.5 | 8.3, 160x544x4096 15.4 | 12.0; B as [K,N] 512x768x768
// 6.1 | 6.1, x2304 10.8 | 9.5; with two per CU 1248x768x768 (468) 5.8 | 6.5, 1024x1024x1024 (512) 6.6 | 7.4, 1280x768x2304 (480) 10.4 | 11.2.
static long split_tiles(int M, int N) { return (long)(M / QB) * ((N + 63) / 64); }
static bool split_tiles_resident(int M, int N, int K) { return K <= TABLE_KB * QB && split_tiles(M, N) <= (long)cu_count(); }
// 64x128 tiles, one block per wave (eight waves that multiply, eight that load): where one workgroup per CU holds them all, but not one of 32x128
// each.  Both put two waves that multiply on a SIMD, but this one loads 6 KB per K block instead of 10, and what a CU can load is what
// two workgroups of 32x128 wait for.  us, 32x128 | these: 2048x768x768 7.25 | 6.98, x3072 16.6 | 15.7, 864x1824x3200 (210) 17.5 | 15.9, B as [K,N] 21.0 | 17.5,
// 640x3072x1600 (240) 12.3 | 10.9, 1024x2048x3200 (256) 19.9 | 17.9, 1664x768x768 (156) 7.19 | 6.64, 4128x256x768 (130) 7.08 | 6.78, 1056x1024x96 (136)
// 4.62 | 4.51.  A ring three deep instead of two: 2048x768x768 7.00, x3072 16.6, 1024x2048x3200 18.7.  Over 3400 drawn sizes these are 5 % faster,
// 2 to 4 % for K up to 256, 5 to 8 % above 512.  Single long rows lose with no size, pitch or layout that tells them from their neighbours: 1056x1024x6240 with B as
// [K,N] 30.1 | 33.6, 3328x288x4416 22.0 | 25.6, but 1056x1024x3072 16.5 | 16.4, 1024x1600x6400 7 % and 544x1984x5600 5 % faster; 34 of the 3400 by more than 2 %.
// Short rows stay with 32x128 where the epilogue is a large part: float results up to K = 256 (2048x544x256 5.7 | 6.0, 1024x1088x224 3 % slower), the
// GELU backward up to 128 (1664x544x128 2.5 % slower).
static bool tall_tiles_resident(int M, int N, int K)
{
    const long cus = cu_count(), cols = (N + 127) / 128;
    return K <= TABLE_KB * QB && (M + 63) / 64 * cols <= cus && (M + 31) / 32 * cols > cus;
}
static bool small_tiles_resident(int M, int N, int K)          // 32x128 tiles, two workgroups per CU
{
    return K <= TABLE_KB * QB && (long)((M + 31) / 32) * ((N + 127) / 128) <= 2L * cu_count();
}

// Tile configuration.  Large launches: 128x128 tiles, 8 waves of two blocks, a 2-deep ring and two workgroups per CU (the
// epilogue of one overlaps the main loop of the other).  A launch whose 32x128 tiles are all resident at once, two workgroups
// of 4 waves and a 3-deep ring per CU, takes those instead: its 128x128 tiles would occupy at most a quarter of the chip with
// 16 products per K block and SIMD pair in sequence, where a wave with one block is bound by the issue of its own 32 vector
// instructions per product.  Measured (one-sequence forward GEMMs, us, 128x128 | 32x128): 32x768x768 9.7 | 5.7, 512x768x3072
// 28.8 | 12.8, 512x3072x768 (384 small tiles) 10.7 | 8.4, 1248x768x768 10.7 | 6.5; beyond two per CU the larger tile's data
// reuse wins: 1248x2304x768 (702) 10.9 | 12.6.  In between: launch_gemm_mixed, and 64x128 tiles (below).
// A [K,N] B operand (and, for the weight gradient, a [K,M] A operand) is read in place.
// a_km (A given as [K,M]) exists for the weight-gradient form only: fp output, B as [K,N].
template <int EPI, typename ST, int BKN> static int launch_gemm_b(const GemmArgs &a, hipStream_t st)
{
    if constexpr (EPI != EPI_S32) {
        if constexpr (EPI != EPI_FP) { if (split_tiles_resident(a.M, a.N, a.K)) return launch_gemm_split<EPI, ST, BKN>(a, st); }
        if (a.splits <= 1 && a.K > (EPI == EPI_FP ? 256 : EPI == EPI_QB ? 128 : 0) && tall_tiles_resident(a.M, a.N, a.K))
            return launch_gemm_cfg<EPI, ST, 1, 2, 4, 2, 1, BKN>(a, st);
        if (a.splits <= 1 && small_tiles_resident(a.M, a.N, a.K))
            return launch_gemm_cfg<EPI, ST, 1, 1, 4, 3, 2, BKN>(a, st);
    }
    if constexpr (EPI == EPI_Q || EPI == EPI_QG || EPI == EPI_QB || EPI == EPI_QD || EPI == EPI_QA) {
        if (const int big = mixed_big_rows(a.M, a.N, a.K)) return launch_gemm_mixed<EPI, ST, BKN>(a, big, st);
    }
    // 64x128 tiles, four waves of two blocks, three workgroups per CU: where they are all resident at once (up to 384 big tiles), the
    // 128x128 tiles would be alone on many of their CUs, and a SIMD's waves belong to workgroups that do not wait for each other.  us,
    // 128x128 | 64x128: 7168x768x768 (336 big tiles) 15.3 | 12.8, 8192x768x768 (384) 15.4 | 13.1, x3072 43.6 | 41.0, 768x8192x2048 (384) 30.3 |
    // 27.8, 3072x1024x4096 (192) 37.5 | 34.9, 2048x1600x1600 (208) 17.6 | 16.9, 1248x2304x768 (180) 10.7 | 10.3; two rounds of them: 2560x2560x2560
    // (400) 37.1 | 47.4.  With a GELU behind it, the longest epilogues, above one big tile per CU: backward 2048x3072x768 (384) 22.0 | 19.8,
    // 1248x3072x768 (240) 15.2 | 15.6, forward 2048x3072x768 18.8 | 18.0, 3072x2048x512 (384) 16.1 | 14.9, 4096x1536x768 (384) 19.0 | 18.1, 1248x3072x768
    // 13.9 | 14.0, 640x6400x1600 (250) 20.7 | 21.8.
    if constexpr (EPI == EPI_Q || EPI == EPI_QB || EPI == EPI_QD || EPI == EPI_QA || EPI == EPI_QG) {
        const long tiles_n = (a.N + 127) / 128;
        if ((a.M + 63) / 64 * tiles_n <= 3L * cu_count() && ((EPI != EPI_QB && EPI != EPI_QG) || (a.M + 127) / 128 * tiles_n > cu_count()))
            return launch_gemm_cfg<EPI, ST, 2, 1, 4, 2, 3, BKN>(a, st);
    }
    return launch_gemm_cfg<EPI, ST, 2, 2, 4, 2, 2, BKN>(a, st);
}
template <int EPI, typename ST> int launch_gemm(const GemmArgs &a, hipStream_t st, bool b_kn, bool a_km = false)
{
    if constexpr (EPI == EPI_QG || EPI == EPI_QA) {           // the forward form only: A [M,K], B [N,K]
        if (a_km || b_kn) return JF_ERR_UNSUPPORTED;
        return launch_gemm_b<EPI, ST, 0>(a, st);
    } else if constexpr (EPI == EPI_QB) {                     // the activation-gradient form only: A [M,K], B [K,N]
        if (a_km || !b_kn) return JF_ERR_UNSUPPORTED;
        return launch_gemm_b<EPI, ST, 1>(a, st);
    } else {
        if (a_km) {
            if constexpr (EPI == EPI_FP) {
                if (b_kn) return launch_gemm_cfg<EPI, ST, 2, 2, 4, 2, 2, 1, 1>(a, st);
            }
            return JF_ERR_UNSUPPORTED;
        }
#ifdef JF_PROF_LIB
        if constexpr (EPI == EPI_Q && std::is_same<ST, float>::value) {
            if (a.phases)                                     // the profiling library: the PROF build of the same kernel
                return b_kn ? launch_gemm_cfg<EPI, ST, 2, 2, 4, 2, 2, 1, 0, 1>(a, st) : launch_gemm_cfg<EPI, ST, 2, 2, 4, 2, 2, 0, 0, 1>(a, st);
        }
#endif
        return b_kn ? launch_gemm_b<EPI, ST, 1>(a, st) : launch_gemm_b<EPI, ST, 0>(a, st);
    }
}

#ifndef JF_PROF_LIB
// x: as for a launch of its own; w: w_wgs workgroups, the longest of them k_per_part deep.
template <int EPI, typename ST, int TILE, bool SMALL_W = false> static int launch_backward(const GemmArgs &x, const GemmGroup &w, long w_wgs, int k_per_part, hipStream_t st)
{
    GemmBackward b = {x, w};
    if (SMALL_W) {
        long at = 0;
        for (int i = 0; i < w.n; ++i) {
            b.w.g[i].tiles_m = w.g[i].M / QB;
            at += ((long)b.w.g[i].tiles_m * b.w.g[i].tiles_n * w.g[i].splits + 7) / 8;
            b.w.end[i] = (int)at;
        }
        w_wgs = at * 8;
    }
    constexpr bool BIG = TILE == TILE_128x128;
    constexpr int BN = TILE == TILE_32x64 ? 64 : 128;
    b.x.tiles_m = BIG ? (x.M + 127) / 128 : x.M / QB; b.x.tiles_n = (x.N + BN - 1) / BN; b.x.splits = 1;
    const long x_wgs = ((long)b.x.tiles_m * b.x.tiles_n + 7) & ~7L;
    b.x.pace = !BIG ? (int)PACE_HARDWARE : pace_of(x_wgs + w_wgs, 2L * cu_count(), std::max(x.K, k_per_part));
    for (int i = 0; i < w.n; ++i) b.w.g[i].pace = SMALL_W ? (int)PACE_HARDWARE : b.x.pace;
    constexpr int SX = BIG ? gemm_lds(EPI, 2, 2, 4, 2) : TILE == TILE_32x128 ? gemm_lds(EPI, 1, 1, 4, 3) : SPLIT_LDS;
    constexpr int SW = SMALL_W ? 2 * 2 * 128 * ROW_BYTES + 4 * (TABLE_KB + KB_STAGE) * 4 : gemm_lds(EPI_FP, 2, 2, 4, 2), SMEM = SX > SW ? SX : SW;
    static std::atomic<bool> opted_in[MAX_DEVICES] = {};
    if (int rc = allow_lds(reinterpret_cast<const void *>(igemm_backward_kernel<EPI, ST, TILE, SMALL_W>), SMEM, opted_in)) return rc;
    hipLaunchKernelGGL((igemm_backward_kernel<EPI, ST, TILE, SMALL_W>), dim3((unsigned)(x_wgs + w_wgs)), dim3(512), SMEM, st, b);
    return (int)hipGetLastError();
}
// One launch for an activation gradient and weight gradients: neither needs the other's result, small ones leave most of the chip
// idle, and larger ones end in a round that is not full, once instead of twice.  The activation gradient's tiles, which are longer, come
// first: 32x128 where one per CU holds them all, and two per CU where K is long and a 128x128 tile would outlast everything else.  us,
// two launches | one, both gradients of a layer, rows x C_in x C_out:
//   32x128: 32x768x768 10.3 | 6.4, 512x768x2304 20.8 | 13.2, 1024x1024x1024 22.8 | 18.7, 1248x768x3072 35.6 | 31.8; two per CU
//   2048x1024x4096 55.5 | 52.5 (128x128: 59.0), 1024x1600x6400 65.7 | 56.7 (62.5);
//   128x128: 2048x768x768 23.6 | 19.4 (32x128: 21.3), 1024x2048x1024 31.8 | 25.8 (28.5), 4096x768x768 35.0 | 26.0, 4096x1024x4096 84.4 | 78.3,
//   12288x768x3072 127.5 | 119.4, 8192x1024x4096 141.4 | 138.2.
// The weight gradients in 128x128 tiles, except where one workgroup per CU holds all of the launch with theirs in 32x128 tiles, one block per wave: a
// turn of those is 0.1 us per K block where a 128x128 tile alone on its CU takes 0.27.  us, 128x128 | 32x128: 480x736x160 8.6 | 5.5, 512x512x512
// 8.7 | 5.6, 64x256x256 4.8 | 4.3, 480x192x2080 8.9 | 8.4, and with K splits 1024x256x1024 11.7 | 9.1, 4096x128x512 12.9 | 9.9; two per CU
// 256x1024x1024 7.3 | 8.6, 512x1024x1024 9.7 | 11.2, 2048x256x768 12.4 | 13.8.
// The activation gradient in 32x64 tiles beside 128x128 ones where its chain over K is the longer one: at three times as many K blocks 32x128 tiles
// (218 cycles each) and the weight gradients (0.27 us) take equally long.  32x128 | 32x64: 800x256x3680 16.8 | 13.1, 576x448x2304 12.4 | 11.0, 480x416x2304 12.1 |
// 10.0, 1024x256x2080 15.3 | 13.9, 1088x256x2016 15.0 | 14.1; not beyond the line 352x992x1056 9.2 | 9.6, 480x672x1024 9.8 | 10.1, 64x5120x192 6.15 | 6.26.
// Above three 128x128 tiles of the activation gradient per CU the rounds even out by themselves: 4096x4096x1024 (1024) 86.1 | 83.7,
// 8192x1600x4800 (832) 248.7 | 263.2, 8192x6400x1600 (3200) 359.4 | 363.9, 4096x4096x4096 (1024) 259.0 | 260.8.
static bool backward_in_one_launch(int R, int C_in, long w_wgs)
{
    return (long)((R + 127) / 128) * ((C_in + 127) / 128) <= 3L * cu_count() && w_wgs <= 0x3fffffffL;
}
template <int EPI, typename ST> int launch_backward_any(const GemmArgs &x, const GemmGroup &w, long w_wgs, int k_per_part, hipStream_t st)
{
    if (x.K <= TABLE_KB * QB) {                                // weight gradients in 32x128 tiles
        const long cus = cu_count(), narrow = split_tiles(x.M, x.N), wide = (long)(x.M / QB) * ((x.N + 127) / 128);
        long small_w = 0;
        for (int i = 0; i < w.n && small_w <= cus; ++i) {
            const GemmArgs &a = w.g[i];
            const bool fits = !a.fold_kb && (a.splits > 1 ? a.kb_per_split : a.K / QB) <= TABLE_KB;
            small_w += fits ? (long)(a.M / QB) * a.tiles_n * a.splits : cus + 1;
        }
        if (narrow + small_w <= cus) return launch_backward<EPI, ST, TILE_32x64, true>(x, w, w_wgs, k_per_part, st);
        if (wide + small_w <= cus) return launch_backward<EPI, ST, TILE_32x128, true>(x, w, w_wgs, k_per_part, st);
    }
    if (x.K > 3 * k_per_part && split_tiles_resident(x.M, x.N, x.K) && split_tiles(x.M, x.N) + w_wgs <= cu_count())
        return launch_backward<EPI, ST, TILE_32x64>(x, w, w_wgs, k_per_part, st);
    const bool small = small_tiles_resident(x.M, x.N, x.K) && (x.K > 2048 || (long)(x.M / QB) * ((x.N + 127) / 128) <= cu_count());
    if (small) return launch_backward<EPI, ST, TILE_32x128>(x, w, w_wgs, k_per_part, st);
    return launch_backward<EPI, ST, TILE_128x128>(x, w, w_wgs, k_per_part, st);
}

#ifdef JF_PART
#define JF_INST(part) JF_INST_##part
#if JF_IN_PART(0)
#define JF_INST_0
#else
#define JF_INST_0 extern
#endif
#if JF_IN_PART(1)
#define JF_INST_1
#else
#define JF_INST_1 extern
#endif
#if JF_IN_PART(2)
#define JF_INST_2
#else
#define JF_INST_2 extern
#endif
#if JF_IN_PART(3)
#define JF_INST_3
#else
#define JF_INST_3 extern
#endif
#if JF_IN_PART(4)
#define JF_INST_4
#else
#define JF_INST_4 extern
#endif
#if JF_IN_PART(5)
#define JF_INST_5
#else
#define JF_INST_5 extern
#endif
#if JF_IN_PART(6)
#define JF_INST_6
#else
#define JF_INST_6 extern
#endif
#if JF_IN_PART(7)
#define JF_INST_7
#else
#define JF_INST_7 extern
#endif
#define JF_GEMM(part, EPI, ST) JF_INST(part) template int launch_gemm<EPI, ST>(const GemmArgs &, hipStream_t, bool, bool)
#define JF_BWD(part, EPI, ST) JF_INST(part) template int launch_backward_any<EPI, ST>(const GemmArgs &, const GemmGroup &, long, int, hipStream_t)
JF_GEMM(0, EPI_S32, float);
JF_GEMM(1, EPI_FP, half_t);
JF_GEMM(1, EPI_FP, float);
JF_GEMM(2, EPI_Q, half_t);
JF_GEMM(3, EPI_Q, float);
JF_GEMM(4, EPI_QD, half_t);
JF_GEMM(5, EPI_QD, float);
JF_GEMM(6, EPI_QG, half_t);
JF_GEMM(7, EPI_QG, float);
JF_GEMM(6, EPI_QB, half_t);
JF_GEMM(7, EPI_QB, float);
JF_BWD(2, EPI_Q, half_t);
JF_BWD(3, EPI_Q, float);
JF_BWD(4, EPI_QD, half_t);
JF_BWD(5, EPI_QD, float);
JF_GEMM(0, EPI_QA, half_t);
JF_GEMM(1, EPI_QA, float);
JF_INST(1) template int launch_wgrad_group<half_t>(const GemmGroup &, unsigned, hipStream_t);
JF_INST(1) template int launch_wgrad_group<float>(const GemmGroup &, unsigned, hipStream_t);
#endif
#endif  // !JF_PROF_LIB

static int check_gemm_common(const void *A, const void *B, const void *C, int M, int N, int K, int b_layout)
{
    if (!A || !B || !C) return JF_ERR_NULL;
    if (!mult32(M) || !mult32(N) || !mult32(K)) return JF_ERR_SHAPE;
    if (b_layout != JF_B_NK && b_layout != JF_B_KN) return JF_ERR_ENUM;
    if (!aligned16(A) || !aligned16(B) || !aligned16(C)) return JF_ERR_ALIGN;
    return JF_OK;
}

}  // namespace jf

using namespace jf;

// element strides (K block, tile block) of a scale operand with `blocks` tile blocks
static bool scale_strides(int layout, int K, int blocks, int &ks, int &is)
{
    if (layout == JF_SCALES_KMAJOR) { ks = blocks; is = 1; return true; }
    if (layout == JF_SCALES_ROWMAJOR) { ks = 1; is = K / QB; return true; }
    return false;
}

// scale arrays need the natural alignment of their element type (binary16 scales are fetched one element at a time)
static bool scale_ptr_ok(const void *p, int scale_dtype)
{
    return (reinterpret_cast<uintptr_t>(p) & (scale_dtype == JF_SCALE_F32 ? 3u : 1u)) == 0;
}

#if !defined(JF_PROF_LIB) && JF_IN_PART(0)
// dX [R, C_in] = G [R, C_out] W [C_out, C_in], requantised or (dx_scales null) dequantised, scales in the tensors' own layout
static GemmArgs dgrad_args(const int8_t *G, const void *sg, const int8_t *W, const void *sw, int R, int C_in, int C_out, void *dx, void *dx_scales,
                           int dx_dtype, uint64_t seed, uint64_t offset)
{
    GemmArgs x = {};
    x.A = G; x.B = W; x.sa = sg; x.sb = sw; x.C = dx; x.sc = dx_scales; x.out_dtype = dx_dtype; x.rounding = JF_ROUND_STOCHASTIC;
    x.seed = seed; x.offset = offset; x.M = R; x.N = C_in; x.K = C_out; x.lda = C_out; x.ldb = C_in;
    x.sa_ks = 1; x.sa_is = C_out / QB; x.sb_ks = C_in / QB; x.sb_is = 1;
    return x;
}
// dW [C_out, C_in] = G^T X, in `splits` parts
static GemmArgs wgrad_args(const int8_t *G, const void *sg, const int8_t *X, const void *sx, int R, int C_in, int C_out, void *out, int out_dtype,
                           int splits, int kb_per_split)
{
    GemmArgs a = {};
    a.A = G; a.B = X; a.sa = sg; a.sb = sx; a.C = out; a.out_dtype = out_dtype; a.splits = splits; a.kb_per_split = kb_per_split;
    a.M = C_out; a.N = C_in; a.K = R; a.lda = C_out; a.ldb = C_in;
    a.sa_ks = C_out / QB; a.sa_is = 1; a.sb_ks = C_in / QB; a.sb_is = 1;
    a.tiles_m = (C_out + 127) / 128; a.tiles_n = (C_in + 127) / 128;
    return a;
}

extern "C" {

const char *jf_error_string(int code)
{
    switch (code) {
    case JF_OK: return "ok";
    case JF_ERR_NULL: return "jetfire_hip: required pointer is NULL";
    case JF_ERR_SHAPE: return "jetfire_hip: dimension is not a positive multiple of 32";
    case JF_ERR_ENUM: return "jetfire_hip: unknown layout/dtype/rounding code";
    case JF_ERR_ALIGN: return "jetfire_hip: pointer not 16-byte aligned";
    case JF_ERR_WORKSPACE: return "jetfire_hip: workspace missing or too small";
    case JF_ERR_DEVICE: return "jetfire_hip: device is not gfx950";
    case JF_ERR_UNSUPPORTED: return "jetfire_hip: this combination of operand layouts is not implemented";
    case JF_ERR_SCRATCH_LIMIT: return "jetfire_hip: the K split of this problem needs more than the built-in scratch buffer (JF_NOALLOC_SCRATCH_BYTES); use jf_igemm_block_fp with a workspace, or splitk = 1";
    case JF_ERR_VALUE: return "jetfire_hip: a number is outside the range this entry point states";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "jetfire_hip: unknown error";
    }
}

int jf_philox_rounds(void) { return PHILOX_ROUNDS; }

size_t jf_igemm_workspace_bytes(int M, int N, int K, int b_layout)
{
    (void)M; (void)N; (void)K; (void)b_layout;                // both B layouts are read in place
    return 0;
}

int jf_igemm_s32(const int8_t *A, const int8_t *B, int32_t *C, int M, int N, int K, int b_layout,
                 void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    (void)workspace; (void)workspace_bytes;
    int rc = check_gemm_common(A, B, C, M, N, K, b_layout);
    if (rc) return rc;
    const bool kn = b_layout == JF_B_KN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.C = C; a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = kn ? N : K;
    return launch_gemm<EPI_S32, float>(a, (hipStream_t)stream, kn);
}

int jf_igemm_block_acc(const int8_t *A, const int8_t *B, int32_t *acc, int M, int N, int K, int b_layout,
                       void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    (void)workspace; (void)workspace_bytes;
    int rc = check_gemm_common(A, B, acc, M, N, K, b_layout);
    if (rc) return rc;
    const bool kn = b_layout == JF_B_KN;
    for (int kb = 0; kb < K / QB; ++kb) {
        GemmArgs a = {};
        a.A = A + kb * QB; a.B = kn ? B + (size_t)kb * QB * N : B + kb * QB; a.C = acc + (size_t)kb * M * N;
        a.M = M; a.N = N; a.K = QB; a.lda = K; a.ldb = kn ? N : K;
        if ((rc = launch_gemm<EPI_S32, float>(a, (hipStream_t)stream, kn))) return rc;
    }
    return JF_OK;
}

int jf_igemm_splitk_plan(int M, int N, int K, int splitk, int *splits, int *kb_per_split)
{
    if (!mult32(M) || !mult32(N) || !mult32(K)) return JF_ERR_SHAPE;
    if (splitk < 0 || !splits || !kb_per_split) return splitk < 0 ? JF_ERR_ENUM : JF_ERR_NULL;
    splitk_plan(M, N, K, splitk, *splits, *kb_per_split);
    return JF_OK;
}

size_t jf_igemm_block_fp_workspace_bytes(int M, int N, int K, int b_layout, int splitk)
{
    (void)b_layout;
    int splits = 1, kb_per = 0;
    if (jf_igemm_splitk_plan(M, N, K, splitk, &splits, &kb_per) != JF_OK) return 0;
    return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}

// The fp-output GEMM behind both of its entry points.  partials: fp32 [splits][M][N] scratch for the K split (only
// touched when the plan has more than one part; every element of it that is read has been written by this call).
static int block_fp_run(const int8_t *A, const int8_t *B, const void *sa, const void *sb, void *C, int M, int N, int K,
                        int a_layout, int b_layout, int scale_dtype, int sa_layout, int sb_layout, int out_dtype,
                        int splits, int kb_per, void *partials, hipStream_t st)
{
    GemmArgs a = {};
    const bool a_km = a_layout == JF_A_KM, kn = b_layout == JF_B_KN;
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = C; a.M = M; a.N = N; a.K = K; a.lda = a_km ? M : K; a.ldb = kn ? N : K;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    a.out_dtype = out_dtype;
    a.splits = splits; a.kb_per_split = kb_per;
    if (splits > 1) a.C = partials;
    int rc = scale_dtype == JF_SCALE_F16 ? launch_gemm<EPI_FP, half_t>(a, st, kn, a_km) : launch_gemm<EPI_FP, float>(a, st, kn, a_km);
    if (rc || splits == 1) return rc;
    return launch_splitk_reduce((const float *)partials, (size_t)M * (size_t)N, splits, C, out_dtype, st);
}

static int block_fp_check(const int8_t *A, const int8_t *B, const void *sa, const void *sb, void *C, int M, int N, int K,
                          int a_layout, int b_layout, int scale_dtype, int out_dtype)
{
    int rc = check_gemm_common(A, B, C, M, N, K, b_layout);
    if (rc) return rc;
    if (a_layout != JF_A_MK && a_layout != JF_A_KM) return JF_ERR_ENUM;
    if (!sa || !sb) return JF_ERR_NULL;
    if ((scale_dtype != JF_SCALE_F16 && scale_dtype != JF_SCALE_F32) ||
        (out_dtype != JF_FP_F16 && out_dtype != JF_FP_F32 && out_dtype != JF_FP_BF16)) return JF_ERR_ENUM;
    if (!scale_ptr_ok(sa, scale_dtype) || !scale_ptr_ok(sb, scale_dtype)) return JF_ERR_ALIGN;
    return JF_OK;
}

int jf_igemm_block_fp(const int8_t *A, const int8_t *B, const void *sa, const void *sb, void *C,
                      int M, int N, int K, int a_layout, int b_layout, int scale_dtype, int sa_layout, int sb_layout,
                      int out_dtype, int splitk, void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    int rc = block_fp_check(A, B, sa, sb, C, M, N, K, a_layout, b_layout, scale_dtype, out_dtype);
    if (rc) return rc;
    int splits = 1, kb_per = 0;
    if ((rc = jf_igemm_splitk_plan(M, N, K, splitk, &splits, &kb_per))) return rc;
    if (splits > 1 && (!workspace || !aligned16(workspace) || workspace_bytes < jf_igemm_block_fp_workspace_bytes(M, N, K, b_layout, splitk)))
        return JF_ERR_WORKSPACE;
    return block_fp_run(A, B, sa, sb, C, M, N, K, a_layout, b_layout, scale_dtype, sa_layout, sb_layout, out_dtype, splits,
                        kb_per, workspace, (hipStream_t)stream);
}

static size_t wgrad_fold_values(int M, int N, int splits)      // of GemmArgs::fold
{
    return (size_t)((M + 127) / 128) * ((N + 127) / 128) * splits * (128 * 128);
}

static size_t wgrad_workspace(int n, const int *M, const int *N, const WgradPlan &plan)
{
    size_t bytes = 0;
    for (int i = 0; i < n; ++i) {
        if (plan.splits[i] > 1) bytes += (size_t)plan.splits[i] * (size_t)M[i] * (size_t)N[i] * sizeof(float);
        if (plan.fold_kb[i]) bytes += wgrad_fold_values(M[i], N[i], plan.splits[i]) * sizeof(float);
    }
    return bytes;
}

size_t jf_wgrad_many_workspace_bytes(int n, const int *M, const int *N, int K)
{
    if (n < 1 || n > WGRAD_MAX || !M || !N || !mult32(K)) return 0;
    WgradPlan plan;
    wgrad_group_plan(n, M, N, K, plan);
    return wgrad_workspace(n, M, N, plan);
}

// The launches of jf_wgrad_many and jf_wgrad_many_dgrad: plan, group of GEMMs and what follows it
struct WgradLaunch {
    GemmGroup grp;
    WgradFinish fin;
    long wgs, fwgs;
    int longest;              // K blocks of a workgroup
};
static int wgrad_launch(int n, const int8_t *const *G, const void *const *SG, const int8_t *const *X, const void *const *SX, void *const *out,
                        const int *M, const int *N, int K, int scale_dtype, int out_dtype, int ncol, const float *const *terms,
                        const int *width, float *const *sum, void *workspace, size_t workspace_bytes, WgradLaunch &l)
{
    if (n < 1 || n > WGRAD_MAX || ncol < 0 || ncol > WGRAD_MAX) return JF_ERR_SHAPE;
    if (!G || !SG || !X || !SX || !out || !M || !N || (ncol && (!terms || !width || !sum))) return JF_ERR_NULL;
    for (int i = 0; i < n; ++i) {
        int rc = block_fp_check(G[i], X[i], SG[i], SX[i], out[i], M[i], N[i], K, JF_A_KM, JF_B_KN, scale_dtype, out_dtype);
        if (rc) return rc;
    }
    for (int i = 0; i < ncol; ++i) {
        if (!terms[i] || !sum[i]) return JF_ERR_NULL;
        if (!mult32(width[i])) return JF_ERR_SHAPE;
    }
    if (!device_is_gfx950()) return JF_ERR_DEVICE;
    WgradPlan plan;
    wgrad_group_plan(n, M, N, K, plan);
    const size_t need = wgrad_workspace(n, M, N, plan);
    if (need && (!workspace || !aligned16(workspace) || workspace_bytes < need)) return JF_ERR_WORKSPACE;
    int order[WGRAD_MAX];                                      // longest parts first: the short ones even out the end of the launch
    for (int i = 0; i < n; ++i) order[i] = i;
    std::stable_sort(order, order + n, [&](int a, int b) { return plan.kb_per_split[a] > plan.kb_per_split[b]; });
    l = {};
    float *part = (float *)workspace;
    for (int j = 0; j < n; ++j) {
        const int i = order[j], splits = plan.splits[i];
        GemmArgs &a = l.grp.g[j];
        a = wgrad_args(G[i], SG[i], X[i], SX[i], K, N[i], M[i], out[i], out_dtype, splits, plan.kb_per_split[i]);
        if (plan.fold_kb[i]) {
            a.fold_kb = plan.fold_kb[i]; a.fold = part;
            part += wgrad_fold_values(M[i], N[i], splits);
        }
        l.wgs += ((long)a.tiles_m * a.tiles_n * splits + 7) / 8;
        l.grp.end[j] = (int)l.wgs;
        if (plan.kb_per_split[i] > l.longest) l.longest = plan.kb_per_split[i];
        if (splits > 1) {
            const size_t count = (size_t)M[i] * (size_t)N[i];
            l.fwgs += (long)((count + 4095) / 4096);
            a.C = part;
            WgradFinish &fin = l.fin;
            fin.part[fin.n] = part; fin.out[fin.n] = out[i]; fin.count[fin.n] = count; fin.splits[fin.n] = splits; fin.end[fin.n] = (int)l.fwgs;
            ++fin.n;
            part += (size_t)splits * count;
        }
    }
    for (int i = 0; i < ncol; ++i) {
        l.fwgs += width[i] / QB;
        l.fin.terms[i] = terms[i]; l.fin.sum[i] = sum[i]; l.fin.width[i] = width[i]; l.fin.cend[i] = (int)l.fwgs;
    }
    l.wgs *= 8;
    if (l.wgs > 0x7fffffffL || l.fwgs > 0x7fffffffL) return JF_ERR_SHAPE;
    l.grp.n = n;
    l.fin.ncol = ncol; l.fin.strips = K / QB; l.fin.out_dtype = out_dtype;
    return JF_OK;
}
static int launch_wgrads(WgradLaunch &l, bool f16, hipStream_t st)
{
    const int pace = pace_of(l.wgs, 2L * cu_count(), l.longest * QB);
    for (int i = 0; i < l.grp.n; ++i) l.grp.g[i].pace = pace;
    return f16 ? launch_wgrad_group<half_t>(l.grp, (unsigned)l.wgs, st) : launch_wgrad_group<float>(l.grp, (unsigned)l.wgs, st);
}
static int launch_finish(const WgradLaunch &l, hipStream_t st)
{
    if (l.fwgs == 0) return JF_OK;
    hipLaunchKernelGGL(wgrad_finish_kernel, dim3((unsigned)l.fwgs), dim3(1024), 0, st, l.fin);
    return (int)hipGetLastError();
}

int jf_wgrad_many(int n, const int8_t *const *G, const void *const *SG, const int8_t *const *X, const void *const *SX, void *const *out,
                  const int *M, const int *N, int K, int scale_dtype, int out_dtype, int ncol, const float *const *terms,
                  const int *width, float *const *sum, void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    WgradLaunch l;
    int rc = wgrad_launch(n, G, SG, X, SX, out, M, N, K, scale_dtype, out_dtype, ncol, terms, width, sum, workspace, workspace_bytes, l);
    if (!rc) rc = launch_wgrads(l, scale_dtype == JF_SCALE_F16, (hipStream_t)stream);
    return rc ? rc : launch_finish(l, (hipStream_t)stream);
}

// A group of weight gradients fills the chip by itself and ends in a short round; the activation gradient's tiles are worth having in it
// where they are few, or the sums over the tokens short.  us of a training step of three blocks, two launches | one, tokens x width (128x128
// tiles of the activation gradient): 1024x768 (48) 733 | 718, 1024x1600 (104) 1348 | 1322, 4096x768 (192) 1279 | 1270, 4096x1024 (256) 1663 |
// 1629, 4096x1600 (416) 3252 | 3219, 8192x256 (128) 674 | 662; on the other side 8192x512 (256) 1225 | 1234, 6144x768 (288) 1576 | 1585,
// 8192x768 (384) 1903 | 1939, 12288x768 (576) 2700 | 2720.
int jf_wgrad_many_dgrad(const int8_t *W, const void *sw, int8_t *dx, void *dx_scales, uint64_t seed, uint64_t offset, int n,
                        const int8_t *const *G, const void *const *SG, const int8_t *const *X, const void *const *SX, void *const *out,
                        const int *M, const int *N, int K, int scale_dtype, int out_dtype, void *workspace, size_t workspace_bytes,
                        jf_stream_t stream)
{
    WgradLaunch l;
    int rc = wgrad_launch(n, G, SG, X, SX, out, M, N, K, scale_dtype, out_dtype, 0, nullptr, nullptr, nullptr, workspace, workspace_bytes, l);
    if (!rc) rc = check_gemm_common(G[0], W, dx, K, N[0], M[0], JF_B_KN);
    if (rc) return rc;
    if (!sw || !dx_scales) return JF_ERR_NULL;
    if (!scale_ptr_ok(sw, scale_dtype)) return JF_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const bool f16 = scale_dtype == JF_SCALE_F16;
    const bool few = (long)((K + 127) / 128) * ((N[0] + 127) / 128) <= cu_count() / 2;
    if (backward_in_one_launch(K, N[0], l.wgs) && (few || K <= 4096)) {
        const GemmArgs x = dgrad_args(G[0], SG[0], W, sw, K, N[0], M[0], dx, dx_scales, 0, seed, offset);
        return f16 ? launch_backward_any<EPI_Q, half_t>(x, l.grp, l.wgs, l.longest * QB, st) : launch_backward_any<EPI_Q, float>(x, l.grp, l.wgs, l.longest * QB, st);
    }
    rc = jf_igemm_block_q(G[0], W, SG[0], sw, nullptr, nullptr, dx, dx_scales, K, N[0], M[0], JF_B_KN, scale_dtype, JF_SCALES_ROWMAJOR,
                          JF_SCALES_KMAJOR, JF_ROUND_STOCHASTIC, seed, offset, nullptr, 0, stream);
    return rc ? rc : launch_wgrads(l, f16, st);
}

int jf_wgrad_many_finish(int n, const int8_t *const *G, const void *const *SG, const int8_t *const *X, const void *const *SX, void *const *out,
                         const int *M, const int *N, int K, int scale_dtype, int out_dtype, int ncol, const float *const *terms,
                         const int *width, float *const *sum, void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    WgradLaunch l;
    const int rc = wgrad_launch(n, G, SG, X, SX, out, M, N, K, scale_dtype, out_dtype, ncol, terms, width, sum, workspace, workspace_bytes, l);
    return rc ? rc : launch_finish(l, (hipStream_t)stream);
}

// ---- the allocation-free weight-gradient entry point ---------------------------------------------------------------
// Scratch of the K split, for callers that cannot hand over a workspace: one array per device, resident until the
// process ends.  In host code `noalloc_scratch` is only a handle; the device address is looked up once per device.
}  // extern "C"
static __device__ __align__(256) unsigned char noalloc_scratch[JF_NOALLOC_SCRATCH_BYTES];
namespace {
std::mutex noalloc_mu;
void *noalloc_ptr[jf::MAX_DEVICES] = {};                       // device address of noalloc_scratch, per device
// rc = 0 and *out = this device's copy of the array (looked up on the first call on the device, with it current)
int noalloc_scratch_of_current_device(void **out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= jf::MAX_DEVICES) return JF_ERR_DEVICE;
    std::lock_guard<std::mutex> g(noalloc_mu);
    if (!noalloc_ptr[dev]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(noalloc_scratch));
        if (e != hipSuccess) return (int)e;
        if (!ptr) return JF_ERR_DEVICE;
        noalloc_ptr[dev] = ptr;
    }
    *out = noalloc_ptr[dev];
    return JF_OK;
}
}  // namespace
extern "C" {

int jf_igemm_block_fp_noalloc(const int8_t *A, const int8_t *B, const void *sa, const void *sb, void *C,
                              int M, int N, int K, int a_layout, int b_layout, int scale_dtype, int sa_layout,
                              int sb_layout, int out_dtype, int splitk, jf_stream_t stream)
{
    int rc = block_fp_check(A, B, sa, sb, C, M, N, K, a_layout, b_layout, scale_dtype, out_dtype);
    if (rc) return rc;
    int splits = 1, kb_per = 0;
    if ((rc = jf_igemm_splitk_plan(M, N, K, splitk, &splits, &kb_per))) return rc;
    void *partials = nullptr;
    if (splits > 1) {
        if ((size_t)splits * (size_t)M * (size_t)N * sizeof(float) > (size_t)JF_NOALLOC_SCRATCH_BYTES) return JF_ERR_SCRATCH_LIMIT;
        if ((rc = noalloc_scratch_of_current_device(&partials))) return rc;
    }
    // nothing in the scratch has to start at zero: every part stores its whole [M][N] partial result before the
    // reduction reads it, so what an earlier (larger) call left behind is never read
    return block_fp_run(A, B, sa, sb, C, M, N, K, a_layout, b_layout, scale_dtype, sa_layout, sb_layout, out_dtype, splits,
                        kb_per, partials, (hipStream_t)stream);
}

int jf_linear_bwd(const int8_t *X, const void *sx, const int8_t *G, const void *sg, const int8_t *W, const void *sw, int R, int C_in, int C_out,
                  int scale_dtype, void *dx, void *dx_scales, int dx_dtype, uint64_t seed, uint64_t offset, void *dw, int dw_dtype, int splitk,
                  void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    int rc = block_fp_check(G, X, sg, sx, dw, C_out, C_in, R, JF_A_KM, JF_B_KN, scale_dtype, dw_dtype);
    if (!rc) rc = check_gemm_common(G, W, dx, R, C_in, C_out, JF_B_KN);
    if (rc) return rc;
    if (!sw) return JF_ERR_NULL;
    if (!scale_ptr_ok(sw, scale_dtype)) return JF_ERR_ALIGN;
    if (!dx_scales && dx_dtype != JF_FP_F16 && dx_dtype != JF_FP_F32 && dx_dtype != JF_FP_BF16) return JF_ERR_ENUM;
    int splits = 1, kb_per = 0;
    if ((rc = jf_igemm_splitk_plan(C_out, C_in, R, splitk, &splits, &kb_per))) return rc;
    if (splits > 1 && (!workspace || !aligned16(workspace) || workspace_bytes < jf_igemm_block_fp_workspace_bytes(C_out, C_in, R, JF_B_KN, splitk)))
        return JF_ERR_WORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    GemmGroup w = {};
    w.n = 1;
    w.g[0] = wgrad_args(G, sg, X, sx, R, C_in, C_out, splits > 1 ? workspace : dw, dw_dtype, splits, kb_per);
    const long w_wgs = ((long)w.g[0].tiles_m * w.g[0].tiles_n * splits + 7) / 8 * 8;
    w.end[0] = (int)(w_wgs / 8);
    if (!backward_in_one_launch(R, C_in, w_wgs)) {
        if (dx_scales)
            rc = jf_igemm_block_q(G, W, sg, sw, nullptr, nullptr, (int8_t *)dx, dx_scales, R, C_in, C_out, JF_B_KN, scale_dtype, JF_SCALES_ROWMAJOR,
                                  JF_SCALES_KMAJOR, JF_ROUND_STOCHASTIC, seed, offset, nullptr, 0, stream);
        else
            rc = jf_igemm_block_q_dequant(G, W, sg, sw, nullptr, nullptr, dx, R, C_in, C_out, JF_B_KN, scale_dtype, JF_SCALES_ROWMAJOR,
                                          JF_SCALES_KMAJOR, dx_dtype, JF_ROUND_STOCHASTIC, seed, offset, stream);
        return rc ? rc : block_fp_run(G, X, sg, sx, dw, C_out, C_in, R, JF_A_KM, JF_B_KN, scale_dtype, JF_SCALES_KMAJOR, JF_SCALES_KMAJOR, dw_dtype,
                                      splits, kb_per, workspace, st);
    }
    if (!device_is_gfx950()) return JF_ERR_DEVICE;
    const GemmArgs x = dgrad_args(G, sg, W, sw, R, C_in, C_out, dx, dx_scales, dx_dtype, seed, offset);
    const bool f16 = scale_dtype == JF_SCALE_F16;
    const int depth = splits > 1 ? kb_per * QB : R;
    if (dx_scales) rc = f16 ? launch_backward_any<EPI_Q, half_t>(x, w, w_wgs, depth, st) : launch_backward_any<EPI_Q, float>(x, w, w_wgs, depth, st);
    else rc = f16 ? launch_backward_any<EPI_QD, half_t>(x, w, w_wgs, depth, st) : launch_backward_any<EPI_QD, float>(x, w, w_wgs, depth, st);
    return rc || splits == 1 ? rc : launch_splitk_reduce((const float *)workspace, (size_t)C_out * (size_t)C_in, splits, dw, dw_dtype, st);
}

int jf_igemm_block_q(const int8_t *A, const int8_t *B, const void *sa, const void *sb,
                     const float *bias, const float *biasmax, int8_t *C, void *sc,
                     int M, int N, int K, int b_layout, int scale_dtype, int sa_layout, int sb_layout, int rounding,
                     uint64_t seed, uint64_t offset,
                     void *workspace, size_t workspace_bytes, jf_stream_t stream)
{
    (void)workspace; (void)workspace_bytes;
    int rc = check_gemm_common(A, B, C, M, N, K, b_layout);
    if (rc) return rc;
    if (!sa || !sb || !sc) return JF_ERR_NULL;
    if ((scale_dtype != JF_SCALE_F16 && scale_dtype != JF_SCALE_F32) ||
        (rounding != JF_ROUND_NEAREST && rounding != JF_ROUND_STOCHASTIC)) return JF_ERR_ENUM;
    if (!scale_ptr_ok(sa, scale_dtype) || !scale_ptr_ok(sb, scale_dtype)) return JF_ERR_ALIGN;
    const bool kn = b_layout == JF_B_KN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = C; a.sc = sc; a.bias = bias; a.biasmax = biasmax;
    a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = kn ? N : K; a.rounding = rounding; a.seed = seed; a.offset = offset;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    hipStream_t st = (hipStream_t)stream;
    return scale_dtype == JF_SCALE_F16 ? launch_gemm<EPI_Q, half_t>(a, st, kn) : launch_gemm<EPI_Q, float>(a, st, kn);
}

int jf_igemm_block_q_dequant(const int8_t *A, const int8_t *B, const void *sa, const void *sb, const float *bias,
                             const float *biasmax, void *out, int M, int N, int K, int b_layout, int scale_dtype,
                             int sa_layout, int sb_layout, int out_dtype, int rounding, uint64_t seed, uint64_t offset,
                             jf_stream_t stream)
{
    int rc = check_gemm_common(A, B, out, M, N, K, b_layout);
    if (rc) return rc;
    if (!sa || !sb) return JF_ERR_NULL;
    if ((scale_dtype != JF_SCALE_F16 && scale_dtype != JF_SCALE_F32) ||
        (rounding != JF_ROUND_NEAREST && rounding != JF_ROUND_STOCHASTIC) ||
        (out_dtype != JF_FP_F16 && out_dtype != JF_FP_F32 && out_dtype != JF_FP_BF16)) return JF_ERR_ENUM;
    if (!scale_ptr_ok(sa, scale_dtype) || !scale_ptr_ok(sb, scale_dtype)) return JF_ERR_ALIGN;
    const bool kn = b_layout == JF_B_KN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = out; a.bias = bias; a.biasmax = biasmax; a.out_dtype = out_dtype;
    a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = kn ? N : K; a.rounding = rounding; a.seed = seed; a.offset = offset;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    hipStream_t st = (hipStream_t)stream;
    return scale_dtype == JF_SCALE_F16 ? launch_gemm<EPI_QD, half_t>(a, st, kn) : launch_gemm<EPI_QD, float>(a, st, kn);
}

// The residual addition reads and writes 13 to 17 bytes per element, of which the GEMM has a third in registers, in a launch of its own.
// us, two launches | this | the GEMM alone, binary16 scales.  Float in and out: 32x768x768 8.7 | 6.3 | 5.3, 512x256x1024 9.6 | 7.2 | 6.0,
// 1248x768x768 10.0 | 7.8 | 5.9, x3072 17.4 | 14.7 | 12.4.  Float in, bfloat16 out: 4096x768x768 18.6 | 16.4 | 12.2, 12288x768x768 40.2 | 34.8 |
// 24.6, x3072 86.5 | 81.5 | 68, 8192x1600x1600 76.3 | 69 | 53, x6400 190 | 187 | 166, 8192x1024x1024 37.1 | 31.7 | 22.9, 12288x768x96 27.0 | 20.6 | 11.6.
// What it adds to a large launch is memory time: the tiles of a round end together, and their 8 bytes per element have nothing to hide behind.
int jf_igemm_block_q_add(const int8_t *A, const int8_t *B, const void *sa, const void *sb, const float *bias, const float *biasmax,
                         const void *x1, int x1_dtype, int add_rounding, void *y, int y_dtype, int8_t *q, void *s, float *rowsum,
                         float *rowsq, int M, int N, int K, int scale_dtype, int sa_layout, int sb_layout, jf_stream_t stream)
{
    int rc = check_gemm_common(A, B, q, M, N, K, JF_B_NK);
    if (rc) return rc;
    if (!sa || !sb || !s || !x1 || !y || (rowsum == nullptr) != (rowsq == nullptr)) return JF_ERR_NULL;
    if ((scale_dtype != JF_SCALE_F16 && scale_dtype != JF_SCALE_F32) || (add_rounding != JF_ROUND_NEAREST && add_rounding != JF_ROUND_TRUNC) ||
        x1_dtype < JF_FP_F16 || x1_dtype > JF_FP_BF16 || y_dtype < JF_FP_F16 || y_dtype > JF_FP_BF16) return JF_ERR_ENUM;
    if (!aligned16(x1) || !aligned16(y) || !scale_ptr_ok(sa, scale_dtype) || !scale_ptr_ok(sb, scale_dtype)) return JF_ERR_ALIGN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = q; a.sc = s; a.bias = bias; a.biasmax = biasmax;
    a.x1 = x1; a.x1_dtype = x1_dtype; a.rounding2 = add_rounding; a.y = y; a.out_dtype = y_dtype; a.rowsum = rowsum; a.rowsq = rowsq;
    a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = K; a.rounding = JF_ROUND_NEAREST;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    hipStream_t st = (hipStream_t)stream;
    return scale_dtype == JF_SCALE_F16 ? launch_gemm<EPI_QA, half_t>(a, st, false) : launch_gemm<EPI_QA, float>(a, st, false);
}

int jf_igemm_block_q_gelu(const int8_t *A, const int8_t *B, const void *sa, const void *sb, const float *bias,
                          const float *biasmax, int8_t *C, void *sc, int8_t *C_gelu, void *sc_gelu, int M, int N, int K,
                          int scale_dtype, int sa_layout, int sb_layout, int gelu_approx, float gelu_amax_eps,
                          jf_stream_t stream)
{
    int rc = check_gemm_common(A, B, C, M, N, K, JF_B_NK);
    if (rc) return rc;
    if (!sa || !sb || !sc || !C_gelu || !sc_gelu) return JF_ERR_NULL;
    if ((scale_dtype != JF_SCALE_F16 && scale_dtype != JF_SCALE_F32) ||
        (gelu_approx != JF_GELU_ERF && gelu_approx != JF_GELU_TANH)) return JF_ERR_ENUM;
    if (!aligned16(C_gelu) || !scale_ptr_ok(sa, scale_dtype) || !scale_ptr_ok(sb, scale_dtype)) return JF_ERR_ALIGN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = C; a.sc = sc; a.bias = bias; a.biasmax = biasmax;
    a.C2 = C_gelu; a.sc2 = sc_gelu; a.gelu_approx = gelu_approx; a.gelu_eps = gelu_amax_eps;
    a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = K; a.rounding = JF_ROUND_NEAREST;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    hipStream_t st = (hipStream_t)stream;
    return scale_dtype == JF_SCALE_F16 ? launch_gemm<EPI_QG, half_t>(a, st, false) : launch_gemm<EPI_QG, float>(a, st, false);
}

int jf_igemm_block_q_gelu_bwd(const int8_t *A, const int8_t *B, const void *sa, const void *sb, const int8_t *Xq,
                              const void *Xs, int8_t *C, void *sc, int M, int N, int K, int scale_dtype, int sa_layout,
                              int sb_layout, int gelu_approx, uint64_t seed, uint64_t offset, int gelu_rounding,
                              uint64_t gelu_seed, uint64_t gelu_offset, jf_stream_t stream)
{
    int rc = check_gemm_common(A, B, C, M, N, K, JF_B_KN);
    if (rc) return rc;
    if (!sa || !sb || !sc || !Xq || !Xs) return JF_ERR_NULL;
    if ((scale_dtype != JF_SCALE_F16 && scale_dtype != JF_SCALE_F32) ||
        (gelu_approx != JF_GELU_ERF && gelu_approx != JF_GELU_TANH) ||
        (gelu_rounding != JF_ROUND_NEAREST && gelu_rounding != JF_ROUND_STOCHASTIC)) return JF_ERR_ENUM;
    if (!aligned16(Xq) || !scale_ptr_ok(sa, scale_dtype) || !scale_ptr_ok(sb, scale_dtype) || !scale_ptr_ok(Xs, scale_dtype))
        return JF_ERR_ALIGN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = C; a.sc = sc; a.Xq = Xq; a.Xs = Xs;
    a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = N;
    a.rounding = JF_ROUND_STOCHASTIC; a.seed = seed; a.offset = offset;
    a.gelu_approx = gelu_approx; a.rounding2 = gelu_rounding; a.seed2 = gelu_seed; a.offset2 = gelu_offset;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    hipStream_t st = (hipStream_t)stream;
    return scale_dtype == JF_SCALE_F16 ? launch_gemm<EPI_QB, half_t>(a, st, true) : launch_gemm<EPI_QB, float>(a, st, true);
}

int jf_transpose_s8(const int8_t *in, int R, int C, int8_t *out, jf_stream_t stream)
{
    if (!in || !out) return JF_ERR_NULL;
    if (R <= 0 || C <= 0 || (R % 16) || (C % 16)) return JF_ERR_SHAPE;
    if (!aligned16(in) || !aligned16(out)) return JF_ERR_ALIGN;
    if (!device_is_gfx950()) return JF_ERR_DEVICE;
    return launch_transpose(in, R, C, out, (hipStream_t)stream);
}

}  // extern "C"
#elif defined(JF_PROF_LIB)   // libjetfire_prof.so

#include "../../include/jetfire_prof.h"

// jf_igemm_block_q with fp32 scales through the PROF instantiation of the kernel: same arithmetic, same bits, plus the
// per-workgroup phase record (include/jetfire_prof.h).
extern "C" int jf_prof_igemm_block_q(const int8_t *A, const int8_t *B, const float *sa, const float *sb, const float *bias,
                                     const float *biasmax, int8_t *C, float *sc, int M, int N, int K, int b_layout,
                                     int sa_layout, int sb_layout, int rounding, uint64_t seed, uint64_t offset,
                                     unsigned long long *phases, int capacity_workgroups, jf_stream_t stream)
{
    int rc = check_gemm_common(A, B, C, M, N, K, b_layout);
    if (rc) return rc;
    if (!sa || !sb || !sc || !phases) return JF_ERR_NULL;
    if (capacity_workgroups <= 0) return JF_ERR_SHAPE;
    if (rounding != JF_ROUND_NEAREST && rounding != JF_ROUND_STOCHASTIC) return JF_ERR_ENUM;
    const bool kn = b_layout == JF_B_KN;
    GemmArgs a = {};
    a.A = A; a.B = B; a.sa = sa; a.sb = sb; a.C = C; a.sc = sc; a.bias = bias; a.biasmax = biasmax;
    a.M = M; a.N = N; a.K = K; a.lda = K; a.ldb = kn ? N : K; a.rounding = rounding; a.seed = seed; a.offset = offset;
    if (!scale_strides(sa_layout, K, M / QB, a.sa_ks, a.sa_is) || !scale_strides(sb_layout, K, N / QB, a.sb_ks, a.sb_is))
        return JF_ERR_ENUM;
    a.phases = phases;
    a.phase_capacity = capacity_workgroups;
    return launch_gemm<EPI_Q, float>(a, (hipStream_t)stream, kn);
}

#endif
