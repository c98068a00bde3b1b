// Causal self-attention of the INT8 recipe for gfx950: forward, and the gradients of Q, K and V.  Between the QKV projection
// and the output projection the recipe leaves the INT8 stream: Q, K, V are the dequantised binary16 output of the projection
// ([tokens, 3C] as the GEMM wrote it; a head is D consecutive columns), the result is binary16 [tokens, C].  (The reference
// calls torch's attention there, INT8_GPT2/qmodel.py:134.)
//
// All products run on v_mfma_f32_32x32x16_f16 (fp32 accumulate).  A wave owns 32 queries (forward, dQ) or 32 keys (dK, dV)
// and walks the other side in tiles of 64 rows that its workgroup shares through LDS.  The products are arranged so that
// the second one of a pair takes the first one's result straight from the registers it was left in:
//   forward   S^T = K Q^T   (lane: query l%32, 16 of the 32 keys)   then   O^T  += V^T P^T      (B operand = P^T)
//   dQ        S^T, dP^T = V dO^T                                     then   dQ^T += K^T dS^T
//   dK, dV    S = Q K^T, dP = dO V^T (lane: key l%32, 16 queries)    then   dV^T += dO^T P,  dK^T += Q^T dS
// A result register set holds, for lane half h = l/32, rows 8g + 4h + 0..3 (g = 0..3); a B operand of 16 deep wants 8
// values per lane.  The order of the contraction index is free as long as both operands agree, so slot (h, j) of step s is
// row 16s + 8(j/4) + 4h + j%4: what the lane already holds.  The A operand is fetched in that order by the transposing LDS
// read (ds_read_b64_tr_b16: 4 rows of one column per lane), so neither V, K, Q nor dO is ever transposed in memory and P and
// dS never leave the registers.  Row statistics of a query are lane-local but for one exchange between lane halves.
//
// What bounds it.  Per 32x32 tile of scores, at D = 64, forward | dQ | dK/dV: 8 | 12 | 16 MFMAs of 32 cycles and 60 to 75 vector
// instructions, 16 of them exponentials at a quarter of the rate; the two kinds share the issue of a SIMD: about 540 | 730 | 810 cycles.
// Eight sequences of 1024 rows with 25 heads have 103 tiles per SIMD: 25 | 34 | 38 us of 44 | 59 | 81 (the tile loop without its loads
// takes 26 us of the forward's; loads and stores outside it, 118 MB, another 15).  Operands are read from LDS a step ahead of the
// products, at immediate offsets (dQ: where it does not fill the chip, see there), and tiles are loaded with scalar addresses: a step's
// instructions are the arithmetic.  us, before | with that, forward and gradient, each as it is launched at its size: 8 x 1024 rows x 25
// heads 50.9 | 44.0, 144.3 | 139.6; 12 x 1024 x 12 36.9 | 33.0, 109.5 | 100.9; 2 x 1024 x 12 21.0 | 17.0, 51.7 | 42.8; 3 x 416 x 12 10.3 | 8.9,
// 27.7 | 23.6; 4 x 256 x 4 7.8 | 7.0, 21.1 | 18.4.  Errors against float64 are the same before and with that, the gradients of keys
// that rise along the sequence 2 % smaller.
// The gradient is two kernels (dQ by query, dK/dV by key: 12 + 16 MFMAs per tile instead of 20) so that every sum has one owner and a
// fixed order: no atomics, the same bits on every run.  Where few workgroups leave CUs idle the two run in one launch.
#include "jf_device.hpp"

#pragma clang diagnostic ignored "-Winline-asm"     // M0 appears in clobber lists on purpose

namespace jf {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) unsigned char lds_byte;

struct AttnArgs {
    const half_t *q, *k, *v;        // [B*T, ld]: head h of a row at column h*D of each
    const half_t *o, *go;           // [B*T, C]: the forward's result and its gradient   (gradient kernels)
    half_t *out;                    // [B*T, C]                                           (forward)
    half_t *gq, *gk, *gv;           // [B*T, ldg]                                         (gradient kernels)
    float *lse;                     // [B*H, T]: log2 of the row sum of exp2(scale * log2(e) * s)
    float *delta;                   // [B*H, T]: minus the sum over D of o * go (left by dQ, read by the dK/dV kernel)
    int ld, ldg, B, H, T;
    float scale;                    // of the scores
    int8_t *cq;                     // codes and scales of the result [B*T, C] or of the gradients [B*T, 3C] (kernels with QUANT)
    half_t *cs;
    uint64_t seed, offset;          // of the gradients' rounding noise
};

constexpr int ATT_ROWS = 64;        // rows of a shared tile
constexpr int ATT_SUB = 32;         // rows of one step
// Waves of a workgroup, sharing every tile: 128 rows, at every size.  Fewer waves make more workgroups where there are few, but each
// then loads its tiles alone.  Measured with one, two and four waves, us (forward | gradient, heads 64 wide): 4 heads of 256 rows
// 9.8 9.5 7.7 | 25.7 25.1 20.7, 36 of 416 15.0 13.5 10.2 | 39.0 35.8 27.4, 24 of 1024 29.4 27.9 21.0 | 75.3 71.1 51.9, 144 of 1024
// 83.0 51.9 36.8 | 213 140 107; heads 32 wide in the same order.  Fewer waves are ahead by at most 1.3 us, and only where a sequence
// has 32 or 64 rows.
constexpr int NW = 4;
constexpr int WG_ROWS = 32 * NW;

// Workgroup -> (head, block of rows).  Workgroups are dealt to the 8 XCDs in turn: the blocks of one head stay on one XCD
// (its K and V are read by all of them), and the longest blocks start first.
__device__ __forceinline__ bool attn_work(const AttnArgs &a, int wg, int nblk, bool longest_is_last, int &bh, int &blk)
{
    const int per = (a.B * a.H + 7) / 8, x = wg & 7, j = wg >> 3;
    bh = (j % per) * 8 + x;
    blk = j / per;
    if (longest_is_last) blk = nblk - 1 - blk;
    return bh < a.B * a.H;
}

// Tile geometry in LDS: rows of D binary16 values, 16-byte chunk c of row r at slot c ^ swz(r): the 16-byte operand reads
// (32 consecutive rows, one chunk) and the transposing reads (8 rows, 64 bytes) then spread over all banks.
template <int D> __device__ __forceinline__ int swz(int r)
{
    if (D == 64) return ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1);
    return (r >> 2) & 3;
}

template <int D> struct TileIO {
    static constexpr int CPR = D / 8, ROWB = D * 2, TILE = ATT_ROWS * ROWB;
    static constexpr int RPI = 64 / CPR;                       // rows one load instruction of a wave moves
    static constexpr int INSTR = ATT_ROWS / RPI;               // load instructions per tensor
    static constexpr int LPW = 2 * INSTR / NW;                 // load instructions per wave: two tensors
    static_assert(2 * INSTR % NW == 0, "loads must split evenly");
    int lane, wave;
    unsigned lx, ly;                                           // this lane's bytes behind the first row of a load, in either tensor
    unsigned rd[D / 16];                                       // operand reads: chunk 2kk + h of row l%32
    unsigned tr[D / 32][2];                                    // transposing reads: column block mb, rows +0..7 / +8..15
    __device__ __forceinline__ TileIO(int lane_, int wave_, int ldx, int ldy) : lane(lane_), wave(wave_)
    {
        const int r0 = (wave * RPI + lane / CPR) % 16;         // (a wave's loads are a multiple of 16 rows apart, the period of swz)
        const unsigned chunk = (unsigned)(((lane % CPR) ^ swz<D>(r0)) << 4);
        lx = (unsigned)(lane / CPR) * (unsigned)ldx * 2u + chunk;
        ly = (unsigned)(lane / CPR) * (unsigned)ldy * 2u + chunk;
        const int h = lane >> 5, r = lane & 31;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) rd[kk] = r * ROWB + (((2 * kk + h) ^ swz<D>(r)) << 4);
        const int g = lane >> 4, i = lane & 15, p = i & 3;
#pragma unroll
        for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int row = 8 * e + 4 * h + (i >> 2), c = mb * 4 + 2 * (g & 1) + (p >> 1);
                tr[mb][e] = row * ROWB + ((c ^ swz<D>(row)) << 4) + (p & 1) * 8;
            }
    }
    // rows row0 .. row0+63 of two tensors (first row of the batch at x / y, ldx / ldy elements apart) into LDS at `lds`.  The first
    // row of a load is wave-uniform: addresses cost no vector instructions.  Loads beyond the T rows (whole ones, T and the rows of a
    // tile are multiples of 32) fetch the tile's first rows instead (never used).
    __device__ __forceinline__ void load(unsigned lds, const half_t *x, int ldx, const half_t *y, int ldy, int row0, int T) const
    {
        static_assert(32 % RPI == 0 && (NW * RPI) % 16 == 0 && INSTR % NW == 0, "whole loads beyond the last row; one swizzle and one tensor per load");
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const bool second = j >= INSTR / NW;
            const int i = wave + (second ? j - INSTR / NW : j) * NW;
            const int row = row0 + i * RPI, src = row < T ? row : row0;
            const half_t *base = second ? y + (unsigned)src * (unsigned)ldy : x + (unsigned)src * (unsigned)ldx;
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         ::"v"(second ? ly : lx), "s"(base), "s"(lds + (unsigned)(second ? TILE : 0) + (unsigned)i * 1024u) : "memory", "m0");
        }
    }
    // LDS addresses of a buffer's operands in vector registers, so that everything else about a read is its immediate offset (left to
    // itself the compiler adds up every read's address: 12 to 24 vector instructions a step)
    struct At {
        unsigned rd[D / 16], tr[D / 32][2];
    };
    __device__ __forceinline__ At at(unsigned buffer) const
    {
        At r;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) { r.rd[kk] = buffer + rd[kk]; asm volatile("" : "+v"(r.rd[kk])); }
#pragma unroll
        for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
            for (int e = 0; e < 2; ++e) { r.tr[mb][e] = buffer + tr[mb][e]; asm volatile("" : "+v"(r.tr[mb][e])); }
        return r;
    }
    // row operands of step `sub` of a buffer's first or second tensor, K step kk
    template <bool SECOND> static __device__ __forceinline__ h8 row_operand(const At &a, int sub, int kk)
    {
        return *(const __attribute__((address_space(3))) h8 *)(uintptr_t)(a.rd[kk] + (SECOND ? TILE : 0) + sub * ATT_SUB * ROWB);
    }
    template <bool SECOND> static __device__ __forceinline__ void row_operands(h8 (&x)[D / 16], const At &a, int sub)
    {
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) x[kk] = row_operand<SECOND>(a, sub, kk);
    }
    // the transposed operands of step `sub`, columns 32mb .. +31; x[st][mb]
    template <bool SECOND> static __device__ __forceinline__ void tr_operands(h8 (&x)[2][D / 32], const At &a, int sub)
    {
        typedef short s4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s4 lds_s4;
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int mb = 0; mb < D / 32; ++mb) {
                h4 half[2];
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    half[e] = __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_s4 *)(uintptr_t)(a.tr[mb][e] + (SECOND ? TILE : 0) + (sub * ATT_SUB + 16 * st) * ROWB)));
                x[st][mb] = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
            }
    }
};

#define ATT_FENCE() __builtin_amdgcn_sched_barrier(0)    // LDS reads above it are under way before what follows
#define ATT_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0)

// KNOWN: with the builtin, so that the compiler knows that its own loads before the tile loop have arrived too.  Left to it, it waits
// for them where they are first used, inside the loop, with a count that takes the next tile's loads along.
template <bool KNOWN = true> __device__ __forceinline__ void attn_tile_ready()
{
    if constexpr (KNOWN) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0F70);                    // vmcnt(0)
        asm volatile("s_barrier" ::: "memory");
    } else {
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
}
// maximum / sum over a lane and its partner in the other lane half
__device__ __forceinline__ float half_max(float x)
{
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __builtin_elementwise_maximum(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float half_sum(float x)
{
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// eight registers of a result as the B operand of a 16-deep step
__device__ __forceinline__ h8 pack8(const v16f &x, int s)
{
    h8 r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = (half_t)x[8 * s + j];
    return r;
}
// a result block times a factor, rounded to binary32 (pinned: the compiler would fold the product into some of the conversions
// to binary16 and not into others, with one rounding less)
__device__ __forceinline__ void scale_t(v16f &x, float f)
{
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        float t = x[v] * f;
        asm volatile("" : "+v"(t));
        x[v] = t;
    }
}
// a transposed result block (lane: row l%32 of the output, columns 8g + 4h + 0..3), stored as binary16
__device__ __forceinline__ void store_t(half_t *row, int h, const v16f &x)
{
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        h4 t;
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = (half_t)x[4 * g + j];
        *reinterpret_cast<h4 *>(row + 8 * g + 4 * h) = t;
    }
}

// The block quantisation (quantize.py:33-117) of a wave's result while it is still in registers: a transposed result block is
// one 32x32 quantisation block (lane: row l%32, columns 8g + 4h + 0..3).  Two 32-lane exchanges per pair of registers give each
// lane 16 consecutive columns (half l/32 of its row), which is what the rounding noise is drawn for.  Values are rounded to
// binary16 first: codes, scales and noise are those of quantising the stored binary16 tensor.  row, col: the block's first
// element in a [., C] tensor.
__device__ __forceinline__ void quantize_t(const v16f &x, int8_t *codes, half_t *scales, int row, int col, int C, int lane, int rounding,
                                           uint64_t seed, uint64_t offset)
{
    float y[16], z[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) y[v] = (float)(half_t)x[v];
    row_halves(y, z);
    const size_t e0 = (size_t)(row + (lane & 31)) * C + col + 16 * (lane >> 5);
    float s;
    *reinterpret_cast<v4i *>(codes + e0) = quantize16(z, 0.0f, rounding, seed, offset, e0, &s);
    if (lane == 0) scales[(size_t)(row / QB) * (C / QB) + col / QB] = (half_t)s;
}

template <int D, bool QUANT>
__global__ __launch_bounds__(64 * NW, 4) void attn_fwd_kernel(AttnArgs a)
{
    using IO = TileIO<D>;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2][2 * IO::TILE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int nblk = (a.T + WG_ROWS - 1) / WG_ROWS;
    int bh, blk;
    if (!attn_work(a, blockIdx.x, nblk, true, bh, blk)) return;
    const int b = bh / a.H, head = bh - b * a.H;
    const size_t first = (size_t)b * a.T * a.ld + (size_t)head * D;
    const half_t *kp = a.k + first, *vp = a.v + first;
    const IO io(lane, wave, a.ld, a.ld);
    const unsigned lds = (unsigned)(uintptr_t)(lds_byte *)smem;
    const int q0 = blk * WG_ROWS + 32 * wave, qend = (blk + 1) * WG_ROWS < a.T ? (blk + 1) * WG_ROWS : a.T;
    const int nt = (qend + ATT_ROWS - 1) / ATT_ROWS;
    const bool active = q0 < a.T;
    const int query = q0 + (lane & 31);
    h8 q[D / 16];
    {
        const half_t *src = a.q + first + (size_t)(active ? query : 0) * a.ld + 8 * h;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) q[kk] = *reinterpret_cast<const h8 *>(src + 16 * kk);
    }
    v16f o[D / 32];
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[mb][v] = 0.0f;
    const float c = a.scale * 1.44269504f;
    // Maximum (shared by the halves), this lane's part of the sum.  The maximum only guards the exponential's range: it is the rows'
    // maximum over the first step and raised, and the sums rescaled, when a lane's 16 probabilities of a step add up to more than 2^8
    // (every later one keeps its relative precision in binary16 up to there).  The sum is taken anyway; so a step has no maximum to
    // form and to exchange before its exponentials can start.  The maximum starts below every finite score but finite: keys whose
    // score is -inf before the first finite one then count for nothing instead of giving -inf - -inf.  (A sum that is NaN takes the
    // slow way and stays one.)
    float m = -1e30f, l = 0.0f;
    io.load(lds, kp, a.ld, vp, a.ld, 0, a.T);
    for (int t = 0; t < nt; ++t) {
        attn_tile_ready();                                     // tile t has landed; nobody reads the other buffer any more
        if (t + 1 < nt) io.load(lds + ((t + 1) & 1) * 2 * IO::TILE, kp, a.ld, vp, a.ld, (t + 1) * ATT_ROWS, a.T);
        const typename IO::At at = io.at(lds + (t & 1) * 2 * IO::TILE);
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int k0 = t * ATT_ROWS + sub * ATT_SUB;
            if (!active || k0 > q0) continue;                  // (wave-uniform) all keys behind the queries
            h8 kr[D / 16], vr[2][D / 32];
            IO::template row_operands<false>(kr, at, sub);
            v16f s;
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = 0.0f;
            ATT_FENCE();
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(kr[kk], q[kk], s);
            IO::template tr_operands<true>(vr, at, sub);
            ATT_FENCE();
            if (k0 == q0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + 4 * h + (v & 3) > (lane & 31) ? -__builtin_inff() : s[v];
            }
            h8 p[2];
            float sum;
            auto probabilities = [&] {
                const float mc = -m * c;
                sum = 0.0f;
#pragma unroll
                for (int st = 0; st < 2; ++st)
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * st + j], c, mc));
                        sum += e;
                        p[st][j] = (half_t)e;
                    }
            };
            const bool first = sub == 0 && t == 0;             // (wave-uniform)
            if (!first) probabilities();
            if (first || __any(!(sum <= 256.0f))) {               // (wave-uniform)
                // (v_maximum3_f32: a NaN stays one, and no operand has to be canonicalised first as for fmaxf)
                float mx = s[0];
#pragma unroll
                for (int v = 1; v < 16; ++v) mx = __builtin_elementwise_maximum(mx, s[v]);
                const float mn = fmaxf(m, half_max(mx)), al = __builtin_amdgcn_exp2f((m - mn) * c);
                l *= al;
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[mb][v] *= al;
                m = mn;
                probabilities();
            }
            l += sum;
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb) o[mb] = ATT_MFMA(vr[st][mb], p[st], o[mb]);
        }
    }
    if (!active) return;
    l = half_sum(l);
    const float r = 1.0f / l;
    half_t *dst = a.out + ((size_t)b * a.T + query) * (a.H * D) + head * D;
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb) {
        scale_t(o[mb], r);
        store_t(dst + 32 * mb, h, o[mb]);
        if (QUANT) quantize_t(o[mb], a.cq, a.cs, b * a.T + q0, head * D + 32 * mb, a.H * D, lane, JF_ROUND_NEAREST, 0, 0);
    }
    if (h == 0) a.lse[(size_t)bh * a.T + query] = m * c + __builtin_amdgcn_logf(l);     // (v_log_f32: base 2)
}

// dQ by blocks of queries; leaves delta for the dK/dV kernel.
// EARLY: operands are read before they are needed and a tile's loads overlap the whole tile before it (140 registers, 3 waves per SIMD).
// It is the faster kernel by itself at every size, us without | with, both with dK/dV: 2 sequences of 1024 rows x 12 heads 45.2 | 42.3, 8 x
// 25 heads 131.6 | 129.4 (on another card than the figures above).  But where it fills the chip, the chip then lowers its clock for everything around it (1.99 -> 1.91 GHz in the
// GEMMs of a training step, read from their clock counters, for as long as the steps go on): three GPT-2 XL blocks 5809 | 5959 us a step,
// three of GPT-2 small 2860 | 2900, three 1024 wide over 8 x 512 tokens 1641 | 1685; two blocks 768 wide over 2 x 1024 tokens 614 | 606.
// So it is taken while no CU has more than one workgroup of it, and in attn_grad_kernel.
template <int D, bool QUANT, bool EARLY> __device__ __forceinline__ void attn_dq(const AttnArgs &a, int wg, unsigned char *smem)
{
    using IO = TileIO<D>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int nblk = (a.T + WG_ROWS - 1) / WG_ROWS;
    int bh, blk;
    if (!attn_work(a, wg, nblk, true, bh, blk)) return;
    const int b = bh / a.H, head = bh - b * a.H;
    const size_t first = (size_t)b * a.T * a.ld + (size_t)head * D;
    const half_t *kp = a.k + first, *vp = a.v + first;
    const IO io(lane, wave, a.ld, a.ld);
    const unsigned lds = (unsigned)(uintptr_t)(lds_byte *)smem;
    const int q0 = blk * WG_ROWS + 32 * wave, qend = (blk + 1) * WG_ROWS < a.T ? (blk + 1) * WG_ROWS : a.T;
    const int nt = (qend + ATT_ROWS - 1) / ATT_ROWS;
    const bool active = q0 < a.T;
    const int query = active ? q0 + (lane & 31) : 0;
    io.load(lds, kp, a.ld, vp, a.ld, 0, a.T);
    h8 q[D / 16], go[D / 16];
    float dl = 0.0f;
    {
        const half_t *src = a.q + first + (size_t)query * a.ld + 8 * h;
        const size_t row = ((size_t)b * a.T + query) * (a.H * D) + head * D + 8 * h;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            q[kk] = *reinterpret_cast<const h8 *>(src + 16 * kk);
            go[kk] = *reinterpret_cast<const h8 *>(a.go + row + 16 * kk);
            const h8 o = *reinterpret_cast<const h8 *>(a.o + row + 16 * kk);
#pragma unroll
            for (int j = 0; j < 8; ++j) dl = __builtin_fmaf((float)o[j], (float)go[kk][j], dl);
        }
    }
    dl = half_sum(dl);
    const float lse = a.lse[(size_t)bh * a.T + query], c = a.scale * 1.44269504f;
    if (active && h == 0) a.delta[(size_t)bh * a.T + query] = -dl;
    v16f acc[D / 32];
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[mb][v] = 0.0f;
    for (int t = 0; t < nt; ++t) {
        attn_tile_ready<EARLY>();
        if (t + 1 < nt) io.load(lds + ((t + 1) & 1) * 2 * IO::TILE, kp, a.ld, vp, a.ld, (t + 1) * ATT_ROWS, a.T);
        const typename IO::At at = io.at(lds + (t & 1) * 2 * IO::TILE);
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int k0 = t * ATT_ROWS + sub * ATT_SUB;
            if (!active || k0 > q0) continue;
            v16f s, dp;
#pragma unroll
            for (int v = 0; v < 16; ++v) { s[v] = 0.0f; dp[v] = 0.0f; }
            h8 kc[2][D / 32];
            if constexpr (EARLY) {
                h8 kr[D / 16], vr[D / 16];
                IO::template row_operands<false>(kr, at, sub);
                IO::template row_operands<true>(vr, at, sub);
                ATT_FENCE();
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(kr[kk], q[kk], s);
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk) dp = ATT_MFMA(vr[kk], go[kk], dp);
                IO::template tr_operands<false>(kc, at, sub);
            } else {
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(IO::template row_operand<false>(at, sub, kk), q[kk], s);
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk) dp = ATT_MFMA(IO::template row_operand<true>(at, sub, kk), go[kk], dp);
            }
            if (k0 == q0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + 4 * h + (v & 3) > (lane & 31) ? -__builtin_inff() : s[v];
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], c, -lse)) * (dp[v] - dl);
            if constexpr (!EARLY) IO::template tr_operands<false>(kc, at, sub);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const h8 ds = pack8(s, st);
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb) acc[mb] = ATT_MFMA(kc[st][mb], ds, acc[mb]);
            }
        }
    }
    if (!active) return;
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb) {
        scale_t(acc[mb], a.scale);
        if (QUANT)
            quantize_t(acc[mb], a.cq, a.cs, b * a.T + q0, head * D + 32 * mb, 3 * a.H * D, lane, JF_ROUND_STOCHASTIC, a.seed, a.offset);
        else
            store_t(a.gq + ((size_t)b * a.T + query) * a.ldg + head * D + 32 * mb, h, acc[mb]);
    }
}

// dK and dV by blocks of keys.  OWN: delta is not read but formed here, for all queries of the block's tiles before the first of them (the
// same operations in the same order as in attn_dq: the same bits).
constexpr int DKV_STAT = 2 * 2 * ATT_ROWS * 4;                 // bytes of LDS behind the tiles: lse, delta of a tile's queries, twice
constexpr int OWN_ROWS = 4096;                                 // queries of a sequence with OWN: 16 KB more
template <int D, bool QUANT, bool OWN> __device__ __forceinline__ void attn_dkv(const AttnArgs &a, int wg, unsigned char *smem)
{
    using IO = TileIO<D>;
    float(*const stat)[2][ATT_ROWS] = reinterpret_cast<float(*)[2][ATT_ROWS]>(smem + 4 * IO::TILE);
    float *const own = reinterpret_cast<float *>(smem + 4 * IO::TILE + DKV_STAT);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int nblk = (a.T + WG_ROWS - 1) / WG_ROWS;
    int bh, blk;
    if (!attn_work(a, wg, nblk, false, bh, blk)) return;
    const int b = bh / a.H, head = bh - b * a.H;
    const size_t first = (size_t)b * a.T * a.ld + (size_t)head * D;
    const half_t *qp = a.q + first, *gp = a.go + (size_t)b * a.T * (a.H * D) + (size_t)head * D;
    const float *lsep = a.lse + (size_t)bh * a.T, *dlp = a.delta + (size_t)bh * a.T;
    const IO io(lane, wave, a.ld, a.H * D);
    const unsigned lds = (unsigned)(uintptr_t)(lds_byte *)smem, stat_lds = (unsigned)(uintptr_t)(lds_byte *)stat;
    const int k0 = blk * WG_ROWS + 32 * wave;
    const int t0 = blk * WG_ROWS / ATT_ROWS, nt = (a.T + ATT_ROWS - 1) / ATT_ROWS;
    const bool active = k0 < a.T;
    const int key = active ? k0 + (lane & 31) : 0;
    auto load = [&](int t) {
        io.load(lds + (t & 1) * 2 * IO::TILE, qp, a.ld, gp, a.H * D, t * ATT_ROWS, a.T);
        if (wave == 0) {
            // (the lane number is made anew: held over the loop it is one register too many, and its reload waits for the whole tile)
            unsigned l;
            asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
            const int r = t * ATT_ROWS + (int)l;
            const unsigned off = (unsigned)(r < a.T ? r : a.T - 1) * 4u, dst = stat_lds + (t & 1) * (2 * ATT_ROWS * 4);
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(lsep), "s"(dst) : "memory", "m0");
            if constexpr (!OWN)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                             ::"v"(off), "s"(dlp), "s"(dst + ATT_ROWS * 4) : "memory", "m0");
        }
    };
    load(t0);
    h8 k[D / 16], vv[D / 16];
    {
        const half_t *ks = a.k + first + (size_t)key * a.ld + 8 * h, *vs = a.v + first + (size_t)key * a.ld + 8 * h;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            k[kk] = *reinterpret_cast<const h8 *>(ks + 16 * kk);
            vv[kk] = *reinterpret_cast<const h8 *>(vs + 16 * kk);
        }
    }
    if constexpr (OWN) {
        for (int r = t0 * ATT_ROWS + 32 * wave; r < a.T; r += 32 * NW) {
            const size_t row = ((size_t)b * a.T + r + (lane & 31)) * (a.H * D) + head * D + 8 * h;
            h8 o[D / 16], go[D / 16];
            float dl = 0.0f;
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) {
                go[kk] = *reinterpret_cast<const h8 *>(a.go + row + 16 * kk);
                o[kk] = *reinterpret_cast<const h8 *>(a.o + row + 16 * kk);
            }
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
                for (int j = 0; j < 8; ++j) dl = __builtin_fmaf((float)o[kk][j], (float)go[kk][j], dl);
            dl = half_sum(dl);
            if (h == 0) own[r - t0 * ATT_ROWS + (lane & 31)] = -dl;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // (the barrier is the first tile's)
    }
    const float c = a.scale * 1.44269504f;
    v16f dk[D / 32], dv[D / 32];
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) { dk[mb][v] = 0.0f; dv[mb][v] = 0.0f; }
    for (int t = t0; t < nt; ++t) {
        attn_tile_ready();
        if (t + 1 < nt) load(t + 1);
        const typename IO::At at = io.at(lds + (t & 1) * 2 * IO::TILE);
        const float *st_l = stat[t & 1][0], *st_d = OWN ? own + (t - t0) * ATT_ROWS : stat[t & 1][1];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int q0 = t * ATT_ROWS + sub * ATT_SUB;
            if (!active || q0 < k0 || q0 >= a.T) continue;     // (wave-uniform) queries before the keys, or none
            h8 qr[D / 16], gr[D / 16];
            IO::template row_operands<false>(qr, at, sub);
            v16f s, dp;
            // (the gradient's product starts from -delta, which the registers of a result are read into as they lie)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const v4f de = *reinterpret_cast<const v4f *>(st_d + sub * ATT_SUB + 8 * g + 4 * h);
#pragma unroll
                for (int j = 0; j < 4; ++j) { s[4 * g + j] = 0.0f; dp[4 * g + j] = de[j]; }
            }
            ATT_FENCE();
            IO::template row_operands<true>(gr, at, sub);
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(qr[kk], k[kk], s);
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) dp = ATT_MFMA(gr[kk], vv[kk], dp);
            ATT_FENCE();
            h8 gc[2][D / 32], qc[2][D / 32];
            v4f ls[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) ls[g] = *reinterpret_cast<const v4f *>(st_l + sub * ATT_SUB + 8 * g + 4 * h);
            IO::template tr_operands<true>(gc, at, sub);
            if (q0 == k0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + 4 * h + (v & 3) < (lane & 31) ? -__builtin_inff() : s[v];
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], c, -ls[v >> 2][v & 3]));
                dp[v] = s[v] * dp[v];
            }
            IO::template tr_operands<false>(qc, at, sub);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const h8 p = pack8(s, st), ds = pack8(dp, st);
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb) {
                    dv[mb] = ATT_MFMA(gc[st][mb], p, dv[mb]);
                    dk[mb] = ATT_MFMA(qc[st][mb], ds, dk[mb]);
                }
            }
        }
    }
    if (!active) return;
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb) scale_t(dk[mb], a.scale);
    if (QUANT) {
        const int C = a.H * D;
#pragma unroll
        for (int mb = 0; mb < D / 32; ++mb) {
            quantize_t(dk[mb], a.cq, a.cs, b * a.T + k0, C + head * D + 32 * mb, 3 * C, lane, JF_ROUND_STOCHASTIC, a.seed, a.offset);
            quantize_t(dv[mb], a.cq, a.cs, b * a.T + k0, 2 * C + head * D + 32 * mb, 3 * C, lane, JF_ROUND_STOCHASTIC, a.seed, a.offset);
        }
        return;
    }
    const size_t row = ((size_t)b * a.T + key) * a.ldg + head * D;
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb) {
        store_t(a.gk + row + 32 * mb, h, dk[mb]);
        store_t(a.gv + row + 32 * mb, h, dv[mb]);
    }
}

template <int D, bool QUANT, bool EARLY> __global__ __launch_bounds__(64 * NW, EARLY ? 3 : 4) void attn_dq_kernel(AttnArgs a)
{
    __shared__ __attribute__((aligned(16))) unsigned char smem[4 * TileIO<D>::TILE];
    attn_dq<D, QUANT, EARLY>(a, blockIdx.x, smem);
}
template <int D, bool QUANT> __global__ __launch_bounds__(64 * NW, 2) void attn_dkv_kernel(AttnArgs a)
{
    __shared__ __attribute__((aligned(16))) unsigned char smem[4 * TileIO<D>::TILE + DKV_STAT];
    attn_dkv<D, QUANT, false>(a, blockIdx.x, smem);
}
// Both in one launch: dK and dV first, the longer of the two.  Where few workgroups leave most of the chip idle each is as long as its
// longest chain of tiles, so side by side they take little more than one of them; the price is that dK/dV forms delta itself (a pass over o and
// its gradient) and dQ runs with dK/dV's 190 registers.  us with codes, two launches | one, by workgroups of each: 4 heads of 256 rows (8) 18.3 | 12.6, 16 of
// 256 (32) 18.6 | 12.8, 32 wide 13.0 | 8.8, 36 of 416 (144) 24.2 | 19.5, 24 of 1024 (192) 44.6 | 36.8, 4 of 2048 (64) 72.7 | 55.0, 8 of 4096 (256) 134.5 |
// 115.7, 36 of 1024 (288) 48.7 | 37.1, 48 of 1024 (384) 51.0 | 46.6, 96 of 512 (384) 34.9 | 31.9; beyond one and a half per CU 60 of 1024 (480)
// 57.6 | 57.8, 144 of 416 (576) 36.6 | 37.2, 144 of 1024 (1152) 106.0 | 117.5, 200 of 1024 (1600) 141.7 | 158.8.  In a training step (three blocks 768 wide, 288 and
// 384 workgroups) 1156 | 1114, 1293 | 1259, with 8 x 512 tokens 1225 | 1212.
// Every operand is read to the end by one half or the other, so a gradient that lies on an operand (dQ on out, dK and dV on out, k or v: what the two
// launches allow) takes the two launches.
template <int D, bool QUANT> __global__ __launch_bounds__(64 * NW, 2) void attn_grad_kernel(AttnArgs a)
{
    __shared__ __attribute__((aligned(16))) unsigned char smem[4 * TileIO<D>::TILE + DKV_STAT + OWN_ROWS * 4];
    const int half = gridDim.x / 2, wg = blockIdx.x;
    if (wg < half) attn_dkv<D, QUANT, true>(a, wg, smem);
    else attn_dq<D, QUANT, true>(a, wg - half, smem);
}

static int attn_check(const void *q, const void *k, const void *v, int ld, int B, int H, int T, int D, float scale)
{
    if (!q || !k || !v) return JF_ERR_NULL;
    if (B <= 0 || H <= 0 || T <= 0 || T % 32 || (D != 32 && D != 64) || ld < H * D || ld % 8) return JF_ERR_SHAPE;
    if ((long)T * ld >= (1L << 30)) return JF_ERR_SHAPE;       // a batch element is addressed with 32-bit byte offsets
    // The kernels work with scale * log2(e) behind the causal mask's -inf and behind a maximum of the unscaled scores: it has to
    // be positive (0 * -inf is no number, a negative factor turns the maximum round) and a normal finite number.
    if (!(scale >= 1.17549435e-38f && scale * 1.44269504f < __builtin_inff())) return JF_ERR_VALUE;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v)) return JF_ERR_ALIGN;
    return device_is_gfx950() ? JF_OK : JF_ERR_DEVICE;
}

static void attn_launch(void (*kernel)(AttnArgs), const AttnArgs &a, hipStream_t st, unsigned parts = 1)
{
    const unsigned grid = 8u * ((a.B * a.H + 7) / 8) * ((a.T + WG_ROWS - 1) / WG_ROWS);
    hipLaunchKernelGGL(kernel, dim3(parts * grid), dim3(64 * NW), 0, st, a);
}
// Whether a result of the gradient kernels lies on one of their operands (as ranges of memory: two columns of one matrix count).
static bool attn_grad_overlaps(const AttnArgs &a, int D)
{
    const size_t rows = (size_t)a.B * a.T, C = (size_t)a.H * D, row = a.H * sizeof(float) * rows;
    struct Range { const void *p; size_t n; };
    const auto matrix = [&](const half_t *p, int ld) { return Range{p, p ? ((rows - 1) * ld + C) * sizeof(half_t) : 0}; };
    const Range in[] = {matrix(a.q, a.ld), matrix(a.k, a.ld), matrix(a.v, a.ld), matrix(a.o, (int)C), matrix(a.go, (int)C), {a.lse, row}};
    const Range out[] = {matrix(a.gq, a.ldg), matrix(a.gk, a.ldg), matrix(a.gv, a.ldg), {a.delta, row},
                         {a.cq, a.cq ? rows * 3 * C : 0}, {a.cs, a.cq ? rows / QB * (3 * C / QB) * sizeof(half_t) : 0}};
    for (const Range &x : out)
        for (const Range &y : in)
            if ((uintptr_t)x.p < (uintptr_t)y.p + y.n && (uintptr_t)y.p < (uintptr_t)x.p + x.n) return true;
    return false;
}
template <int D, bool QUANT> static void attn_launch_grad(const AttnArgs &a, hipStream_t st)
{
    const long wgs = (long)a.B * a.H * ((a.T + WG_ROWS - 1) / WG_ROWS), cus = cu_count();
    if (2 * wgs <= 3 * cus && a.T <= OWN_ROWS && !attn_grad_overlaps(a, D)) return attn_launch(attn_grad_kernel<D, QUANT>, a, st, 2);   // (see the kernels)
    const bool alone = wgs <= cus;
    attn_launch(alone ? attn_dq_kernel<D, QUANT, true> : attn_dq_kernel<D, QUANT, false>, a, st);
    attn_launch(attn_dkv_kernel<D, QUANT>, a, st);
}

}  // namespace jf

using namespace jf;

static int attention_fwd(const void *q, const void *k, const void *v, int ld, int B, int H, int T, int D, float scale, void *out, float *lse,
                         int8_t *codes, void *scales, jf_stream_t stream)
{
    int rc = attn_check(q, k, v, ld, B, H, T, D, scale);
    if (rc) return rc;
    if (!out || !lse) return JF_ERR_NULL;
    if (!aligned16(out) || !aligned16(codes)) return JF_ERR_ALIGN;
    AttnArgs a = {};
    a.q = (const half_t *)q; a.k = (const half_t *)k; a.v = (const half_t *)v; a.ld = ld;
    a.out = (half_t *)out; a.lse = lse; a.B = B; a.H = H; a.T = T; a.scale = scale;
    a.cq = codes; a.cs = (half_t *)scales;
    if (D == 64) attn_launch(codes ? attn_fwd_kernel<64, true> : attn_fwd_kernel<64, false>, a, (hipStream_t)stream);
    else attn_launch(codes ? attn_fwd_kernel<32, true> : attn_fwd_kernel<32, false>, a, (hipStream_t)stream);
    return (int)hipGetLastError();
}

static int attention_bwd(const void *q, const void *k, const void *v, int ld, const void *out, const void *gout, const float *lse, int B, int H,
                         int T, int D, float scale, void *gq, void *gk, void *gv, int ldg, float *delta, int8_t *codes, void *scales,
                         uint64_t seed, uint64_t offset, jf_stream_t stream)
{
    int rc = attn_check(q, k, v, ld, B, H, T, D, scale);
    if (rc) return rc;
    if (!out || !gout || !lse || !delta) return JF_ERR_NULL;
    if ((long)T * H * D >= (1L << 30)) return JF_ERR_SHAPE;
    if (!aligned16(out) || !aligned16(gout) || !aligned16(codes)) return JF_ERR_ALIGN;
    AttnArgs a = {};
    a.q = (const half_t *)q; a.k = (const half_t *)k; a.v = (const half_t *)v; a.ld = ld;
    a.o = (const half_t *)out; a.go = (const half_t *)gout; a.lse = const_cast<float *>(lse); a.delta = delta;
    a.gq = (half_t *)gq; a.gk = (half_t *)gk; a.gv = (half_t *)gv; a.ldg = ldg; a.B = B; a.H = H; a.T = T; a.scale = scale;
    a.cq = codes; a.cs = (half_t *)scales; a.seed = seed; a.offset = offset;
    hipStream_t st = (hipStream_t)stream;
    if (D == 64) codes ? attn_launch_grad<64, true>(a, st) : attn_launch_grad<64, false>(a, st);
    else codes ? attn_launch_grad<32, true>(a, st) : attn_launch_grad<32, false>(a, st);
    return (int)hipGetLastError();
}

extern "C" {

int jf_attention_fwd(const void *q, const void *k, const void *v, int ld, int B, int H, int T, int D, float scale, void *out,
                     float *lse, jf_stream_t stream)
{
    return attention_fwd(q, k, v, ld, B, H, T, D, scale, out, lse, nullptr, nullptr, stream);
}

int jf_attention_fwd_q(const void *q, const void *k, const void *v, int ld, int B, int H, int T, int D, float scale, void *out,
                       float *lse, int8_t *codes, void *scales, jf_stream_t stream)
{
    if (!codes || !scales) return JF_ERR_NULL;
    return attention_fwd(q, k, v, ld, B, H, T, D, scale, out, lse, codes, scales, stream);
}

int jf_attention_bwd(const void *q, const void *k, const void *v, int ld, const void *out, const void *gout, const float *lse,
                     int B, int H, int T, int D, float scale, void *gq, void *gk, void *gv, int ldg, float *delta, jf_stream_t stream)
{
    if (!gq || !gk || !gv) return JF_ERR_NULL;
    if (ldg < H * D || ldg % 8) return JF_ERR_SHAPE;
    if (!aligned16(gq) || !aligned16(gk) || !aligned16(gv)) return JF_ERR_ALIGN;
    return attention_bwd(q, k, v, ld, out, gout, lse, B, H, T, D, scale, gq, gk, gv, ldg, delta, nullptr, nullptr, 0, 0, stream);
}

int jf_attention_bwd_q(const void *q, const void *k, const void *v, int ld, const void *out, const void *gout, const float *lse,
                       int B, int H, int T, int D, float scale, int8_t *codes, void *scales, uint64_t seed, uint64_t offset, float *delta,
                       jf_stream_t stream)
{
    if (!codes || !scales) return JF_ERR_NULL;
    return attention_bwd(q, k, v, ld, out, gout, lse, B, H, T, D, scale, nullptr, nullptr, nullptr, 0, delta, codes, scales, seed, offset, stream);
}

}  // extern "C"
