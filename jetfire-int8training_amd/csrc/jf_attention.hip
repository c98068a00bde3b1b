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
// What bounds it: vector instructions.  At D = 64 a 32x32 tile of scores is 8 MFMAs forward (256 cycles) and about 130 vector
// instructions (8 per score register, one of them the quarter-rate exponential), at 4 cycles each.  8 x 25 heads of 1024 rows,
// counters per SIMD, in 1000 cycles (forward | dQ | dK/dV): vector ALU 64 | 75 | 99, matrix pipe 26 | 40 | 53, of 121 | 143 | 194;
// 50.7 | 62.9 | 80.0 us, no LDS bank conflicts.  The rest is waiting: the register operands' own loads are waited for inside the
// tile loop, where the compiler's count takes the next tile's loads with them, so that a tile's loads overlap only part of the one
// before.  The gradient is two kernels (dQ by query, dK/dV by key: 12 + 16 MFMAs per tile instead of 20) so that every sum has one
// owner and a fixed order: no atomics, the same bits on every run.
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
    float *delta;                   // [B*H, T]: sum over D of o * go (left by the dQ kernel, read by the dK/dV kernel)
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
__device__ __forceinline__ bool attn_work(const AttnArgs &a, int nblk, bool longest_is_last, int &bh, int &blk)
{
    const int per = (a.B * a.H + 7) / 8, x = blockIdx.x & 7, j = blockIdx.x >> 3;
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
    unsigned rd[D / 16];                                       // operand reads: chunk 2kk + h of row l%32
    unsigned tr[D / 32][2];                                    // transposing reads: column block mb, rows +0..7 / +8..15
    __device__ __forceinline__ TileIO(int lane_, int wave_) : lane(lane_), wave(wave_)
    {
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
    // rows row0 .. row0+63 of two tensors (first row of the batch at x / y, ldx / ldy elements apart) into LDS at `lds`;
    // rows beyond the last are replaced by the last (never used)
    __device__ __forceinline__ void load(unsigned lds, const half_t *x, int ldx, const half_t *y, int ldy, int row0, int last) const
    {
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const int idx = wave + j * NW;                     // wave-uniform
            const bool second = idx >= INSTR;
            const int i = second ? idx - INSTR : idx;
            const int row = i * RPI + lane / CPR, src = row0 + row < last ? row0 + row : last;
            const unsigned off = (unsigned)src * (unsigned)(second ? ldy : ldx) * 2u + (((lane % CPR) ^ swz<D>(row)) << 4);
            const half_t *base = second ? y : x;
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         ::"v"(off), "s"(base), "s"(lds + (unsigned)(second ? TILE : 0) + (unsigned)i * 1024u) : "memory", "m0");
        }
    }
    __device__ __forceinline__ h8 row_operand(unsigned tile, int sub, int kk) const
    {
        return *(const __attribute__((address_space(3))) h8 *)(uintptr_t)(tile + rd[kk] + sub * ATT_SUB * ROWB);
    }
    __device__ __forceinline__ h8 tr_operand(unsigned tile, int sub, int s, int mb) const
    {
        typedef short s4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s4 lds_s4;
        const unsigned b = tile + (sub * ATT_SUB + 16 * s) * ROWB;
        const h4 lo = __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(uintptr_t)(b + tr[mb][0])));
        const h4 hi = __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(uintptr_t)(b + tr[mb][1])));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
};

#define ATT_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0)

__device__ __forceinline__ void attn_tile_ready()
{
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ float half_swap(float x)            // the value of lane l ^ 32
{
    return __shfl_xor(x, 32, WAVE);
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
    if (!attn_work(a, nblk, true, bh, blk)) return;
    const int b = bh / a.H, head = bh - b * a.H;
    const size_t first = (size_t)b * a.T * a.ld + (size_t)head * D;
    const half_t *kp = a.k + first, *vp = a.v + first;
    const IO io(lane, wave);
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
    // Running maximum (shared by the halves), this lane's part of the sum.  The maximum starts below every finite score but
    // finite: keys whose score is -inf before the first finite one then count for nothing instead of giving -inf - -inf.
    float m = -1e30f, l = 0.0f;
    io.load(lds, kp, a.ld, vp, a.ld, 0, a.T - 1);
    for (int t = 0; t < nt; ++t) {
        attn_tile_ready();                                     // tile t has landed; nobody reads the other buffer any more
        if (t + 1 < nt) io.load(lds + ((t + 1) & 1) * 2 * IO::TILE, kp, a.ld, vp, a.ld, (t + 1) * ATT_ROWS, a.T - 1);
        const unsigned kt = lds + (t & 1) * 2 * IO::TILE, vt = kt + IO::TILE;
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int k0 = t * ATT_ROWS + sub * ATT_SUB;
            if (!active || k0 > q0) continue;                  // (wave-uniform) all keys behind the queries
            v16f s;
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = 0.0f;
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(io.row_operand(kt, sub, kk), q[kk], s);
            if (k0 == q0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + 4 * h + (v & 3) > (lane & 31) ? -__builtin_inff() : s[v];
            }
            // (v_maximum3_f32: a NaN stays one, and no operand has to be canonicalised first as for fmaxf)
            float mx = s[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) mx = __builtin_elementwise_maximum(mx, s[v]);
            mx = __builtin_elementwise_maximum(mx, half_swap(mx));
            // The maximum only guards the exponential's range: it is raised, and the sums rescaled, when a score exceeds it
            // by more than a factor of 2^8 (every later probability keeps its relative precision in binary16 up to there).
            if (__any((mx - m) * c > 8.0f)) {
                const float mn = fmaxf(m, mx), al = __builtin_amdgcn_exp2f((m - mn) * c);
                l *= al;
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[mb][v] *= al;
                m = mn;
            }
            const float mc = -m * c;
#pragma unroll
            for (int v = 0; v < 16; ++v) { s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], c, mc)); l += s[v]; }
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const h8 p = pack8(s, st);
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb) o[mb] = ATT_MFMA(io.tr_operand(vt, sub, st, mb), p, o[mb]);
            }
        }
    }
    if (!active) return;
    l += half_swap(l);
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

// dQ by blocks of queries; leaves delta for the dK/dV kernel
template <int D, bool QUANT>
__global__ __launch_bounds__(64 * NW, 4) void attn_dq_kernel(AttnArgs a)
{
    using IO = TileIO<D>;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2][2 * IO::TILE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int nblk = (a.T + WG_ROWS - 1) / WG_ROWS;
    int bh, blk;
    if (!attn_work(a, nblk, true, bh, blk)) return;
    const int b = bh / a.H, head = bh - b * a.H;
    const size_t first = (size_t)b * a.T * a.ld + (size_t)head * D;
    const half_t *kp = a.k + first, *vp = a.v + first;
    const IO io(lane, wave);
    const unsigned lds = (unsigned)(uintptr_t)(lds_byte *)smem;
    const int q0 = blk * WG_ROWS + 32 * wave, qend = (blk + 1) * WG_ROWS < a.T ? (blk + 1) * WG_ROWS : a.T;
    const int nt = (qend + ATT_ROWS - 1) / ATT_ROWS;
    const bool active = q0 < a.T;
    const int query = active ? q0 + (lane & 31) : 0;
    io.load(lds, kp, a.ld, vp, a.ld, 0, a.T - 1);
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
    dl += half_swap(dl);
    const float lse = a.lse[(size_t)bh * a.T + query], c = a.scale * 1.44269504f;
    if (active && h == 0) a.delta[(size_t)bh * a.T + query] = dl;
    v16f acc[D / 32];
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[mb][v] = 0.0f;
    for (int t = 0; t < nt; ++t) {
        attn_tile_ready();
        if (t + 1 < nt) io.load(lds + ((t + 1) & 1) * 2 * IO::TILE, kp, a.ld, vp, a.ld, (t + 1) * ATT_ROWS, a.T - 1);
        const unsigned kt = lds + (t & 1) * 2 * IO::TILE, vt = kt + IO::TILE;
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int k0 = t * ATT_ROWS + sub * ATT_SUB;
            if (!active || k0 > q0) continue;
            v16f s, dp;
#pragma unroll
            for (int v = 0; v < 16; ++v) { s[v] = 0.0f; dp[v] = 0.0f; }
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(io.row_operand(kt, sub, kk), q[kk], s);
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) dp = ATT_MFMA(io.row_operand(vt, sub, kk), go[kk], dp);
            if (k0 == q0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + 4 * h + (v & 3) > (lane & 31) ? -__builtin_inff() : s[v];
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], c, -lse)) * (dp[v] - dl);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const h8 ds = pack8(s, st);
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb) acc[mb] = ATT_MFMA(io.tr_operand(kt, sub, st, mb), ds, acc[mb]);
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

// dK and dV by blocks of keys
template <int D, bool QUANT>
__global__ __launch_bounds__(64 * NW, 3) void attn_dkv_kernel(AttnArgs a)
{
    using IO = TileIO<D>;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2][2 * IO::TILE];
    __shared__ __attribute__((aligned(16))) float stat[2][2][ATT_ROWS];        // lse, delta of the tile's queries
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int nblk = (a.T + WG_ROWS - 1) / WG_ROWS;
    int bh, blk;
    if (!attn_work(a, nblk, false, bh, blk)) return;
    const int b = bh / a.H, head = bh - b * a.H;
    const size_t first = (size_t)b * a.T * a.ld + (size_t)head * D;
    const half_t *qp = a.q + first, *gp = a.go + (size_t)b * a.T * (a.H * D) + (size_t)head * D;
    const float *lsep = a.lse + (size_t)bh * a.T, *dlp = a.delta + (size_t)bh * a.T;
    const IO io(lane, wave);
    const unsigned lds = (unsigned)(uintptr_t)(lds_byte *)smem, stat_lds = (unsigned)(uintptr_t)(lds_byte *)stat;
    const int k0 = blk * WG_ROWS + 32 * wave;
    const int t0 = blk * WG_ROWS / ATT_ROWS, nt = (a.T + ATT_ROWS - 1) / ATT_ROWS;
    const bool active = k0 < a.T;
    const int key = active ? k0 + (lane & 31) : 0;
    auto load = [&](int t) {
        io.load(lds + (t & 1) * 2 * IO::TILE, qp, a.ld, gp, a.H * D, t * ATT_ROWS, a.T - 1);
        if (wave == 0) {
            // (the lane number is made anew: held over the loop it is one register too many, and its reload waits for the whole tile)
            unsigned l;
            asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
            const int r = t * ATT_ROWS + (int)l;
            const unsigned off = (unsigned)(r < a.T ? r : a.T - 1) * 4u, dst = stat_lds + (t & 1) * (2 * ATT_ROWS * 4);
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(lsep), "s"(dst) : "memory", "m0");
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
    const float c = a.scale * 1.44269504f;
    v16f dk[D / 32], dv[D / 32];
#pragma unroll
    for (int mb = 0; mb < D / 32; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) { dk[mb][v] = 0.0f; dv[mb][v] = 0.0f; }
    for (int t = t0; t < nt; ++t) {
        attn_tile_ready();
        if (t + 1 < nt) load(t + 1);
        const unsigned qt = lds + (t & 1) * 2 * IO::TILE, gt = qt + IO::TILE;
        const float *st_l = stat[t & 1][0], *st_d = stat[t & 1][1];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int q0 = t * ATT_ROWS + sub * ATT_SUB;
            if (!active || q0 < k0 || q0 >= a.T) continue;     // (wave-uniform) queries before the keys, or none
            v16f s, dp;
#pragma unroll
            for (int v = 0; v < 16; ++v) { s[v] = 0.0f; dp[v] = 0.0f; }
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) s = ATT_MFMA(io.row_operand(qt, sub, kk), k[kk], s);
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) dp = ATT_MFMA(io.row_operand(gt, sub, kk), vv[kk], dp);
            if (q0 == k0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + 4 * h + (v & 3) < (lane & 31) ? -__builtin_inff() : s[v];
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const v4f ls = *reinterpret_cast<const v4f *>(st_l + sub * ATT_SUB + 8 * g + 4 * h);
                const v4f de = *reinterpret_cast<const v4f *>(st_d + sub * ATT_SUB + 8 * g + 4 * h);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[4 * g + j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * g + j], c, -ls[j]));
                    dp[4 * g + j] = s[4 * g + j] * (dp[4 * g + j] - de[j]);
                }
            }
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const h8 p = pack8(s, st), ds = pack8(dp, st);
#pragma unroll
                for (int mb = 0; mb < D / 32; ++mb) {
                    dv[mb] = ATT_MFMA(io.tr_operand(gt, sub, st, mb), p, dv[mb]);
                    dk[mb] = ATT_MFMA(io.tr_operand(qt, sub, st, mb), ds, dk[mb]);
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

#define JF_ATT_D(KERN, D, a, st)                                                                                            \
    do {                                                                                                                    \
        const unsigned grid = 8u * (((a).B * (a).H + 7) / 8) * (((a).T + WG_ROWS - 1) / WG_ROWS);                           \
        if ((a).cq) hipLaunchKernelGGL((KERN<D, true>), dim3(grid), dim3(64 * NW), 0, st, a);                               \
        else hipLaunchKernelGGL((KERN<D, false>), dim3(grid), dim3(64 * NW), 0, st, a);                                     \
    } while (0)
#define JF_ATT(KERN, D, a, st) do { if (D == 64) JF_ATT_D(KERN, 64, a, st); else JF_ATT_D(KERN, 32, a, st); } while (0)

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
    JF_ATT(attn_fwd_kernel, D, a, (hipStream_t)stream);
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
    JF_ATT(attn_dq_kernel, D, a, (hipStream_t)stream);
    JF_ATT(attn_dkv_kernel, D, a, (hipStream_t)stream);
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
